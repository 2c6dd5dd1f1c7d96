"""Scores far beyond any softmax in use (K scales times 2^14 to 2^100): the probability operands stay
finite and a row returns the value of its largest score, on the kernels that take the exponents'
arguments from the dots; a NaN in a query reaches its head's output and no other."""
import numpy as np
import pytest

from kvcase import rel_l2, upload_cache
from test_gpu_attention import REL_L2, build_case, run_decode, run_prefill
from test_gpu_verify_rows import verify

pytestmark = pytest.mark.gpu

# decode in one split, in several; prefill chunks on the decode kernel and the multi-row kernel, in one
# split and in several; verify blocks in one and in several
CASES = [("decode", 50, 1), ("decode", 900, 3), ("prefill", 1000, 16), ("prefill", 0, 100), ("prefill", 3000, 40),
         ("verify", 60, 2), ("verify", 1500, 8)]


def run(device, kind, q, gate, host, rows, history):
    cache = upload_cache(device, *host)
    if kind == "verify":
        y = verify(device, q, gate, cache, rows, history)
    else:
        y = (run_decode if kind == "decode" else run_prefill)(device, q, gate, cache, rows, history)
        assert np.isnan(y[-1]), "output guard overwritten"
        y = y[:-1]
    cache.dispose()
    return y


@pytest.mark.parametrize("power", [14, 18, 22, 27, 40, 100])
@pytest.mark.parametrize("kind,history,rows", CASES)
def test_large_scores(device, oracle, kind, history, rows, power):
    """Against FP64, whose rows hold one key here (the two largest scores lie thousands apart): 5e-6
    where the operands are FP32-accurate, the prefill bar otherwise."""
    q, gate, host = build_case(oracle, history, rows)
    host = (host[0], host[1], host[2] * np.float32(2.0 ** power), host[3])
    y = run(device, kind, q, gate, host, rows, history)
    assert np.all(np.isfinite(y))
    ref = oracle.attention(q, *host, gate, rows, history, round_q_half=int(kind == "prefill"))
    assert rel_l2(y, ref) <= (REL_L2 if kind == "prefill" else 5e-6)


@pytest.mark.parametrize("kind,history,rows", CASES)
def test_nan_query(device, oracle, kind, history, rows):
    """The head holding the NaN is NaN as the reference's float arithmetic has it; every other head is
    bitwise what it is without."""
    q, gate, host = build_case(oracle, history, rows)
    plain = run(device, kind, q, gate, host, rows, history).reshape(rows, 16, 256)
    q.reshape(rows, 16, 256)[rows // 2, 3, 7] = np.nan
    y = run(device, kind, q, gate, host, rows, history).reshape(rows, 16, 256)
    assert np.all(np.isnan(y[rows // 2, 3]))
    y[rows // 2, 3] = plain[rows // 2, 3]
    assert np.array_equal(y.view(np.uint32), plain.view(np.uint32))
