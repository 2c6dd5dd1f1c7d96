"""V vectors near either end of FP32's range on the kernels that scale the probability operands by a
split's largest V scale: a split (or a row's whole range) of vectors around 1e-36 beside ordinary
ones, alone, and before a later token whose V a row does not see; and vectors around 3e38, whose sums
before the division by the softmax's denominator lie beyond FP32, alone, in one split and in one token."""
import numpy as np
import pytest

from kvcase import reference_kv, rel_l2, upload_cache
from test_gpu_attention import REL_L2, build_case, run_decode, run_prefill
from test_gpu_verify_rows import verify

pytestmark = pytest.mark.gpu

TINY = np.float32(1e-36)   # scales around 7.9e-39: 128 over one of them overflows FP32


def tiny_values(values, where):
    """Which tokens' V are scaled: one 128-token split of several, all, or all but the last token, which
    becomes large (its scale over the others' overflows FP32)."""
    values = values.copy()
    values[{"split": slice(128, 256), "all": slice(None), "before_last": slice(0, -1)}[where]] *= TINY
    if where == "before_last":
        values[-1] *= np.float32(1e4)
    return values


@pytest.mark.parametrize("where", ["split", "all", "before_last"])
@pytest.mark.parametrize("kind,history,rows", [
    ("decode", 200, 1), ("decode", 4092, 1), ("decode", 1000, 5),
    ("prefill", 1000, 16), ("prefill", 0, 98), ("prefill", 2031, 18),      # decode kernel; multi-row kernel, one split, several
    ("verify", 300, 2), ("verify", 1500, 8)])
def test_tiny_values(device, oracle, kind, history, rows, where):
    """Each row against FP64: 5e-6 where the operands are FP32-accurate (as the other decode tests;
    FP32's subnormals add at most 2^-149 to outputs above 1e-39), the prefill bar otherwise."""
    keys, values = reference_kv(history + rows)
    q, gate, host = build_case(oracle, history, rows, kv=(keys, tiny_values(values, where)))
    cache = upload_cache(device, *host)
    if kind == "verify":
        y = verify(device, q, gate, cache, rows, history)
    else:
        y = (run_decode if kind == "decode" else run_prefill)(device, q, gate, cache, rows, history)
        assert np.isnan(y[-1]), "output guard overwritten"
        y = y[:-1]
    assert np.all(np.isfinite(y))
    ref = oracle.attention(q, *host, gate, rows, history, round_q_half=int(kind == "prefill"))
    for r, (a, b) in enumerate(zip(y.reshape(rows, 4096), np.asarray(ref).reshape(rows, 4096))):
        scale = np.abs(b).max()   # (norms of values around 1e-37 would underflow)
        assert rel_l2(a.astype(np.float64) / scale, b / scale) <= (REL_L2 if kind == "prefill" else 5e-6), r
    cache.dispose()


@pytest.mark.parametrize("where", ["split", "all", "last"])
@pytest.mark.parametrize("kind,history,rows", [
    ("decode", 200, 1), ("decode", 4092, 1), ("decode", 1000, 5), ("prefill", 1000, 16), ("prefill", 0, 98),
    ("prefill", 2031, 18), ("verify", 300, 2), ("verify", 1500, 8)])
def test_huge_values(device, oracle, kind, history, rows, where):
    """Flat rows (queries a tenth of the others') against FP64, each row at the bounds above."""
    keys, values = reference_kv(history + rows)
    values[{"split": slice(128, 256), "all": slice(None), "last": slice(-1, None)}[where]] *= np.float32(3e38)
    q, gate, host = build_case(oracle, history, rows, kv=(keys, values))
    q = q * np.float32(0.1)
    cache = upload_cache(device, *host)
    if kind == "verify":
        y = verify(device, q, gate, cache, rows, history)
    else:
        y = (run_decode if kind == "decode" else run_prefill)(device, q, gate, cache, rows, history)[:-1]
    assert np.all(np.isfinite(y))
    ref = oracle.attention(q, *host, gate, rows, history, round_q_half=int(kind == "prefill"))
    for r, (a, b) in enumerate(zip(y.reshape(rows, 4096), np.asarray(ref).reshape(rows, 4096))):
        scale = np.abs(b).max()
        assert rel_l2(a.astype(np.float64) / scale, b / scale) <= (REL_L2 if kind == "prefill" else 5e-6), r
    cache.dispose()
