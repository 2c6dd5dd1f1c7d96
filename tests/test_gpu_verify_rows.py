"""attention_verify_int8 (the verify block's one-dispatch attention, several rows per work-group)
against the FP64 oracle, in place, and row by row against dispatches of one row."""
import numpy as np
import pytest

from bootstrap_hip import KernelArgs
from kvcase import fp32_reader, rel_l2, upload, upload_cache
from test_gpu_attention import build_case

pytestmark = pytest.mark.gpu


def verify(device, q, gate, cache, rows, pos):
    """The rows' outputs, written over the query as the engine does; the guard after them stays."""
    qb = upload(device, np.append(q, np.float32(np.nan)))
    gb = upload(device, gate)
    device.begin()
    device.dispatch("attention_verify_int8", KernelArgs(M=rows, K=pos + rows, Position=pos), rows * 4096, 256, qb,
                    cache.kc, cache.vc, gb, qb, cache.ks, cache.vs)
    device.end()
    y = qb.read(np.float32, rows * 4096 + 1)
    qb.dispose()
    gb.dispose()
    assert np.isnan(y[-1]), "output guard overwritten"
    return y[:-1]


# one, two, three and four rows per work-group and several row blocks; blocks across the ends of a
# chunk (128), a page (256) and a split's size (8192 tokens: 64 splits of one chunk, then of two;
# 65536: eight chunks, then five)
@pytest.mark.parametrize("history,rows", [(0, 1), (0, 8), (126, 2), (127, 3), (125, 5), (250, 8), (511, 4), (1500, 7),
                                          (8188, 6), (8191, 1), (33000, 4), (65533, 6), (700, 64)])
def test_verify_rows_match_fp64(device, oracle, history, rows):
    """rel-L2 within 1.5 times the reference reader's own float32 error + 1e-6 (the bound of the other
    FP32-query paths), and every row bitwise that of a dispatch holding it alone."""
    q, gate, host = build_case(oracle, history, rows)
    cache = upload_cache(device, *host)
    y = verify(device, q, gate, cache, rows, history)
    assert np.all(np.isfinite(y))
    ref = oracle.attention(q, *host, gate, rows, history, round_q_half=0)
    if history + rows <= 2000 and rows <= 8:
        bound = 1.5 * rel_l2(fp32_reader(q, *host, gate, rows, history), ref) + 1e-6
    else:
        bound = 4e-6   # 8 rounding steps of 2^-24 on base-2 scores up to about 2^3
    assert rel_l2(y, ref) <= bound, (rel_l2(y, ref), bound)
    for r in range(rows):
        one = verify(device, q[r * 4096:(r + 1) * 4096], gate[r * 4096:(r + 1) * 4096], cache, 1, history + r)
        assert np.array_equal(one.view(np.uint32), y[r * 4096:(r + 1) * 4096].view(np.uint32)), r
    cache.dispose()
