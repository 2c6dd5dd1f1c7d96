"""Prefill chunks over short key ranges: one or two 32-key tiles per split, the last one ragged,
and row tiles whose causal end lies splits before the range's end."""
import numpy as np
import pytest

from kvcase import rel_l2, upload_cache
from test_gpu_attention import MAX_ABS, REL_L2, build_case, run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("history,rows", [(0, 65), (0, 96), (0, 97), (7, 120), (0, 255), (31, 257), (500, 480), (993, 513)])
def test_prefill_short_ranges(device, oracle, history, rows):
    """Against FP64 at the bounds of the other prefill tests: rel-L2 1e-3, max-abs 2e-3 and the
    reference's per-element bound (FP16 operands and FP16 split partials, 2^-12 relative each)."""
    q, gate, host = build_case(oracle, history, rows)
    cache = upload_cache(device, *host)
    y = run_prefill(device, q, gate, cache, rows, history)
    assert np.isnan(y[-1]), "output guard overwritten"
    y = y[:-1]
    ref, bound = oracle.attention(q, *host, gate, rows, history, round_q_half=1, with_bound=True)
    err = np.abs(y - ref)
    assert rel_l2(y, ref) <= REL_L2 and err.max() <= MAX_ABS, (rel_l2(y, ref), err.max())
    assert np.all(err <= bound / 256 + 1e-4)
    cache.dispose()
