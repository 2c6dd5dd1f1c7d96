"""Prefill chunks over short key ranges and of few rows: the multi-row kernel (whole and partial row
blocks, row blocks whose causal end lies chunks or splits before the range's end, one split and
several), its edges against the decode kernel and the 256-row kernel, and that kernel next to those
edges (splits of two to seven 32-key tiles, the last one ragged); decodes around two chunks of keys,
which take one split."""
import numpy as np
import pytest

from kvcase import rel_l2, upload_cache
from test_gpu_attention import MAX_ABS, REL_L2, build_case, run_decode, run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("history,rows", [
    (0, 65), (0, 97), (7, 120), (0, 255), (31, 257), (500, 480), (1023, 512),      # multi-row, one split
    (112, 17), (1000, 33), (2031, 17), (8128, 64), (4000, 8), (60000, 5),          # multi-row, few rows
    (64, 64), (112, 16), (2000, 16), (2033, 16),                                   # around the decode kernel
    (801, 100), (1025, 512), (993, 513), (0, 600)])                                # 256-row kernel
def test_prefill_short_ranges(device, oracle, history, rows):
    """Against FP64 at the bounds of the other prefill tests: rel-L2 1e-3, max-abs 2e-3 and the
    reference's per-element bound (the 256-row kernel's FP16 operands and partials, 2^-12 relative
    each; the others are FP32-accurate)."""
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


@pytest.mark.parametrize("history,rows", [(126, 2), (128, 1), (100, 64), (192, 64), (254, 2), (255, 2), (240, 17)])
def test_decode_two_chunks(device, oracle, history, rows):
    """129 to 256 keys in one split (rows that end in its first chunk among them), and 257 in several:
    against FP64 at the bound of the fused decode's FP32-accurate operands, 5e-6 (FP16 hi + lo
    probabilities 2^-22 relative, query parts 6.1e-8 of the row's maximum)."""
    q, gate, host = build_case(oracle, history, rows)
    cache = upload_cache(device, *host)
    y = run_decode(device, q, gate, cache, rows, history)
    assert np.isnan(y[-1]), "output guard overwritten"
    ref = oracle.attention(q, *host, gate, rows, history, round_q_half=0)
    assert rel_l2(y[:-1], ref) <= 5e-6, rel_l2(y[:-1], ref)
    cache.dispose()
