"""The 256-row prefill kernel at the split counts its rules give few rows (a split of one key tile, of
two, of several, and more than eight combine steps) and ragged last splits, on both storage formats."""
import pytest

from test_gpu_fp16_control import test_online_fp16_matches_fp64 as check_fp16
from test_gpu_short_chunks import test_prefill_short_ranges as check_int8

pytestmark = pytest.mark.gpu


# on 256 CUs: 16, 24 and 17 splits of one 32-key tile, 26 and 32 of two, 63 and 64 of four, 72 of seven
@pytest.mark.parametrize("history,rows", [(511, 1), (668, 100), (511, 33), (1600, 32), (2000, 16), (8000, 8), (8131, 32),
                                          (16000, 1)])
def test_fp16_few_rows(device, oracle, history, rows):
    """Against FP64 at the bounds of the FP16 control's other shapes."""
    check_fp16(device, oracle, history, rows, False)


# 15 splits of two tiles (928 keys, whole), 22 and 27 of three, 33 of four
@pytest.mark.parametrize("history,rows", [(828, 100), (2000, 65), (2500, 70), (4100, 65)])
def test_int8_few_rows(device, oracle, history, rows):
    """Against FP64 at the bounds of the other prefill tests."""
    check_int8(device, oracle, history, rows)


# more work-groups than CUs: 1500 and 1600 rows in three splits, 2200 in two; and next to them, in one
# round, 1600 rows after a longer history and 1300 rows
@pytest.mark.parametrize("history,rows", [(0, 1600), (1500, 1500), (2000, 1500), (0, 2200), (1000, 1600), (700, 1300)])
def test_int8_second_round(device, oracle, history, rows):
    """Against FP64 at the bounds of the other prefill tests."""
    check_int8(device, oracle, history, rows)


@pytest.mark.parametrize("history,rows", [(1000, 1450)])
def test_fp16_second_round(device, oracle, history, rows):
    check_fp16(device, oracle, history, rows, False)
