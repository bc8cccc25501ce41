"""Arguments the entry of a joined launch refuses before anything is launched (no GPU needed)."""
import ctypes

import pytest

from warpconvnet_amd._lib import lib

FAKE = ctypes.c_void_p(4096)
NULL = ctypes.c_void_p(0)


def _starts(*v):
    return (ctypes.c_int64 * len(v))(*v)


@pytest.mark.parametrize("rows,starts,items", [(10, (0, 4, 9), 2), (10, (1, 10), 1), (10, (0, 7, 5, 10), 3), (0, (0, 0), 1),
                                               (10, tuple([0] * 65 + [10]), 65)])
def test_table_over_items_refuses_offsets_that_are_none(rows, starts, items):
    assert lib().wcn_table_build_items(FAKE, rows, _starts(*starts), items, FAKE, FAKE, 1024, NULL) == -1


def test_table_over_items_refuses_null_and_odd_arguments():
    L = lib()
    assert L.wcn_table_build_items(NULL, 10, _starts(0, 10), 1, FAKE, FAKE, 1024, NULL) == -1
    assert L.wcn_table_build_items(FAKE, 10, _starts(0, 10), 1, ctypes.c_void_p(4100), FAKE, 1024, NULL) == -1
    assert L.wcn_table_build_items(FAKE, 10, _starts(0, 10), 1, FAKE, FAKE, 1000, NULL) == -1


@pytest.mark.parametrize("rows", [0, 1, 64, 65, 1_000_000])
@pytest.mark.parametrize("offsets", [1, 8, 27, 125, 1024])
def test_what_stays_with_a_map_is_what_is_read_of_it(rows, offsets):
    """The head of a builder's workspace: offsets and status, totals, a counter, and a row of group starts for every offset."""
    up = lambda n: (n + 255) // 256 * 256
    groups = (rows + 63) // 64
    assert lib().wcn_kmap_head_bytes(rows, offsets) == (up(8 * (offsets + 3)) + up(8 * offsets) + 256
                                                        + up(4 * offsets * (groups + 1)))
