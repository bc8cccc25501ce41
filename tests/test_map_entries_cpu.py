"""Arguments the entries of joined launches refuse before anything is launched (no GPU needed)."""
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


def test_joined_entries_refuse_null_and_odd_arguments():
    ks, bad = (ctypes.c_int32 * 3)(3, 3, 3), (ctypes.c_int32 * 3)(3, 0, 3)
    L = lib()
    assert L.wcn_table_build_items(NULL, 10, _starts(0, 10), 1, FAKE, FAKE, 1024, NULL) == -1
    assert L.wcn_table_build_items(FAKE, 10, _starts(0, 10), 1, ctypes.c_void_p(4100), FAKE, 1024, NULL) == -1
    assert L.wcn_table_build_items(FAKE, 10, _starts(0, 10), 1, FAKE, FAKE, 1000, NULL) == -1
    for args in ((bad, ks, None, None, FAKE, 100, FAKE, FAKE), (ks, ks, ks, None, FAKE, 100, FAKE, FAKE),
                 (ks, ks, None, None, NULL, 100, FAKE, FAKE), (ks, ks, None, None, FAKE, 100, NULL, FAKE),
                 (ks, ks, None, None, FAKE, -1, FAKE, FAKE)):
        assert L.wcn_kmap_count_fill(FAKE, 10, 1024, FAKE, 5, *args, NULL) == -1
