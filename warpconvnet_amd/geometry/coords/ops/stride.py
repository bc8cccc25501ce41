"""Strided (down-sampled) output coordinates (reference:
warpconvnet/geometry/coords/ops/stride.py:17-54 and warpconvnet/utils/unique.py:125-144)."""
import ctypes
from typing import Tuple

import torch
from torch import Tensor

from ...._lib import ERR_TABLE_OVERFLOW, check, int3, lib, ptr, stream_ptr, workspace
from ...._lib import host as native
from .batch_index import offsets_from_batch_index
from ..search.torch_hashmap import _four_columns, more_slots


def stride_coords(batch_indexed_coords: Tensor, stride: Tuple[int, ...],
                  order="random", batch_sorted: bool = False) -> Tuple[Tensor, Tensor]:
    """Unique rows of floor(coords / [1, *stride]) and their batch offsets.

    One call into the HIP library (floor division, table build over the coarse rows, selection of
    the lowest source row per coarse voxel, order-preserving compaction) and one host read for the
    row count.  Output rows ascend in their representative's source row, so a batch-sorted input
    yields a batch-sorted output (the reference sorts by batch afterwards, stride.py:44-48, with an
    order inside a batch that depends on a thread race; as sets the results are identical).
    Any other `order` sorts the coarse voxels of every batch item along that curve.
    `batch_sorted=True` (not in the reference) vouches that the input's batch column does not
    descend, which makes the batch offsets of the output one device search and one read.
    """
    num_spatial_dims = batch_indexed_coords.shape[1] - 1
    assert len(stride) == num_spatial_dims, \
        (f"Stride must match the number of spatial dimensions. Got {len(stride)} spatial "
         f"dimensions for but coordinates with {num_spatial_dims} spatial dimensions.")
    if all(s == 1 for s in stride):
        return batch_indexed_coords, offsets_from_batch_index(batch_indexed_coords[:, 0], ascending=batch_sorted)
    unique_coords, out_offsets, _ = _unique_floor_div(batch_indexed_coords, stride, batch_sorted)
    if num_spatial_dims != 3:
        unique_coords = unique_coords[:, : num_spatial_dims + 1].contiguous()
    if out_offsets is None:
        out_offsets = offsets_from_batch_index(unique_coords[:, 0], ascending=batch_sorted)
    if str(getattr(order, "name", order)).lower() not in ("random", "point_ordering.random"):
        # The coarse voxels of every batch item along a space-filling curve.  (The reference hands
        # the four-column rows to `encode`, whose code function accepts three columns and raises,
        # stride.py:49-51; the evident intent is the ordering of the spatial columns per batch item.)
        from .serialization import encode
        code = encode(unique_coords[:, 1:].contiguous(), batch_offsets=out_offsets, order=order,
                      return_perm=True)
        unique_coords = unique_coords[code.perm].contiguous()
    return unique_coords, out_offsets


def _unique_floor_div(batch_indexed_coords: Tensor, stride: Tuple[int, ...], batch_sorted: bool = False):
    """((M, 4) rows, batch offsets or None, the same as int32 or None): the distinct rows of
    floor(coords / [1, *stride]), ascending in the first source row of each (one library call and one
    host read).  `batch_sorted`: for an input whose batch column does not descend the batch items'
    first rows are looked up behind the compaction and come with the row count: what
    offsets_from_batch_index(..., ascending=True) computes (None beyond 1024 items)."""
    assert batch_indexed_coords.dtype == torch.int32
    num_spatial_dims = batch_indexed_coords.shape[1] - 1
    strides = [int(s) for s in stride] + [1] * (3 - num_spatial_dims)
    if batch_indexed_coords.shape[0] > 0 and all(v in (1, 2, 4) for v in strides):
        # Cells of 1, 2 or 4 voxels per dimension lie inside the 4x4x4 blocks of the table of the
        # fine coordinates (the one this resolution's kernel maps use, kept on the tensor object):
        # the distinct coarse rows come out of that table, no second table is built.
        from ..search.torch_discrete import _table_of
        from ..search.torch_hashmap import HashMethod
        table = _table_of(batch_indexed_coords, HashMethod.CITY, batch_indexed_coords.device)
        return native().stride_cells(table, strides, batch_sorted)
    device = batch_indexed_coords.device
    coords = _four_columns(batch_indexed_coords)
    n = coords.shape[0]
    L = lib()
    st = int3(strides)
    out = torch.empty((n, 4), dtype=torch.int32, device=device)
    first = torch.empty(n, dtype=torch.int32, device=device)
    count = ctypes.c_int64(0)
    bounds = (ctypes.c_int64 * 1025)() if batch_sorted else None

    def read(ws, slots):
        if batch_sorted:
            return L.wcn_stride_unique_read_bounds(ptr(ws), n, slots, ctypes.byref(count), bounds,
                                                   stream_ptr(device))
        return L.wcn_stride_unique_read_count(ptr(ws), n, slots, ctypes.byref(count), stream_ptr(device))

    slots = L.wcn_table_default_capacity(n)
    while True:
        ws = workspace(L.wcn_stride_unique_workspace_bytes(n, slots), device)
        check(L.wcn_stride_unique(ptr(coords), n, st, ptr(ws), slots, ptr(out), ptr(first),
                                  stream_ptr(device)), "wcn_stride_unique")
        status = read(ws, slots)
        if status == ERR_TABLE_OVERFLOW:
            slots = more_slots(slots)
            continue
        check(status, "wcn_stride_unique")
        break
    m = int(count.value)
    batches = sum(1 for b in bounds if b < m) if batch_sorted else 0  # the last batch item with rows, plus one
    if not 0 < batches < 1025:
        return out[:m], None, None
    offsets = torch.tensor(list(bounds[:batches]) + [m], dtype=torch.int64)
    return out[:m], offsets, offsets.int()
