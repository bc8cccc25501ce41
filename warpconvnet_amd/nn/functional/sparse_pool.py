"""Pooling of sparse voxel tensors over a kernel map (reference:
warpconvnet/nn/functional/sparse_pool.py).

`sparse_reduce` keeps the reference's bookkeeping (strided output coordinates, the kernel-map
cache entry shared with a strided convolution of the same geometry, tensor stride, zeros for
output voxels without any input) and sends the reduction itself to the HIP library: the pairs are
grouped by output row (`wcn_map_rows_build`) and reduced with fp32 accumulation
(`wcn_sparse_pool_fwd_offsets`); the gradient runs in the same library (`wcn_sparse_pool_bwd_offsets`).
"""
from typing import Optional, Tuple, Union

import torch
from torch import Tensor

from ..._lib import host as native
from ...geometry.coords.integer import IntCoords
from ...geometry.coords.ops.stride import stride_coords
from ...geometry.coords.search.cache import IntSearchCache, IntSearchCacheKey
from ...geometry.coords.search.torch_discrete import generate_kernel_map, rows_with_table
from ...geometry.types.voxels import Voxels
from ...ops.reductions import REDUCTIONS
from ...utils.ntuple import ntuple
from ...utils.gather import take_rows

_MODE = {REDUCTIONS.SUM: 0, REDUCTIONS.MEAN: 1, REDUCTIONS.MAX: 2, REDUCTIONS.MIN: 3}


def sparse_reduce(voxels: Voxels, kernel_size: Union[int, Tuple[int, ...]],
                  stride: Optional[Union[int, Tuple[int, ...]]] = None,
                  reduction: Union[REDUCTIONS, str] = REDUCTIONS.MAX, order="random") -> Voxels:
    """Reduce the features of every strided output voxel's kernel window
    (reference: sparse_pool.py:25-120)."""
    if isinstance(reduction, str):
        reduction = REDUCTIONS(reduction)
    if reduction not in _MODE:
        raise NotImplementedError(f"reduction {reduction.value!r} is not built (min, max, mean, sum are)")
    if stride is None:
        stride = kernel_size
    ndim = voxels.num_spatial_dims
    stride = ntuple(stride, ndim=ndim)
    kernel_size = ntuple(kernel_size, ndim=ndim)
    in_tensor_stride = voxels.stride
    if in_tensor_stride is None:
        in_tensor_stride = ntuple(1, ndim=ndim)
    out_tensor_stride = tuple(o * s for o, s in zip(stride, in_tensor_stride))

    in_coords = (rows_with_table(voxels.batched_coordinates) if type(voxels.batched_coordinates) is IntCoords
                 else voxels.batch_indexed_coordinates)
    out_coords, out_offsets = stride_coords(in_coords, stride, order=order, batch_sorted=True)
    from .sparse_conv import STRIDED_CONV_MODE
    key = IntSearchCacheKey(kernel_size=kernel_size, kernel_dilation=ntuple(1, ndim=ndim),
                            transposed=False, generative=False,
                            stride_mode=str(STRIDED_CONV_MODE.STRIDE_ONLY),
                            skip_symmetric_kernel_map=False, in_offsets=voxels.offsets,
                            out_offsets=out_offsets)
    kernel_map = voxels.cache.get(key) if voxels.cache is not None else None
    if kernel_map is None:
        kernel_map = generate_kernel_map(in_coords, out_coords, in_to_out_stride_ratio=stride,
                                         kernel_size=kernel_size,
                                         kernel_dilation=ntuple(1, ndim=ndim),
                                         skip_symmetric_kernel_map=False)
    if voxels.cache is None:
        voxels._extra_attributes["_cache"] = IntSearchCache()
    voxels.cache.put(key, kernel_map)

    # kernel as large as the stride over voxels without repeats: every input row is in one pair
    single_in = kernel_size == stride and kernel_map._from_builder and kernel_map._keys_unique
    out_features = native().pool_autograd(voxels.feature_tensor, kernel_map, out_coords.shape[0], _MODE[reduction],
                                          single_in)
    new_coords = IntCoords(out_coords[:, 1:], offsets=out_offsets.cpu().int())
    new_coords._batch_indexed = out_coords
    return voxels.replace(batched_coordinates=new_coords, batched_features=out_features,
                          stride=out_tensor_stride)


def sparse_max_pool(voxels: Voxels, kernel_size, stride=None) -> Voxels:
    return sparse_reduce(voxels, kernel_size, stride, reduction=REDUCTIONS.MAX)


def sparse_avg_pool(voxels: Voxels, kernel_size, stride=None) -> Voxels:
    return sparse_reduce(voxels, kernel_size, stride, reduction=REDUCTIONS.MEAN)


def sparse_unpool(pooled_voxels: Voxels, unpooled_voxels: Voxels, kernel_size, stride,
                  concat_unpooled_voxels: bool = False) -> Voxels:
    """Copy every pooled voxel's features back to the fine voxels of its window, through the kernel
    map the pooling left in the cache (reference: sparse_pool.py:145-188: the same torch indexing,
    differentiable by torch)."""
    ndim = pooled_voxels.num_spatial_dims
    stride = ntuple(stride, ndim=ndim)
    kernel_size = ntuple(kernel_size, ndim=ndim)
    from .sparse_conv import STRIDED_CONV_MODE
    key = IntSearchCacheKey(kernel_size=kernel_size, kernel_dilation=ntuple(1, ndim=ndim),
                            transposed=False, generative=False,
                            stride_mode=str(STRIDED_CONV_MODE.STRIDE_ONLY),
                            skip_symmetric_kernel_map=False, in_offsets=unpooled_voxels.offsets,
                            out_offsets=pooled_voxels.offsets)
    assert pooled_voxels.cache is not None
    kernel_map = pooled_voxels.cache.get(key)
    assert kernel_map is not None
    unpooled_maps, pooled_maps = kernel_map._lists()
    perm = torch.argsort(unpooled_maps)
    rep_feats = take_rows(pooled_voxels.feature_tensor, pooled_maps[perm].long())
    if concat_unpooled_voxels:
        rep_feats = torch.cat([unpooled_voxels.feature_tensor, rep_feats], dim=-1)
    return unpooled_voxels.replace(batched_features=rep_feats)
