"""A layer over a map that a layer before it has left goes a shorter way through the host (_over_kept_map); every kind of call
against the general way, bit for bit: output, coordinates, stride, cache, and what is refused; and which calls take it."""
import contextlib

import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features
from warpconvnet_amd.utils import synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
C_IN, C_OUT = 32, 48


def _voxels(strided, rows=2500):
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    items = [synthetic.random_cloud(7 + b, n, 22)[:, 1:] for b, n in enumerate((rows, rows // 3))] if rows else [np.zeros((0, 3), np.int32)]
    xyz = np.concatenate(items).astype(np.int32)
    x = normal_features(len(xyz), C_IN, seed=4, dtype=torch.float16).to(DEV)
    vox = Voxels(torch.as_tensor(np.ascontiguousarray(xyz), device=DEV), x, offsets=torch.as_tensor(np.cumsum([0] + [len(i) for i in items])))
    if strided:
        vox = spatially_sparse_conv(vox, kaiming_weight(8, C_IN, C_IN, seed=1, dtype=torch.float16).to(DEV), 2, stride=2)
    return vox


class _Ways:
    """How often the short way gave an answer; `open` False closes it."""

    def __init__(self, monkeypatch):
        from warpconvnet_amd.nn.functional import sparse_conv
        real, self.taken, self.open = sparse_conv._over_kept_map, 0, True

        def spied(*args):
            out = real(*args) if self.open else None
            self.taken += out is not None
            return out

        monkeypatch.setattr(sparse_conv, "_over_kept_map", spied)


def _kinds(n):
    bias = (torch.randn(C_OUT, generator=torch.Generator().manual_seed(8)) * 0.1).half().to(DEV)
    res = normal_features(n, C_OUT, seed=9, dtype=torch.float16).to(DEV)
    return {"plain": {}, "bias": {"bias": bias}, "fp32 bias": {"bias": bias.float()}, "one value": {"bias": bias[:1]},
            "residual": {"bias": bias, "residual": res, "relu": True}, "residual voxels": {"residual": "voxels"}, "relu": {"relu": True},
            "bf16": {"compute_dtype": torch.bfloat16, "bias": bias}, "fp32": {"compute_dtype": torch.float32},
            "kept weight": {"keep_prepared_weight": True, "bias": bias}, "dilated": {"kernel_dilation": 2},
            "tuples": {"kernel_dilation": (1, 1, 1), "stride": (1, 1, 1)}, "reduce": {"stride_mode": "REDUCE_AND_STRIDE"},
            "bias that asks": {"bias": bias.clone().requires_grad_()}}


@pytest.mark.parametrize("strided", [False, True], ids=["fine", "strided"])
@pytest.mark.parametrize("ksize", [3, (3, 1, 3), 2], ids=["k3", "k313", "k2"])
def test_the_short_way_gives_what_the_general_one_gives(monkeypatch, strided, ksize):
    from warpconvnet_amd.nn.functional.sparse_conv import STRIDED_CONV_MODE, spatially_sparse_conv
    vox = _voxels(strided)
    K = int(np.prod(ksize)) if isinstance(ksize, tuple) else ksize ** 3
    w = kaiming_weight(K, C_IN, C_OUT, seed=2, dtype=torch.float16).to(DEV)
    ways = _Ways(monkeypatch)
    for name, kind in _kinds(len(vox)).items():
        if kind.get("residual") == "voxels":
            kind["residual"] = vox.replace(batched_features=normal_features(len(vox), C_OUT, seed=3, dtype=torch.float16).to(DEV))
        if "stride_mode" in kind:
            kind["stride_mode"] = STRIDED_CONV_MODE[kind["stride_mode"]]
        for mode in (torch.no_grad, contextlib.nullcontext):
            with mode():
                first = spatially_sparse_conv(vox, w, ksize, **kind)  # leaves the map, where it is not there yet
                maps, before = len(list(vox.cache.values())), ways.taken
                short = spatially_sparse_conv(vox, w, ksize, **kind)
                assert ways.taken == before + 1, name
                ways.open = False
                general = spatially_sparse_conv(vox, w, ksize, **kind)
                ways.open = True
            assert ways.taken == before + 1
            assert torch.equal(short.feature_tensor, general.feature_tensor) and torch.equal(short.feature_tensor, first.feature_tensor), name
            assert short.feature_tensor.dtype == general.feature_tensor.dtype and not short.feature_tensor.requires_grad
            assert short.batched_coordinates is general.batched_coordinates is vox.batched_coordinates
            assert short.tensor_stride == general.tensor_stride == ((2, 2, 2) if strided else (1, 1, 1)), name
            assert short.cache is general.cache is vox.cache and torch.equal(short.offsets, general.offsets)
            assert len(list(vox.cache.values())) == maps and type(short) is type(general)


def test_other_layers_take_the_general_way(monkeypatch):
    """Gradients of any input, autocast, other outputs, orders and maps, no rows."""
    from warpconvnet_amd.geometry.coords.ops.serialization import POINT_ORDERING
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    vox = _voxels(False)
    w = kaiming_weight(27, C_IN, C_OUT, seed=2, dtype=torch.float16).to(DEV)
    res = normal_features(len(vox), C_OUT, seed=9, dtype=torch.float16).to(DEV)
    want = spatially_sparse_conv(vox, w, 3)
    ways = _Ways(monkeypatch)
    out = spatially_sparse_conv(vox, w.clone().requires_grad_(), 3)
    assert out.feature_tensor.requires_grad
    asks = vox.replace(batched_features=vox.feature_tensor.clone().requires_grad_())
    assert spatially_sparse_conv(asks, w, 3).feature_tensor.requires_grad
    added = spatially_sparse_conv(vox, w, 3, residual=res.clone().requires_grad_(), relu=True)
    assert added.feature_tensor.requires_grad
    with torch.autocast("cuda", dtype=torch.bfloat16):
        spatially_sparse_conv(vox, w, 3)
    spatially_sparse_conv(vox, w, 3, output_spatially_sparse_tensor=vox)
    spatially_sparse_conv(vox, w[:8].contiguous(), 2, stride=2)
    spatially_sparse_conv(vox, w, 3, order=POINT_ORDERING.MORTON_XYZ)
    spatially_sparse_conv(vox, w, 3, generative=True)
    assert ways.taken == 0
    assert torch.equal(spatially_sparse_conv(vox, w, 3).feature_tensor, want.feature_tensor) and ways.taken == 1
    none = _voxels(False, rows=0)
    for _ in range(2):
        assert spatially_sparse_conv(none, w, 3).feature_tensor.shape == (0, C_OUT)
    assert ways.taken == 1


def test_what_is_refused_is_refused_on_both_ways(monkeypatch):
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    vox = _voxels(False)
    w = kaiming_weight(27, C_IN, C_OUT, seed=2, dtype=torch.float16).to(DEV)
    spatially_sparse_conv(vox, w, 3)
    res = normal_features(len(vox), C_OUT, seed=9, dtype=torch.float16).to(DEV)
    ways = _Ways(monkeypatch)
    for args, kw in (((w[:26], 3), {}), ((w[:, :16], 3), {}), ((w[0], 3), {}), ((w.cpu(), 3), {}), ((w, 3), {"residual": res[:-1]}),
                     ((w, 3), {"residual": res[:, :8]}), ((w, 3), {"compute_dtype": torch.int32}), ((w, 3), {"bias": res[:5, 0]})):
        seen = []
        for ways.open in (True, False):
            with pytest.raises(Exception) as e:
                spatially_sparse_conv(vox, *args, **kw)
            seen.append((type(e.value), str(e.value)))
        assert seen[0] == seen[1], seen
