"""The convolution of one voxel (csrc/wcn_conv_point.hip) at the edges of its tiles, and the calls that stay with torch."""
import pytest
import torch

from helpers import kaiming_weight, normal_features
from warpconvnet_amd.geometry.types.voxels import Voxels
from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}  # unit roundoff: 11 and 8 significant bits, half a place


def _voxels(rows, c, dtype, seed=3):
    coords = torch.arange(rows, dtype=torch.int32)
    coords = torch.stack([coords % 64, coords // 64 % 64, coords // 4096], 1)
    return Voxels(coords.to(DEV), normal_features(rows, c, seed=seed, dtype=dtype).to(DEV), offsets=torch.tensor([0, rows]))


def _kernel():
    from warpconvnet_amd._lib import lib
    return lib().wcn_conv_last_kernel().decode()


_SHAPES = [(32, 32, 1), (32, 8, 257), (32, 96, 255), (64, 32, 127), (64, 24, 129), (64, 64, 40_000), (96, 40, 128), (96, 96, 1000),
           (96, 16, 300_001), (128, 72, 100_000), (192, 96, 100_001), (256, 128, 100_031)]


@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("c_in,c_out,rows", _SHAPES)
def test_one_voxel_kernels_match_float64(c_in, c_out, rows, dtype, bias):
    vox = _voxels(rows, c_in, dtype)
    w = kaiming_weight(1, c_in, c_out, seed=4, dtype=dtype).to(DEV)
    b = (torch.randn(c_out, generator=torch.Generator().manual_seed(5)) * 0.1).to(dtype).to(DEV) if bias else None
    with torch.no_grad():
        got = spatially_sparse_conv(vox, w, kernel_size=1, stride=1, bias=b).feature_tensor
    assert _kernel().startswith("pointwise_fwd<"), _kernel()
    assert got.shape == (rows, c_out) and got.dtype == dtype
    x64, w64 = vox.feature_tensor.double(), w[0].double()
    want = x64 @ w64 + (b.double() if bias else 0.0)
    # fp32 sums of c_in products (and the bias), then one rounding
    sums = (c_in + 1) * 2.0 ** -24 * (x64.abs() @ w64.abs() + (b.double().abs() if bias else 0.0))
    assert bool(((got.double() - want).abs() <= UNIT[dtype] * (want.abs() + sums) + sums + 2.0 ** -25).all())


@pytest.mark.parametrize("dtype,c_in,c_out,rows", [(torch.float32, 64, 64, 500), (torch.float16, 40, 64, 500), (torch.float16, 64, 20, 500),
                                                   (torch.bfloat16, 128, 64, 99_999), (torch.bfloat16, 160, 64, 100_000)],
                         ids=["fp32", "c_in_40", "c_out_20", "wide_few_rows", "c_in_160"])
def test_other_calls_stay_with_the_library(dtype, c_in, c_out, rows):
    from warpconvnet_amd._lib import lib
    w = kaiming_weight(1, c_in, c_out, seed=4, dtype=dtype).to(DEV)
    with torch.no_grad():
        spatially_sparse_conv(_voxels(10, 32, torch.float16), kaiming_weight(1, 32, 16, seed=1, dtype=torch.float16).to(DEV),
                              kernel_size=1)
        assert _kernel() == "pointwise_fwd<f16, 1, 4>"
        vox = _voxels(rows, c_in, dtype)
        got = spatially_sparse_conv(vox, w, kernel_size=1).feature_tensor
        assert torch.equal(got, vox.feature_tensor @ w[0])
    assert not lib().wcn_pointwise_takes(rows, c_in, c_out, {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype])


@pytest.mark.parametrize("c_in,c_out,rows,own", [(128, 64, 1, True), (256, 128, 300, True), (192, 96, 32_767, True),
                                                 (128, 128, 32_768, True), (128, 128, 32_769, False), (256, 128, 99_999, False)])
def test_wide_rows_over_few_voxels(c_in, c_out, rows, own):
    w = kaiming_weight(1, c_in, c_out, seed=4, dtype=torch.bfloat16).to(DEV)
    vox = _voxels(rows, c_in, torch.bfloat16)
    with torch.no_grad():
        spatially_sparse_conv(_voxels(10, 32, torch.float16), kaiming_weight(1, 32, 16, seed=1, dtype=torch.float16).to(DEV),
                              kernel_size=1)
        before = _kernel()
        got = spatially_sparse_conv(vox, w, kernel_size=1).feature_tensor
    assert (_kernel() != before) == own
    x64, w64 = vox.feature_tensor.double(), w[0].double()
    want, sums = x64 @ w64, c_in * 2.0 ** -24 * (x64.abs() @ w64.abs())  # fp32 sums of c_in products, then one rounding
    assert bool(((got.double() - want).abs() <= UNIT[torch.bfloat16] * (want.abs() + sums) + sums + 2.0 ** -25).all())


def test_gradients_transforms_and_modes_see_the_product():
    w = kaiming_weight(1, 64, 32, seed=4, dtype=torch.float16).to(DEV)
    vox = _voxels(300, 64, torch.float16)
    conv = lambda v, weight: spatially_sparse_conv(v, weight, kernel_size=1).feature_tensor
    leaf = w.clone().requires_grad_(True)
    conv(vox, leaf).float().sum().backward()
    assert torch.allclose(leaf.grad[0].float(), vox.feature_tensor.float().sum(0)[:, None].expand(64, 32), atol=0.1, rtol=1e-2)
    with torch.no_grad():
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(w, torch.ones_like(w))
            tangent = torch.autograd.forward_ad.unpack_dual(conv(vox, dual)).tangent
        assert tangent is not None
        batch = torch.func.vmap(lambda weight: conv(vox, weight))(torch.stack([w, 2 * w]))
        assert torch.equal(batch[0], conv(vox, w)) and batch.shape == (2, 300, 32)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert conv(vox, w).dtype == torch.bfloat16
        # a view that is no dense matrix, one off the 16-byte grid, and no rows at all
        wide = torch.cat([w, w], 2)
        assert torch.equal(conv(vox, wide[:, :, :32]), conv(vox, w))
        off = torch.empty(64 * 32 + 4, dtype=w.dtype, device=DEV)[4:].view(1, 64, 32).copy_(w)
        assert torch.equal(conv(vox, off), conv(vox, w))
        with pytest.raises(RuntimeError):
            conv(vox, w.float())
        with torch.inference_mode():
            assert torch.equal(conv(vox, w), conv(vox, w.clone()))


def test_replays_of_a_captured_call_follow_the_rows():
    vox = _voxels(5000, 64, torch.bfloat16)
    w = kaiming_weight(1, 64, 32, seed=4, dtype=torch.bfloat16).to(DEV)
    with torch.no_grad():
        spatially_sparse_conv(vox, w, kernel_size=1)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = spatially_sparse_conv(vox, w, kernel_size=1).feature_tensor
        for seed in (7, 8, 9):
            vox.feature_tensor.copy_(normal_features(5000, 64, seed=seed, dtype=torch.bfloat16))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, spatially_sparse_conv(vox, w, kernel_size=1).feature_tensor)
