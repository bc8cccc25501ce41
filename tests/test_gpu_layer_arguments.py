"""What the layers' native host side takes and refuses, against the torch operations it stands for: biases of other
shapes, types, places and alignments, weights in host memory."""
import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features
from warpconvnet_amd.utils import synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _voxels(n, c, dtype, seed=3, extent=24):
    from warpconvnet_amd.geometry.types.voxels import Voxels
    bc = synthetic.random_cloud(seed, n, extent)
    x = normal_features(len(bc), c, seed=seed, dtype=dtype).to(DEV)
    return Voxels(torch.as_tensor(np.ascontiguousarray(bc[:, 1:]), device=DEV), x, offsets=torch.tensor([0, len(bc)]))


def _biases(c_out, n):
    """Everything that `out + bias` takes, by name."""
    g = torch.Generator().manual_seed(5)
    full = torch.randn(c_out + 1, generator=g).to(DEV)
    return {"one value": full[:1].clone(), "row": full[None, :c_out].clone(), "per row": torch.randn(n, c_out, generator=g).to(DEV),
            "host scalar": torch.tensor(0.25), "fp64": full[:c_out].double(), "misaligned": full.half()[1:],
            "misaligned fp32": full[1:], "strided": torch.randn(c_out, 2, generator=g).to(DEV)[:, 0]}


@pytest.mark.parametrize("grad", [True, False], ids=["gradients", "inference"])
@pytest.mark.parametrize("c_in,c_out,stride", [(32, 64, 1), (32, 32, 2)], ids=["k3", "up_sampling"])
def test_convolution_biases_are_what_an_addition_takes(c_in, c_out, stride, grad):
    """k3: the general contraction; up_sampling: the one for maps with one pair per output row."""
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    vox = _voxels(3000, c_in, torch.float16)
    w = kaiming_weight(27 if stride == 1 else 8, c_in, c_out, seed=2, dtype=torch.float16).to(DEV)
    coarse = None
    if stride == 2:
        coarse = spatially_sparse_conv(vox, kaiming_weight(8, c_in, c_in, seed=1, dtype=torch.float16).to(DEV), 2, stride=2)

    def layer(weight, bias):
        if coarse is None:
            return spatially_sparse_conv(vox, weight, 3, bias=bias).feature_tensor
        return spatially_sparse_conv(coarse, weight, 2, stride=2, bias=bias, transposed=True,
                                     output_spatially_sparse_tensor=vox).feature_tensor

    gy = normal_features(len(vox), c_out, seed=9, dtype=torch.float16).to(DEV)
    for name, b in _biases(c_out, len(vox)).items():
        wg, wr = (w.clone().requires_grad_(grad) for _ in range(2))
        bg, br = (b.clone().requires_grad_(grad) if name == "one value" else b for _ in range(2))
        got = layer(wg, bg)
        want = layer(wr, None) + br.half()
        # without gradients a (c_out) bias goes into the sums: one rounding instead of two (2^-11 of a value of at most 8 each)
        assert float((got.detach().float() - want.detach().float()).abs().max()) <= (0.0 if grad else 2 * 2 ** -11 * 8), name
        if grad:
            got.backward(gy)
            want.backward(gy)
            assert torch.equal(wg.grad, wr.grad), name
            if bg.requires_grad:
                assert bg.grad.shape == b.shape and torch.equal(bg.grad, br.grad), name
    for bad in (torch.zeros(c_out - 1, device=DEV), torch.zeros(c_out + 1, device=DEV), torch.zeros(c_out)):
        with pytest.raises(RuntimeError):
            layer(w.clone().requires_grad_(grad), bad)
    with pytest.raises((ValueError, RuntimeError)):
        layer(w.cpu().requires_grad_(grad), None)


@pytest.mark.parametrize("grad", [True, False], ids=["gradients", "inference"])
def test_depthwise_biases_are_what_an_addition_takes(grad):
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv_depth import spatially_sparse_depthwise_conv
    vox = _voxels(3000, 32, torch.float16)
    c, n = vox.batch_indexed_coordinates, len(vox)
    km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
    w = kaiming_weight(27, 32, 1, seed=2, dtype=torch.float16)[..., 0].to(DEV)
    for name, b in _biases(32, n).items():
        bg, br = (b.clone().requires_grad_(grad) if name == "one value" else b for _ in range(2))
        got = spatially_sparse_depthwise_conv(vox.feature_tensor, w, km, n, bias=bg)
        want = spatially_sparse_depthwise_conv(vox.feature_tensor, w, km, n) + br.half()
        assert torch.equal(got, want), name
        if bg.requires_grad:
            got.sum().backward()
            want.sum().backward()
            assert torch.equal(bg.grad, br.grad)
    for bad in (torch.zeros(31, device=DEV), torch.zeros(33, device=DEV), torch.zeros(32)):
        with pytest.raises(RuntimeError):
            spatially_sparse_depthwise_conv(vox.feature_tensor, w, km, n, bias=bad)
    with pytest.raises(ValueError):
        spatially_sparse_depthwise_conv(vox.feature_tensor, w.cpu(), km, n)


def test_forward_mode_tangents_are_refused_and_those_of_a_bias_carried():
    from torch.autograd import forward_ad
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    from warpconvnet_amd.nn.functional.sparse_conv_depth import spatially_sparse_depthwise_conv
    from warpconvnet_amd.nn.functional.sparse_pool import sparse_max_pool
    vox = _voxels(500, 32, torch.float32)
    x, n = vox.feature_tensor, len(vox)
    w = kaiming_weight(27, 32, 32, seed=2).to(DEV).requires_grad_(True)
    wd = kaiming_weight(27, 32, 1, seed=2)[..., 0].to(DEV)
    b = torch.randn(32, device=DEV)
    spatially_sparse_conv(vox, w, 3)
    km = next(iter(vox.cache.values()))
    with forward_ad.dual_level():
        dx, dw, dwd, db = (forward_ad.make_dual(t.detach(), torch.ones_like(t)) for t in (x, w, wd, b))
        dual = vox.replace(batched_features=dx)
        for call in (lambda: spatially_sparse_conv(dual, w, 3), lambda: spatially_sparse_conv(vox, dw.requires_grad_(True), 3),
                     lambda: spatially_sparse_depthwise_conv(dx, wd, km, n), lambda: spatially_sparse_depthwise_conv(x, dwd, km, n),
                     lambda: sparse_max_pool(dual, 2)):
            with pytest.raises(NotImplementedError):
                call()
        for out in (spatially_sparse_conv(vox, w, 3, bias=db).feature_tensor,
                    spatially_sparse_depthwise_conv(x, wd, km, n, bias=db)):
            tangent = forward_ad.unpack_dual(out).tangent
            assert tangent is not None and bool((tangent == 1).all())


def test_errors_inside_a_backward_pass_are_the_package_s_own():
    """The map's host offsets no longer ascend when the gradient is asked for: the library refuses them, on a thread of the
    autograd engine, before anything is launched."""
    from warpconvnet_amd._lib import WcnError
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    vox = _voxels(500, 32, torch.float32)
    x = vox.feature_tensor.clone().requires_grad_(True)
    out = spatially_sparse_conv(vox.replace(batched_features=x), kaiming_weight(27, 32, 32, seed=2).to(DEV), 3)
    offsets = next(iter(out.cache.values()))._offsets64
    out = out.feature_tensor
    right = offsets.clone()
    offsets[3] = offsets[-1] + 1
    with pytest.raises(WcnError) as failed:
        out.backward(torch.ones_like(out), retain_graph=True)
    assert failed.value.status == -1
    offsets.copy_(right)
    out.backward(torch.ones_like(out))
    assert x.grad is not None


@pytest.mark.parametrize("n", [63, 3000, 20_001])
@pytest.mark.parametrize("dtype,c_in,c_out,kernel,name", [
    (torch.float16, 32, 32, 3, "group"), (torch.bfloat16, 16, 24, 3, "group"), (torch.float32, 16, 13, 3, "group"), (torch.float16, 8, 9, 5, "group"),
    (torch.float16, 32, 64, 3, "pack"), (torch.bfloat16, 64, 40, 3, "pack"), (torch.float32, 32, 32, 3, "pack"), (torch.float16, 64, 13, 3, "pack"),
    (torch.bfloat16, 256, 128, 3, "ring")])
def test_a_bias_is_added_to_the_rounded_product(n, dtype, c_in, c_out, kernel, name):
    """A layer with gradients: the bits of the product and an addition behind it, in the kernel or as a launch of its own."""
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    vox = _voxels(n, c_in, dtype)
    w = kaiming_weight(kernel ** 3, c_in, c_out, seed=2, dtype=torch.float32).to(DEV).requires_grad_(True)
    weight = w if dtype == torch.float32 else w.to(dtype)
    product = spatially_sparse_conv(vox, weight, kernel).feature_tensor
    for b in (normal_features(1, c_out, seed=4, dtype=dtype)[0].to(DEV), normal_features(1, c_out, seed=4, dtype=torch.float32)[0].to(DEV)):
        got = spatially_sparse_conv(vox, weight, kernel, bias=b).feature_tensor
        assert lib().wcn_conv_last_kernel().decode().startswith(f"conv_fwd_{name}<")
        assert torch.equal(got, product + b.to(dtype))
