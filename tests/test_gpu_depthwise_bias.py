"""Weight and bias gradient of a depthwise convolution in one call against the two calls, bit for bit, and the bias against
float64 sums: channel counts around the 16 and 64 that a workgroup finishes, rows around the parts of the first pass and the
ranges of the weight gradient, rows that are no whole vectors or not aligned, no rows on either side, every type of bias."""
import numpy as np
import pytest
import torch

from warpconvnet_amd._lib import check, lib, ptr, stream_ptr, workspace
from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
ROUNDING = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _close_to_sums(got, gy):
    # fp32 sums: each addition rounds by 2^-24 of a partial sum, which is at most the sum of the magnitudes; then the bias's type
    want = gy.double().sum(0)
    bound = gy.double().abs().sum(0) * 2.0 ** -20 + want.abs() * ROUNDING[got.dtype]
    return bool(((got.double() - want).abs() <= bound + 1e-7).all())


def _voxels(n, seed):
    g = np.random.default_rng(seed)
    side = int(np.ceil((4 * n) ** (1 / 3))) + 1
    cells = g.choice(side ** 3, size=n, replace=False)
    c = np.stack([np.zeros(n, np.int64), cells // side ** 2, cells // side % side, cells % side], 1)
    return torch.as_tensor(c.astype(np.int32), device=DEV)


@pytest.mark.parametrize("channels,n,dtype,bias_dtype,shift", [
    (8, 1, torch.float16, torch.float32, 0), (16, 63, torch.bfloat16, torch.bfloat16, 0), (72, 513, torch.float16, torch.float16, 0),
    (64, 40_000, torch.float16, torch.float32, 0), (96, 9000, torch.bfloat16, torch.float32, 0), (13, 300, torch.float16, torch.bfloat16, 0),
    (130, 700, torch.float32, torch.float32, 0), (32, 300, torch.float16, torch.float32, 4), (2056, 129, torch.bfloat16, torch.float32, 0)])
@pytest.mark.parametrize("empty", [None, "in", "out"])
def test_weight_and_bias_gradient_in_one_call(channels, n, dtype, bias_dtype, shift, empty):
    c = _voxels(n, n)
    km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
    iden = -1 if km.identity_map_index is None else km.identity_map_index
    n_in, n_out = 0 if empty == "in" else n, 0 if empty == "out" else n
    g = torch.Generator().manual_seed(channels + n)
    x = torch.randn(n, channels, generator=g).to(dtype).to(DEV)
    gy = torch.randn(n * channels + shift, generator=g).to(dtype).to(DEV)[shift:].view(n, channels)
    L, s, K = lib(), stream_ptr(DEV), len(km)

    def run(joined):
        gw = torch.full((K, channels), float("nan"), device=DEV, dtype=dtype)
        gb = torch.full((channels,), float("nan"), dtype=bias_dtype, device=DEV)
        ws = workspace(L.wcn_depthwise_wgrad_grouped_workspace_bytes(K, channels, n_out), DEV)
        bws = workspace(L.wcn_column_sums_workspace_bytes(channels), DEV)
        args = (ptr(x), n_in, ptr(gy), n_out, channels, CODE[dtype], ptr(km.in_maps), ptr(km.out_maps), ptr(km._device_offsets),
                km._group_start[1], K, iden, ptr(gw), CODE[dtype], ptr(ws), ws.numel())
        if joined:
            check(L.wcn_sparse_depthwise_wgrad_grouped_bias(*args, ptr(gb), CODE[bias_dtype], ptr(bws), bws.numel(), s), "joined")
            assert L.wcn_sparse_depthwise_wgrad_grouped_bias(*args, ptr(gb), CODE[bias_dtype], ptr(bws), 4, s) != 0
            assert L.wcn_sparse_depthwise_wgrad_grouped_bias(*args, None, CODE[bias_dtype], ptr(bws), bws.numel(), s) == -1
        else:
            check(L.wcn_sparse_depthwise_wgrad_grouped(*args, s), "wgrad")
            check(L.wcn_column_sums(ptr(gy), n_out, channels, CODE[dtype], ptr(gb), CODE[bias_dtype], ptr(bws), bws.numel(), s), "sums")
        return gw, gb

    (gw, gb), (gw2, gb2) = run(True), run(False)
    assert torch.equal(gw, gw2) and torch.equal(gb, gb2)
    assert _close_to_sums(gb, gy[:n_out])


@pytest.mark.parametrize("needs", ["both", "bias", "weight"])
@pytest.mark.parametrize("compute_dtype", [None, torch.float16])
def test_layer_gradients(needs, compute_dtype):
    """Which of the two are asked for, and a product in another type than the gradient's (whose sums stay calls of their own)."""
    from warpconvnet_amd.nn.functional.sparse_conv_depth import spatially_sparse_depthwise_conv
    c = _voxels(2000, 5)
    km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
    g = torch.Generator().manual_seed(1)
    dtype = torch.float32 if compute_dtype else torch.bfloat16
    x = torch.randn(2000, 48, generator=g).to(dtype).to(DEV)
    w, b = torch.randn(27, 48, generator=g).to(DEV), torch.randn(48, generator=g).to(DEV)
    w.requires_grad_(needs != "bias")
    b.requires_grad_(needs != "weight")
    x.requires_grad_()
    out = spatially_sparse_depthwise_conv(x, w, km, 2000, compute_dtype=compute_dtype, bias=b)
    gy = torch.randn(2000, 48, generator=g).to(dtype).to(DEV)
    out.backward(gy)
    assert (w.grad is None) == (needs == "bias") and (b.grad is None) == (needs == "weight")
    if b.grad is not None:
        assert _close_to_sums(b.grad, gy)
    if w.grad is not None:
        before = w.grad.clone()
        w.grad = None
        spatially_sparse_depthwise_conv(x, w, km, 2000, compute_dtype=compute_dtype).backward(gy)
        assert torch.equal(w.grad, before)
