"""The contraction over a tile plan against the fp64 oracle and, bit for bit, against the same product over
the bare pair lists: row counts around a tile of 128, channel counts around the instances' widths and slices,
maps of 8 and 27 offsets, with and without identity, every form of the weight and the epilogue's extras."""
import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features, rel_err
from warpconvnet_amd.utils import synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.float16: 1, torch.bfloat16: 2}


def _surface(n, seed):
    """n distinct voxels of three planes that meet, in random order."""
    side = int(np.ceil(np.sqrt(n / 2.0))) + 2
    g = np.random.default_rng(seed)
    uv = np.stack(np.meshgrid(np.arange(side), np.arange(side), indexing="ij"), -1).reshape(-1, 2)
    z = np.zeros((len(uv), 1), dtype=np.int64)
    c = np.unique(np.concatenate([np.hstack([uv, z]), np.hstack([uv[:, :1], z, uv[:, 1:]]), np.hstack([z, uv])]), axis=0)
    c = c[g.permutation(len(c))[:n]]
    return np.hstack([np.zeros((len(c), 1), dtype=np.int64), c]).astype(np.int32)


def _tiled(km, x, w, form, n_out, c_out, bias=None, rounded=0, residual=None, relu=0):
    from warpconvnet_amd._lib import check, lib, ptr, stream_ptr, workspace
    L, K, pairs = lib(), len(km), km.in_maps.shape[0]
    iden = -1 if km.identity_map_index is None else km.identity_map_index
    s = stream_ptr(x.device)
    plan = workspace(L.wcn_tile_plan_bytes(n_out, K), x.device)
    ws = workspace(L.wcn_tile_plan_workspace_bytes(n_out, K, pairs), x.device)
    check(L.wcn_tile_plan_build(ptr(km.in_maps), ptr(km.out_maps), ptr(km._device_offsets), km._group_start[1], K, iden,
                                x.shape[0], n_out, pairs, ptr(plan), plan.numel(), ptr(ws), ws.numel(), s), "plan")
    out = torch.full((n_out, c_out), float("nan"), dtype=x.dtype, device=x.device)
    wb = L.wcn_conv_prepared_weight_bytes(K, x.shape[1], c_out, CODE[x.dtype])
    tiles = workspace(wb, x.device)
    wcode = 0 if w.dtype == torch.float32 else CODE[w.dtype]
    if form == 1:
        check(L.wcn_conv_prepare_weight(ptr(w), wcode, K, x.shape[1], c_out, CODE[x.dtype], ptr(tiles), wb, s), "prep")
        w = tiles
    check(L.wcn_sparse_conv_fwd_tiled(ptr(x), x.shape[0], x.shape[1], CODE[x.dtype], ptr(w), wcode, form, K, c_out,
                                      ptr(bias), CODE[x.dtype], rounded, ptr(plan), ptr(residual), relu, ptr(out), n_out, ptr(tiles),
                                      wb, s), "wcn_sparse_conv_fwd_tiled")
    return out


@pytest.mark.parametrize("n", [1, 127, 128, 129, 1000, 5003])
@pytest.mark.parametrize("dtype,c_in,c_out,ksize,stride", [
    (torch.bfloat16, 64, 64, 3, 1), (torch.float16, 96, 96, 3, 1), (torch.bfloat16, 128, 256, 3, 1),
    (torch.float16, 8, 24, 3, 1), (torch.float16, 40, 72, 3, 2), (torch.bfloat16, 64, 128, 2, 2),
    (torch.float16, 200, 136, 3, 1)])
def test_tiled_contraction_matches_the_oracle(oracle, n, dtype, c_in, c_out, ksize, stride):
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    bc = _surface(n, n)
    c = torch.as_tensor(bc, device=DEV)
    out_c = c if stride == 1 else stride_coords(c, (stride,) * 3)[0]
    m = len(out_c)
    km = generate_kernel_map(c, out_c, (stride,) * 3, (ksize,) * 3)
    x = normal_features(len(bc), c_in, seed=1, dtype=dtype)
    w = kaiming_weight(ksize ** 3, c_in, c_out, seed=2, dtype=dtype)
    bias = (torch.randn(c_out, generator=torch.Generator().manual_seed(3)) * 0.1).to(dtype)
    res = normal_features(m, c_out, seed=4, dtype=dtype)
    im, om, off, iden = oracle.kernel_map(bc, out_c.cpu().numpy(), (ksize,) * 3, (stride,) * 3)
    want = oracle.explicit_conv_f64(x.double().numpy(), w.double().numpy(), im, om, off, iden, m)
    xd, wd = x.to(DEV), w.to(DEV)
    plain = _tiled(km, xd, wd, 0, m, c_out)
    assert rel_err(plain.double().cpu().numpy(), want) <= 1e-2
    assert torch.equal(plain, _tiled(km, xd, wd, 1, m, c_out))
    assert torch.equal(plain, _tiled(km, xd, wd.transpose(1, 2).contiguous(), 2, m, c_out))
    assert torch.equal(plain, _tiled(km, xd, wd.flip(0).transpose(1, 2).contiguous(), 3, m, c_out))
    bd, rd = bias.to(DEV), res.to(DEV)
    assert torch.equal(_tiled(km, xd, wd, 0, m, c_out, bias=bd, rounded=1), plain + bd)
    got = _tiled(km, xd, wd, 0, m, c_out, bias=bd, residual=rd, relu=1)
    full = np.maximum(want + bias.double().numpy() + res.double().numpy(), 0.0)
    assert rel_err(got.double().cpu().numpy(), full) <= 1e-2


def test_layers_over_one_map_take_the_plan_and_give_the_same_bits():
    """A surface large enough for the plan: the first layer over the map runs without, the second makes it; forward
    and gradients agree with those over the bare lists."""
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.geometry.coords.search.search_results import IntSearchResult
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_backward, sparse_conv_forward
    c = torch.as_tensor(_surface(40_000, 9), device=DEV)
    n = len(c)
    km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
    bare = IntSearchResult(km.in_maps, km.out_maps, km.offsets, km.identity_map_index)
    bare._out_ascend = True
    x = normal_features(n, 64, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 64, 64, seed=2, dtype=torch.float16).to(DEV)
    gy = normal_features(n, 64, seed=3, dtype=torch.float16).to(DEV)
    names, outs = [], []
    for m in (km, km, bare):
        outs.append(sparse_conv_forward(x, w, m, n))
        names.append(lib().wcn_conv_last_kernel().decode())
    assert [name.startswith("conv_fwd_tiles<") for name in names] == [False, True, False], names
    assert torch.equal(outs[1], outs[2]) and torch.equal(outs[0], outs[2])
    gx, _ = sparse_conv_backward(gy, x, w, km, need_weight_grad=False)
    assert lib().wcn_conv_last_kernel().decode().startswith("conv_fwd_tiles<")
    want, _ = sparse_conv_backward(gy, x, w, bare, need_weight_grad=False)
    assert float((gx.float() - want.float()).norm() / want.float().norm()) <= 1e-3


@pytest.mark.parametrize("dtype,c_in,c_out,n", [
    (torch.float16, 64, 64, 40_000),     # the pair-packed kernel stands behind the plan
    (torch.bfloat16, 128, 128, 20_000),  # the one for small maps: its waves' sums are added last
    (torch.bfloat16, 128, 128, 40_000),  # the one for wide rows
    (torch.float16, 32, 32, 40_000),     # narrow rows: small maps, and beyond them the kernel that starts with the
    (torch.float16, 24, 32, 90_000),     # identity's product
    (torch.float16, 320, 64, 90_000),    # the ring kernel: channels outside the offsets
    (torch.bfloat16, 512, 32, 34_000)],  # the same with its slices apart
    ids=["f16_64_64", "bf16_128_128_small", "bf16_128_128", "f16_32_32", "f16_24_32", "f16_320_64", "bf16_512_32"])
def test_results_do_not_depend_on_the_layers_before(dtype, c_in, c_out, n):
    """The same layer three times over one map, then over a map that a wider layer has left its plan on: the same
    bits each time, with and without gradients, and in the input gradient."""
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_backward, sparse_conv_forward, spatially_sparse_conv
    coords = torch.as_tensor(_surface(n, 12)[:, 1:].copy(), device=DEV)
    x = normal_features(n, c_in, seed=1, dtype=dtype).to(DEV)
    wide = normal_features(n, 256, seed=1, dtype=dtype).to(DEV)
    w = kaiming_weight(27, c_in, c_out, seed=2, dtype=dtype).to(DEV)
    res = normal_features(n, c_out, seed=4, dtype=dtype).to(DEV)
    gy = normal_features(n, c_out, seed=3, dtype=dtype).to(DEV)
    w_wide = kaiming_weight(27, 256, 256, seed=5, dtype=dtype).to(DEV)

    def fresh():
        return Voxels(coords, x, offsets=torch.tensor([0, n]))

    def calls(vox):
        plain = spatially_sparse_conv(vox, w, 3, residual=res, relu=True).feature_tensor
        km = next(iter(vox.cache.values()))
        wg = w.clone().requires_grad_(True)
        graph = spatially_sparse_conv(vox, wg, 3).feature_tensor.detach()
        gx, _ = sparse_conv_backward(gy, x, w, km, need_weight_grad=False)
        return km, (plain, graph, gx)

    vox = fresh()
    km, first = calls(vox)
    for _ in range(2):
        assert all(torch.equal(a, b) for a, b in zip(calls(vox)[1], first))
    vox = fresh()
    calls(vox)  # (leaves the map in the cache)
    km = next(iter(vox.cache.values()))
    km._tile_plan = None
    sparse_conv_forward(wide, w_wide, km, n)
    assert km._tile_plan is not None
    assert all(torch.equal(a, b) for a, b in zip(calls(vox)[1], first))


def _with_infinities(w):
    """An infinite, a NaN and (fp32: of fp16 features) a too large weight in three offsets that few rows have pairs in."""
    w = w.clone()
    w[2, 3, 7], w[11, 0, 0], w[20, 5, 9] = float("inf"), float("nan"), 1e6 if w.dtype == torch.float32 else -float("inf")
    return w


@pytest.mark.parametrize("kernel,dtype,c_in,c_out,n", [
    ("tiles", torch.float16, 64, 64, 5003), ("tiles", torch.bfloat16, 128, 256, 5003), ("tiles", torch.float16, 40, 24, 700),
    ("tiles", torch.float16, 96, 96, 3000), ("small", torch.float16, 64, 64, 5003), ("small", torch.bfloat16, 32, 32, 700),
    ("small", torch.float32, 32, 64, 3000)])
@pytest.mark.parametrize("wide_weight", [False, True], ids=["", "fp32_weight"])
def test_infinite_weights_reach_only_rows_with_pairs_in_their_offsets(oracle, kernel, dtype, c_in, c_out, n, wide_weight):
    """A place without a pair multiplies zeros, and zero times infinity is no zero: those rows stay as they are."""
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    bc = _surface(n, n)
    c = torch.as_tensor(bc, device=DEV)
    km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
    x = normal_features(n, c_in, seed=1, dtype=dtype)
    w = _with_infinities(kaiming_weight(27, c_in, c_out, seed=2, dtype=torch.float32 if wide_weight else dtype))
    im, om, off, iden = oracle.kernel_map(bc, bc, (3, 3, 3), (1, 1, 1))
    want = oracle.explicit_conv_f64(x.double().numpy(), w.to(dtype).double().numpy(), im, om, off, iden, n)
    some = np.isfinite(want)
    assert 0.01 < (~some).any(axis=1).mean() < 0.9
    xd, wd = x.to(DEV), w.to(DEV)
    if kernel == "tiles":
        got = _tiled(km, xd, wd, 0, n, c_out)
    else:
        got = sparse_conv_forward(xd, wd, km, n)
        assert lib().wcn_conv_last_kernel().decode().startswith("conv_fwd_small<")
    got = got.double().cpu().numpy()
    assert np.array_equal(np.isfinite(got), some) and np.array_equal(np.isnan(got), np.isnan(want))
    assert rel_err(got[some], want[some]) <= (1e-5 if dtype == torch.float32 else 1e-2)
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])


def test_no_plan_for_an_input_gradient_nobody_asks_for():
    """512 -> 64 with gradients: the forward product takes no plan (its slices are summed apart), the input gradient
    does, where there is one."""
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_backward, spatially_sparse_conv
    n = 40_000
    coords = torch.as_tensor(_surface(n, 14)[:, 1:].copy(), device=DEV)
    w = kaiming_weight(27, 512, 64, seed=2, dtype=torch.float16).to(DEV).requires_grad_(True)
    gy = normal_features(n, 64, seed=3, dtype=torch.float16).to(DEV)
    for wanted in (False, True):
        x = normal_features(n, 512, seed=1, dtype=torch.float16).to(DEV).requires_grad_(wanted)
        vox = Voxels(coords, x, offsets=torch.tensor([0, n]))
        out = spatially_sparse_conv(vox, w, 3).feature_tensor
        km = next(iter(vox.cache.values()))
        assert (km._tile_plan is not None) == wanted
        out.backward(gy)
        assert (x.grad is not None) == wanted
        km._tile_plan = None
        sparse_conv_backward(gy, x.detach(), w.detach(), km, need_input_grad=wanted)
        assert (km._tile_plan is not None) == wanted
