"""The contraction for small maps (csrc/wcn_conv_split.hip: the offsets of a tile dealt to the waves of a
workgroup) at the edges of its tiles, and the kernels it stands in front of at the sizes they keep."""
import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features, rel_err
from warpconvnet_amd.utils import synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {torch.float32: 1e-5, torch.float16: 1e-2, torch.bfloat16: 1e-2}


def _run(oracle, dtype, c_in, c_out, rows, extent, ksize, stride=(1, 1, 1), residual=False, seed=5):
    """(output twice, fp64 oracle, kernel) of one contraction over `rows` random voxels."""
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    bc = synthetic.random_cloud(seed, 2 * rows, extent)[:rows]
    c = torch.as_tensor(np.ascontiguousarray(bc), device=DEV)
    out_c = c if stride == (1, 1, 1) else stride_coords(c, stride)[0]
    out_bc = out_c.cpu().numpy()
    km = generate_kernel_map(c, out_c, stride, ksize)
    K = int(np.prod(ksize))
    x = normal_features(len(bc), c_in, seed=6, dtype=dtype)
    w = kaiming_weight(K, c_in, c_out, seed=7, dtype=dtype)
    bias = (torch.randn(c_out, generator=torch.Generator().manual_seed(8)) * 0.1).to(dtype)
    res = normal_features(len(out_bc), c_out, seed=9, dtype=dtype) if residual else None
    im, om, off, iden = oracle.kernel_map(bc, out_bc, ksize, stride)
    want = oracle.explicit_conv_f64(x.double().numpy(), w.double().numpy(), im, om, off, iden, len(out_bc))
    want = want + bias.double().numpy()
    if residual:
        want = np.maximum(want + res.double().numpy(), 0.0)
    wd = w.to(DEV)
    got = [sparse_conv_forward(x.to(DEV), wd, km, len(out_bc), bias=bias.to(DEV),
                               residual=None if res is None else res.to(DEV), relu=residual,
                               keep_prepared_weight=keep) for keep in (False, True)]
    return got, want, lib().wcn_conv_last_kernel().decode()


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 64, 65, 700])
@pytest.mark.parametrize("dtype,c_in,c_out,ksize,residual", [
    (torch.bfloat16, 32, 32, (3, 3, 3), True), (torch.float16, 40, 72, (3, 3, 3), True),
    (torch.float16, 72, 20, (3, 3, 3), False), (torch.bfloat16, 256, 192, (3, 3, 3), True),
    (torch.float32, 32, 64, (3, 3, 3), True), (torch.float32, 68, 24, (2, 3, 2), False),
    (torch.float16, 16, 16, (5, 5, 5), False)],
    ids=["bf16_32_32", "f16_40_72", "f16_72_20", "bf16_256_192", "f32_32_64", "f32_68_24", "f16_16_16_k5"])
def test_small_maps_match_the_oracle(oracle, dtype, c_in, c_out, ksize, residual, rows):
    got, want, kernel = _run(oracle, dtype, c_in, c_out, rows, 12, ksize, residual=residual)
    assert kernel.startswith("conv_fwd_small<"), kernel
    assert torch.equal(got[0], got[1])  # kept tiles and tiles made in the call, and one order of additions
    assert rel_err(got[0].double().cpu().numpy(), want) <= TOL[dtype]


def test_small_strided_map_without_identity(oracle):
    got, want, kernel = _run(oracle, torch.float16, 64, 64, 900, 14, (3, 3, 3), stride=(2, 2, 2))
    assert kernel.startswith("conv_fwd_small<"), kernel
    assert torch.equal(got[0], got[1]) and rel_err(got[0].double().cpu().numpy(), want) <= 1e-2


@pytest.mark.parametrize("dtype,c_in,c_out,rows,extent,ksize,kernel", [
    (torch.bfloat16, 32, 32, 90_000, 70, (3, 3, 3), "conv_fwd_group<bf16, 2, false"),
    (torch.float16, 12, 20, 90_000, 70, (3, 3, 3), "conv_fwd_group<f16, 2, true"),
    (torch.float16, 16, 16, 80_000, 80, (5, 5, 5), "conv_fwd_group<f16, 1, true"),
    (torch.float16, 64, 64, 60_000, 60, (3, 3, 3), "conv_fwd_pack<"),
    (torch.float32, 32, 24, 60_000, 60, (3, 3, 3), "conv_fwd_pack<"),
    (torch.bfloat16, 160, 64, 60_000, 70, (3, 3, 3), "conv_fwd_ring<")],
    ids=["group", "group_narrow", "group_k5", "pack", "pack_f32", "ring"])
def test_larger_maps_keep_their_kernels(oracle, dtype, c_in, c_out, rows, extent, ksize, kernel):
    got, want, name = _run(oracle, dtype, c_in, c_out, rows, extent, ksize, residual=True)
    assert name.startswith(kernel), name
    assert torch.equal(got[0], got[1]) and rel_err(got[0].double().cpu().numpy(), want) <= TOL[dtype]


def test_kept_tiles_are_those_that_are_read():
    """One weight over a small map, a large one and the small one again: a half of the tiles for each kind of map, made
    when first asked for and found again, with the bits of the calls that make their own."""
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    w = kaiming_weight(27, 64, 64, seed=2, dtype=torch.float16).to(DEV)
    half = lib().wcn_conv_prepared_weight_bytes(27, 64, 64, 1) // 2
    seen = []
    for n, extent in ((3000, 20), (60_000, 60), (3000, 20), (60_000, 60)):
        c = torch.as_tensor(np.ascontiguousarray(synthetic.random_cloud(3, n, extent)), device=DEV)
        km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
        x = normal_features(len(c), 64, seed=4, dtype=torch.float16).to(DEV)
        before = torch.cuda.memory_allocated()
        kept = sparse_conv_forward(x, w, km, len(c), keep_prepared_weight=True)
        seen.append((lib().wcn_conv_last_kernel().decode().startswith("conv_fwd_small<"),
                     torch.cuda.memory_allocated() - before - (kept.numel() * 2 + 511) // 512 * 512))
        assert torch.equal(kept, sparse_conv_forward(x, w, km, len(c)))
        del kept
    assert [small for small, _ in seen] == [True, False, True, False]
    assert [bytes_ for _, bytes_ in seen] == [half, half, 0, 0]


# (dtype, C_in, C_out, rows, instance): sixteen, thirty-two or sixty-four channels a tile, as long as every tile has one of the 256 CUs
# (forty-eight where that leaves less over), and eight or sixteen waves (from 100 units on)
_TILES = [(torch.bfloat16, 32, 32, 4096, "1, 8"), (torch.bfloat16, 32, 32, 4097, "2, 8"), (torch.bfloat16, 64, 64, 2080, "2, 8"),
          (torch.float16, 128, 128, 1024, "1, 16"), (torch.float16, 128, 128, 1025, "2, 16"),
          (torch.float16, 128, 128, 2049, "4, 16"), (torch.float16, 120, 100, 4097, "4, 8"),
          (torch.float32, 64, 40, 2048, "1, 16"), (torch.float32, 64, 72, 2049, "2, 16"), (torch.float32, 16, 20, 60, "1, 8"),
          (torch.float32, 64, 64, 4097, "4, 8"), (torch.float16, 32, 16, 8193, "1, 8"), (torch.float32, 64, 12, 8193, "1, 8"),
          (torch.bfloat16, 96, 96, 4097, "3, 8"), (torch.float16, 64, 136, 2100, "3, 8"), (torch.float32, 48, 40, 8193, "3, 8")]


@pytest.mark.parametrize("infinite", [False, True], ids=["finite", "infinite_weight"])
@pytest.mark.parametrize("dtype,c_in,c_out,rows,tile", _TILES, ids=[f"{t[1]}_{t[2]}_{t[3]}_{t[4].replace(', ', 'x')}" for t in _TILES])
def test_tiles_get_wider_when_the_cus_are_taken(oracle, dtype, c_in, c_out, rows, tile, infinite):
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    bc = synthetic.random_cloud(11, 2 * rows, max(8, int(round((3 * rows) ** (1 / 3)))))[:rows]
    assert len(bc) == rows
    c = torch.as_tensor(np.ascontiguousarray(bc), device=DEV)
    km = generate_kernel_map(c, c, (1, 1, 1), (3, 3, 3))
    x, w = normal_features(rows, c_in, seed=6, dtype=dtype), kaiming_weight(27, c_in, c_out, seed=7, dtype=dtype)
    if infinite:
        w[2, 3, 7], w[20, 5, 9] = float("inf"), float("nan")
    im, om, off, iden = oracle.kernel_map(bc, bc, (3, 3, 3))
    with np.errstate(invalid="ignore"):
        want = oracle.explicit_conv_f64(x.double().numpy(), w.double().numpy(), im, om, off, iden, rows)
    got = sparse_conv_forward(x.to(DEV), w.to(DEV), km, rows).double().cpu().numpy()
    text = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "float"}[dtype]
    assert lib().wcn_conv_last_kernel().decode() == f"conv_fwd_small<{text}, {tile}>"
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert rel_err(np.where(np.isfinite(want), got, 0.0), np.where(np.isfinite(want), want, 0.0)) <= TOL[dtype]


@pytest.mark.parametrize("dtype,c_in,c_out,rows,extent,ksize,kernel", [
    (torch.float32, 96, 96, 24_000, 60, (3, 3, 3), "conv_fwd_pack<float"), (torch.float32, 128, 40, 48_000, 60, (3, 3, 3), "conv_fwd_pack<float"),
    (torch.float32, 36, 64, 45_000, 60, (3, 3, 3), "conv_fwd_pack<float"), (torch.float32, 160, 64, 12_000, 40, (3, 3, 3), "conv_fwd_small<float, 4, 8"),
    (torch.float32, 64, 64, 2500, 30, (5, 5, 5), "conv_fwd_small<float, 2, 16"), (torch.float16, 256, 256, 12_000, 50, (3, 3, 3), "conv_fwd_ring<"),
    (torch.float16, 128, 128, 12_000, 50, (2, 2, 2), "conv_fwd_small<f16, 4, 8"),
    # narrow layers: what comes behind is the kernel of their own, or the pair-packed one where their weights are too many for it
    (torch.float32, 16, 16, 49_000, 70, (5, 5, 5), "conv_fwd_small<float, 1, 8"), (torch.float32, 16, 16, 51_000, 70, (5, 5, 5), "conv_fwd_group<float, 1, true, 2"),
    (torch.float32, 16, 16, 55_000, 70, (3, 3, 3), "conv_fwd_small<float, 1, 8"), (torch.float32, 16, 16, 58_000, 70, (3, 3, 3), "conv_fwd_group<float, 1, true, 1"),
    (torch.float32, 32, 16, 44_000, 70, (3, 3, 3), "conv_fwd_small<float, 1, 8"), (torch.float32, 32, 16, 46_000, 70, (3, 3, 3), "conv_fwd_group<float, 1, false"),
    (torch.float32, 12, 32, 48_000, 70, (3, 3, 3), "conv_fwd_small<float, 2, 8"), (torch.float32, 12, 32, 50_000, 70, (3, 3, 3), "conv_fwd_group<float, 2, true"),
    (torch.bfloat16, 16, 32, 90_000, 90, (4, 4, 4), "conv_fwd_small<bf16, 2, 8"), (torch.bfloat16, 16, 32, 95_000, 90, (4, 4, 4), "conv_fwd_pack<"),
    (torch.bfloat16, 16, 16, 66_000, 80, (4, 4, 4), "conv_fwd_group<bf16, 1, true")],
    ids=["f32_three_slices", "f32_four_slices", "f32_part_of_a_slice", "f32_five_slices", "f32_k5", "f16_ring", "f16_k2", "f32_narrow_k5_below",
         "f32_narrow_k5_above", "f32_narrow_below", "f32_narrow_above", "f32_32_16_below", "f32_32_16_above", "f32_12_32_below", "f32_12_32_above",
         "bf16_narrow_k4_below", "bf16_narrow_k4_above", "bf16_narrow_k4_group"])
def test_lines_between_the_kernels(oracle, dtype, c_in, c_out, rows, extent, ksize, kernel):
    got, want, name = _run(oracle, dtype, c_in, c_out, rows, extent, ksize, residual=True)
    assert name.startswith(kernel), name
    assert torch.equal(got[0], got[1]) and rel_err(got[0].double().cpu().numpy(), want) <= TOL[dtype]
