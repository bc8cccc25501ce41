"""The kernel for narrow layers on fp32 rows: every instance against the fp64 oracle and the pair-packed kernel, rows that are
narrower than the 16 or 32 channels an instance is made for, infinite features, and what stays with the pair-packed kernel."""
import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features, rel_err
from warpconvnet_amd.utils import synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # c_in, c_out, kernel, voxels per item, extent, epilogue
    (24, 12, (3, 3, 3), 70000, 60, "plain"),   # the last quarter of a row is not there
    (32, 16, (3, 3, 3), 70000, 60, "fused"),
    (16, 16, (3, 3, 3), 70000, 60, "plain"),
    (16, 32, (3, 3, 3), 70000, 60, "fused"),
    (4, 13, (3, 3, 3), 70000, 60, "plain"),    # three quarters are not there, output rows of no whole vectors
    (12, 28, (3, 3, 3), 70000, 60, "fused"),
    (16, 16, (5, 5, 5), 90000, 70, "plain"),   # 125 KB of weights beside eight waves' sums
    (8, 8, (5, 4, 4), 90000, 70, "fused"),     # more than 64 offsets, sixteen waves' worth of LDS
    (32, 16, (4, 4, 3), 70000, 60, "plain"),
]


def _run(bc, items, x, w, ksize, bias, residual, relu):
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    offsets = torch.as_tensor(np.cumsum([0] + [len(i) for i in items]))
    vox = Voxels(torch.as_tensor(bc[:, 1:].copy(), device=DEV), x.to(DEV), offsets=offsets)
    res = None if residual is None else vox.replace(batched_features=residual.to(DEV))
    out = spatially_sparse_conv(vox, w.to(DEV), ksize, bias=bias.to(DEV), residual=res, relu=relu).feature_tensor
    return out, lib().wcn_conv_last_kernel().decode()


@pytest.mark.parametrize("c_in,c_out,ksize,n,extent,epilogue", CASES, ids=[f"{c[0]}_{c[1]}_{''.join(map(str, c[2]))}" for c in CASES])
def test_fp32_rows_of_narrow_layers(oracle, monkeypatch, c_in, c_out, ksize, n, extent, epilogue):
    items = [synthetic.random_cloud(90 + b, n, extent)[:, 1:] for b in range(2)]
    bc = synthetic.batch_indexed(items)
    K = int(np.prod(ksize))
    x = normal_features(len(bc), c_in, seed=31)
    w = kaiming_weight(K, c_in, c_out, seed=32)
    bias = torch.randn(c_out, generator=torch.Generator().manual_seed(33)) * 0.1
    residual = normal_features(len(bc), c_out, seed=34) if epilogue == "fused" else None
    got, kernel = _run(bc, items, x, w, ksize, bias, residual, epilogue == "fused")
    name = "conv_fwd_group<float, %d, %s, %d," % ((c_out + 15) // 16, "true" if c_in <= 16 else "false", 1 if K <= 64 else 2)
    assert kernel.startswith(name), kernel
    im, om, off, iden = oracle.kernel_map(bc, bc, ksize)
    want = oracle.explicit_conv_f64(x.double().numpy(), w.double().numpy(), im, om, off, iden, len(bc)) + bias.double().numpy()
    if residual is not None:
        want = np.maximum(want + residual.double().numpy(), 0)
    # at most K * c_in products a sum, each with one rounding of 2^-24, which add up like a random walk
    assert rel_err(got.cpu().numpy(), want) <= 1e-5
    again, _ = _run(bc, items, x, w, ksize, bias, residual, epilogue == "fused")
    assert torch.equal(got, again)
    # an infinite feature reaches what it reaches in the kernel these rows went to before, as the same value
    x[len(x) // 2, 0] = float("inf")
    got, kernel = _run(bc, items, x, w, ksize, bias, residual, epilogue == "fused")
    assert kernel.startswith(name), kernel
    monkeypatch.setenv("WCN_CONV_KERNEL", "pack")
    before, kernel = _run(bc, items, x, w, ksize, bias, residual, epilogue == "fused")
    assert kernel.startswith("conv_fwd_pack<float"), kernel
    assert torch.equal(torch.isnan(got), torch.isnan(before)) and torch.equal(torch.isinf(got), torch.isinf(before))
    finite = torch.isfinite(got)
    assert torch.allclose(got[finite], before[finite], rtol=1e-4, atol=1e-5)


def test_more_than_16_channels_on_both_sides_stay_with_the_pair_packed_kernel():
    bc = synthetic.batch_indexed([synthetic.random_cloud(95, 80000, 80)[:, 1:]])
    for c_in, c_out, name in ((24, 20, "conv_fwd_pack<float"), (24, 16, "conv_fwd_group<float"), (16, 20, "conv_fwd_group<float")):
        x, w = normal_features(len(bc), c_in, seed=35), kaiming_weight(27, c_in, c_out, seed=36)
        _, kernel = _run(bc, [bc], x, w, (3, 3, 3), torch.zeros(c_out), None, False)
        assert kernel.startswith(name), kernel
