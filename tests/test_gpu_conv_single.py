"""The contraction for one pair per output row (csrc/wcn_conv_single.hip) where its tiles end: runs of pairs around whole
tiles, empty offsets, and entries that name no row."""
import ctypes

import numpy as np
import pytest
import torch

from warpconvnet_amd._lib import check, lib, ptr, stream_ptr, workspace

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("c_in,c_out", [(32, 24), (64, 64), (96, 8), (128, 104), (192, 32), (256, 256)])
def test_runs_around_whole_tiles(c_in, c_out, dtype):
    counts = [0, 1, 64, 65, 0, 127, 128, 129, 255, 256, 257, 700, 0]
    g = torch.Generator().manual_seed(c_in + c_out)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    n, n_in, K = int(offsets[-1]), 911, len(counts)
    x = torch.randn(n_in, c_in, generator=g).to(dtype).to(DEV)
    w = (torch.randn(K, c_in, c_out, generator=g) / c_in ** 0.5).to(dtype).to(DEV)
    res = torch.randn(n, c_out, generator=g).to(dtype).to(DEV)
    im = torch.randint(0, n_in, (n,), generator=g, dtype=torch.int32)
    om = torch.randperm(n, generator=g).int()
    im[5], om[70], im[300] = -1, n, n_in  # name no row: leave theirs as it is
    im, om = im.to(DEV), om.to(DEV)
    out = torch.full((n, c_out), 7.0, dtype=dtype, device=DEV)
    L, code = lib(), 1 if dtype is torch.float16 else 2
    ws = workspace(L.wcn_conv_prepared_weight_bytes(K, c_in, c_out, code), DEV)
    check(L.wcn_sparse_conv_fwd_single(ptr(x), n_in, c_in, code, ptr(w), code, 0, K, c_out, None, ptr(im), ptr(om),
                                       (ctypes.c_int64 * (K + 1))(*offsets), ptr(res), 1, ptr(out), n, ptr(ws), ws.numel(),
                                       stream_ptr(DEV)), "single")
    want = torch.full((n, c_out), 7.0, dtype=torch.float64, device=DEV)
    room = torch.zeros_like(want)
    for k in range(K):
        i, o = im[offsets[k]:offsets[k + 1]].long(), om[offsets[k]:offsets[k + 1]].long()
        ok = (i >= 0) & (i < n_in) & (o < n)
        i, o = i[ok], o[ok]
        want[o] = (x[i].double() @ w[k].double() + res[o].double()).clamp(min=0.0)
        room[o] = x[i].double().abs() @ w[k].double().abs() + res[o].double().abs()
    # fp32 sums of c_in products and the residual, one rounding
    sums = (c_in + 1) * 2.0 ** -24 * room
    unit = 2.0 ** -11 if dtype is torch.float16 else 2.0 ** -8
    assert bool(((out.double() - want).abs() <= unit * (want.abs() + sums) + sums + 2.0 ** -25).all())
