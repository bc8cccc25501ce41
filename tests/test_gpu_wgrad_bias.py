"""Weight and bias gradient in one call against the two calls, bit for bit, and the bias against float64 sums: channel
counts around the 16 a workgroup finishes, rows around the parts of the first pass, rows that are no whole vectors or not aligned (finished in
a launch of their own), every type of bias."""
import ctypes

import numpy as np
import pytest
import torch

from warpconvnet_amd._lib import check, lib, ptr, stream_ptr, workspace

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


@pytest.mark.parametrize("c_out,rows,dtype,bias_dtype,shift", [
    (8, 1, torch.float16, torch.float32, 0), (16, 63, torch.bfloat16, torch.bfloat16, 0), (24, 2047, torch.float16, torch.float16, 0),
    (96, 40000, torch.bfloat16, torch.float32, 0), (200, 5000, torch.float16, torch.float32, 0), (13, 300, torch.float16, torch.float32, 0),
    (32, 300, torch.float32, torch.float32, 0), (32, 300, torch.float16, torch.float32, 4)])
def test_weight_and_bias_gradient_in_one_call(c_out, rows, dtype, bias_dtype, shift):
    g = torch.Generator().manual_seed(c_out + rows)
    n_in, c_in, counts = 500, 40, [0, 65, 300]
    x = torch.randn(n_in, c_in, generator=g).to(dtype).to(DEV)
    gy = torch.randn(rows * c_out + shift, generator=g).to(dtype).to(DEV)[shift:].view(rows, c_out)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    im = torch.randint(0, n_in, (int(offsets[-1]),), generator=g, dtype=torch.int32).to(DEV)
    om = torch.randint(0, rows, (int(offsets[-1]),), generator=g, dtype=torch.int32).to(DEV)
    host = (ctypes.c_int64 * 4)(*offsets)
    L, s = lib(), stream_ptr(DEV)

    def run(joined):
        gw = torch.empty(3, c_in, c_out, device=DEV)
        gb = torch.empty(c_out, dtype=bias_dtype, device=DEV)
        ws = workspace(L.wcn_conv_wgrad_workspace_bytes(3, c_in, c_out, int(offsets[-1]), 0), DEV)
        bws = workspace(L.wcn_column_sums_workspace_bytes(c_out), DEV)
        args = (ptr(x), n_in, c_in, ptr(gy), rows, c_out, CODE[dtype], ptr(im), ptr(om), host, None, 3, -1, ptr(gw), 0, ptr(ws),
                ws.numel())
        if joined:
            check(L.wcn_sparse_conv_wgrad_bias(*args, ptr(gb), CODE[bias_dtype], ptr(bws), bws.numel(), s), "wgrad_bias")
            assert L.wcn_sparse_conv_wgrad_bias(*args, ptr(gb), CODE[bias_dtype], ptr(bws), 4, s) != 0
            assert L.wcn_sparse_conv_wgrad_bias(*args, None, CODE[bias_dtype], ptr(bws), bws.numel(), s) == -1
        else:
            check(L.wcn_sparse_conv_wgrad_mapped(*args, s), "wgrad")
            check(L.wcn_column_sums(ptr(gy), rows, c_out, CODE[dtype], ptr(gb), CODE[bias_dtype], ptr(bws), bws.numel(), s), "sums")
        return gw, gb

    (gw, gb), (gw2, gb2) = run(True), run(False)
    assert torch.equal(gw, gw2) and torch.equal(gb, gb2)
    want = gy.double().sum(0)
    # fp32 sums: each addition rounds by 2^-24 of a partial sum, which is at most the sum of the magnitudes; then the bias's type
    bound = gy.double().abs().sum(0) * 2.0 ** -20 + want.abs() * {torch.float32: 0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[bias_dtype]
    assert ((gb.double() - want).abs() <= bound + 1e-7).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out,rows,pairs", [(8, 8, 0, 0), (8, 8, 5, 0), (32, 32, 3000, 1), (64, 264, 70_001, 5000), (136, 64, 33_000, 64),
                                                   (96, 96, 300_000, 20_000)])
def test_column_sums_beside_any_weight_gradient(c_in, c_out, rows, pairs, dtype):
    """The sums ride on the weight gradient's launches, also where that has no pair, and no row, to work on."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(700, c_in, generator=g).to(dtype).to(DEV)
    gy = torch.randn(rows, c_out, generator=g).to(dtype).to(DEV)
    im = torch.randint(0, 700, (max(pairs, 1),), generator=g, dtype=torch.int32).to(DEV)
    om = torch.randint(0, max(rows, 1), (max(pairs, 1),), generator=g, dtype=torch.int32).to(DEV)
    host = (ctypes.c_int64 * 3)(0, pairs // 3, pairs)
    L, s = lib(), stream_ptr(DEV)
    ws = workspace(L.wcn_conv_wgrad_workspace_bytes(2, c_in, c_out, pairs, 0), DEV)
    bws = workspace(L.wcn_column_sums_workspace_bytes(c_out), DEV)
    gw, gw2 = (torch.full((2, c_in, c_out), 9.0, device=DEV) for _ in range(2))
    gb, gb2 = (torch.full((c_out,), 9.0, device=DEV) for _ in range(2))
    args = (ptr(x), 700, c_in, ptr(gy) if rows else None, rows, c_out, CODE[dtype], ptr(im), ptr(om), host, None, 2, -1)
    check(L.wcn_sparse_conv_wgrad_bias(*args, ptr(gw), 0, ptr(ws), ws.numel(), ptr(gb), 0, ptr(bws), bws.numel(), s), "wgrad_bias")
    check(L.wcn_sparse_conv_wgrad_mapped(*args, ptr(gw2), 0, ptr(ws), ws.numel(), s), "wgrad")
    check(L.wcn_column_sums(ptr(gy) if rows else None, rows, c_out, CODE[dtype], ptr(gb2), 0, ptr(bws), bws.numel(), s), "sums")
    assert torch.equal(gw, gw2) and torch.equal(gb, gb2)
    assert pairs > 0 or not gw.any()
    assert ((gb.double() - gy.double().sum(0)).abs() <= gy.double().abs().sum(0) * 2.0 ** -20 + 1e-7).all()
