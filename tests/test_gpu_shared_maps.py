"""What layers leave on a map for the layers after them (tile plan, rows forms, re-ordered lists): read from a
stream other than the one that made it, while that one is still busy, and from inside a captured graph."""
import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _surface(n, seed):
    """n distinct voxels of three planes that meet, in random order."""
    side = int(np.ceil(np.sqrt(n / 2.0))) + 2
    uv = np.stack(np.meshgrid(np.arange(side), np.arange(side), indexing="ij"), -1).reshape(-1, 2)
    z = np.zeros((len(uv), 1), dtype=np.int64)
    c = np.unique(np.concatenate([np.hstack([uv, z]), np.hstack([uv[:, :1], z, uv[:, 1:]]), np.hstack([z, uv])]), axis=0)
    c = c[np.random.default_rng(seed).permutation(len(c))[:n]]
    return torch.as_tensor(np.hstack([np.zeros((len(c), 1), dtype=np.int64), c]).astype(np.int32), device=DEV)


def _map(c, out=None, stride=1, ksize=3):
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    return generate_kernel_map(c, c if out is None else out, (stride,) * 3, (ksize,) * 3)


def _occupy(big):
    """Some 10 ms of work in front of whatever the current stream is given next."""
    for _ in range(8):
        big = torch.mm(big, big)
    return big


def _on_two_streams(call):
    """call() behind a long queue on one stream, and at once on another: both results."""
    big = torch.zeros(8192, 8192, device=DEV)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        _occupy(big)
        first = call()
    assert not a.query()  # still busy
    with torch.cuda.stream(b):
        second = call()
    torch.cuda.synchronize()
    return first, second


def test_a_tile_plan_serves_layers_on_other_streams():
    from warpconvnet_amd._lib import lib
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    c = _surface(40_000, 1)
    n, km = len(c), _map(c)
    x = normal_features(n, 128, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 128, 256, seed=2, dtype=torch.float16).to(DEV)
    want = sparse_conv_forward(x, w, _map(c.clone()), n)
    assert lib().wcn_conv_last_kernel().decode().startswith("conv_fwd_tiles<")
    for got in _on_two_streams(lambda: sparse_conv_forward(x, w, km, n)):
        assert torch.equal(got, want)
    assert km._tile_plan is not None


def test_a_tile_plan_in_a_captured_graph():
    """A plan made before the capture, on another stream, is read by the graph; one that would be made inside the
    capture stays the graph's own.  Every replay gives the eager result."""
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    c = _surface(40_000, 3)
    n = len(c)
    x = normal_features(n, 128, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 128, 256, seed=2, dtype=torch.float16).to(DEV)
    for planned in (True, False):
        km = _map(c)
        if planned:
            sparse_conv_forward(x, w, km, n)
            assert km._tile_plan is not None
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            out = sparse_conv_forward(x, w, km, n)
        assert (km._tile_plan is not None) == planned
        for i in range(3):
            x.copy_(normal_features(n, 128, seed=10 + i, dtype=torch.float16))
            want = sparse_conv_forward(x, w, _map(c), n)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), (planned, i)


def test_rows_forms_serve_layers_on_other_streams():
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    from warpconvnet_amd.nn.functional.sparse_conv_depth import spatially_sparse_depthwise_conv
    c = _surface(40_000, 5)
    coarse = stride_coords(c, (2, 2, 2))[0]
    n, m = len(c), len(coarse)
    x = normal_features(n, 32, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(8, 32, 1, seed=2, dtype=torch.float16)[..., 0].to(DEV)
    gy = normal_features(m, 32, seed=3, dtype=torch.float16).to(DEV)

    def step(km):  # the forward reads the form by output row, the input gradient the one by input row
        xg = x.clone().requires_grad_(True)
        out = spatially_sparse_depthwise_conv(xg, w, km, m)
        out.backward(gy)
        return out.detach(), xg.grad

    want = step(_map(c, coarse, 2, 2))
    km = _map(c.clone(), coarse, 2, 2)
    for got in _on_two_streams(lambda: step(km)):
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert len(km._rows_forms) == 2


def test_reordered_lists_serve_layers_on_other_streams():
    """The lists by output row of a map made by hand, and those by input row for its input gradient."""
    from warpconvnet_amd.geometry.coords.search.search_results import IntSearchResult
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_backward, sparse_conv_forward
    c = _surface(40_000, 7)
    n, km = len(c), _map(c)
    x = normal_features(n, 64, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 64, 64, seed=2, dtype=torch.float16).to(DEV)

    def by_hand():  # the pairs of a symmetric map with in and out exchanged, and no word of their order
        m = IntSearchResult(km.out_maps, km.in_maps, km.offsets, km.identity_map_index)
        m._from_builder = m._keys_unique = True
        return m

    def step(m):
        return sparse_conv_forward(x, w, m, n), sparse_conv_backward(x, x, w, m, need_weight_grad=False)[0]

    want = step(by_hand())
    shared = by_hand()
    for got in _on_two_streams(lambda: step(shared)):
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert shared._by_out is not None and shared._by_in is not None


def test_kept_weight_tiles_serve_other_streams_and_are_not_kept_from_a_capture():
    """Tiles made behind a busy queue and read from another stream; tiles that a capture makes are the graph's own."""
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    c = _surface(3_000, 9)
    n, km = len(c), _map(c)
    x = normal_features(n, 64, seed=1, dtype=torch.float16).to(DEV)
    w0 = kaiming_weight(27, 64, 64, seed=2, dtype=torch.float16).to(DEV)
    want = sparse_conv_forward(x, w0, km, n)
    w = w0.clone()
    for got in _on_two_streams(lambda: sparse_conv_forward(x, w, km, n, keep_prepared_weight=True)):
        assert torch.equal(got, want)
    w = w0.clone()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = sparse_conv_forward(x, w, km, n, keep_prepared_weight=True)
    assert not hasattr(w, "_wcn_prepared")
    for i in range(3):
        assert torch.equal(sparse_conv_forward(x, w, km, n, keep_prepared_weight=True), want)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i


def test_a_map_given_back_while_another_stream_reads_it():
    """A layer waits in a busy queue; the map, made on the default stream, is dropped and memory of its sizes is taken
    and overwritten there."""
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    c = _surface(40_000, 11)
    n = len(c)
    x = normal_features(n, 64, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 64, 64, seed=2, dtype=torch.float16).to(DEV)
    want = sparse_conv_forward(x, w, _map(c.clone()), n)
    big = torch.zeros(8192, 8192, device=DEV)
    side = torch.cuda.Stream()
    km = _map(c)
    sizes = [t.untyped_storage().nbytes() for t in (km.in_maps, km.out_maps, km._group_start[0])]
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        _occupy(big)
        got = sparse_conv_forward(x, w, km, n)
    assert not side.query()
    del km
    taken = [torch.empty(s, dtype=torch.uint8, device=DEV).zero_() for s in sizes for _ in range(2)]
    torch.cuda.synchronize()
    assert len(taken) == 6 and torch.equal(got, want)


@pytest.mark.parametrize("rows,ksize,width,assumed", [(1_000_000, 5, 16, None),   # scan, then lists and group starts
                                                      (200_000, 3, 16, None),     # all three in one launch
                                                      (200_000, 3, 16, 0.1),      # lists filled behind the host's wait
                                                      (1_000_000, 3, 16, 27.0)])  # copied there: far fewer than assumed
def test_a_map_just_made_serves_layers_on_other_streams(rows, ksize, width, assumed):
    """The host knows the counts of a map before its lists and group starts are complete: a layer on an idle stream, at once
    and without a synchronisation, waits for them."""
    from warpconvnet_amd._lib import host
    from warpconvnet_amd.geometry.coords.search import torch_discrete
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    c = _surface(rows, 19)
    n = len(c)
    x = normal_features(n, width, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(ksize ** 3, width, width, seed=2, dtype=torch.float16).to(DEV)
    want = sparse_conv_forward(x, w, _map(c, ksize=ksize), n)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(4):
        if assumed is not None:
            torch_discrete._PAIRS_PER_ROW.update({k: assumed for k in torch_discrete._PAIRS_PER_ROW})
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            km = _map(c, ksize=ksize)
        with torch.cuda.stream(b):
            got = sparse_conv_forward(x, w, km, n)
        assert isinstance(km._made, host().MadeOn)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        del km


def test_maps_put_together_of_others_serve_layers_on_other_streams():
    """Over four spatial dimensions the lists are joined behind the builder's wait; half a map has the whole one's lists."""
    from warpconvnet_amd._lib import host
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.nn.functional.sparse_conv import sparse_conv_forward
    at = torch.as_tensor(np.random.default_rng(23).permutation(24 ** 4)[:60_000], device=DEV)
    c = torch.stack([torch.zeros_like(at), at // 24 ** 3, at // 24 ** 2 % 24, at // 24 % 24, at % 24], 1).int()
    n = len(c)
    x = normal_features(n, 16, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(81, 16, 16, seed=2, dtype=torch.float16).to(DEV)
    make = lambda **kw: generate_kernel_map(c, c, (1,) * 4, (3,) * 4, **kw)
    want = sparse_conv_forward(x, w, make(), n)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        km = make()
    with torch.cuda.stream(b):
        got = sparse_conv_forward(x, w, km, n)
    assert isinstance(km._made, host().MadeOn)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    for half, whole in ((make(skip_symmetric_kernel_map=True), km),
                        (generate_kernel_map(c[:, :4].contiguous(), c[:, :4].contiguous(), (1,) * 3, (3,) * 3,
                                             skip_symmetric_kernel_map=True), None)):
        assert isinstance(half._made, host().MadeOn) and half.in_maps.shape[0] == int(half.offsets[-1])
        if whole is not None:
            assert torch.equal(half.in_maps, whole.in_maps[:len(half.in_maps)]) and len(half) == 40


def test_copies_and_files_of_voxels_with_maps():
    """copy.deepcopy and pickle of a tensor whose cache holds maps with everything the layers left on them: the copy
    makes its own and gives the same results after the original is gone."""
    import copy
    import pickle
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    from warpconvnet_amd.nn.functional.sparse_pool import sparse_max_pool
    rows = _surface(40_000, 13)
    x = normal_features(len(rows), 128, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 128, 256, seed=2, dtype=torch.float16).to(DEV)
    w_up = kaiming_weight(8, 128, 32, seed=3, dtype=torch.float16).to(DEV)

    def use(vox):
        pooled = sparse_max_pool(vox, 2)
        up = spatially_sparse_conv(pooled, w_up, 2, stride=2, transposed=True, output_spatially_sparse_tensor=vox)
        return (spatially_sparse_conv(vox, w, 3).feature_tensor, pooled.feature_tensor, up.feature_tensor)

    vox = Voxels(rows[:, 1:].contiguous(), x, offsets=torch.tensor([0, len(rows)]))
    want = use(vox)
    copies = [copy.deepcopy(vox), pickle.loads(pickle.dumps(vox))]
    del vox
    taken = [torch.full((1 << 24,), 0x7f, dtype=torch.uint8, device=DEV) for _ in range(16)]
    for other in copies:
        assert other.cache and all(km._group_start is None and km._made is None for km in other.cache.values())
        for _ in range(2):
            assert all(torch.equal(a, b) for a, b in zip(use(other), want))
    del taken


def test_a_coordinate_table_nobody_has_waited_for_is_its_stream_s_own():
    from warpconvnet_amd.geometry.coords.search.torch_discrete import _table_of
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import HashMethod
    c = _surface(3_000, 17)
    torch.cuda.synchronize()
    first = _table_of(c, HashMethod.CITY, c.device)
    assert _table_of(c, HashMethod.CITY, c.device) is first
    with torch.cuda.stream(torch.cuda.Stream()):
        own = _table_of(c, HashMethod.CITY, c.device)
        assert own is not first
        km = _map(c)  # waits
        assert own._checked
    assert _table_of(c, HashMethod.CITY, c.device) is own
    other = _map(c.clone())
    assert torch.equal(km.in_maps, other.in_maps) and torch.equal(km.out_maps, other.out_maps)


@pytest.mark.parametrize("kernel,stride", [(2, 2), (3, 1), (3, 2), (5, 1)])
@pytest.mark.parametrize("scene", ["cube", "sheet", "cloud", "one"])
def test_rows_form_of_a_builders_map_is_that_of_its_lists(kernel, stride, scene):
    """Groups of few pairs, of 384 and more (a chunk of a thin map) and of 1,024 and more (a chunk of a dense one), rows that end
    inside a group: a depthwise layer over the one-pass form against the form made from the lists alone, bit for bit."""
    from warpconvnet_amd.nn.functional.sparse_conv import native
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    rng = np.random.default_rng(kernel + stride)
    if scene == "cube":
        cells = np.stack(np.meshgrid(*[np.arange(23)] * 3, indexing="ij"), -1).reshape(-1, 3)
    elif scene == "sheet":
        cells = np.stack([rng.permutation(200 * 200)[:20_011] // 200, rng.permutation(200 * 200)[:20_011] % 200, np.zeros(20_011, int)], 1)
    elif scene == "cloud":
        at = rng.permutation(60 ** 3)[:9001]
        cells = np.stack([at // 3600, at // 60 % 60, at % 60], 1)
    else:
        cells = np.zeros((1, 3), int)
    cells = np.unique(cells, axis=0)
    rows = torch.as_tensor(np.concatenate([np.zeros((len(cells), 1), int), cells], 1).astype(np.int32), device=DEV)
    out = stride_coords(rows, (stride,) * 3)[0] if stride > 1 else rows
    km = generate_kernel_map(rows, out, (stride,) * 3, (kernel,) * 3)
    K, n, m = kernel ** 3, len(rows), len(out)
    x = torch.randn(n, 8, device=DEV, generator=torch.Generator(DEV).manual_seed(1))
    w = torch.randn(K, 8, device=DEV, generator=torch.Generator(DEV).manual_seed(2))
    got = native().depthwise_forward(x, w, km, m, torch.float32)
    km._rows_forms, km._from_builder = None, False
    want = native().depthwise_forward(x, w, km, m, torch.float32)
    assert torch.equal(got, want)
    ins, outs, offsets = km.in_maps.long(), km.out_maps.long(), km.offsets.tolist()
    sums = torch.zeros(m, 8, dtype=torch.float64, device=DEV)
    for k in range(K):
        at = slice(offsets[k], offsets[k + 1])
        sums.index_add_(0, outs[at], x[ins[at]].double() * w[k].double())
    assert float((got - sums).abs().max()) <= K * 2.0 ** -22 * 16  # K fp32 steps on sums of a few units
