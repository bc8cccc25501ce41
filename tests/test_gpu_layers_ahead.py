"""Layers that are launched before the map's offsets have reached the host: the same bits as over the kept
map, with every extra of the epilogue; lists that turn out too short, and calls that have to wait for the map."""
import numpy as np
import pytest
import torch

from helpers import kaiming_weight, normal_features

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _voxels(n, c_in, dtype, seed=0):
    from warpconvnet_amd.geometry.types.voxels import Voxels
    rng = np.random.default_rng(seed)
    side = int(np.ceil(np.sqrt(n / 0.5)))
    cells = rng.permutation(side * side)[:n]
    coords = np.stack([cells // side, cells % side, cells % 3 // 2], axis=1).astype(np.int32) - 7
    return Voxels(torch.as_tensor(coords, device=DEV), normal_features(n, c_in, seed=seed, dtype=dtype).to(DEV),
                  offsets=torch.tensor([0, n // 3, n]))


def _spied(monkeypatch):
    """What the layers that ran ahead of their maps have left: one entry per LayerAhead made.  The lists are sized as if no map had
    been made before."""
    from warpconvnet_amd.geometry.coords.search import torch_discrete
    from warpconvnet_amd.nn.functional import sparse_conv as f
    monkeypatch.setattr(torch_discrete, "_PAIRS_PER_ROW", {})
    made = []
    native = f.native()

    class Spy:
        def __getattr__(self, name):
            if name != "LayerAhead":
                return getattr(native, name)

            def make(*args):
                made.append(native.LayerAhead(*args))
                return made[-1]
            return make
    monkeypatch.setattr(f, "native", lambda: Spy())
    return made


@pytest.mark.parametrize("n", [1, 31, 33, 1800, 5000])
@pytest.mark.parametrize("dtype,c_in,c_out,kernel,stride", [
    (torch.float16, 32, 64, 3, 1), (torch.bfloat16, 64, 64, 3, 1), (torch.float32, 32, 32, 3, 1), (torch.bfloat16, 64, 128, 2, 2),
    (torch.float16, 16, 24, 5, 1), (torch.float16, 32, 32, 3, 2), (torch.bfloat16, 256, 256, 3, 1)])
@pytest.mark.parametrize("extras", [False, True])
def test_same_bits_as_over_the_kept_map(monkeypatch, n, dtype, c_in, c_out, kernel, stride, extras):
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    w = kaiming_weight(kernel ** 3, c_in, c_out, seed=2, dtype=dtype).to(DEV)
    vox = _voxels(n, c_in, dtype, seed=n)
    kw = {"stride": stride}
    if extras:
        kw.update(bias=normal_features(1, c_out, seed=3, dtype=dtype)[0].to(DEV), relu=True, keep_prepared_weight=True)
        if stride == 1:
            kw["residual"] = normal_features(n, c_out, seed=4, dtype=dtype).to(DEV)
    first = spatially_sparse_conv(vox, w, kernel, **kw).feature_tensor
    assert len(made) == 1 and made[0].out is not None
    again = spatially_sparse_conv(vox, w, kernel, **kw).feature_tensor
    assert all(a.out is None for a in made[1:])  # the map is there
    assert torch.equal(first, again)
    # new voxels in the same rows: the layer's own map, and the bits of the first
    assert torch.equal(first, spatially_sparse_conv(_voxels(n, c_in, dtype, seed=n), w, kernel, **kw).feature_tensor)


def test_lists_that_turn_out_too_short(monkeypatch):
    """27 pairs per voxel where ten are assumed: the layer that ran ahead has found no lists, and runs again."""
    from warpconvnet_amd.geometry.coords.search import torch_discrete
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    monkeypatch.setattr(torch_discrete, "_PAIRS_PER_ROW", {})
    cube = np.stack(np.meshgrid(*[np.arange(20)] * 3, indexing="ij"), axis=-1).reshape(-1, 3).astype(np.int32)
    n = len(cube)
    x = normal_features(n, 64, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 64, 64, seed=2, dtype=torch.float16).to(DEV)
    vox = Voxels(torch.as_tensor(cube, device=DEV), x, offsets=torch.tensor([0, n]))
    first = spatially_sparse_conv(vox, w, 3).feature_tensor
    assert len(made) == 1 and made[0].out is None
    km = next(iter(vox.cache.values()))
    assert km.in_maps.shape[0] == (20 * 3 - 2) ** 3
    assert torch.equal(first, spatially_sparse_conv(vox, w, 3).feature_tensor)
    # the next map of this size assumes what this one held
    vox = Voxels(torch.as_tensor(cube, device=DEV), x, offsets=torch.tensor([0, n]))
    assert torch.equal(first, spatially_sparse_conv(vox, w, 3).feature_tensor)
    assert made[-1].out is not None


def _kernel():
    from warpconvnet_amd._lib import lib
    return lib().wcn_conv_last_kernel().decode()


@pytest.mark.parametrize("n,dtype,c_in,c_out,kernel,stride,name", [
    (70_001, torch.float16, 32, 32, 3, 1, "group"), (240_000, torch.bfloat16, 16, 13, 3, 2, "group"), (140_000, torch.float16, 8, 8, 5, 1, "group"),
    (200_000, torch.float32, 16, 13, 3, 2, "group"), (60_007, torch.float32, 32, 16, 3, 1, "group"),
    (50_001, torch.float32, 32, 32, 3, 1, "pack"), (30_000, torch.float32, 128, 128, 3, 1, "pack"), (160_000, torch.float32, 40, 72, 2, 2, "pack"),
    (64_000, torch.float16, 64, 20, 3, 1, "pack"), (90_031, torch.bfloat16, 32, 60, 3, 1, "pack")])
@pytest.mark.parametrize("extras", [False, True])
def test_narrow_and_packed_kernels_give_the_same_bits(monkeypatch, n, dtype, c_in, c_out, kernel, stride, name, extras):
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    w = kaiming_weight(kernel ** 3, c_in, c_out, seed=2, dtype=dtype).to(DEV)
    kw = {"stride": stride}
    if extras:
        kw.update(bias=normal_features(1, c_out, seed=3, dtype=dtype)[0].to(DEV), relu=True, keep_prepared_weight=True)
        if stride == 1:
            kw["residual"] = normal_features(n, c_out, seed=4, dtype=dtype).to(DEV)
    vox = _voxels(n, c_in, dtype, seed=n)
    first = spatially_sparse_conv(vox, w, kernel, **kw).feature_tensor
    assert len(made) == 1 and made[0].out is not None
    assert _kernel().startswith(f"conv_fwd_{name}<"), _kernel()
    again = spatially_sparse_conv(vox, w, kernel, **kw).feature_tensor  # the pairs are known now
    assert made[1:] == [] or made[-1].out is None
    assert _kernel().startswith(f"conv_fwd_{name}<"), _kernel()
    assert torch.equal(first, again)


@pytest.mark.parametrize("dtype,c_in,c_out,name", [(torch.float16, 32, 32, "group"), (torch.float32, 32, 32, "pack")])
def test_narrow_and_packed_kernels_find_no_lists(monkeypatch, dtype, c_in, c_out, name):
    from warpconvnet_amd.geometry.coords.search import torch_discrete
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    monkeypatch.setattr(torch_discrete, "_PAIRS_PER_ROW", {})
    cube = np.stack(np.meshgrid(*[np.arange(40)] * 3, indexing="ij"), axis=-1).reshape(-1, 3).astype(np.int32)
    n = len(cube)
    x = normal_features(n, c_in, seed=1, dtype=dtype).to(DEV)
    w = kaiming_weight(27, c_in, c_out, seed=2, dtype=dtype).to(DEV)
    vox = Voxels(torch.as_tensor(cube, device=DEV), x, offsets=torch.tensor([0, n]))
    first = spatially_sparse_conv(vox, w, 3).feature_tensor
    assert len(made) == 1 and made[0].out is None
    assert _kernel().startswith(f"conv_fwd_{name}<"), _kernel()
    vox = Voxels(torch.as_tensor(cube, device=DEV), x, offsets=torch.tensor([0, n]))
    assert torch.equal(first, spatially_sparse_conv(vox, w, 3).feature_tensor)
    assert made[-1].out is not None


@pytest.mark.parametrize("dtype,num_offsets,c_in,c_out,rows,capacity,half", [
    (1, 27, 32, 64, 1000, 27_000, 1), (1, 27, 32, 32, 70_000, 10 ** 6, 0), (0, 27, 32, 32, 100_000, 10 ** 6, 0),
    (1, 27, 64, 64, 32_768, 10 ** 6, -1),  # a tile plan may be taken: the pairs decide
    (1, 27, 20, 32, 70_000, 10 ** 6, -1),  # rows of other than whole 16-byte vectors
    (2, 200, 128, 128, 5000, 10 ** 6, -1),  # slices of channels over workgroups
    (1, 27, 32, 32, 100_000_000, 1 << 30, -1)])  # more pairs than the kernels' offsets reach
def test_half_of_the_weight(dtype, num_offsets, c_in, c_out, rows, capacity, half):
    from warpconvnet_amd._lib import lib
    assert lib().wcn_conv_ahead_half(dtype, num_offsets, c_in, c_out, rows, rows, capacity) == half


@pytest.mark.parametrize("n,dtype,c_in,c_out,kernel,stride,ahead", [
    (900, torch.float16, 32, 64, 3, 1, True), (24_000, torch.float16, 32, 32, 3, 1, True), (12_000, torch.float16, 32, 64, 2, 2, True),
    (8000, torch.bfloat16, 64, 64, 3, 1, True), (5000, torch.float32, 16, 16, 3, 1, True), (9000, torch.float32, 32, 32, 3, 2, True),
    (4000, torch.bfloat16, 256, 256, 3, 1, False), (40_000, torch.float16, 64, 64, 3, 1, False), (500, torch.float16, 3, 16, 3, 1, False)])
@pytest.mark.parametrize("bias", [None, "own", "fp32", "per_row", "requires_grad"])
@pytest.mark.parametrize("master", [False, True])
def test_layers_with_gradients(monkeypatch, n, dtype, c_in, c_out, kernel, stride, ahead, bias, master):
    """Product and gradients ahead of the map are those over the kept map, bit for bit."""
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    vox = _voxels(n, c_in, dtype, seed=n)
    w = kaiming_weight(kernel ** 3, c_in, c_out, seed=2, dtype=torch.float32 if master else dtype).to(DEV)
    b = normal_features(1, c_out, seed=3, dtype=torch.float32)[0].to(DEV)
    if bias in ("own", "requires_grad"):
        b = b.to(dtype)

    def step(vox, times):
        x = vox.feature_tensor.detach().requires_grad_(True)
        weight, extra = w.clone().requires_grad_(True), None if bias is None else b.clone().requires_grad_(bias == "requires_grad")
        if bias == "per_row":
            extra = b[None]
        vox = vox.replace(batched_features=x)
        for _ in range(times):  # (the first call of several makes the map)
            out = spatially_sparse_conv(vox, weight, kernel, stride=stride, bias=extra).feature_tensor
        gy = normal_features(len(out), c_out, seed=7, dtype=dtype).to(DEV)
        wanted = [x, weight] + ([extra] if bias == "requires_grad" else [])
        return [out.detach()] + list(torch.autograd.grad(out, wanted, gy))

    first = step(vox, 1)
    assert len(made) == 1 and (made[0].out is not None) == (ahead and bias != "per_row")
    over_kept = step(_voxels(n, c_in, dtype, seed=n), 2)
    assert made[-1].out is None
    assert all(torch.equal(p, q) for p, q in zip(first, over_kept))


def test_lists_too_short_for_a_layer_with_gradients(monkeypatch):
    from warpconvnet_amd.geometry.coords.search import torch_discrete
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    cube = np.stack(np.meshgrid(*[np.arange(20)] * 3, indexing="ij"), axis=-1).reshape(-1, 3).astype(np.int32)
    n, got = len(cube), []
    x = normal_features(n, 32, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 32, 64, seed=2, dtype=torch.float32).to(DEV).requires_grad_(True)
    b = torch.linspace(-1, 1, 64, device=DEV)
    monkeypatch.setattr(torch_discrete, "_PAIRS_PER_ROW", {})
    for assumed in ("too few", "enough"):
        vox = Voxels(torch.as_tensor(cube, device=DEV), x, offsets=torch.tensor([0, n]))
        got.append(spatially_sparse_conv(vox, w, 3, bias=b).feature_tensor)
        assert (made[-1].out is None) == (assumed == "too few")
    assert torch.equal(*got)


@pytest.mark.parametrize("case", ["columns", "fp32_bias", "one_bias", "half_weight", "residual_type", "three_channels", "converted"])
def test_calls_that_wait_for_the_map(monkeypatch, case):
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    n, c_in, c_out, dtype = 900, 3 if case == "three_channels" else 32, 32, torch.float16
    vox = _voxels(n, c_in, dtype)
    w = kaiming_weight(27, c_in, c_out, seed=2, dtype=torch.bfloat16 if case == "half_weight" else dtype).to(DEV)
    kw = {}
    if case == "columns":
        wide = normal_features(n, 2 * c_in, seed=5, dtype=dtype).to(DEV)
        vox = vox.replace(batched_features=wide[:, ::2])
    elif case == "fp32_bias":
        kw["bias"] = torch.randn(c_out, device=DEV)
    elif case == "one_bias":
        kw["bias"] = torch.ones(1, device=DEV, dtype=dtype)
    elif case == "residual_type":
        kw["residual"] = torch.randn(n, c_out, device=DEV)
    elif case == "converted":
        kw["compute_dtype"] = torch.bfloat16
    first = spatially_sparse_conv(vox, w, 3, **kw).feature_tensor
    assert len(made) == 1 and made[0].out is None
    assert torch.equal(first, spatially_sparse_conv(vox, w, 3, **kw).feature_tensor)


def test_dilated_and_plain_layers_keep_their_own_estimates(monkeypatch):
    """Over voxels of even places a row has one pair, and nine with a dilation of two: neither layer makes the other's lists too short."""
    from warpconvnet_amd.geometry.types.voxels import Voxels
    from warpconvnet_amd.nn.functional.sparse_conv import spatially_sparse_conv
    made = _spied(monkeypatch)
    cells = np.stack(np.meshgrid(np.arange(200), np.arange(200), [0], indexing="ij"), axis=-1).reshape(-1, 3).astype(np.int32) * 2
    n = len(cells)
    x = normal_features(n, 32, seed=1, dtype=torch.float16).to(DEV)
    w = kaiming_weight(27, 32, 32, seed=2, dtype=torch.float16).to(DEV)
    for turn in range(3):
        for dilation, pairs in ((1, n), (2, (200 * 3 - 2) ** 2)):
            vox = Voxels(torch.as_tensor(cells, device=DEV), x, offsets=torch.tensor([0, n]))
            got = spatially_sparse_conv(vox, w, 3, kernel_dilation=dilation).feature_tensor
            assert next(iter(vox.cache.values())).in_maps.shape[0] == pairs
            if turn > 0:
                assert made[-1].out is not None, dilation
                assert torch.equal(got, spatially_sparse_conv(vox, w, 3, kernel_dilation=dilation).feature_tensor)
