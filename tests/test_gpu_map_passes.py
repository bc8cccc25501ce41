"""The map passes where their lists are full or nearly empty: every offset of every row hits (a solid
cube), rows that end inside a group, a workgroup or a stretch of workgroups, and maps of more offsets
than one workgroup of the emit pass takes for eight groups.  Bit-exact against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cube(edge):
    g = np.stack(np.meshgrid(*[np.arange(edge)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return np.concatenate([np.zeros((len(g), 1), np.int64), g - 3], axis=1).astype(np.int32)


@pytest.mark.parametrize("ksize,stride", [((3, 3, 3), (1, 1, 1)), ((5, 5, 5), (1, 1, 1)), ((2, 2, 2), (2, 2, 2)),
                                          ((3, 3, 3), (2, 2, 2)), ((4, 3, 2), (1, 1, 1)), ((7, 7, 7), (1, 1, 1))],
                         ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 256, 257, 513, 2049, 4913])
def test_solid_cubes_and_ragged_ends(oracle, ksize, stride, rows):
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    rng = np.random.default_rng(rows)
    cube = _cube(17)
    rng.shuffle(cube)
    keys = cube if ksize != (7, 7, 7) else cube[:2500]
    if stride == (1, 1, 1) and rows <= len(keys):
        out = keys[:rows]  # any rows may be asked for, not only the keys
    else:
        out = np.unique(np.concatenate([keys[:, :1], keys[:, 1:] // np.asarray(stride)], axis=1), axis=0)[:rows]
    out = np.ascontiguousarray(out, dtype=np.int32)
    want = oracle.kernel_map(keys, out, ksize, stride)
    got = generate_kernel_map(torch.as_tensor(keys, device=DEV), torch.as_tensor(out, device=DEV), stride, ksize)
    assert np.array_equal(got.offsets.numpy().astype(np.int64), want[2])
    assert np.array_equal(got.in_maps.cpu().numpy(), want[0])
    assert np.array_equal(got.out_maps.cpu().numpy(), want[1])


@pytest.mark.parametrize("sizes", [(1,), (64, 0, 1), (255, 257), (16384,), (16385,), (4096, 0, 0, 4097, 9000), tuple([7] * 64)],
                         ids=lambda v: f"{len(v)}_{sum(v)}")
def test_rows_and_table_by_the_same_launches(sizes):
    """The batch column, and the table over the rows, for few keys and many, empty items and the most items that
    travel with a launch; a second tensor of the same rows takes the launches of their own."""
    from warpconvnet_amd.geometry.coords.integer import IntCoords
    from warpconvnet_amd.geometry.coords.search.torch_discrete import rows_with_table
    n = sum(sizes)
    rng = np.random.default_rng(n)
    xyz = np.unique(rng.integers(-60, 60, size=(3 * n + 100, 3)), axis=0)
    xyz = torch.as_tensor(rng.permutation(xyz)[:n].astype(np.int32), device=DEV)
    offsets = torch.as_tensor(np.concatenate([[0], np.cumsum(sizes)]))
    coords, plain = IntCoords(xyz, offsets), IntCoords(xyz, offsets)
    rows = rows_with_table(coords)
    assert torch.equal(rows, plain.batch_indexed_coordinates) and rows_with_table(coords) is rows
    table = rows._wcn_table[1]
    want = torch.arange(n, dtype=torch.int32, device=DEV)
    assert torch.equal(table.search(rows), want) and torch.equal(plain.hashmap.search(rows), want)
    absent = rows + torch.tensor([0, 500, 0, 0], dtype=torch.int32, device=DEV)
    assert (table.search(absent) == -1).all()


@pytest.mark.parametrize("stride", [(2, 2, 2), (4, 1, 2)], ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("sizes", [(1,), (256,), (300, 0, 0, 513), (64, 192, 1, 0), (9000, 3), (1_100_000, 5)],
                         ids=lambda v: f"{len(v)}_{sum(v)}")
def test_strided_rows_and_their_batch_offsets(sizes, stride):
    """Items that end inside a group, a workgroup's rows and beyond the parts that are added up without a scan."""
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    n = sum(sizes)
    rng = np.random.default_rng(n)
    edge = max(3, int(round((2.5 * n) ** (1 / 3))))
    cells = rng.permutation(edge ** 3)[:n] if max(sizes) <= edge ** 3 else None
    assert cells is not None
    xyz = np.stack([cells // edge ** 2, cells // edge % edge, cells % edge], axis=1).astype(np.int32) - 7
    item = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    rows = np.concatenate([item[:, None], xyz], axis=1)
    coarse = np.concatenate([item[:, None], xyz // np.asarray(stride)], axis=1)
    _, first = np.unique(coarse, axis=0, return_index=True)
    want = coarse[np.sort(first)]
    got, offsets = stride_coords(torch.as_tensor(rows, device=DEV), stride, batch_sorted=True)
    assert np.array_equal(got.cpu().numpy(), want)
    counts = np.bincount(want[:, 0], minlength=len(sizes))[: int(want[-1, 0]) + 1]
    assert offsets.tolist() == np.concatenate([[0], np.cumsum(counts)]).tolist()


@pytest.mark.parametrize("bounds", [False, True], ids=["count", "bounds"])
@pytest.mark.parametrize("left", ["count", "dilated", "self", "cells"])
def test_a_result_that_nobody_read_is_not_the_next_one(left, bounds):
    """A map (or strided rows) whose result is not read, as after an error in between, then strided rows of another kind in
    the same workspace: their number is theirs."""
    from warpconvnet_amd._lib import check, int3, lib, ptr, stream_ptr, workspace
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    dev = torch.device(DEV)
    rows = torch.as_tensor(_cube(9), device=DEV)
    n, L, s = len(rows), lib(), stream_ptr(dev)
    table, _, slots = TorchHashTable.from_keys(rows)._raw()
    out = torch.empty(n, 4, dtype=torch.int32, device=DEV)
    first = torch.empty(n, dtype=torch.int32, device=DEV)
    ws = workspace(max(L.wcn_kmap_workspace_bytes(n, 27), L.wcn_stride_unique_workspace_bytes(n, slots),
                       L.wcn_stride_unique_cells_workspace_bytes(n)), dev)
    k3, one, two, three = (int3((v,) * 3) for v in (3, 1, 2, 3))
    if left == "count":
        check(L.wcn_kmap_count(ptr(table), n, slots, ptr(rows), n, k3, one, ptr(ws), s), "count")
    elif left == "dilated":
        check(L.wcn_kmap_count_dilated(ptr(table), n, slots, ptr(rows), n, k3, one, two, one, ptr(ws), s), "count")
    elif left == "self":
        check(L.wcn_kmap_count_self(ptr(table), n, slots, k3, ptr(ws), s), "count")
    else:
        check(L.wcn_stride_unique_cells(ptr(table), n, slots, ptr(rows), two, ptr(ws), ptr(out), ptr(first), s), "cells")
    torch.cuda.synchronize()
    check(L.wcn_stride_unique(ptr(rows), n, three, ptr(ws), slots, ptr(out), ptr(first), s), "stride")
    got, marks = ctypes.c_int64(-1), (ctypes.c_int64 * 1025)()
    if bounds:
        check(L.wcn_stride_unique_read_bounds(ptr(ws), n, slots, ctypes.byref(got), marks, s), "read")
        assert marks[0] == 0 and marks[1] == 27 and marks[1024] == 27
    else:
        check(L.wcn_stride_unique_read_count(ptr(ws), n, slots, ctypes.byref(got), s), "read")
    assert got.value == 27  # -3 .. 5 in cells of three
    assert torch.equal(out[:27].unique(dim=0), torch.unique(torch.cat([rows[:, :1], rows[:, 1:] // 3], dim=1), dim=0))


@pytest.mark.parametrize("then", ["map", "cells"])
def test_a_result_on_its_way_does_not_reach_the_next_one(oracle, then):
    """A map's result that nobody reads, behind a long queue of another stream; results asked for meanwhile come from the
    device, and later ones from the mailbox again."""
    from warpconvnet_amd._lib import check, int3, lib, ptr, stream_ptr, workspace
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    dev, cube = torch.device(DEV), _cube(9)
    rows = torch.as_tensor(cube, device=DEV)
    n, L = len(rows), lib()
    table, _, slots = TorchHashTable.from_keys(rows)._raw()
    ws = workspace(L.wcn_kmap_workspace_bytes(n, 125), dev)
    want = oracle.kernel_map(cube, cube, (3, 3, 3))
    a = torch.randn(8192, 8192, device=DEV)
    (a @ a).sum().item()
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        for _ in range(20):
            a = a @ a * 1e-4
        check(L.wcn_kmap_count(ptr(table), n, slots, ptr(rows), n, int3((5, 5, 5)), int3((1, 1, 1)), ptr(ws), stream_ptr(dev)), "count")
        done = torch.cuda.Event()
        done.record()
    for turn in range(3):
        if then == "map":
            got = generate_kernel_map(rows.clone(), rows, (1, 1, 1), (3, 3, 3))
            assert np.array_equal(got.offsets.numpy().astype(np.int64), want[2])
            assert np.array_equal(got.in_maps.cpu().numpy(), want[0]) and np.array_equal(got.out_maps.cpu().numpy(), want[1])
        else:
            coarse, offsets = stride_coords(rows.clone(), (2, 2, 2), batch_sorted=True)
            assert offsets.tolist() == [0, 125] and len(coarse.unique(dim=0)) == 125
        if turn == 0:
            assert not done.query()  # the queue was longer than this
        if turn == 1:
            torch.cuda.synchronize()


@pytest.mark.parametrize("kernel,stride,dilation", [(3, 1, 1), (3, 2, 1), (2, 2, 1), (2, 1, 1), (5, 1, 1), (3, 1, 2), ((1, 3, 2), 1, 1)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 256, 257, 511, 513, 2049, 30_011, 131_073, (1 << 18), (1 << 18) + 1, 700_003])
def test_one_call_leaves_what_two_leave(n, kernel, stride, dilation):
    """wcn_kmap_count_fill against wcn_kmap_count and wcn_kmap_fill: offsets, status, group starts and lists, also where the lists
    are too short and a fill follows."""
    import math

    from warpconvnet_amd._lib import check, int3, lib, ptr, stream_ptr, workspace
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    dev, L = torch.device(DEV), lib()
    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n / 0.6)))
    cells = rng.permutation(side * side)[:n]
    rows = torch.as_tensor(np.stack([cells % 2, cells // side - 40, cells % side, cells % 5 // 3], axis=1).astype(np.int32), device=DEV)
    table, _, slots = TorchHashTable.from_keys(rows)._raw()
    ks = (kernel,) * 3 if isinstance(kernel, int) else kernel
    K, k3, st, dil, centre = math.prod(ks), int3(ks), int3((stride,) * 3), int3((dilation,) * 3), int3(tuple(k // 2 for k in ks))
    s, groups = stream_ptr(dev), (n + 63) // 64

    def run(fill):
        ws = workspace(L.wcn_kmap_workspace_bytes(n, K), dev)
        ws.fill_(0xEE)
        ins, outs = (torch.full((K * n + 64,), -7, dtype=torch.int32, device=DEV) for _ in range(2))
        fill(ws, ins, outs)
        offsets = (ctypes.c_int64 * (K + 1))()
        check(L.wcn_kmap_read_result(ptr(ws), n, K, offsets, s), "read")
        begin = L.wcn_kmap_group_start(ptr(ws), n, K) - ws.data_ptr()
        starts = ws[begin:begin + 4 * K * (groups + 1)].clone()
        return list(offsets), L.wcn_kmap_last_table_flags(), starts, ins, outs, ws[:8 * (K + 3)].clone(), ws

    def two(ws, ins, outs):
        if dilation == 1:
            check(L.wcn_kmap_count(ptr(table), n, slots, ptr(rows), n, k3, st, ptr(ws), s), "count")
        else:
            check(L.wcn_kmap_count_dilated(ptr(table), n, slots, ptr(rows), n, k3, st, dil, centre, ptr(ws), s), "count")
        check(L.wcn_kmap_fill(ptr(table), n, slots, ptr(rows), n, k3, st, ptr(ws), K * n, ptr(ins), ptr(outs), s), "fill")

    def one(capacity):
        def fill(ws, ins, outs):
            extra = (dil, centre) if dilation != 1 else (None, None)
            check(L.wcn_kmap_count_fill(ptr(table), n, slots, ptr(rows), n, k3, st, *extra, ptr(ws), capacity, ptr(ins), ptr(outs), s),
                  "count_fill")
        return fill

    want = run(two)
    pairs = want[0][K]
    got = run(one(K * n))
    assert got[0] == want[0] and got[1] == want[1]
    assert all(torch.equal(a, b) for a, b in zip(got[2:6], want[2:6]))
    if pairs:
        exact = run(one(pairs))
        assert all(torch.equal(a, b) for a, b in zip(exact[2:6], want[2:6]))
        short = run(one(pairs - 1))
        assert short[0] == want[0] and torch.equal(short[2], want[2]) and bool((short[3] == -7).all()) and bool((short[4] == -7).all())
        check(L.wcn_kmap_fill(ptr(table), n, slots, ptr(rows), n, k3, st, ptr(short[6]), K * n, ptr(short[3]), ptr(short[4]), s), "fill")
        assert torch.equal(short[3], want[3]) and torch.equal(short[4], want[4])


@pytest.mark.parametrize("kernel,stride,dilation", [(3, 1, 1), (2, 2, 1), (5, 1, 1), (3, 1, 2), ((1, 3, 2), 1, 1)])
@pytest.mark.parametrize("n", [1, 65, 30_011, (1 << 18) + 1])
@pytest.mark.parametrize("short", [False, True])
def test_maps_whose_head_lies_apart(monkeypatch, n, kernel, stride, dilation, short):
    """A workspace in two pieces (that of maps over a size) against one in one piece: lists, offsets and group starts, also where the
    lists were taken for shorter than they are and are emitted again."""
    from warpconvnet_amd.geometry.coords.search import torch_discrete
    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n / 0.6)))
    cells = rng.permutation(side * side)[:n]
    rows = torch.as_tensor(np.stack([cells * 0, cells // side, cells % side, cells % 5 // 3], axis=1).astype(np.int32), device=DEV)
    ks = (kernel,) * 3 if isinstance(kernel, int) else kernel

    def build(keep):
        monkeypatch.setattr(torch_discrete, "_KEEP_WORKSPACE_BYTES", keep)
        monkeypatch.setattr(torch_discrete, "_PAIRS_PER_ROW", torch_discrete._PAIRS_PER_ROW.__class__())
        if short:
            octave = (tuple(ks), (stride,) * 3, -n.bit_length())
            torch_discrete._PAIRS_PER_ROW[octave] = 0.01
        args = dict(kernel_dilation=(dilation,) * 3, method="offset") if dilation != 1 else {}
        km = torch_discrete.generate_kernel_map(rows, rows, (stride,) * 3, ks, **args)
        torch.cuda.synchronize()
        return km

    want, got = build(1 << 40), build(0)
    assert torch.equal(got.in_maps, want.in_maps) and torch.equal(got.out_maps, want.out_maps)
    assert torch.equal(got.offsets, want.offsets) and torch.equal(got._device_offsets, want._device_offsets)
    starts = 4 * len(want) * ((n + 63) // 64 + 1)
    assert torch.equal(got._group_start[0][:starts], want._group_start[0][:starts])


@pytest.mark.parametrize("since", ["cells", "count", "stride", "release"])
def test_the_event_of_a_map_is_not_that_of_a_later_call(since):
    """wcn_kmap_take_event is asked after the same thread has made something else: the event is behind that by then, maybe on
    another stream, and none is handed out."""
    from warpconvnet_amd._lib import check, int3, lib, ptr, stream_ptr, workspace
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    dev, L = torch.device(DEV), lib()
    rows = torch.as_tensor(_cube(9), device=DEV)
    n, s = len(rows), stream_ptr(dev)
    table, _, slots = TorchHashTable.from_keys(rows)._raw()
    k3, one, two, three = (int3((v,) * 3) for v in (3, 1, 2, 3))
    ws, other = (workspace(max(L.wcn_kmap_workspace_bytes(n, 27), L.wcn_stride_unique_workspace_bytes(n, slots),
                               L.wcn_stride_unique_cells_workspace_bytes(n)), dev) for _ in range(2))
    ins, outs = (torch.empty(27 * n, dtype=torch.int32, device=DEV) for _ in range(2))
    out, first = torch.empty(n, 4, dtype=torch.int32, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV)
    offsets, got = (ctypes.c_int64 * 28)(), ctypes.c_int64(0)
    check(L.wcn_kmap_count_fill(ptr(table), n, slots, ptr(rows), n, k3, one, None, None, ptr(ws), 27 * n, ptr(ins), ptr(outs), s), "fill")
    check(L.wcn_kmap_read_result(ptr(ws), n, 27, offsets, s), "read")
    if since == "cells":
        check(L.wcn_stride_unique_cells(ptr(table), n, slots, ptr(rows), two, ptr(other), ptr(out), ptr(first), s), "cells")
        check(L.wcn_stride_unique_read_count(ptr(other), n, slots, ctypes.byref(got), s), "read")
    elif since == "count":
        check(L.wcn_kmap_count(ptr(table), n, slots, ptr(rows), n, k3, one, ptr(other), s), "count")
        check(L.wcn_kmap_read_result(ptr(other), n, 27, offsets, s), "read")
    elif since == "stride":
        check(L.wcn_stride_unique(ptr(rows), n, three, ptr(other), slots, ptr(out), ptr(first), s), "stride")
        check(L.wcn_stride_unique_read_count(ptr(other), n, slots, ctypes.byref(got), s), "read")
    else:
        torch.cuda.synchronize()
        check(L.wcn_thread_release(), "release")
    device = ctypes.c_int32(-1)
    assert not L.wcn_kmap_take_event(ptr(ws), ctypes.byref(device)) and device.value == -1


def test_the_events_of_maps_are_handed_back():
    """As many events as maps are alive; what is handed back, on whichever thread, is used again; a bounded number is kept."""
    import threading

    from warpconvnet_amd._lib import check, int3, lib, ptr, stream_ptr, workspace
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    dev, L = torch.device(DEV), lib()
    rows = torch.as_tensor(_cube(9), device=DEV)
    n, s = len(rows), stream_ptr(dev)
    table, _, slots = TorchHashTable.from_keys(rows)._raw()
    k3, one = int3((3, 3, 3)), int3((1, 1, 1))
    ws = workspace(L.wcn_kmap_workspace_bytes(n, 27), dev)
    ins, outs = (torch.empty(27 * n, dtype=torch.int32, device=DEV) for _ in range(2))
    offsets, device = (ctypes.c_int64 * 28)(), ctypes.c_int32(-1)

    def event():
        check(L.wcn_kmap_count_fill(ptr(table), n, slots, ptr(rows), n, k3, one, None, None, ptr(ws), 27 * n, ptr(ins), ptr(outs), s),
              "fill")
        check(L.wcn_kmap_read_result(ptr(ws), n, 27, offsets, s), "read")
        taken = L.wcn_kmap_take_event(ptr(ws), ctypes.byref(device))
        assert taken and device.value == dev.index and not L.wcn_kmap_take_event(ptr(ws), ctypes.byref(device))
        return taken

    torch.cuda.synchronize()
    check(L.wcn_thread_release(), "release")  # none are kept
    alive = [event() for _ in range(100)]
    assert len(set(alive)) == 100
    other = threading.Thread(target=lambda: [L.wcn_kmap_return_event(e, dev.index) for e in alive])
    other.start()
    other.join()
    again = [event() for _ in range(64)]
    assert set(again) == set(alive[:64])  # the other 36 were destroyed
    for e in again:
        L.wcn_kmap_return_event(e, dev.index)
    torch.cuda.synchronize()
    check(L.wcn_thread_release(), "release")
