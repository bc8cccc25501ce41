"""Slots of the coordinate table whose tag is the block coordinate (boxes of up to 31 bits of block
coordinates) and slots whose tag is a hash of it (wider boxes): look-ups, kernel maps and strided
coordinates against the oracle, bit-exact, either side of the line."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.int32, device=DEV)


def _clusters(n, field_bits, seed):
    """Voxels in clumps over a box whose block coordinates take field_bits[d] bits per column, its far
    corners among them."""
    rng = np.random.default_rng(seed)
    span = np.array([(1 << field_bits[0]) - 1] + [(4 << b) - 1 for b in field_bits[1:]], dtype=np.int64)
    centres = np.stack([rng.integers(0, s + 1, size=40) for s in span], axis=1)
    centres[0], centres[1] = 0, span
    rows = centres[rng.integers(0, 40, size=2 * n)]
    rows[:, 1:] += rng.integers(-9, 10, size=(2 * n, 3))
    rows = np.concatenate([np.clip(rows, 0, span), [span * 0, span]])
    rows[:, 1:] -= (span[1:] // 8) * 4  # the box's corner is a multiple of four below zero
    rows = np.unique(rows, axis=0)
    rng.shuffle(rows)
    # batch items one after the other
    return rows[np.argsort(rows[:, 0], kind="stable")].astype(np.int32)


# bits of (batch, x, y, z): 6 to 63 in all; 31 is the last with the block coordinate as the tag
FIELDS = [(0, 2, 2, 2), (1, 10, 10, 9), (1, 10, 10, 10), (2, 10, 10, 10), (0, 11, 0, 20), (0, 0, 0, 29), (3, 20, 20, 20)]


@pytest.mark.parametrize("n", [900, 30_000])
@pytest.mark.parametrize("fields", FIELDS, ids=["_".join(map(str, f)) for f in FIELDS])
def test_look_ups_and_maps_either_side_of_the_tags_width(oracle, fields, n):
    from warpconvnet_amd.geometry.coords.ops.stride import stride_coords
    from warpconvnet_amd.geometry.coords.search.torch_discrete import generate_kernel_map
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    rows = _clusters(n, fields, seed=sum(fields))
    table = TorchHashTable.from_keys(_dev(rows), device=DEV)
    assert np.array_equal(table.search(_dev(rows)).cpu().numpy(), np.arange(len(rows), dtype=np.int32))
    near = rows + np.array([0, 1, 0, -1], np.int32)
    assert np.array_equal(table.search(_dev(near)).cpu().numpy(), oracle.HashTable(rows).search(near))
    for ksize in ((3, 3, 3), (5, 5, 5), (3, 1, 2)):
        km = generate_kernel_map(_dev(rows), _dev(rows), (1, 1, 1), ksize)
        ref_in, ref_out, ref_off, _ = oracle.kernel_map(rows, rows, ksize, (1, 1, 1))
        assert np.array_equal(km.offsets.numpy().astype(np.int64), ref_off)
        assert np.array_equal(km.in_maps.cpu().numpy(), ref_in)
        assert np.array_equal(km.out_maps.cpu().numpy(), ref_out)
    for stride in ((2, 2, 2), (3, 2, 1)):
        coarse, _ = stride_coords(_dev(rows), stride)
        cells = np.floor_divide(rows, np.array([1, *stride], np.int32))  # (the oracle divides in fp32, as the reference does)
        first = np.sort(np.unique(cells, axis=0, return_index=True)[1])
        assert np.array_equal(coarse.cpu().numpy(), cells[first])


@pytest.mark.parametrize("step", [4, 8, 64])
@pytest.mark.parametrize("n", [3_000, 40_000])
def test_blocks_at_the_same_place_of_their_cells(n, step):
    """Voxels at multiples of a block, of a cell of eight blocks and of more: one place of a line would
    hold them all if the cell's hash did not turn it."""
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    side = int(np.ceil(n ** (1 / 3)))
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)[:n] * step - 5 * step
    rows = np.concatenate([np.zeros((n, 1)), grid], axis=1).astype(np.int32)
    np.random.default_rng(step).shuffle(rows)
    table = TorchHashTable.from_keys(_dev(rows), device=DEV)
    assert np.array_equal(table.search(_dev(rows)).cpu().numpy(), np.arange(n, dtype=np.int32))
    assert (table.search(_dev(rows + np.array([0, 1, 0, 0], np.int32))).cpu().numpy() == -1).all()


# (one workgroup of the sort and more, 256 of them and more keys in each)
@pytest.mark.parametrize("n", [16_385, 131_073, 262_143, 262_145, 300_000])
@pytest.mark.parametrize("repeats", [False, True])
def test_tables_of_several_parts(n, repeats):
    from warpconvnet_amd.geometry.coords.search.torch_hashmap import TorchHashTable
    rng = np.random.default_rng(n)
    cells = rng.choice(4 * 90 ** 3, n, replace=repeats)
    rows = np.stack([cells // 90 ** 3, cells // 8100 % 90 - 31, cells // 90 % 90, cells % 90 - 60], axis=1).astype(np.int32)
    _, first, back = np.unique(cells, return_index=True, return_inverse=True)
    table = TorchHashTable.from_keys(_dev(rows), device=DEV)
    assert np.array_equal(table.search(_dev(rows)).cpu().numpy(), first[back])


@pytest.mark.parametrize("n,slots", [(16_385, 1 << 16), (262_144, 1 << 20), (262_145, 1 << 20), (20_000, 1 << 24), (70_001, 1 << 22),
                                     (1 << 20, 1 << 21), ((1 << 20) + 1, 1 << 22), (1_300_007, 1 << 24)])
@pytest.mark.parametrize("items", [False, True], ids=["rows", "items"])
def test_parts_that_stay_in_registers_and_parts_that_do_not(n, slots, items):
    """Up to 4,096 keys a part and more of them (read twice), up to 4,096 bins and more (not through LDS), rows given and made of
    three columns and offsets; some keys twice, all of one corner in one bin."""
    import ctypes

    from warpconvnet_amd._lib import check, lib, ptr, stream_ptr
    rng = np.random.default_rng(n)
    cells = np.sort(rng.integers(0, 3, n)) * 10 ** 7 + rng.integers(0, 128 ** 3, n)
    cells[: min(n // 4, 5000)] = np.arange(min(n // 4, 5000)) % 4096  # (16 x 16 x 16 voxels: one bin)
    cells = np.sort(cells)
    at = cells % 10 ** 7
    rows = np.stack([cells // 10 ** 7, at % 16 + at // 4096 % 8 * 16 - 31, at // 16 % 16 + at // 32768 % 8 * 16,
                     at // 256 % 16 + at // 262144 * 16 - 60], axis=1).astype(np.int32)
    order = np.argsort(rows[:, 0], kind="stable")
    rows = rows[order]
    for b in range(3):  # no order inside an item
        mine = np.flatnonzero(rows[:, 0] == b)
        rows[mine] = rows[rng.permutation(mine)]
    key = rows.astype(np.int64) @ np.array([10 ** 9, 10 ** 6, 10 ** 3, 1])
    _, first, back = np.unique(key, return_index=True, return_inverse=True)
    L, s = lib(), stream_ptr(torch.device(DEV))
    table = torch.empty(L.wcn_table_bytes(n, slots), dtype=torch.uint8, device=DEV)
    if items:
        bounds = (ctypes.c_int64 * 4)(0, *np.cumsum(np.bincount(rows[:, 0], minlength=3)).tolist())
        made = torch.empty(n, 4, dtype=torch.int32, device=DEV)
        columns = _dev(rows[:, 1:])
        check(L.wcn_table_build_items(ptr(columns), n, bounds, 3, ptr(made), ptr(table), slots, s), "build")
        assert torch.equal(made, _dev(rows))
    else:
        made = _dev(rows)
        check(L.wcn_table_build(ptr(made), n, ptr(table), slots, s), "build")
    found = torch.empty(n, dtype=torch.int32, device=DEV)
    check(L.wcn_table_query(ptr(table), n, slots, ptr(made), n, ptr(found), s), "query")
    assert np.array_equal(found.cpu().numpy(), first[back])
