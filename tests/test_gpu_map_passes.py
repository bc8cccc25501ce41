"""The map passes where their lists are full or nearly empty: every offset of every row hits (a solid
cube), rows that end inside a group, a workgroup or a stretch of workgroups, and maps of more offsets
than one workgroup of the emit pass takes for eight groups.  Bit-exact against the CPU oracle."""
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
