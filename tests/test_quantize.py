"""sparse_quantize on the native path against numpy's sort, where its digits and words can go wrong."""
import numpy as np
import pytest

from torchsparse_amd import backend
from torchsparse_amd.utils.quantize import ravel_hash, sparse_quantize


def by_numpy(points, voxel):
    cells = np.floor(points / np.asarray(voxel)).astype(np.int32)
    _, index, inverse = np.unique(ravel_hash(cells), return_index=True, return_inverse=True)
    return cells[index], index, inverse


@pytest.mark.parametrize("n,extent,voxel,dtype", [
    (1, 1.0, (0.1,) * 3, np.float32), (2, 1e-3, (0.5,) * 3, np.float64),      # one voxel, no digit that varies
    (2047, 3.0, (0.05, 0.05, 4.0), np.float32), (4097, 40.0, (1.0,) * 3, np.float64),
    (70000, 60.0, (0.05,) * 3, np.float32),                                    # three digits and a bit
    (5000, 4e5, (1e-3,) * 3, np.float64),                                      # keys beyond 64 bits: numpy's way
    (3001, 1000, (7, 2, 1), np.int32), (3000, 1000, (3, 3, 3), np.int64)])
def test_native_voxels_are_numpys(n, extent, voxel, dtype):
    rng = np.random.default_rng(n)
    wide = (rng.uniform(-extent, extent, (n, 4))).astype(dtype)
    wide[::3] = wide[0]                                                        # many points in one voxel
    for points in (wide[:, :3], np.asfortranarray(wide[:, 1:]), wide[::-1, 2::-1]):
        want = by_numpy(points, voxel)
        got = sparse_quantize(points, voxel, return_index=True, return_inverse=True)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and a.shape == b.shape and np.array_equal(a, b)
        assert np.array_equal(sparse_quantize(points, voxel), want[0])
        assert np.array_equal(sparse_quantize(points, voxel, return_inverse=True)[1], want[2])


def test_what_the_native_path_leaves_to_numpy():
    points = np.array([[0.0, 1.0, 2.0], [np.nan, 0.0, 0.0]])
    assert backend.host_voxelize(points, (1.0,) * 3, True, True) is None
    assert backend.host_voxelize(points[:1] * 1e12, (1.0,) * 3, True, True) is None
    assert backend.host_voxelize(points[:0], (1.0,) * 3, True, True) is None
    assert backend.host_voxelize(points.astype(np.float16), (1.0,) * 3, True, True) is None
