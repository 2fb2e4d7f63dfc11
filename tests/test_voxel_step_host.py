"""The voxel step's quick geometry against the general functions, bit for bit
(host builds of the same code): points on and around faces, at the nudging
distance, at the edge of the volume; directions along axes, on either side of
the parallel limit and at random; grids of the largest coordinates and the
thinnest voxels it takes, and those it must leave to the general step."""

import numpy as np
import pytest

from ggems_amd.engine import host_voxel_exit

F = np.float32
TOL = F(5e-4)
N = 400_000


def _points(rng, lo, voxel, dims, n):
    lo, voxel, dims = np.asarray(lo, F), np.asarray(voxel, F), np.asarray(dims)
    face = (lo + (rng.integers(0, dims + 1, (n, 3)).astype(F) * voxel).astype(F)).astype(F)
    inside = (lo + rng.uniform(0, 1, (n, 3)) * dims * voxel).astype(F)
    off = rng.choice([0, 1, -1], (n, 3)).astype(F) * TOL
    p = (face + off).astype(F)
    ulps = rng.integers(-3, 4, (n, 3))
    p = np.where(ulps == 0, p, (p + ulps * np.spacing(np.abs(p) + F(1e-6))).astype(F))
    return np.where(rng.random((n, 3)) < 0.5, p, inside).astype(F)


def _directions(rng, n):
    d = rng.normal(size=(n, 3))
    small = rng.choice([0.0, 1.0, 9.9e-7, 1.0e-6, 1.01e-6, 3e-5, 1e-12], (n, 3)) * rng.choice([-1, 1], (n, 3))
    d = np.where(rng.random((n, 3)) < 0.3, np.where(np.abs(small) == 1.0, d, small), d)
    norm = np.linalg.norm(d, axis=1, keepdims=True)
    d = np.where(norm < 1e-3, [[1.0, 0.0, 0.0]], d / np.maximum(norm, 1e-30))
    return d.astype(F)


@pytest.mark.parametrize("lo,voxel,dims", [
    ((-50, -50, -50), (1, 1, 1), (100, 100, 100)),
    ((-204.8, -204.8, -102.4), (0.8, 0.8, 0.8), (512, 512, 256)),
    ((-153.75, -113.75, -96.25), (2.5, 2.5, 2.5), (123, 91, 77)),
    ((-0.02, -0.03, -0.025), (0.002, 0.002, 0.0025), (20, 30, 20)),   # the thinnest voxels
    ((-2048, -2000, 1900), (0.7, 3.1, 0.9), (800, 1290, 160)),        # the largest coordinates
    ((0, 0, 0), (0.3, 0.01, 40), (7, 5, 3)),
])
def test_quick_equals_general(lo, voxel, dims):
    rng = np.random.default_rng(7)
    p, d = _points(rng, lo, voxel, dims, N), _directions(rng, N)
    general, quick, took = host_voxel_exit(p, d, lo, voxel, dims)
    assert took
    assert np.count_nonzero(general[:, 3]) > N // 3
    assert np.array_equal(general.view(np.uint32), quick.view(np.uint32))


@pytest.mark.parametrize("lo,voxel,dims", [
    ((-1, -1, -1), (0.0019, 1, 1), (1000, 2, 2)),       # thinner than 4 tolerances
    ((-2049, 0, 0), (1, 1, 1), (5, 5, 5)),              # too far out on one side
    ((0, 0, 0), (1, 1, 1), (5, 5, 2049)),               # and on the other
    ((0, 0, np.nan), (1, 1, 1), (5, 5, 5)),
])
def test_other_grids_take_the_general_step(lo, voxel, dims):
    assert not host_voxel_exit(np.zeros((1, 3)), [[1, 0, 0]], lo, voxel, dims)[2]
