"""The ray tracer's split of a ray over threads and of a panel over tiles,
against Siddon path lengths in FP64: panels that end inside a tile, volumes of
fewer voxels than a ray has parts, rays along an axis, an axis the walk
leaves early, a turned volume, and as many materials as it takes."""

import numpy as np
import pytest

import drr as R
import plain_scene as S

pytestmark = pytest.mark.gpu

TURNED = np.array([[0.8, -0.6, 0, 3.0], [0.6, 0.8, 0, -2.0], [0, 0, 1, 1.0], [0, 0, 0, 1]], np.float64)


@pytest.mark.parametrize("shape,voxel,panel,pixel,n_mat,matrix", [
    ((1, 1, 1), (40.0, 30.0, 20.0), (9, 5), 12.0, 3, np.eye(4)),       # one voxel
    ((3, 2, 5), (7.0, 9.0, 11.0), (8, 4), 8.0, 4, np.eye(4)),          # fewer voxels than parts
    ((33, 41, 57), (1.1, 0.9, 1.3), (17, 33), 5.0, 6, TURNED),         # odd sides, remainders of tiles
    ((4, 5, 130), (1.0, 1.0, 1.0), (1, 1), 1.0, 5, np.eye(4)),         # one ray, along x between voxels
    ((64, 64, 64), (2.0, 2.0, 2.0), (24, 31), 9.0, 32, TURNED),        # the most materials; rays past the volume
])
def test_parts_and_tiles_match_siddon(shape, voxel, panel, pixel, n_mat, matrix):
    rng = np.random.default_rng(sum(shape))
    labels = rng.integers(0, n_mat - 1, shape).astype(np.uint8)
    eng = S.engine(n_mat)
    S.add_voxels(eng, labels, voxel, matrix)
    k = S.add_panel(eng, *panel, pixel, n_mat - 1)
    S.add_source(eng)
    got = eng.drr(k)
    eng.close()
    t = S.tables(n_mat)
    b = R.left_bin(t["energy_bins"], np.float32(0.06))
    mu = t["cross_sections"].astype(np.float64).sum(0)[:, b]
    nz, ny, nx = shape
    half = np.array([nx, ny, nz]) * np.asarray(voxel) / 2
    inv = np.linalg.inv(matrix)
    src = (inv @ [-600.0, 0, 0, 1])[:3]
    want = np.ones_like(got, np.float64)
    for iy in range(panel[1]):
        for ix in range(panel[0]):
            at = [400.0, (iy + 0.5 - panel[1] / 2) * pixel, -(ix + 0.5 - panel[0] / 2) * pixel, 1]
            path = R.siddon_lengths(src, (inv @ at)[:3], -half, half, voxel, (nx, ny, nz))
            want[iy, ix] = np.exp(-sum(mu[labels.reshape(-1)[v]] * l for v, l in path))
    # end points in FP32: about 1e-4 mm of path at up to 0.1 / mm
    assert np.abs(got - want).max() < 2e-5
    assert got.shape == (panel[1], panel[0])
