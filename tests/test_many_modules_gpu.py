"""Photons that leave a phantom look for their next solid at once with few
solids and in the next pass with many: the histories are the same."""

import numpy as np
import pytest

import plain_scene

pytestmark = pytest.mark.gpu


def _engine(aside, tau, phantoms):
    eng = plain_scene.engine(3)
    z, y, x = np.mgrid[-20:20, -20:20, -20:20]
    labels = (x * x + y * y < 9 ** 2).astype(np.uint8)
    for k in range(phantoms):
        m = np.eye(4)
        m[0, 3] = 90.0 * (k - 0.5 * (phantoms - 1))
        plain_scene.add_voxels(eng, labels, (2.0,) * 3, m)
    eng.panels = []
    for j in range(2):
        m = plain_scene.PANEL_AT.copy()
        m[1, 3] = (j - 0.5) * 48.0
        eng.panels.append(plain_scene.add_panel(eng, 24, 24, 2.0, 2, m))
    for j in range(aside):  # behind the source, and so far that no photon meets them
        m = np.eye(4, dtype=np.float32)
        m[0, 3], m[1, 3] = -5e5, 1e3 * j
        plain_scene.add_panel(eng, 4, 4, 1e-2, 2, m)
    plain_scene.add_source(eng, 0.1)
    eng.set_sampling("tau" if tau else "reference")
    return eng


@pytest.mark.parametrize("tau", [False, True])
@pytest.mark.parametrize("phantoms", [1, 2, 3])
def test_solids_out_of_reach_do_not_change_histories(phantoms, tau):
    few, many = _engine(0, tau, phantoms), _engine(40, tau, phantoms)
    for n in (1, 900, 500_000):
        got = []
        for eng in (few, many):
            eng.reset_tallies()
            eng.seed(13)
            eng.run(n)
            got.append((eng.stats(), [eng.histogram(k) for k in eng.panels]))
        assert got[0][0] == got[1][0] and got[0][0]["primaries"] == n
        for a, b in zip(got[0][1], got[1][1]):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    few.close()
    many.close()
