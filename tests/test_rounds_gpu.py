"""Rounds of any length, and those whose length follows the photons that stop,
regroup photons and nothing else: a part of a block, one block, more photons
than lanes, both samplings, both kernels, grids of quick and of thin voxels."""

import numpy as np
import pytest

import plain_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("voxel", [4.0, 0.0015])
@pytest.mark.parametrize("tau", [False, True])
@pytest.mark.parametrize("n", [1, 300, 513, 400_000])
def test_rounds_do_not_change_histories(n, tau, voxel):
    eng = plain_scene.engine(3)
    labels = np.random.default_rng(3).integers(0, 2, (20, 24, 28)).astype(np.uint8)
    plain_scene.add_voxels(eng, labels, (voxel,) * 3)
    panel = plain_scene.add_panel(eng, 24, 24, 8.0, 2)
    half = np.array([28, 24, 20]) * voxel / 2
    eng.set_dosimetry(0, (voxel,) * 3, (28, 24, 20), tuple(-half), tuple(half))
    plain_scene.add_source(eng, 0.06 if voxel > 1 else 2e-5)
    eng.set_sampling("tau" if tau else "reference")
    base = None
    for general in (False, True):
        for steps in (0, 1, 8, 20, 77):
            eng.set_launch(round_steps=steps, general_kernel=general)
            eng.reset_tallies()
            eng.seed(11)
            eng.run(n)
            got = (eng.stats(), eng.histogram(panel), eng.dose_tallies())
            assert got[0]["primaries"] == n
            if base is None:
                base = got
            assert got[0] == base[0], (steps, general)
            assert all(np.array_equal(a, b) for a, b in zip(got[1], base[1]))
            assert np.array_equal(got[2][2], base[2][2])
            # FP64 sums whose order follows the atomics
            np.testing.assert_allclose(got[2][0], base[2][0], rtol=1e-12, atol=1e-18)
    eng.close()
