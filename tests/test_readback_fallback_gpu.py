"""Readbacks without pinned host memory, in chunks of a megabyte over device
memory, give what the pinned slots give: less than a chunk, several, and parts
of one."""

import numpy as np
import pytest

import plain_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split,panel", [((1, 1, 1), (1, 1)), ((5, 4, 3), (300, 437)), ((16, 16, 16), (701, 703))])
def test_same_results(split, panel):
    eng = plain_scene.engine(3)
    labels = np.zeros((11, 13, 21), np.uint8)
    labels[4:7, 5:9, 8:15] = 1
    plain_scene.add_voxels(eng, labels, (8.0, 8.0, 8.0))
    k = plain_scene.add_panel(eng, panel[0], panel[1], 0.5, 2)
    half = np.array([84.0, 52.0, 44.0])
    n = np.array((21, 13, 11)) * split
    eng.set_dosimetry(0, tuple(2 * half / n), n, tuple(-half), tuple(half), photon_tracking=True)
    plain_scene.add_source(eng)
    eng.seed(5)
    eng.run(200_000)
    eng.set_acquisition(plain_scene.SOURCE_AT[None], plain_scene.PANEL_AT[None, None], (100_000,))
    eng.run_acquisition()
    got = []
    for off in (False, True, False):
        eng.debug_no_pinned(off)
        got.append([*eng.dose_tallies(), *eng.compute_dose(1.0, True), eng.compute_dose(1.0, uncertainty=False)[0],
                    *eng.histogram(k), *eng.projection(k, 0), eng.drr(k)])
    assert got[0][2].sum() > 0 and got[0][3].sum() > 0
    for other in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], other))
    eng.close()
