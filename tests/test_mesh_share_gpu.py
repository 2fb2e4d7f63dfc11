"""Meshes that few of the source's photons meet take each lane's track loop at
any number of photons: against the oracle, and an acquisition of large and
small meshes against single runs, which choose for themselves."""

import numpy as np
import pytest

import plain_scene
from ggems_amd import authoring
from plain_oracle import PlainScene, assert_same_histories, plain_oracle  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("meshes", [[(3.0, 2, (0, 0, 0))], [(2.0, 3, (0, 9, 0)), (1.5, 1, (30, -8, 4))],
                                    [(2.0, 2, (0, 0, 0)), (30.0, 3, (0, 0, 0))]])
def test_few_photons_in_meshes_match_the_oracle(plain_oracle, meshes):  # noqa: F811
    sc = PlainScene(nbins=64)
    for k, (radius, level, at) in enumerate(meshes):
        sc.add_mesh(authoring.icosphere(radius, level).astype(np.float32) + np.asarray(at, np.float32), str(k),
                    dosimetry={"dosel_size": (1.0, 1.0, 1.0), "photon_tracking": True} if k == 0 else None)
    sc.add_ct_flat("panel", (1, 2), (32, 32, 1), (2.0, 2.0, 1.0), 600.0, 1000.0, 10e-3)
    sc.set_source((-600.0, 0.0, 0.0), 6.0, [0.08], mono=True)
    sc.build()
    n = 2_000_000
    ref, got = sc.run_oracle(n, 9), sc.run_engine(n, 9)
    assert got["stats"]["primaries"] == n and got["stats"]["mesh_steps"] > 100
    assert_same_histories(ref, got, ("mesh_steps", "mesh_interactions", "hops", "detector_interactions"),
                          ("hit", "photon_tracking"))


@pytest.mark.parametrize("radius", [2.0, 40.0])
def test_acquisitions_equal_single_runs(radius):
    eng = plain_scene.engine(3)
    tri = authoring.icosphere(radius, 3).astype(np.float32)
    half = np.abs(tri).reshape(-1, 3).max(0) + np.float32(1e-3)
    eng.add_mesh_solid(tri, -half, half, 0)
    panel = plain_scene.add_panel(eng, 32, 32, 4.0, 2)
    plain_scene.add_source(eng)
    budgets = (1_500_000, 300, 40_000)
    eng.seed(9)
    images, before = [], 0
    for n in budgets:
        eng.run(n)
        now = np.stack(eng.histogram(panel))
        images.append(now - before)
        before = now
    assert eng.stats()["mesh_interactions"] > 0
    eng.seed(9)
    eng.set_acquisition(np.stack([plain_scene.SOURCE_AT] * 3), np.stack([plain_scene.PANEL_AT[None]] * 3), budgets)
    eng.run_acquisition()
    for p, want in enumerate(images):
        assert np.array_equal(np.stack(eng.projection(panel, p)), want), p
    eng.close()
