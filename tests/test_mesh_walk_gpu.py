"""Meshed scenes whose photons differ most in steps and nodes: one photon, a
wave's worth and a few thousand, meshes of a few triangles and of many, solids
inside one another and beside each other, with an acquisition's placements,
against the oracle."""

import numpy as np
import pytest

import plain_scene
from ggems_amd import authoring
from scene import Scene

pytestmark = pytest.mark.gpu


def _scene(meshes, aperture=4.0):
    sc = Scene()
    for k, (radius, level, at) in enumerate(meshes):
        sc.add_mesh(authoring.icosphere(radius, level).astype(np.float32) + np.asarray(at, np.float32),
                    ("SoftTissus_15", "RibBone", "Water")[k % 3],
                    dosimetry={"dosel_size": (2.0, 2.0, 2.0), "photon_tracking": k == 0} if k == 0 else None)
    sc.add_ct_flat("GOS", (1, 2), (32, 32, 1), (2.0, 2.0, 1.0), 600.0, 1000.0, 10e-3)
    sc.set_source((-600.0, 0.0, 0.0), aperture, [0.08], mono=True)
    return sc.build()


@pytest.mark.parametrize("n", [1, 64, 5_000, 40_000])
@pytest.mark.parametrize("meshes", [
    [(40.0, 0, (0, 0, 0))],                                            # 20 triangles
    [(40.0, 4, (0, 0, 0)), (12.0, 2, (0, 0, 0)), (6.0, 3, (0, 60, 0))],  # inside and beside
])
def test_histories_match_the_oracle(meshes, n):
    sc = _scene(meshes)
    ref, got = sc.run_oracle(n, 9), sc.run_engine(n, 9)
    assert got["stats"]["primaries"] == n
    # histories are equal up to the transcendentals' last bits, which move a few of them
    for k in ("mesh_steps", "mesh_interactions", "hops"):
        assert abs(ref["stats"][k] - got["stats"][k]) <= 20 + 3e-3 * ref["stats"][k], (k, ref["stats"], got["stats"])
    for k in ("hit", "photon_tracking"):
        l1 = int(np.abs(ref[k].astype(np.int64) - got[k]).sum())
        assert l1 <= 40 + 0.02 * int(ref[k].sum()), (k, l1)


def test_acquisition_equals_single_runs():
    sc = _scene([(40.0, 3, (0, 0, 0)), (12.0, 2, (0, 50, 0))])
    rot, n = [(0.0, 0.0, 0.0), (0.0, 0.0, 1.1)], [3_000, 20_000]
    eng = sc.engine_acquisition(rot, n, 4)
    eng.run_acquisition()
    got = sc.read_acquisition(eng)
    ref = sc.run_oracle_acquisition(rot, n, 4)
    assert got["stats"]["primaries"] == sum(n)
    for a, b in zip(ref["hist"], got["hist"]):
        assert int(np.abs(a.astype(np.int64) - b).sum()) <= 20 + 0.02 * int(a.sum())
    eng.close()


@pytest.mark.parametrize("meshes", [[(40.0, 0)], [(40.0, 4), (12.0, 2)]])
def test_few_and_many_photons_a_lane_take_the_same_histories(meshes):
    """600,000 photons are fewer than four for each lane of the whole card and
    more than four for each lane of one block per compute unit: the first launch
    runs each lane's track loop, the second the shared walk."""
    eng = plain_scene.engine(3)
    for k, (radius, level) in enumerate(meshes):
        tri = authoring.icosphere(radius, level).astype(np.float32)
        half = np.abs(tri).reshape(-1, 3).max(0) + np.float32(1e-3)
        eng.add_mesh_solid(tri, -half, half, k)
    panel = plain_scene.add_panel(eng, 32, 32, 4.0, 2)
    eng.set_dosimetry(0, (4.0, 4.0, 4.0), (20, 20, 20), (-40.0,) * 3, (40.0,) * 3, photon_tracking=True)
    plain_scene.add_source(eng)
    got = []
    for blocks in (0, 1):
        eng.set_launch(blocks_per_cu=blocks)
        eng.reset_tallies()
        eng.seed(77)
        eng.run(600_000)
        edep, _, hit, track = eng.dose_tallies()
        got.append((eng.stats(), eng.histogram(panel)[0], hit, track, edep))
    a, b = got
    assert a[0] == b[0] and a[0]["primaries"] == 600_000 and a[0]["mesh_interactions"] > 0
    for x, y in zip(a[1:4], b[1:4]):
        assert np.array_equal(x, y)
    # FP64 sums whose order follows the atomics
    np.testing.assert_allclose(a[4], b[4], rtol=1e-12, atol=1e-18)
    eng.close()
