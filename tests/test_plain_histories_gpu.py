"""Whole histories against the CPU oracle on made-up tables: the quick voxel
step at the edges of its geometry and the general one, both samplings, fewer
processes and another order of them, photon tracking, several phantoms before
several modules, acquisitions, and the shared walk through meshes."""

import numpy as np
import pytest

from ggems_amd import authoring
from plain_oracle import PlainScene, assert_same_histories, plain_oracle  # noqa: F401

pytestmark = pytest.mark.gpu


def _voxels(shape=(9, 21, 17), voxel=(4.0, 3.0, 5.0), processes=(0, 1, 2), aperture=None, modules=(1, 1),
            tracking=False, phantoms=1, sid=600.0, sdd=1000.0, nbins=64):
    rng = np.random.default_rng(3)
    sc = PlainScene(nbins=nbins, processes=processes)
    for k in range(phantoms):
        sc.add_phantom(rng.integers(0, 2, shape).astype(np.uint8), ["a", "b"], voxel,
                       position=((k - 0.5 * (phantoms - 1)) * 1.2 * shape[2] * voxel[0], 0.0, 0.0),
                       dosimetry={"photon_tracking": tracking} if k == 0 else None)
    sc.add_ct_flat("panel", modules, (32, 32, 1), (4.0, 4.0, 1.0), sid, sdd, 10e-3)
    half = shape[1] * voxel[1] / 2
    sc.set_source((-sid, 0.0, 0.0), np.degrees(np.arctan(half / sid)) if aperture is None else aperture, [0.06],
                  mono=True)
    return sc.build()


@pytest.mark.parametrize("tau", [False, True])
@pytest.mark.parametrize("kw", [
    dict(),
    dict(processes=(1,)), dict(processes=(0, 1)), dict(processes=(2, 1, 0)),
    dict(tracking=True), dict(tracking=True, processes=(1, 0)),
    dict(shape=(30, 40, 20), voxel=(0.0015, 0.0015, 0.002)),                       # thin voxels: the general step
    dict(shape=(20, 30, 25), voxel=(0.002, 0.0025, 0.003)),                        # the thinnest of the quick step
    dict(shape=(3, 3, 3), voxel=(1500.0, 90.0, 90.0), sid=4000.0, sdd=8000.0),     # far coordinates: the general step
    dict(shape=(30, 40, 20), voxel=(0.0015, 0.0015, 0.002), processes=(0, 1), tracking=True),
    dict(aperture=0.0), dict(aperture=1e-5),                                       # rays along x, and next to it
    dict(voxel=(40.0, 30.0, 50.0)),                                                # steps of several free paths
    dict(modules=(3, 5), phantoms=3),                                              # hops between solids
    dict(modules=(3, 5), phantoms=2, shape=(30, 40, 20), voxel=(0.0015, 0.0015, 0.002)),
    dict(nbins=1000),                                                              # tables beyond LDS
], ids=lambda kw: "-".join("%s=%s" % i for i in kw.items()) or "plain")
def test_voxel_histories_match_the_oracle(plain_oracle, kw, tau):  # noqa: F811
    sc = _voxels(**kw)
    sc.tau = tau
    n = 40_000
    ref, got = sc.run_oracle(n, 5), sc.run_engine(n, 5)
    assert got["stats"]["primaries"] == n and ref["stats"]["voxel_steps"] > 0
    assert_same_histories(ref, got, images=("hit", "photon_tracking") if kw.get("tracking") else ("hit",))


@pytest.mark.parametrize("tau", [False, True])
@pytest.mark.parametrize("thin", [False, True])
def test_acquisitions_match_the_oracle(plain_oracle, thin, tau):  # noqa: F811
    sc = _voxels(modules=(1, 3), **(dict(shape=(30, 40, 20), voxel=(0.0015, 0.0015, 0.002)) if thin else {}))
    sc.tau = tau
    rot, n = [(0.0, 0.0, 0.0), (0.0, 0.0, 1.1), (0.0, 0.0, 2.5)], [3_000, 20_000, 700]
    eng = sc.engine_acquisition(rot, n, 4)
    eng.run_acquisition()
    got, ref = sc.read_acquisition(eng), sc.run_oracle_acquisition(rot, n, 4)
    eng.close()
    assert got["stats"]["primaries"] == sum(n)
    assert_same_histories(ref, got, images=())


@pytest.mark.parametrize("n", [64, 5_000, 40_000, 2_000_000])
@pytest.mark.parametrize("meshes", [
    [(40.0, 0, (0, 0, 0))],                                            # 20 triangles
    [(40.0, 4, (0, 0, 0)), (12.0, 2, (0, 0, 0)), (6.0, 3, (0, 60, 0))],  # inside and beside
])
def test_mesh_histories_match_the_oracle(plain_oracle, meshes, n):  # noqa: F811
    """the most photons take the shared walk, fewer than four a lane each lane's own loop"""
    sc = PlainScene(nbins=64)
    for k, (radius, level, at) in enumerate(meshes):
        sc.add_mesh(authoring.icosphere(radius, level).astype(np.float32) + np.asarray(at, np.float32), str(k),
                    dosimetry={"dosel_size": (2.0, 2.0, 2.0), "photon_tracking": True} if k == 0 else None)
    sc.add_ct_flat("panel", (1, 2), (32, 32, 1), (2.0, 2.0, 1.0), 600.0, 1000.0, 10e-3)
    sc.set_source((-600.0, 0.0, 0.0), 4.0, [0.08], mono=True)
    sc.build()
    ref, got = sc.run_oracle(n, 9), sc.run_engine(n, 9)
    assert got["stats"]["primaries"] == n
    assert_same_histories(ref, got, ("mesh_steps", "mesh_interactions", "hops"), ("hit", "photon_tracking"))
