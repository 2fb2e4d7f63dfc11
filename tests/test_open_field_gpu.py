"""Scenes of detector modules alone (an open field) against the oracle: tables
in LDS and beyond it, fewer processes, several modules, acquisitions, photons
that leave the last module's pixels."""

import pytest

from plain_oracle import PlainScene, assert_same_histories, plain_oracle  # noqa: F401

pytestmark = pytest.mark.gpu


def _scene(nbins=64, processes=(0, 1, 2), modules=(1, 1), thick=1.0, aperture=6.0):
    sc = PlainScene(nbins=nbins, processes=processes)
    sc.add_ct_flat("panel", modules, (32, 32, 1), (2.0, 2.0, thick), 600.0, 1000.0, 10e-3)
    sc.set_source((-600.0, 0.0, 0.0), aperture, [0.03, 0.06, 0.1], [1.0, 2.0, 1.0])
    return sc.build()


@pytest.mark.parametrize("kw", [dict(), dict(nbins=1500), dict(processes=(0,)), dict(processes=(2, 1), thick=20.0),
                                dict(modules=(2, 7)), dict(thick=40.0, aperture=0.0)],
                         ids=lambda kw: "-".join("%s=%s" % i for i in kw.items()) or "plain")
@pytest.mark.parametrize("tau", [False, True])
def test_open_field_matches_the_oracle(plain_oracle, kw, tau):  # noqa: F811
    sc = _scene(**kw)
    sc.tau = tau  # boxes keep GGEMS's sampling
    for n in (1, 700, 60_000):
        ref, got = sc.run_oracle(n, 3), sc.run_engine(n, 3)
        assert got["stats"]["primaries"] == n and (n == 1 or got["stats"]["detector_interactions"] > 0)
        assert_same_histories(ref, got, ("detector_steps", "detector_interactions", "hops"), ())


def test_open_field_acquisition_matches_the_oracle(plain_oracle):  # noqa: F811
    sc = _scene(modules=(1, 3))
    rot, n = [(0.0, 0.0, 0.0), (0.0, 0.0, 1.1), (0.0, 0.0, 2.5)], [3_000, 40_000, 700]
    eng = sc.engine_acquisition(rot, n, 4)
    eng.run_acquisition()
    got, ref = sc.read_acquisition(eng), sc.run_oracle_acquisition(rot, n, 4)
    eng.close()
    assert_same_histories(ref, got, ("detector_steps", "detector_interactions", "hops"), ())
