"""The voxel step's short cuts on the GPU: the bound by which it rules an
interaction out, and whole histories on grids and beams at the edges of its
quick geometry, against the oracle."""

import numpy as np
import pytest

import plain_scene as S
from scene import Scene

pytestmark = pytest.mark.gpu


def test_no_interaction_bound_holds_for_the_device_logarithm():
    """A draw that the step's bound rules out has -log(u) / sigma beyond the
    boundary: with 2^-32 sum + 1.01 a < 1 - 2^-19 in the step's arithmetic,
    -log(u) >= a.  Checked at the largest a that still passes."""
    eng = S.engine(2)
    top = (2 ** 32 - 1 - np.arange(1 << 21, dtype=np.uint64)).astype(np.uint32)
    spread = np.random.default_rng(1).integers(1, 2 ** 32, 1 << 21, dtype=np.uint64).astype(np.uint32)
    steps = (2 ** 32 - np.unique(np.geomspace(1, 2 ** 31, 1 << 18).astype(np.uint64))).astype(np.uint32)
    sums = np.concatenate([top, spread, steps])
    lg, _ = eng.debug_neg_log(sums)
    eng.close()
    room = 1.0 - 2.0 ** -19 - sums.astype(np.float32).astype(np.float64) * 2.0 ** -32
    a = room / 1.01 * (1 + 1e-6) + 2.0 ** -24  # rounding of the product and of the sum
    ruled = room > 0
    assert ruled.sum() > 1 << 20
    assert (lg[ruled] >= a[ruled]).all()


def _scene(shape, voxel, aperture=None, sdd=1000.0, sid=600.0):
    rng = np.random.default_rng(3)
    sc = Scene()
    sc.add_phantom(rng.integers(0, 2, shape).astype(np.uint8), ["Water", "RibBone"], voxel,
                   dosimetry={"photon_tracking": False})
    sc.add_ct_flat("GOS", (1, 1), (32, 32, 1), (4.0, 4.0, 1.0), sid, sdd, 10e-3)
    half = shape[1] * voxel[1] / 2
    sc.set_source((-sid, 0.0, 0.0), np.degrees(np.arctan(half / sid)) if aperture is None else aperture, [0.06],
                  mono=True)
    return sc.build()


@pytest.mark.parametrize("tau", [False, True])
@pytest.mark.parametrize("shape,voxel,kw", [
    ((30, 40, 20), (0.0015, 0.0015, 0.002), {}),                       # thin voxels: the general step
    ((20, 30, 25), (0.002, 0.0025, 0.003), {}),                        # the thinnest of the quick step
    ((3, 3, 3), (1500.0, 90.0, 90.0), dict(sid=4000.0, sdd=8000.0)),   # coordinates past 2,048 mm: the general step
    ((9, 21, 17), (4.0, 3.0, 5.0), dict(aperture=0.0)),                # rays along x, between voxels
    ((9, 21, 17), (4.0, 3.0, 5.0), dict(aperture=1e-5)),               # and next to it
    ((9, 21, 17), (40.0, 30.0, 50.0), {}),                             # steps of several free paths
])
def test_histories_match_the_oracle(shape, voxel, kw, tau):
    sc = _scene(shape, voxel, **kw)
    sc.tau = tau
    n = 40_000
    ref, got = sc.run_oracle(n, 5), sc.run_engine(n, 5)
    a, b = ref["stats"], got["stats"]
    assert b["primaries"] == n
    # histories are equal up to the transcendentals' last bits, which move a few of them
    for k in ("voxel_steps", "interactions", "hops"):
        assert abs(a[k] - b[k]) <= 20 + 2e-3 * a[k], (k, a[k], b[k])
    l1 = int(np.abs(ref["hit"].astype(np.int64) - got["hit"]).sum())
    assert l1 <= 20 + 0.01 * int(ref["hit"].sum()), l1
