"""Grids that take the general voxel step: it makes the quick step's histories
bit for bit, and such scenes run every kernel variant that others do."""

import numpy as np
import pytest

import plain_scene

pytestmark = pytest.mark.gpu

ASIDE = np.array([[1, 0, 0, 0], [0, 1, 0, 500.0], [0, 0, 1, 0], [0, 0, 0, 1]], np.float32)


def _engine(voxel=4.0, processes=(0, 1, 2), tracking=False, tau=False, thin_aside=False, nbins=64, modules=1,
            phantoms=1):
    t = plain_scene.tables(3, nbins)
    t["process_ids"] = processes
    eng = plain_scene.Engine(0)
    eng.set_physics(**t)
    labels = np.random.default_rng(3).integers(0, 2, (20, 24, 28)).astype(np.uint8)
    for k in range(phantoms):
        m = np.eye(4)
        m[0, 3] = (k - 0.5 * (phantoms - 1)) * 30 * voxel
        plain_scene.add_voxels(eng, labels, (voxel,) * 3, m)
    half = np.array([28, 24, 20]) * voxel / 2
    eng.set_dosimetry(0, (voxel,) * 3, (28, 24, 20), tuple(-half), tuple(half), photon_tracking=tracking)
    eng.panels = []
    for j in range(modules):
        m = plain_scene.PANEL_AT.copy()
        m[1, 3] = (j - 0.5 * (modules - 1)) * 48.0
        eng.panels.append(plain_scene.add_panel(eng, 24, 24, 2.0, 2, m))
    if thin_aside:  # out of the beam, and too thin for the quick step, which no solid then takes
        plain_scene.add_voxels(eng, np.zeros((2, 2, 2), np.uint8), (1e-3,) * 3, ASIDE)
    plain_scene.add_source(eng, 0.06 if voxel > 1 else 2e-5)
    eng.set_sampling("tau" if tau else "reference")
    return eng


def _results(eng, n, seed):
    eng.reset_tallies()
    eng.seed(seed)
    eng.run(n)
    tallies = eng.dose_tallies()
    return eng.stats(), [eng.histogram(k) for k in eng.panels], tallies[2], tallies[3], tallies[0]


@pytest.mark.parametrize("tau", [False, True])
@pytest.mark.parametrize("tracking", [False, True])
@pytest.mark.parametrize("processes", [(0, 1, 2), (2, 0, 1), (1,), (0, 2), ()])
def test_quick_steps_make_the_general_steps_histories(processes, tracking, tau):
    quick = _engine(processes=processes, tracking=tracking, tau=tau)
    general = _engine(processes=processes, tracking=tracking, tau=tau, thin_aside=True)
    for n, seed in ((1, 1), (700, 2), (300_000, 3)):
        a, b = _results(quick, n, seed), _results(general, n, seed)
        assert a[0] == b[0] and a[0]["primaries"] == n and a[0]["voxel_steps"] > 0
        for (x, xs), (y, ys) in zip(a[1], b[1]):
            assert np.array_equal(x, y) and np.array_equal(xs, ys)
        assert np.array_equal(a[2], b[2])
        if tracking:
            assert np.array_equal(a[3], b[3]) and a[3].sum() > 0
        # FP64 sums whose order follows the atomics
        np.testing.assert_allclose(a[4], b[4], rtol=1e-12, atol=1e-18)
    quick.close()
    general.close()


@pytest.mark.parametrize("kw,variant", [
    (dict(), 0), (dict(tau=True), 0), (dict(tracking=True), 1), (dict(processes=(0, 1)), 1), (dict(phantoms=2), 2),
    (dict(phantoms=2, tau=True), 2), (dict(nbins=1000), 1), (dict(nbins=1000, tau=True), 1),
])
def test_thin_grids_run_every_variant(kw, variant):
    """the specialised kernels as for thicker voxels, each against the general
    one, and an acquisition of each against single runs"""
    eng = _engine(voxel=0.0015, modules=2, **kw)
    base = None
    for general in (False, True):
        eng.set_launch(general_kernel=general)
        got = _results(eng, 100_000, 7)
        assert eng.last_grid()[2] == (1 if general else variant)
        base = base or got
        assert got[0] == base[0] and got[0]["voxel_steps"] > 0
        assert all(np.array_equal(x, y) for a, b in zip(got[1], base[1]) for x, y in zip(a, b))
        assert np.array_equal(got[2], base[2])
    budgets = (40_000, 300, 20_000)
    eng.seed(9)
    eng.reset_tallies()
    images, before = [], 0
    for n in budgets:
        eng.run(n)
        now = np.stack([np.stack(eng.histogram(k)) for k in eng.panels])
        images.append(now - before)
        before = now
    box = np.stack([plain_scene.PANEL_AT] * 2)
    box[:, 1, 3] = (-24.0, 24.0)
    for general in (False, True):
        eng.set_launch(general_kernel=general)
        eng.seed(9)
        eng.set_acquisition(np.stack([plain_scene.SOURCE_AT] * 3), np.stack([box] * 3), budgets)
        eng.run_acquisition()
        assert eng.last_grid()[2] == (1 if general else variant)
        for p, want in enumerate(images):
            got = np.stack([np.stack(eng.projection(k, p)) for k in eng.panels])
            assert np.array_equal(got, want), p
    eng.close()
