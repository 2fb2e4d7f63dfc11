"""Results that leave in several chunks: dose tallies, dose maps, detector and
ray-traced images larger and smaller than a chunk, whole and not, and several
threads that read one engine."""

import threading

import numpy as np
import pytest
import torch

import plain_scene

pytestmark = pytest.mark.gpu


def _engine(n_dosels, panel=(24, 24)):
    eng = plain_scene.engine(3)
    labels = np.zeros((11, 13, 21), np.uint8)
    labels[4:7, 5:9, 8:15] = 1
    plain_scene.add_voxels(eng, labels, (8.0, 8.0, 8.0))
    eng.panel = plain_scene.add_panel(eng, panel[0], panel[1], 2.0, 2)
    half = np.array([84.0, 52.0, 44.0])
    eng.set_dosimetry(0, tuple(2 * half / n_dosels), n_dosels, tuple(-half), tuple(half), photon_tracking=True)
    plain_scene.add_source(eng)
    eng.seed(5)
    return eng


def _run(eng):
    eng.reset_tallies()
    eng.run(200_000)
    return eng.dose_tallies()


# dosels of 8, 4, 1 and 1/2 mm: 3,003 (a part of a chunk) to 12.3 million
@pytest.mark.parametrize("split", [(2, 2, 2), (8, 8, 4), (16, 16, 16)])
def test_tallies_of_fine_dosels_add_up_to_the_coarse_ones(split):
    """Dosimetry does not touch the histories and the borders are exact, so a
    coarse dosel's counts are the sum of its parts'."""
    coarse = _engine((21, 13, 11))
    ref = _run(coarse)
    coarse.close()
    n = tuple(a * b for a, b in zip((21, 13, 11), split))
    eng = _engine(n)
    got = _run(eng)
    assert int(ref[2].sum()) > 10_000
    shape = (11, split[2], 13, split[1], 21, split[0])
    for k, (a, b) in enumerate(zip(ref, got)):
        if k == 1:  # squares: of the same deposits
            np.testing.assert_allclose(b.reshape(shape).sum((1, 3, 5)), a, rtol=1e-11, atol=1e-18)
        elif a.dtype == np.float64:
            np.testing.assert_allclose(b.reshape(shape).sum((1, 3, 5)), a, rtol=1e-11, atol=1e-18)
        else:
            assert np.array_equal(b.reshape(shape).sum((1, 3, 5)), a), k
    # the maps from the tallies read: one material density where labels are 0
    dose, unc = eng.compute_dose(1.0, True)
    edep, edep2, hit, _ = got
    vol = float(np.prod(2 * np.array([84.0, 52.0, 44.0]) / n))
    want = edep / (6.241509704e21 / 1e3) / vol / 1e-12
    np.testing.assert_allclose(dose, want, rtol=1e-5)  # FP32 density, volume and result
    many = (hit > 1) & (edep != 0)
    assert np.all(unc[~many] == 1.0)
    h, s2 = hit[many].astype(np.float64), edep[many] ** 2
    np.testing.assert_allclose(unc[many], np.sqrt((h * edep2[many] - s2) / ((h - 1) * s2)), rtol=1e-6, atol=1e-6)
    eng.close()


@pytest.mark.parametrize("panel", [(1, 1), (5, 13), (300, 437), (701, 703)])
def test_images(panel):
    eng = _engine((21, 13, 11), panel)
    ny, nx, _ = eng.box_elements[eng.panel]
    image = torch.zeros(ny, nx, device="cuda")
    eng.drr(eng.panel)  # the solid table goes to the device
    eng.drr_noalloc(eng.panel, image.data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
    assert np.array_equal(eng.drr(eng.panel), image.cpu().numpy())
    eng.run(100_000)
    counts, scatter = eng.histogram(eng.panel)
    assert np.all(scatter <= counts) and np.all(scatter >= 0)
    if min(panel) > 100:
        assert 0 < scatter.sum() < counts.sum()
    eng.close()


def test_threads_share_an_engine():
    eng = _engine((84, 52, 44))
    ref = _run(eng)
    bad = []

    def read():
        for _ in range(5):
            if not all(np.array_equal(a, b) for a, b in zip(ref, eng.dose_tallies())):
                bad.append(1)

    threads = [threading.Thread(target=read) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    eng.close()
