"""The ray tracer's spectrum table follows the source and the physics tables:
images after any order of changes equal those of a new engine."""

import numpy as np
import pytest

import plain_scene as S

pytestmark = pytest.mark.gpu

LINE = (np.array([0.06, 0.06], S.F), np.array([0, 1], S.F), False)
TWO = (np.array([0.03, 0.09, 0.09], S.F), np.array([0, 0.25, 1], S.F), False)
SPREAD = (np.array([0.03, 0.09, 0.09], S.F), np.array([0, 0.25, 1], S.F), True)  # the same numbers, interpolated
OTHER = (np.array([0.03, 0.09, 0.09], S.F), np.array([0, 0.75, 1], S.F), False)
MOVED = np.array([[0, 0, -1, -650], [0, 1, 0, 10], [1, 0, 0, -5], [0, 0, 0, 1]], S.F)


def _tables(density=1.0, nbins=64):
    t = S.tables(4, nbins)
    t["cross_sections"] = (t["cross_sections"] * S.F(density)).astype(S.F)
    return t


def _image(eng, panel):
    import torch
    a = eng.drr(panel)
    b = torch.full(a.shape, -1.0, device="cuda")
    eng.drr_noalloc(panel, b.data_ptr())
    eng.synchronize()
    assert np.array_equal(a, b.cpu().numpy())
    return a


def _scene(tables, matrix, spectrum):
    eng = S.Engine(0)
    eng.set_physics(**tables)
    labels = np.random.default_rng(8).integers(0, 3, (10, 14, 12)).astype(np.uint8)
    S.add_voxels(eng, labels, (6.0, 5.0, 7.0))
    panel = S.add_panel(eng, 20, 24, 6.0, 3)
    eng.set_xray_source(matrix, 0.1, (0.0, 0.0, 0.0), *spectrum)
    return eng, panel


def test_images_follow_the_source_and_the_tables():
    eng, panel = _scene(_tables(), S.SOURCE_AT, LINE)
    tables = _tables()
    images = []
    for matrix, spectrum, new in ((S.SOURCE_AT, LINE, None), (MOVED, LINE, None), (MOVED, TWO, None),
                                  (S.SOURCE_AT, TWO, None), (S.SOURCE_AT, SPREAD, None), (S.SOURCE_AT, OTHER, None),
                                  (S.SOURCE_AT, OTHER, dict(density=0.5)), (MOVED, OTHER, None),
                                  (MOVED, OTHER, dict(nbins=200)), (S.SOURCE_AT, LINE, None)):
        if new is not None:
            tables = _tables(**new)
            eng.set_physics(**tables)
        eng.set_xray_source(matrix, 0.1, (0.0, 0.0, 0.0), *spectrum)
        images.append(_image(eng, panel))
        fresh, k = _scene(tables, matrix, spectrum)
        assert np.array_equal(images[-1], _image(fresh, k))
        fresh.close()
    assert len({i.tobytes() for i in images}) == len(images)
    # tables set after the source
    eng.set_physics(**_tables(density=2.0))
    fresh, k = _scene(_tables(density=2.0), S.SOURCE_AT, LINE)
    assert np.array_equal(_image(eng, panel), _image(fresh, k))
    fresh.close()
    eng.close()
