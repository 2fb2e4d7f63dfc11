"""A readback that asks for no array still waits for the engine's stream."""

import numpy as np
import pytest
import torch

import plain_scene
from ggems_amd.engine import library

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["ggh_get_histogram", "ggh_get_projection", "ggh_get_dose_tallies"])
def test_waits_without_an_array(call):
    eng = plain_scene.engine(3)
    plain_scene.add_voxels(eng, np.zeros((128, 128, 128), np.uint8), (1.0,) * 3)
    panel = plain_scene.add_panel(eng, 512, 512, 0.5, 2)
    eng.set_dosimetry(0, (8.0,) * 3, (16, 16, 16), (-64.0,) * 3, (64.0,) * 3)
    plain_scene.add_source(eng)
    eng.seed(1)
    eng.set_acquisition(plain_scene.SOURCE_AT[None], plain_scene.PANEL_AT[None, None], (1000,))
    eng.run_acquisition()
    eng.drr(panel)
    scratch, image = torch.empty(512, 512, device="cuda"), torch.full((512, 512), -1.0, device="cuda")
    torch.cuda.synchronize()
    for _ in range(300):  # some ten milliseconds of work on the engine's stream
        eng.drr_noalloc(panel, scratch.data_ptr())
    eng.drr_noalloc(panel, image.data_ptr())
    args = {"ggh_get_histogram": (panel, None, None), "ggh_get_projection": (panel, 0, None, None),
            "ggh_get_dose_tallies": (None, None, None, None)}[call]
    assert getattr(library(), call)(eng.h, *args) == 0
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        seen = image.clone()
    side.synchronize()
    assert (seen >= 0).all()
    eng.close()
