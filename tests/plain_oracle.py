"""The CPU oracle and the engine on plain_scene's made-up tables, for history
tests that need no physics data.  The oracle reads the Rayleigh form factors
from a data file; a copy of its library, loaded beside the one that holds
GGEMS's data, reads a made-up one."""

import os
import shutil
import sys

import numpy as np
import pytest

import plain_scene
import ggems_oracle as O
from scene import F, Scene

sys.path.insert(0, os.path.join(O.REPO, "ggems_amd", "data"))
from extract_physics_data import write_blob  # noqa: E402


@pytest.fixture
def plain_oracle(tmp_path, monkeypatch):
    if not os.path.exists(O.LIB_PATH):
        O.build()
    pp = plain_scene.tables(2)["rayleigh_pp"]
    blob = {"rayleigh_pp%d" % k: ("f32", pp[k].tolist()) for k in range(9)}
    blob["rayleigh_factor"] = ("f32", [plain_scene.tables(2)["rayleigh_factor"]])
    blob["element_names"], blob["element_z"] = ("i8", list(b"Hydrogen") + [0]), ("i32", [1])
    write_blob(blob, str(tmp_path / "physics.bin"))
    (tmp_path / "materials.txt").write_text("Nothing: d=1.0 g/cm3; n=1\n+el: name=Hydrogen; f=1.0\n")
    monkeypatch.setattr(O, "LIB_PATH", shutil.copy(O.LIB_PATH, str(tmp_path / "liboracle.so")))
    monkeypatch.setattr(O, "PHYSICS_BLOB", str(tmp_path / "physics.bin"))
    monkeypatch.setattr(O, "MATERIALS_TXT", str(tmp_path / "materials.txt"))
    monkeypatch.setattr(O, "_lib", None)
    return O.lib()


class PlainScene(Scene):
    """a Scene whose materials are rows of plain_scene.tables: 0, 1, ... of its
    phantoms in the order of their navigators, the last one the detector's"""

    def build(self):
        self.materials, self.offsets = [], []
        for _, materials, _ in self.navigators:
            self.offsets.append(len(self.materials))
            self.materials.extend(materials)
        n = len(self.materials)
        t = plain_scene.tables(n, self.nbins)
        self.ebins, self.cs, self.cs_atom = t["energy_bins"], t["cross_sections"], t["cs_atom_rayleigh"]
        self.arrays = dict(n_elements=np.array(t["n_elements"], np.int32),
                           elem_index=np.array(t["element_index"], np.int32),
                           z=np.array(t["atomic_number"], np.uint8),
                           atom_density=np.array(t["atom_density"], np.float32),
                           density=np.array(t["density"], F), photon_cut=np.array(t["photon_cut"], F))
        self.pp, self.factor = t["rayleigh_pp"], t["rayleigh_factor"]
        return self


def assert_same_histories(ref, got, steps=("voxel_steps", "interactions", "hops"), images=("hit",)):
    """equal up to the transcendentals' last bits, which move a few histories
    (the margins of the tests on GGEMS's data)"""
    for k in steps:
        a, b = ref["stats"][k], got["stats"][k]
        assert abs(a - b) <= 20 + 3e-3 * a, (k, a, b)
    for k in images:
        l1 = int(np.abs(ref[k].astype(np.int64) - got[k]).sum())
        assert l1 <= 40 + 0.02 * int(ref[k].sum()), (k, l1, int(ref[k].sum()))
    for a, b in zip(ref["hist"], got["hist"]):
        assert int(np.abs(a.astype(np.int64) - b).sum()) <= 20 + 0.02 * int(a.sum())
