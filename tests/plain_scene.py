"""Engine scenes on made-up tables, for tests that need no physics data: the
cross sections are smooth in energy and of the right size, nothing more."""

import numpy as np

from ggems_amd.engine import Engine

F = np.float32
SOURCE_AT = np.array([[0, 0, -1, -600], [0, 1, 0, 0], [1, 0, 0, 0], [0, 0, 0, 1]], F)
PANEL_AT = np.array([[0, 0, 1, 400], [0, 1, 0, 0], [-1, 0, 0, 0], [0, 0, 0, 1]], F)


def tables(n_mat, nbins=64):
    e = np.exp(np.linspace(np.log(1e-3), 0.0, nbins)).astype(F)
    dens = np.linspace(0.3, 2.0, n_mat)
    dens[-1] = 8.0  # the detector's
    k = e.astype(np.float64) * 1e3
    cs = np.stack([np.outer(dens, 0.03 / (1 + k / 200)), np.outer(dens, 600.0 / k ** 3),
                   np.outer(dens, 6.0 / k ** 2 / (1 + 1 / k))]).astype(F)
    pp = np.zeros((9, 101), F)
    pp[:, 1:] = np.array([0.6, 0.3, 0.1, 2.0, 0.3, 0.04, 3.0, 4.0, 5.0], F)[:, None]
    return dict(energy_bins=e, cross_sections=cs, cs_atom_rayleigh=np.ones((101, nbins), F),
                n_elements=[1] * n_mat, element_index=[0] * n_mat, atomic_number=[8], atom_density=[1.0],
                photon_cut=[1e-3] * n_mat, density=list(dens * 6.24e18), rayleigh_pp=pp, rayleigh_factor=3252.7,
                process_ids=(0, 1, 2))


def engine(n_mat, nbins=64):
    eng = Engine(0)
    eng.set_physics(**tables(n_mat, nbins))
    return eng


def add_voxels(eng, labels, voxel, matrix=None):
    nz, ny, nx = labels.shape
    half = np.array([nx, ny, nz]) * np.asarray(voxel) / 2
    return eng.add_voxel_solid(np.eye(4) if matrix is None else matrix, -half, half, labels, voxel, 0)


def add_panel(eng, rows, cols, pixel, material, matrix=PANEL_AT):
    size = np.array([rows * pixel, cols * pixel, 1.0])
    return eng.add_box_solid(matrix, -size / 2, size / 2, (rows, cols, 1), size, 10e-3, material, True)


def add_source(eng, aperture=0.1, energy=0.06):
    eng.set_xray_source(SOURCE_AT, aperture, (0.0, 0.0, 0.0), np.array([energy, energy], F), np.array([0, 1], F),
                        False)
