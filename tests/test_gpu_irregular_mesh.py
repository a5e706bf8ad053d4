"""Residuals on mesh arrays that list a face twice in a cell, in one of its
cells only, or between a cell and itself (runs on an MI355X): each cell sums
the fluxes of its own slots, here slot by slot from the Riemann operator. Two
orders of at most four terms differ by a few units in the last place."""
import numpy as np
import pytest

from test_face_lists import IRREGULAR, irregular
from test_gpu_flux_blocks import random_state

pytestmark = pytest.mark.gpu


def slot_by_slot(mlr, a, U):
    f, cof = a["faces_of_cell"].astype(int), a["cells_of_face"]
    xy, nof, noc = a["node_coords"].reshape(-1, 2), a["nodes_of_face"].reshape(-1, 2), a["nodes_of_cell"].reshape(-1, 4)
    n_cells = len(f)
    corner = xy[noc]
    center = corner.mean(1)
    d1, d2 = corner[:, 2] - corner[:, 0], corner[:, 3] - corner[:, 1]
    vol = 0.5 * np.abs(d1[:, 0] * d2[:, 1] - d1[:, 1] * d2[:, 0])
    e = xy[nof[:, 1]] - xy[nof[:, 0]]
    area = np.hypot(e[:, 0], e[:, 1])
    n = np.stack([e[:, 1], -e[:, 0]], 1) / area[:, None]
    mid = 0.5 * (xy[nof[:, 0]] + xy[nof[:, 1]])
    n[((mid - center[cof[:, 0]]) * n).sum(1) < 0] *= -1.0
    rho = U[:, 0]
    u, v = U[:, 1] / rho, U[:, 2] / rho
    ee = U[:, 3] / rho - 0.5 * (u * u + v * v)
    p = 0.4 * rho * ee
    P = np.stack([rho, u, v, p, np.full(n_cells, 1.4), ee + p / rho], 1)
    cell = np.repeat(np.arange(n_cells), 4)
    face = f.ravel()
    bnd = cof[face, 1] < 0
    side = ~bnd & (cof[face, 1] == cell)
    left, right = P[cof[face, 0]].copy(), P[np.where(bnd, cof[face, 0], cof[face, 1])].copy()
    un = (left[:, 1:3] * n[face]).sum(1)
    right[bnd, 1:3] = (left[:, 1:3] - 2.0 * un[:, None] * n[face])[bnd]
    F = mlr.riemann_flux("Rusanov", n[face], left, right)
    r = np.where(side, 1.0, -1.0)[:, None] * area[face][:, None] * F
    return r.reshape(n_cells, 4, 4).sum(1) / vol[:, None]


@pytest.mark.parametrize("how,nx,ny", IRREGULAR)
def test_residual(mlr, oracle, how, nx, ny):
    a = irregular(oracle, how, nx, ny)
    s = mlr.Solver(mesh=a, num=mlr.numerics(recon="FO", riemann="Rusanov", p_ref=1.0, T_ref=1.0 / 287.0, rho_ref=1.0))
    U = random_state(nx * ny, nx + ny)
    want = slot_by_slot(mlr, a, U)
    for block in (64, 128, 256):
        s.set_tune(0, block, 256)
        assert np.abs(s.calc_rhs_of(U) - want).max() <= 1e-12 * np.abs(want).max()
