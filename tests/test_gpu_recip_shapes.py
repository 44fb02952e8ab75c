"""The matrix passes of the Ewald sum over k against the oracle, at the k lists and site counts
where their tiles end: one n, less than a tile of 8 n, one past a tile, more than the four tiles
a block takes at a time; a partly filled group of 16 (l, m) pairs; sites that do not fill a
step of 4 or a tile of 16; unequal and triclinic cells, whose runs of n are not symmetric.

Bars as test_gpu_elec.compare: both sides sum the same terms in FP64, in different orders.
"""
import importlib

import numpy as np
import pytest

import oracle_lib as o
from test_gpu_elec import compare, run_gpu

pytestmark = pytest.mark.gpu

CASES = [
    # waters, cell vectors, imcon, kmax
    (1, (12.42, 12.42, 12.42), 1, (1, 1, 1)),
    (3, (12.42, 12.42, 12.42), 1, (3, 3, 2)),
    (5, (12.42, 12.42, 12.42), 1, (8, 8, 8)),
    (11, (12.42, 12.42, 12.42), 1, (9, 9, 9)),
    (16, (12.42, 12.42, 12.42), 1, (7, 10, 17)),
    (22, (12.42, 13.5, 62.0), 2, (8, 9, 41)),
    (13, (62.0, 12.42, 12.42), 2, (40, 8, 8)),
    (43, (14.0, 13.0, 15.0), 3, (9, 8, 10)),
]


@pytest.mark.parametrize("nw,edges,imcon,kmax", CASES)
def test_k_list_shapes(pkg, waterbox, nw, edges, imcon, kmax):
    ep = importlib.import_module("dlpoly2-mbpol-heat_amd.elec_params")
    box = waterbox.make_waterbox(nw, 12.42, 4, seed=100 + nw)
    box.imcon = imcon
    cell = np.diag(edges).astype(float)
    if imcon == 3:
        cell[1, 0], cell[2, 0], cell[2, 1] = 1.7, -2.1, 1.3
    box.cell = cell.reshape(9)
    # the k lists are compared as they are, converged or not
    p = ep.ElecParams(rcut=5.5, alpha=0.5, kmax=kmax, max_iter=2000)
    r = o.elec_forces(box, p)
    _, g = run_gpu(pkg, box, p)
    compare(g, r)
    p.solver = 1
    _, g = run_gpu(pkg, box, p)
    r = dict(r, niter=g["niter"])            # (the solvers take different counts)
    compare(g, r)
