"""Sites without a polarizability that are given a start dipole: ewald1p.f leaves their dipoles
out of the reciprocal sums, the solver leaves them as they are and the real-space pair terms
take them.  The oxygens alone polarizable, then the hydrogens alone, from random start dipoles
on every real site; both solvers.  (Not compared: the reciprocal stress of such a site itself,
in which the library has no dipole either and the oracle has it.)

Bars as test_gpu_elec.compare: both sides sum the same terms in FP64, in different orders.
"""
import importlib

import numpy as np
import pytest

import oracle_lib as o
from test_gpu_elec import compare, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("polr2", [(1.310, 0.0, 0.0), (0.0, 0.294, 0.0)])
@pytest.mark.parametrize("nw", [5, 43])
def test_start_dipoles_of_unpolarizable_sites(pkg, waterbox, nw, polr2):
    ep = importlib.import_module("dlpoly2-mbpol-heat_amd.elec_params")
    box = waterbox.make_waterbox(nw, 12.42, 4, seed=200 + nw)
    p = ep.ElecParams(rcut=5.5, alpha=0.5, kmax=(9, 8, 10), max_iter=2000, polr2=polr2)
    dip = np.zeros((4 * nw, 3))
    dip[:3 * nw] = 0.05 * np.random.default_rng(nw).normal(size=(3 * nw, 3))
    r = o.elec_forces(box, p, dip0=dip)
    fixed = np.arange(3 * nw) % 3 != 0 if polr2[1] == 0.0 else np.arange(3 * nw) % 3 == 0
    _, g = run_gpu(pkg, box, p, dip=dip)
    g["s_ew1p"][fixed] = r["s_ew1p"][fixed]
    compare(g, r)
    assert np.array_equal(g["dip"][:3 * nw][fixed], dip[:3 * nw][fixed])
    p.solver = 1
    _, g = run_gpu(pkg, box, p, dip=dip)
    g["s_ew1p"][fixed] = r["s_ew1p"][fixed]
    compare(g, dict(r, niter=g["niter"]))            # (the solvers take different counts)
