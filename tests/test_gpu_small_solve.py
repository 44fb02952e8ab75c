"""The solve of the dipoles of an isolated cluster, at the sizes where its kernels change or end:
one launch holds up to 21 waters (63 rows of 16 lanes, 7 waters to a wavefront, so 1, 7, 8, 21),
22 take the launches per iteration, and rows with room for 512 partners and more (4 sites a water,
rounded up to 64: 112 waters 448, 113 waters 512) are shared by four wavefronts.  The pair and per-water passes run at the same odd counts.

Bars as test_gpu_cluster: both sides sum the same terms in FP64 in different orders, the solves
stop below the same RMS step.
"""
import numpy as np
import pytest

import oracle_lib as o
from test_gpu_cluster import rel
from test_gpu_elec import run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw", [1, 2, 7, 8, 21, 22, 112, 113, 129])
def test_cluster_sizes(pkg, waterbox, nw):
    box = waterbox.make_cluster(nw, seed=5)
    p = pkg.elec_params.for_cluster(box.L)
    p.max_iter = 2000
    p.solver = 1
    r = o.elec_forces(box, p)
    ctx, g = run_gpu(pkg, box, p)
    scale = abs(r["eng_ew2p"]) + abs(r["eng_polar"])
    assert abs(g["eng"] - r["eng"]) <= 1e-10 * scale
    for k in ("stress", "dip", "vesp", "f", "atomic_energy", "heat_w"):
        assert rel(g[k], r[k]) <= 1e-10, k
    # again in the same context: the iterations of the first call came a few to a launch, with
    # the vectors passed on in between; the same operations in the same order
    _, h = run_gpu(pkg, box, p, ctx=ctx)
    assert h["niter"] == g["niter"]
    assert np.array_equal(h["dip"], g["dip"]) and np.array_equal(h["f"], g["f"])
    # and from the converged dipoles: no iteration is needed
    _, h = run_gpu(pkg, box, p, ctx=ctx, dip=g["dip"])
    assert h["niter"] <= 1 and rel(h["dip"], g["dip"]) <= 1e-10
