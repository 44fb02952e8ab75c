"""max_iter in a context whose earlier solves took many iterations (and which enqueues as many at
once): a solve that needs more than the limit, rounded up to the batch that reaches it (64, then
8 at a time), is an error, as in a context that solves for the first time; one within the limit
is the same solve as before.  The parts called one by one and the complete evaluation in one
call, with graph replay and without.
"""
import dataclasses
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("graphs", [False, True])
def test_lower_limit_in_a_warm_context(pkg, waterbox, fused, graphs):
    engine = importlib.import_module("dlpoly2-mbpol-heat_amd.engine")
    box = waterbox.box_64()
    # (omega: the weight of the old dipole; a heavier one takes more iterations)
    e = dataclasses.replace(pkg.elec_params.for_box(box.L), omega=0.7, max_iter=2000)
    s = engine.Slot(box, solver=0, elec=e, fused=fused)
    s.ctx.set_graphs(graphs)
    for _ in range(3):
        r = s.evaluate()
    n = r["dipole_iterations"]
    assert n > 100
    f = s.forces()
    reach = lambda limit: 64 + 8 * ((max(limit - 64, 0) + 7) // 8)     # iterations done at the limit
    for limit in (10, 64, 65, n - 20, n - 8, n - 1, n):
        print(f"{n} iterations, max_iter {limit}, one call {fused}, graphs {graphs}", flush=True)
        s.set_params(dataclasses.replace(e, max_iter=limit), pkg.water_params.for_box(box.L))
        if reach(limit) < n:
            with pytest.raises(pkg.MbgpuError, match="did not converge in"):
                s.evaluate()
        else:
            assert s.evaluate()["dipole_iterations"] == n and np.array_equal(s.forces(), f)
    assert reach(n - 8) < n <= reach(n)
