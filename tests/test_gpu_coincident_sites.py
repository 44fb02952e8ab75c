"""A 2-body leaf whose monomer has its hydrogens at one point: the distance is 0 there, the
variable and the energy finite (its direction, and with it the gradient, is not defined).

Bar as the golden leaves: 1e-15 of the polynomial's cancellation scale.
"""
import numpy as np
import pytest

import oracle_lib as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("second", [False, True])
def test_energy_of_coincident_hydrogens(pkg, golden, second):
    n = 0
    for w in golden["d_w"]:
        w = w.copy()
        if np.linalg.norm(w[:3] - w[9:12]) > 6.5:
            continue
        k = 9 * second
        w[k + 6:k + 9] = w[k + 3:k + 6]
        e, _ = o.leaf_2b(w[:9], w[9:])
        assert np.isfinite(e)
        g, _, _ = pkg.mbpol_2b_poly(w[:9], w[9:], np.zeros(9), np.zeros(9))
        assert abs(g - e) <= 1e-15 * o.poly_scale(2, o.vars_2b(w[:9], w[9:]))
        n += 1
    assert n
