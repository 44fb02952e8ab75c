"""No kernel reads an element that it did not write in the same evaluation, on the paths that
test_gpu_engine.test_no_read_of_unwritten_memory does not reach: clusters solved in one launch (up
to 21 waters) and the first one past them, the particle mesh, a box whose sites fill no tile, more
than four tiles of n.  A context on memory filled with NaN gives bit for bit what one on memory
left as it is gives, in the first evaluation and in a replayed one.
"""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def system(pkg, wb, kind):
    if kind.startswith("cluster"):
        b = wb.make_cluster(int(kind[8:]), seed=5)
        return b, pkg.elec_params.for_cluster(b.L), pkg.water_params.for_cluster(b.L), None
    b = wb.box_64() if kind == "mesh" else wb.make_waterbox(43, 12.42, 4, seed=143)
    e = pkg.elec_params.for_box(b.L)
    if kind == "long k list":
        b.imcon, b.cell = 2, np.diag([12.42, 13.5, 62.0]).reshape(9)
        e.kmax = (8, 9, 41)
    return b, e, pkg.water_params.for_box(b.L), ("spme", 6, (32, 32, 32)) if kind == "mesh" else None


@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("kind", ["cluster 1", "cluster 9", "cluster 21", "cluster 22", "mesh", "box", "long k list"])
def test_results_on_memory_full_of_nan(pkg, waterbox, kind, solver, monkeypatch):
    engine = importlib.import_module("dlpoly2-mbpol-heat_amd.engine")
    box, e, w, recip = system(pkg, waterbox, kind)
    out = []
    for poison in ("0", "1"):
        monkeypatch.setenv("MBGPU_POISON", poison)
        print(f"{kind}, solver {solver}, poison {poison}", flush=True)
        s = engine.Slot(box, solver=solver, elec=e, water=w, recip=recip)
        for _ in range(3):
            r = s.evaluate()
            d, t = s.ctx.elec_details(), s.ctx.water_details()
            out.append((poison, [r["eng"], r["vir"], r["stress"], r["jtot"], s.forces(), d["atomic_energy"], d["heat_w"],
                                 d["s_ew1p"], d["vesp"], t["atomic_energy"], t["heat_w"], *s.ctx.decomposition()]))
        s.close()
    want = out[0][1]
    assert all(np.isfinite(a).all() for a in want)
    for poison, got in out[1:]:
        for a, b in zip(want, got):
            assert np.array_equal(a, b), poison
