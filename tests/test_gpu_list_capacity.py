"""The one-call evaluation of a configuration whose lists do not fit what the context holds: its
launches go on with the clusters that fit, in bounds, and the evaluation is repeated with larger
buffers, or refused where a neighbour row is full.

* One dimer too many and more (72 waters, whose dimers lie about the first capacity of 1536), and
  several times as many dimers and trimers (waters spread over the cell, then drawn together):
  the results of a context that never held another configuration, bit for bit.
* More than 128 O-O partners: an error, and the context's next evaluation is as before.
"""
import importlib
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    return importlib.import_module("dlpoly2-mbpol-heat_amd.engine")


def same(a, b):
    (ra, sa), (rb, sb) = a, b
    assert ra["eng"] == rb["eng"] and ra["vir"] == rb["vir"] and np.array_equal(ra["jtot"], rb["jtot"])
    assert np.array_equal(sa.forces(), sb.forces())
    for u, v in zip(sa.ctx.decomposition(), sb.ctx.decomposition()):
        assert np.array_equal(u, v)


def compact(box, size):
    """The box's waters, whole, on a lattice inside a cube of this size in the same cell."""
    nw, L = box.nw, box.L
    x = box.xyz[:3 * nw].reshape(nw, 3, 3).copy()
    d = x[:, 1:] - x[:, :1]
    d -= L * np.round(d / L)
    n = math.ceil(nw ** (1.0 / 3.0) - 1e-9)
    g = np.array([(i, j, k) for i in range(n) for j in range(n) for k in range(n)][:nw], float)
    x[:, 0] = 1.0 + g * (size / n)
    x[:, 1:] = x[:, :1] + d
    wb = importlib.import_module("dlpoly2-mbpol-heat_amd.waterbox")
    xyz = box.xyz.copy()
    xyz[:3 * nw] = x.reshape(-1, 3)
    return wb.WaterBox(nw, L, xyz, box.vel, box.mass, box.listttm2)


def test_dimers_about_the_first_capacity(pkg, waterbox, engine):
    L = (72 / waterbox.RHO_WATER) ** (1.0 / 3.0)
    boxes = [waterbox.make_waterbox(72, L, 5, seed) for seed in (23501, *range(33000, 33014))]
    slot = engine.Slot(boxes[0])
    over = 0
    for b in boxes:
        slot.load(b)
        r = slot.evaluate()
        over += len(slot.ctx.lists()[0]) > 1536
        fresh = engine.Slot(b)
        rf = fresh.evaluate()
        same((r, slot), (rf, fresh))
        fresh.close()
    print("configurations past 1536 dimers:", over, flush=True)
    assert over and len(boxes) - over > 1


def test_many_times_the_clusters(pkg, waterbox, engine):
    sparse = waterbox.make_waterbox(216, 30.0, 6, seed=3)
    dense = compact(sparse, 18.0)
    slot = engine.Slot(sparse)
    few = [slot.evaluate() for _ in range(3)][-1]
    n2, n3 = (len(a) for a in slot.ctx.lists())
    f = slot.forces()
    for _ in range(3):
        slot.load(dense)
        r = slot.evaluate()
        m2, m3 = (len(a) for a in slot.ctx.lists())
        assert m2 > 1536 and m3 > 1536 and n2 < 1536 and n3 < 1536
        fresh = engine.Slot(dense)
        same((r, slot), (fresh.evaluate(), fresh))
        fresh.close()
        slot.load(sparse)
        assert slot.evaluate()["eng"] == few["eng"] and np.array_equal(slot.forces(), f)


def test_full_neighbour_rows_are_an_error(pkg, waterbox, engine):
    sparse = waterbox.make_waterbox(343, 26.0, 7, seed=4)
    dense = compact(sparse, 10.5)                     # 1.5 A apart
    slot = engine.Slot(sparse)
    for _ in range(2):
        slot.evaluate()
    e, f = slot.evaluate()["eng"], slot.forces()
    for _ in range(2):
        slot.load(dense)
        with pytest.raises(pkg.MbgpuError, match="neighbour list capacity"):
            slot.evaluate()
        slot.load(sparse)
        assert slot.evaluate()["eng"] == e and np.array_equal(slot.forces(), f)
