"""Queued edits reach the device grouped by word, those of a word in call order: calls in ascending
cell order (no sort needed), in descending and in random order with repeated cells, over all fields
that they touch, on a context and on a batch member. Zero tolerance: the same float32 operations
in the same order as the oracle's."""
import numpy as np
import pytest

from fluid_amd import Fluid, FluidBatch
from oracle.pyoracle import OracleFluid

pytestmark = pytest.mark.gpu


def calls(w, h, order, n, seed):
    rng = np.random.default_rng(seed)
    cells = [(int(i), int(j)) for i, j in zip(rng.integers(1, w + 1, n), rng.integers(1, h + 1, n))]
    if order != "random":
        cells.sort(reverse=order == "descending")
    kinds = rng.integers(0, 4, n)
    vals = rng.standard_normal((n, 2)).astype(np.float32)
    return [(int(k), i, j, float(a), float(b)) for k, (i, j), (a, b) in zip(kinds, cells, vals)]


def edit(f, ops):
    for k, i, j, a, b in ops:
        if k == 0:
            f.ApplyForce(i, j, a, b)
        elif k == 1:
            f.SetVelocity(i, j, a, b)
        elif k == 2:
            f.SetSolid(i, j, a < -1.0)
        else:
            f.AddSmoke(i, j, abs(a))


@pytest.mark.parametrize("order", ["ascending", "descending", "random"])
@pytest.mark.parametrize("w,h,n", [(1, 1, 1), (7, 5, 300), (40, 33, 2000)])
def test_edits_in_call_order(w, h, n, order):
    o = OracleFluid(1000.0, w, h, 0.01)
    g = Fluid(1000.0, w, h, 0.01)
    b = FluidBatch(1000.0, [(5, 6), (w, h)], 0.01)
    m = b.members[1]
    for f in (o, g, m):
        for i in range(w + 2):
            for j in range(h + 2):
                f.SetSolid(i, j, False)
    ops = calls(w, h, order, n, [w, h, n])
    for f in (o, g, m):
        edit(f, ops)
    for k in ("U", "V", "newU", "newV", "S", "M"):
        want = o.get(k).view(np.uint32)
        assert np.array_equal(g.get(k).view(np.uint32), want), k
        assert np.array_equal(m.get(k).view(np.uint32), want), k
    # queued again and applied by the step's own batch-wide launch
    again = calls(w, h, order, n, [n, w, h])
    for f in (g, m):
        edit(f, again)
    b.PressureIters = g.PressureIters = 3
    b.update(0.1)
    g.update(0.1)
    for k in ("U", "V", "p", "S", "M"):
        assert np.array_equal(m.get(k).view(np.uint32), g.get(k).view(np.uint32)), k
    b.close()
