"""States of the temporal-blocked solve that a program reaches by chance or after hours, bit for bit
against the oracle (zero tolerance: the same float32 operations in the same order): 16-sweep tiles
handed out from one queue because an XCD did not start (their K streams then cross the XCDs' L2s),
the solve's number passing the range of its tags, and a sweep count that changes from step to
step, so that every solve plans its layout anew."""
import ctypes

import numpy as np
import pytest

from fluid_amd import Fluid, FluidBatch
from oracle.pyoracle import OracleFluid

pytestmark = pytest.mark.gpu


def state(w, h, scale=0.5):
    rng = np.random.default_rng([w, h, 2])
    shape = (w + 2, h + 2)
    st = {"S": (rng.random(shape) >= 0.03).astype(np.float32)}
    for k in ("U", "V", "newU", "newV"):
        st[k] = (scale * rng.standard_normal(shape)).astype(np.float32)
    return st


def far(f, on=1, number=0):
    fn, h = (f._L.fl_test_batch_solve, f._b) if isinstance(f, FluidBatch) else (f._L.fl_test_solve, f._ctx)
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int]
    assert fn(h, on, number) == 0


def same(g, o):
    assert g.stats()["sweeps_run"] == o.last_sweeps()
    for k in ("U", "V", "p"):
        assert np.array_equal(g.get(k).view(np.uint32), o.get(k).view(np.uint32)), k


# scale 3e-5: the early exit keeps some of the sweeps and runs them again
@pytest.mark.parametrize("w,h,sweeps,scale", [(62, 7, 5, 0.5), (150, 41, 40, 0.5), (150, 41, 40, 3e-5), (513, 300, 100, 0.5),
                                              (1200, 900, 48, 0.5)])
@pytest.mark.parametrize("blk", [4, 8])
def test_tiles_from_one_queue(w, h, sweeps, scale, blk):
    g, o = Fluid(1000.0, w, h, 0.01), OracleFluid(1000.0, w, h, 0.01, threads=8)
    g.Solver, g.BlockSweeps, g.BlockCols = 2, 16, blk
    for f in (g, o):
        f.load_state(state(w, h, scale))
        f.PressureIters = sweeps
    for step, on in enumerate((1, 0, 1)):  # and from the XCDs' queues in between, on the same words
        far(g, on)
        g.Simulate(0.1)
        o.Simulate(0.1)
        if scale < 0.1 and step == 0:
            assert 1 < o.last_sweeps() < sweeps
        same(g, o)
    g.close()


@pytest.mark.parametrize("graph", [False, True])
def test_batch_tiles_from_one_queue(graph):
    sizes, scales = [(150, 41), (40, 30), (300, 200)], [3e-5, 0.5, 0.5]
    b = FluidBatch(1000.0, sizes, 0.01)
    b.PressureIters, b.BlockSweeps = 40, 16
    b.set_graph(graph)
    oracles = []
    for m, (w, h), sc in zip(b.members, sizes, scales):
        oracles.append(OracleFluid(1000.0, w, h, 0.01))
        for f in (m, oracles[-1]):
            f.load_state(state(w, h, sc))
            f.PressureIters = 40
    for on in (1, 1, 0, 1):
        far(b, on)
        b.update(0.1)
        for m, o in zip(b.members, oracles):
            o.update(0.1)
            same(m, o)
    b.close()


@pytest.mark.parametrize("tk", [4, 8, 16])
@pytest.mark.parametrize("scale", [0.5, 3e-5])
def test_tags_repeat(tk, scale):
    """Solve 32768 has the tag 0 that the cleared words carry, the next ones those of the first
    solves; 65536 the same again, at the end of the tag's other half."""
    w, h, sweeps = 150, 41, 40
    g, o = Fluid(1000.0, w, h, 0.01), OracleFluid(1000.0, w, h, 0.01)
    g.Solver, g.BlockSweeps = 2, tk
    for f in (g, o):
        f.PressureIters = sweeps
    for number in (0, 0, 32766, 0, 0, 0, 0, 65535, 0, 0):
        if number:
            far(g, 0, number)
        for f in (g, o):
            f.load_state(state(w, h, scale))
            f.Simulate(0.1)
        same(g, o)
    g.close()


@pytest.mark.parametrize("tk", [0, 8, 16])
def test_sweep_count_changes(tk):
    w, h = 150, 141
    g, o = Fluid(1000.0, w, h, 0.01), OracleFluid(1000.0, w, h, 0.01)
    b = FluidBatch(1000.0, [(20, 30), (w, h)], 0.01)
    b.set_graph(True)
    g.Solver, g.BlockSweeps, b.BlockSweeps = 2, tk, tk
    for f in (g, o, b.members[1]):
        f.load_state(state(w, h))
    for sweeps in (8, 40, 8, 7, 41, 40, 8, 100, 1, 8):
        g.PressureIters = o.PressureIters = b.PressureIters = sweeps
        for f in (g, o, b):
            f.update(0.1)
        same(g, o)
        same(b.members[1], o)
    b.close()
    g.close()
