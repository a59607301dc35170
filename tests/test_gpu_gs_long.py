"""The temporal-blocked solve on grids at the lengths where its handoff words pass 4 GB, bit for bit
against the oracle. A tile of 64 rows writes 1 KB of words a column, so its words lie beyond
32-bit byte offsets from column 2^22 on, and its buffers begin anew after every 2^16 blocks of columns: one row-tile with three blocks of sweeps, two row-tiles
(63 sweeps on one interior row), a batch member, and the other way round a grid of more than
2^15 row-tiles. The tolerance is zero: the oracle's float32 operations in the oracle's order."""
import numpy as np
import pytest

from fluid_amd import Fluid, FluidBatch
from oracle.pyoracle import OracleFluid

pytestmark = pytest.mark.gpu

LONG = (1 << 22) + 300


def state(w, h):
    rng = np.random.default_rng([w, h])
    shape = (w + 2, h + 2)
    st = {"S": (rng.random(shape, dtype=np.float32) >= 0.03).astype(np.float32)}
    st["S"][0, :] = 0
    for k in ("U", "V"):
        st[k] = rng.random(shape, dtype=np.float32) - 0.5
    return st


def compare(g, o):
    for k in ("U", "V", "p"):
        a, b = g.get(k), o.get(k)
        bad = a.view(np.uint32) != b.view(np.uint32)
        assert not bad.any(), "%s differs at %d cells, first %s" % (k, int(bad.sum()), np.argwhere(bad)[0])


@pytest.mark.parametrize("w,h,sweeps,tk,blk", [(1, LONG, 5, 2, 8), (1, LONG, 63, 16, 8), (64 * ((1 << 15) + 3), 1, 5, 0, 8),
                                               (63, (1 << 18) - 70, 21, 8, 4), (3, (1 << 19) + 1, 64, 4, 8)])
def test_long_grids_bit_exact(w, h, sweeps, tk, blk):
    st = state(w, h)
    g, o = Fluid(1000.0, w, h, 0.01), OracleFluid(1000.0, w, h, 0.01, threads=8)
    g.Solver, g.BlockSweeps, g.BlockCols = 2, tk, blk
    for f in (g, o):
        f.load_state(st)
        f.PressureIters, f.EarlyExit = sweeps, False
        f.Simulate(0.1)
    compare(g, o)
    g.close()


def test_long_batch_member_bit_exact():
    sizes = [(1, LONG), (5, 7)]
    b = FluidBatch(1000.0, sizes, 0.01)
    b.PressureIters = 3
    for m, (w, h) in zip(b.members, sizes):
        m.load_state(state(w, h))
    b.update(0.1)
    for m, (w, h) in zip(b.members, sizes):
        o = OracleFluid(1000.0, w, h, 0.01, threads=8)
        o.load_state(state(w, h))
        o.PressureIters = 3
        o.update(0.1)
        compare(m, o)
    b.close()
