"""The temporal-blocked solve at the edges of its tiles, bit for bit against the oracle: grids of
one cell, one lane more or less than a 64-row tile and one column more or less than a block of
columns; sweep counts that do not fill a tile or a wave's pair of sweeps; blocks of cells with all
neighbours, walls only and scattered solids; the multigrid's coarse solve on the same tiles; the parameters that need the selecting update
(damping, negative relaxation and dt); faces that are infinite or NaN. The tolerance is zero: the
solve performs the oracle's float32 operations in the oracle's order (NaN compares by position)."""
import numpy as np
import pytest

from fluid_amd import Fluid, FluidBatch
from oracle.pyoracle import OracleFluid

pytestmark = pytest.mark.gpu


def run(w, h, sweeps, tk, blk, solid=0.03, early=False, dt=0.1, special=False, steps=2, **knobs):
    rng = np.random.default_rng([w, h, sweeps])
    shape = (w + 2, h + 2)
    st = {"S": (rng.random(shape) >= solid).astype(np.float32)}
    st["S"][0, :] = 0
    for k in ("U", "V", "newU", "newV"):
        st[k] = (0.5 * rng.standard_normal(shape)).astype(np.float32)
    if special:
        for k, v in (("U", np.inf), ("V", -np.inf), ("U", np.nan), ("V", 1e-42), ("U", -0.0)):
            st[k][tuple(rng.integers(0, n) for n in shape)] = v
    g, o = Fluid(1000.0, w, h, 0.01), OracleFluid(1000.0, w, h, 0.01)
    for f in (g, o):
        f.load_state(st)
        f.PressureIters, f.EarlyExit = sweeps, early
        for k, v in knobs.items():
            setattr(f, k, v)
    g.Solver, g.BlockSweeps, g.BlockCols = 2, tk, blk
    for step in range(steps):
        g.Simulate(dt)
        o.Simulate(dt)
        for k in ("U", "V", "p"):
            a, b = g.get(k), o.get(k)
            bad = (a.view(np.uint32) != b.view(np.uint32)) & ~(np.isnan(a) & np.isnan(b))
            assert not bad.any(), "step %d: %s differs at %d cells, first %s" % (
                step, k, int(bad.sum()), np.argwhere(bad)[0])
    g.close()


@pytest.mark.parametrize("tk,blk", [(tk, blk) for tk in (0, 2, 4, 8, 16) for blk in (4, 8)])
@pytest.mark.parametrize("w,h,sweeps", [(1, 1, 1), (1, 9, 3), (62, 7, 5), (63, 8, 16), (65, 17, 19), (130, 33, 33)])
def test_edges_of_tiles(w, h, sweeps, tk, blk):
    run(w, h, sweeps, tk, blk)


@pytest.mark.parametrize("tk,blk", [(2, 8), (4, 4), (8, 8), (16, 8)])
@pytest.mark.parametrize("case", [dict(solid=0.0), dict(solid=0.5), dict(PressureDamping=0.75),
                                  dict(Relaxation=-0.5), dict(dt=-0.05), dict(early=True, solid=0.9),
                                  dict(special=True, steps=1)], ids=str)
def test_cells_and_parameters(case, tk, blk):
    run(150, 41, 21, tk, blk, **case)


@pytest.mark.parametrize("w,h", [(3, 3), (4, 130), (122, 12), (126, 30), (130, 31), (3300, 3900)])
@pytest.mark.parametrize("solid", [0.0, 0.05])
def test_multigrid_coarse_tiles(w, h, solid):
    """Coarse interiors of one cell, one row more or less than a tile, and (the last) more than
    256 tiles of four sweeps in flight, so tiles of eight."""
    run(w, h, 1, 0, 0, solid=solid, steps=2 if w < 1000 else 1, UseMultigrid=True)


@pytest.mark.parametrize("w,h,early", [(1022, 1021, False), (1022, 1022, False), (1022, 1022, True), (4094, 255, False),
                                       (90, 12001, False)])
def test_turbulence_with_the_solve(w, h, early):
    """From 2^20 cells the solve's last kernel adds the turbulence; (1022, 1021) is the largest below.
    early: with a tolerance met after some sweeps the result is the re-run's."""
    run(w, h, 5, 0, 0, early=early, solid=0.9 if early else 0.05)


def test_turbulence_with_a_batch_solve():
    """Members that alone stay below 2^20 cells, together above; and each on its own."""
    sizes = [(800, 798), (631, 700), (5, 7)]
    b = FluidBatch(1000.0, sizes, 0.01)
    alone = [Fluid(1000.0, w, h, 0.01) for w, h in sizes]
    for e, (m, f) in enumerate(zip(b.members, alone)):
        rng = np.random.default_rng(e)
        shape = (sizes[e][0] + 2, sizes[e][1] + 2)
        st = {"S": (rng.random(shape) >= 0.05).astype(np.float32)}
        for k in ("U", "V", "newU", "newV"):
            st[k] = (0.5 * rng.standard_normal(shape)).astype(np.float32)
        m.load_state(st)
        f.load_state(st)
        f.PressureIters = 9
    b.PressureIters = 9
    for step in range(2):
        b.update(0.1)
        for f in alone:
            f.update(0.1)
        for e, (m, f) in enumerate(zip(b.members, alone)):
            for k in ("U", "V", "p", "M"):
                assert np.array_equal(m.get(k).view(np.uint32), f.get(k).view(np.uint32)), (step, e, k)
    b.close()
