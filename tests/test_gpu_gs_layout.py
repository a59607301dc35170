"""The temporal-blocked solve's layout (its handoff buffers and tile lists) from solve to solve: a
layout that does not fit the device is an error each time it is asked for, and leaves nothing
behind: the sweep counts before it run again, bit for bit the oracle's (zero tolerance: the same
float32 operations in the same order). Where only deeper tiles fit, the solve takes those."""
import contextlib

import numpy as np
import pytest
import torch

from fluid_amd import Fluid, FluidBatch
from oracle.pyoracle import OracleFluid

pytestmark = pytest.mark.gpu


def pair(w, h, make=None):
    rng = np.random.default_rng([w, h])
    shape = (w + 2, h + 2)
    st = {"S": (rng.random(shape) >= 0.05).astype(np.float32)}
    for k in ("U", "V", "newU", "newV"):
        st[k] = (0.5 * rng.standard_normal(shape)).astype(np.float32)
    g, o = make or Fluid(1000.0, w, h, 0.01), OracleFluid(1000.0, w, h, 0.01, threads=8)
    for f in (g, o):
        f.load_state(st)
        f.EarlyExit = False
    return g, o


def same(g, o):
    for k in ("U", "V", "p"):
        a, b = g.get(k), o.get(k)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), k


def test_layout_that_does_not_fit():
    """60,000 sweeps of 64 x 64 cells ask for 518 GB of words."""
    g, o = pair(62, 62)
    g.Solver = 2
    for sweeps in (8, 60000, 60000, 8, 5):
        g.PressureIters = o.PressureIters = sweeps
        if sweeps == 60000:
            with pytest.raises(RuntimeError, match="hipMalloc"):
                g.Simulate(0.1)
            continue
        g.Simulate(0.1)
        o.Simulate(0.1)
        same(g, o)
    g.close()


@pytest.mark.parametrize("graph", [False, True])
def test_batch_layout_that_does_not_fit(graph):
    """1024 sweeps of a grid of a million columns ask for 1.1 TB of words."""
    sizes = [(1, 1000000), (30, 20)]
    b = FluidBatch(1000.0, sizes, 0.01)
    oracles = [pair(w, h, m)[1] for m, (w, h) in zip(b.members, sizes)]
    b.EarlyExit = False
    b.set_graph(graph)
    for sweeps in (8, 1024, 1024, 8, 3):
        b.PressureIters = sweeps
        if sweeps == 1024:
            with pytest.raises(RuntimeError, match="hipMalloc"):
                b.update(0.1)
            continue
        b.update(0.1)
        for m, o in zip(b.members, oracles):
            o.PressureIters = sweeps
            o.update(0.1)
            same(m, o)
    b.close()


@contextlib.contextmanager
def device_memory_left(bytes_left):
    """The rest of the device's memory is taken while the block runs."""
    torch.cuda.empty_cache()
    hog = [torch.empty(max(0, torch.cuda.mem_get_info()[0] - bytes_left), dtype=torch.uint8, device="cuda")]
    try:
        yield
    finally:
        hog.clear()
        torch.cuda.empty_cache()


def test_deeper_tiles_where_shallow_ones_do_not_fit():
    """40 sweeps of a million columns: 12 GB of words in the tiles of 4 sweeps that the size picks,
    6.9 GB in tiles of 8, 5.1 GB in tiles of 16."""
    g, o = pair(1, 1000000)
    b = FluidBatch(1000.0, [(1, 1000000)], 0.01)
    m, ob = pair(1, 1000000, b.members[0])
    b.EarlyExit = False
    g.PressureIters = o.PressureIters = b.PressureIters = ob.PressureIters = 40
    with device_memory_left(6 << 30):
        for _ in range(2):
            g.Simulate(0.1)
        assert g.gs_layout()["sweeps_per_tile"] > 4
    for _ in range(2):
        o.Simulate(0.1)
    same(g, o)
    g.close()
    with device_memory_left(6 << 30):
        for _ in range(2):
            b.update(0.1)
        b.sync()
    for _ in range(2):
        ob.update(0.1)
    same(m, ob)
    b.close()
