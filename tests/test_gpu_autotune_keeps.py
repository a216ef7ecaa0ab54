"""The autotuner times the tuning in force too: it stays where no candidate fits the grid (4 cells a
side) and where it is the fastest, tiles of 64 cells are among the candidates of FP32 grids, and
whatever is kept, the run goes on as if it had not been tuned."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib  # noqa: E402
from test_gpu_default_tuning import case  # noqa: E402


def test_grid_below_every_candidate():
    cfg, parts = case(4, 4, 500, _lib.PIC_FP32, 0.05, 1)
    with Simulation(cfg) as sim:
        sim.set_particles(*parts)
        t = sim.tuning()
        ms = sim.autotune(8)
        assert 0.0 < ms < 10.0 and sim.tuning() == t


@pytest.mark.parametrize("precision,n,m", [(_lib.PIC_FP32, 64, 30_000), (_lib.PIC_FP64, 128, 30_000),
                                           (_lib.PIC_FP32, 8, 1000)])
def test_run_goes_on(precision, n, m):
    cfg, parts = case(n, n, m, precision, 0.05, 2)
    out = []
    for tuned in (False, True):
        with Simulation(cfg) as sim:
            sim.set_particles(*parts)
            sim.step(5)
            if tuned:
                sim.autotune(4)
            sim.step(12)
            sim.sync()
            out.append(sim.particles(sync=False) + (sim.diagnostics(0, 17)[:, 0],))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_batch_goes_on():
    runs = [case(32, 32, 5000, _lib.PIC_FP32, 0.05, 3), case(4, 8, 300, _lib.PIC_FP32, 0.05, 4)]
    out = []
    for tuned in (False, True):
        with Batch([c for c, _ in runs]) as b:
            for k, (_, p) in enumerate(runs):
                b.set_particles(*p, run=k)
            if tuned:
                b.autotune(4)
            b.step(9)
            b.sync()
            out.append([v for k in range(2) for v in b.particles(run=k, sync=False)])
    for a, c in zip(*out):
        assert np.array_equal(a, c)


def test_not_slower_than_the_default():
    """1024^2 FP32, whose default takes tiles of 64 cells: a tenth is left for timing noise."""
    cfg, parts = case(1024, 1024, 4_000_000, _lib.PIC_FP32, 0.01, 5)

    def per_step(sim):
        best = 1e9
        for _ in range(5):
            sim.sync()
            t = time.perf_counter()
            sim.step(48)
            sim.sync()
            best = min(best, time.perf_counter() - t)
        return best

    with Simulation(cfg) as sim:
        sim.set_particles(*parts)
        sim.step(48)
        default = per_step(sim)
        sim.autotune(8)
        sim.step(48)
        assert per_step(sim) <= 1.1 * default
