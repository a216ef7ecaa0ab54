"""The form of the DSMC push goes by the particles held, not by the capacity: spare capacity changes
nothing, down to the last bit of the diagnostics (whose FP32 partial sums group other particles in
the other form), below and above the line of 16 particles per cell, also when a run is given more or
fewer particles than before, with captured steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Simulation  # noqa: E402
from test_gpu_cell_sort import clumps  # noqa: E402


def rows(cfg, sets, capacity, splits):
    cfg.capacity = capacity
    out = []
    with Simulation(cfg) as sim:
        sim.set_tuning(8, 4, splits, 1)
        for parts in sets:
            sim.set_particles(*parts)
            sim.step(17)
            sim.sync()
            out.append(sim.diagnostics(0, 17))
            out += list(sim.particles(sync=False))
    return out


@pytest.mark.parametrize("splits", [0, 2])
@pytest.mark.parametrize("per_cell", [(5,), (20,), (5, 20, 6)])
def test_spare_capacity_changes_nothing(per_cell, splits):
    sets = []
    for k in per_cell:
        cfg, parts = clumps(64, 64, (), 4096 * k, 100 + k)
        sets.append(parts)
    cfg.dsmc_coeff = 1e-6
    most = 4096 * max(per_cell)
    a = rows(cfg, sets, most, splits)
    b = rows(cfg, sets, 20 * most, splits)
    for u, v in zip(a, b):
        assert np.array_equal(u, v)
    if len(sets) > 1:  # and each set of particles goes as in a context of its own
        for i, parts in enumerate(sets):
            c = rows(cfg, [parts], parts[0].size, splits)
            for u, v in zip(a[5 * i:5 * i + 5], c):
                assert np.array_equal(u, v)
