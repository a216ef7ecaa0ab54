"""The push of cell-ordered particles: shares of the order that start and end inside tiles, span
several tiles, tiles without particles, one cell with most of them; the same particles in items
per tile.  Whole DSMC steps against the oracle: particles bit for bit, and the charge and the
kinetic energy through the steps that follow from them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Simulation  # noqa: E402
from test_gpu_cell_sort import clumps  # noqa: E402
from test_gpu_collide_engine import engine_run, oracle_run  # noqa: E402


@pytest.mark.parametrize("tiling", [None, (8, 3, 3, 1), (4, 5, 1, 1)])
@pytest.mark.parametrize("nx,ny,sizes,background", [
    (16, 16, (), 40_000),
    (16, 32, (30_000, 5000, 900), 20_001),
    (32, 16, (52_000,), 3),
    (64, 64, (1500,) * 8, 300_001),
])
def test_against_oracle(oracle, nx, ny, sizes, background, tiling):
    print(f"{nx}x{ny} clumps {sizes} + {background} tiling {tiling}", flush=True)
    cfg, parts = clumps(nx, ny, sizes, background, nx + 3 * ny + background)
    cfg.dsmc_coeff = 1e-7
    want, counts = oracle_run(oracle, cfg, parts, 3)
    out = engine_run(cfg, parts, 3, tiling=tiling)
    for g, w in zip(out[0], want):
        assert np.array_equal(g, w)
    assert out[1][0] == counts[0]


@pytest.mark.parametrize("nx,ny,sizes,background", [
    (16, 32, (30_000, 5000, 900), 20_001), (64, 64, (1500,) * 8, 300_001)])
def test_diagnostics_of_shares(nx, ny, sizes, background):
    """Kinetic energy and momentum of a step: FP32 sums of at most 4 particles in FP64 sums, so
    each term is off by a few times 2^-24 and the rows of shares and of items per tile agree to
    1e-6; the field energy is of the same charge, word for word."""
    cfg, parts = clumps(nx, ny, sizes, background, nx * ny)
    cfg.dsmc_coeff = 1e-7
    rows = []
    for tiling in (None, (8, 3, 3, 1)):
        with Simulation(cfg) as sim:
            if tiling:
                sim.set_tuning(*tiling)
            sim.set_particles(*parts)
            sim.step(3)
            rows.append(sim.diagnostics(0, 3))
    mp = cfg.qp / cfg.qm
    assert np.allclose(rows[0], rows[1], rtol=1e-6, atol=1e-6 * mp * parts[0].size)
    assert np.array_equal(rows[0][:, 0], rows[1][:, 0])
