"""DSMC collisions where the kernel's workgroups change: more first-round candidates than a batch
(1024) in one workgroup's 64 cells, cells that need several rounds, fewer cells than a
workgroup takes, fewer workgroups than counters of accepted pairs (32), more of them, and an
uneven share.  Whole steps against the oracle, bit for bit, with the counts of accepted pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_cell_sort import clumps  # noqa: E402
from test_gpu_collide_engine import engine_run, oracle_run  # noqa: E402


@pytest.mark.parametrize("nx,ny,sizes,background,coeff", [
    (4, 4, (), 3000, 2e-3),               # 16 cells, 200 each
    (16, 16, (), 40_000, 5e-3),           # 160 each: about 4000 candidates per workgroup
    (64, 32, (900, 900, 300), 10_000, 5e-3),  # several rounds in three cells
    (64, 64, (), 30_000, 3e-2),
    (128, 64, (600,) * 12, 60_000, 1e-3),
])
def test_against_oracle(oracle, nx, ny, sizes, background, coeff):
    print(f"{nx}x{ny} clumps {sizes} + {background}, coeff {coeff}", flush=True)
    cfg, parts = clumps(nx, ny, sizes, background, nx * ny + background)
    cfg.dsmc_coeff = coeff
    want, counts = oracle_run(oracle, cfg, parts, 3)
    out = engine_run(cfg, parts, 3)
    for g, w in zip(out[0], want):
        assert np.array_equal(g, w)
    assert counts[0] > 0 and out[1][0] == counts[0]
