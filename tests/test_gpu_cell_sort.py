"""The engine's cell sort where its kernels change: cells at and one past the size ranked by
counting (512) and past the one sorted in LDS (4096), cells that span several of the ordering
kernel's 1024-slot workgroups, a particle count just past a 4096-particle chunk, grids whose
neighbouring tiles' cell numbers lie far apart, and a few particles on many cells.  Whole DSMC
steps against the oracle's composition (cells ordered by key, then id), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from test_gpu_collide_engine import engine_run, oracle_run  # noqa: E402


def clumps(nx, ny, sizes, background, seed):
    """`sizes` cold particles at the centres of scattered cells, the rest spread out."""
    rng = np.random.default_rng(seed)
    cells = rng.choice(nx * ny, len(sizes), replace=False)
    x = [np.full(m, c // ny + 0.5) for m, c in zip(sizes, cells)]
    y = [np.full(m, c % ny + 0.5) for m, c in zip(sizes, cells)]
    x = np.concatenate(x + [rng.uniform(0, nx, background)])
    y = np.concatenate(y + [rng.uniform(0, ny, background)])
    p = rng.permutation(x.size)
    cfg = _lib.default_config(nx=nx, ny=ny, lx=float(nx), ly=float(ny), dt=0.2, qm=-1.0,
                              precision=_lib.PIC_FP32, seed=seed,
                              collide=_lib.PIC_COLLIDE_DSMC, dsmc_coeff=2e-5, dsmc_gmax0=1.0,
                              capacity=x.size)
    cfg.qp = -1e-6 * nx * ny / x.size
    v = rng.normal(0, 0.3, (2, x.size))
    return cfg, (x[p], y[p], v[0], v[1])


@pytest.mark.parametrize("nx,ny,sizes,background,tiling", [
    (32, 32, (511, 512, 513, 1, 1024, 1025), 4000, None),
    (64, 16, (4095, 4096, 4097, 700), 1000, (8, 4, 0, 1)),
    (256, 256, (5000, 600, 40), 90_000, (16, 8, 0, 1)),
    (512, 256, (300,), 40_000, (8, 4, 0, 1)),
    (16, 16, (8191,), 2, None),
    (128, 128, (), 4097, (32, 8, 0, 1)),
    (64, 64, (), 1, None)])
def test_cells_in_id_order(oracle, nx, ny, sizes, background, tiling):
    print(f"{nx}x{ny} clumps {sizes} + {background}", flush=True)
    cfg, parts = clumps(nx, ny, sizes, background, nx + ny + len(sizes))
    want, counts = oracle_run(oracle, cfg, parts, 3)
    out = engine_run(cfg, parts, 3, tiling=tiling)
    for g, w in zip(out[0], want):
        assert np.array_equal(g, w)
    assert out[1][0] == counts[0]
