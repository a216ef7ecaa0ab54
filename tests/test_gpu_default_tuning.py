"""The default tiling over grid shapes, particle counts and precisions (each branch of its
rule: tiles of 8 to 64 cells, halos cut by small grids, one and many workgroups per tile, both
cadences, a batch's shares): what it picks is legal, and since no tiling changes a trajectory,
a run under it equals the run under small tiles sorted every step, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib  # noqa: E402


def case(nx, ny, n, precision, dt, seed):
    rng = np.random.default_rng(seed)
    cfg = _lib.default_config(nx=nx, ny=ny, lx=12.0, ly=12.0 * ny / nx, dt=dt, qm=-1.0,
                              precision=precision, seed=seed, capacity=n)
    return cfg, (rng.uniform(0, cfg.lx, n), rng.uniform(0, cfg.ly, n), rng.normal(size=n),
                 rng.normal(size=n))


def run(cfg, parts, tuning, steps=10):
    with Simulation(cfg) as sim:
        sim.set_particles(*parts)
        if tuning:
            sim.set_tuning(**tuning)
        t = sim.tuning()
        sim.step(steps)
        sim.sync()
        return t, sim.particles(sync=False)


@pytest.mark.parametrize("precision", [_lib.PIC_FP32, _lib.PIC_FP64])
@pytest.mark.parametrize("nx,ny,n,dt,want", [
    (4, 4, 300, 0.05, dict(tile=2, sort_every=8)), (8, 2048, 5000, 0.001, dict(tile=4)),
    (32, 32, 70_000, 0.05, dict(tile=8, splits=16)), (64, 64, 70_000, 0.05, dict(tile=8, splits=4)),
    (128, 128, 60_000, 0.02, dict(tile=8, halo=8)), (256, 256, 200_000, 0.05, dict(tile=16)),
    (512, 64, 100_000, 0.5, dict(tile=16, halo=16, sort_every=4)),
    (1024, 1024, 200_000, 0.02, dict())])
def test_default_equals_small_tiles(nx, ny, n, dt, want, precision):
    print(f"{nx}x{ny} n={n} precision {precision}", flush=True)
    cfg, parts = case(nx, ny, n, precision, dt, nx + ny)
    t, got = run(cfg, parts, None)
    for k, v in want.items():
        assert t[k] == v, t
    m = min(nx, ny)
    assert t["tile"] <= m // 2 and t["tile"] + 2 * t["halo"] + 1 <= m and 1 <= t["splits"] <= 64
    if nx == 1024:
        assert t["tile"] == (64 if precision == _lib.PIC_FP32 else 32)
    small = dict(tile=min(16, m // 2), halo=1, splits=1, sort_every=1)
    _, ref = run(cfg, parts, small)
    assert all(np.array_equal(a, b) for a, b in zip(got, ref))


def test_batch_shares_its_workgroups():
    """Runs of a batch are tiled by their share of the particles; each equals itself alone."""
    runs = [case(nx, nx, n, _lib.PIC_FP32, 0.05, n) for nx, n in
            ((64, 3000), (128, 400_000), (256, 90_000), (32, 70_000))]
    with Batch([c for c, _ in runs]) as b:
        for k, (_, p) in enumerate(runs):
            b.set_particles(*p, run=k)
        b.step(10)
        got = [b.particles(run=k, sync=False) for k in range(len(runs))]
    for (cfg, parts), g in zip(runs, got):
        _, ref = run(cfg, parts, None)
        assert all(np.array_equal(a, r) for a, r in zip(g, ref))
