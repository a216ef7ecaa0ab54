"""The default sort cadence and halo follow the speeds of the particles that a run holds: thermal
and beam speeds either side of the lines, along either axis, one fast run in a batch, explicit
values kept; new particles change them again.  Whatever is picked, the trajectory is the one under
small tiles sorted every step, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib  # noqa: E402
from test_gpu_default_tuning import case, run  # noqa: E402


def with_speeds(cfg, parts, vx, vy, beams=False):
    """Speeds of vx, vy cells per step: thermal (one normal per component) or beams of +- it."""
    n = parts[0].size
    dx, dy = cfg.lx / cfg.nx, cfg.ly / cfg.ny
    sx, sy = vx * dx / cfg.dt, vy * dy / cfg.dt
    if beams:
        s = np.where(np.arange(n) & 1, 1.0, -1.0)
        return parts[0], parts[1], s * sx, s * sy
    return parts[0], parts[1], parts[2] * sx, parts[3] * sy


# cells per step; 2.6 thermal cells per step is the cadence's line, beams' 4.65; the halo's is
# 0.64 thermal at a cadence of 8, beams' 1.14
@pytest.mark.parametrize("precision", [_lib.PIC_FP32, _lib.PIC_FP64])
@pytest.mark.parametrize("vx,vy,beams,every,halo", [
    (0.3, 0.3, False, 8, 8), (2.2, 0.1, False, 8, 16), (3.1, 0.1, False, 4, 16),
    (0.1, 3.1, False, 4, 16), (0.9, 0.1, True, 8, 8), (4.0, 0.5, True, 8, 16),
    (0.5, 6.0, True, 4, 16), (40.0, 40.0, False, 4, 16), (0.0, 0.0, False, 8, 8)])
def test_follows_the_speeds(vx, vy, beams, every, halo, precision):
    cfg, parts = case(256, 128, 60_000, precision, 0.01, 11)
    cfg.ly = cfg.lx  # cells of different sides
    parts = (parts[0], parts[1] * (cfg.ly / parts[1].max()) * (1 - 1e-6), parts[2], parts[3])
    parts = with_speeds(cfg, parts, vx, vy, beams)
    t, got = run(cfg, parts, None)
    assert (t["sort_every"], t["halo"]) == (every, halo), t
    _, ref = run(cfg, parts, dict(tile=8, halo=1, splits=1, sort_every=1))
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)


def test_new_particles_change_them_again():
    cfg, parts = case(256, 256, 50_000, _lib.PIC_FP32, 0.01, 12)
    slow, fast = (with_speeds(cfg, parts, v, v) for v in (0.3, 8.0))
    _, want = run(cfg, slow, dict(tile=8, halo=1, splits=1, sort_every=1), 9)
    with Simulation(cfg) as sim:
        for p, every in ((fast, 4), (slow, 8), (fast, 4), (slow, 8)):
            sim.set_particles(*p)
            assert sim.tuning()["sort_every"] == every
            sim.step(9)
        for a, b in zip(sim.particles(sync=False), want):
            assert np.array_equal(a, b)
        sim.set_tuning(sort_every=6)      # asked for: kept from here on
        sim.set_particles(*fast)
        assert sim.tuning()["sort_every"] == 6 and sim.tuning()["halo"] == 16


def test_asked_values_are_kept():
    cfg, parts = case(256, 256, 50_000, _lib.PIC_FP32, 0.01, 13)
    cfg.halo, cfg.sort_every = 4, 5
    t, _ = run(cfg, with_speeds(cfg, parts, 9.0, 9.0), None, 2)
    assert t["halo"] == 4 and t["sort_every"] == 5


def test_a_fast_run_of_a_batch():
    """The cadence is the batch's, the halo each run's; both runs equal themselves alone."""
    runs = []
    for k, v in enumerate((0.2, 7.0, 0.2)):
        cfg, p = case(128, 128, 20_000, _lib.PIC_FP32, 0.01, 14 + k)
        runs.append((cfg, with_speeds(cfg, p, v, v)))
    with Batch([c for c, _ in runs]) as b:
        for k, (_, p) in enumerate(runs):
            b.set_particles(*p, run=k)
        assert b.tuning()["sort_every"] == 4
        b.step(10)
        got = [b.particles(run=k, sync=False) for k in range(3)]
    for (cfg, p), g in zip(runs, got):
        _, ref = run(cfg, p, None)
        assert all(np.array_equal(a, r) for a, r in zip(g, ref))


@pytest.mark.parametrize("order", [(0, 1, 2), (2, 0, 1)])
def test_a_batch_is_laid_out_when_its_last_run_is_set(order):
    """Whichever run comes last, also one whose own values are given; and again when a run of a
    full batch gets other particles."""
    runs = []
    for k, v in enumerate((0.2, 7.0, 0.2)):
        cfg, p = case(128, 128, 20_000, _lib.PIC_FP32, 0.01, 24 + k)
        runs.append((cfg, with_speeds(cfg, p, v, v)))
    runs[2][0].halo = 8
    slow = with_speeds(runs[1][0], case(128, 128, 20_000, _lib.PIC_FP32, 0.01, 25)[1], 0.2, 0.2)
    with Batch([c for c, _ in runs]) as b:
        for k in order:
            b.set_particles(*runs[k][1], run=k)
        assert b.tuning()["sort_every"] == 4
        b.step(10)
        got = [b.particles(run=k, sync=False) for k in range(3)]
        b.set_particles(*slow, run=1)
        assert b.tuning()["sort_every"] == 8
        b.step(10)
        again = b.particles(run=1, sync=False)
    for (cfg, p), g in zip(runs, got):
        _, ref = run(cfg, p, None)
        assert all(np.array_equal(a, r) for a, r in zip(g, ref))
    _, ref = run(runs[1][0], slow, None)
    assert all(np.array_equal(a, r) for a, r in zip(again, ref))


def test_mcc_reach():
    """With MCC the keys are not led: the line is 1.44 cells per step, the halo's 0.36."""
    for v, every, halo in ((0.2, 8, 8), (0.5, 8, 16), (1.2, 8, 16), (1.7, 4, 16)):
        cfg, parts = case(256, 256, 30_000, _lib.PIC_FP32, 0.01, 15)
        _lib.check(_lib.lib.pic_mcc_preset(cfg, 1e19, 2.0, 1e15))
        cfg.dt, cfg.capacity = 0.01, 40_000
        t, _ = run(cfg, with_speeds(cfg, parts, v, v), None, 3)
        assert (t["sort_every"], t["halo"]) == (every, halo), (v, t)
