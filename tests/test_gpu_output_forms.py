"""Particles out in id order around the size where the output changes form (straight to the
arrays, or records that are then split), host and device destinations, with and without the
pending half kick, into some of the arrays only, and in a batch.  Device output must equal
host output bit for bit, and reading must not change the run."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib, presets  # noqa: E402

DEV = "cuda:0"


def device_out(sim, n, dtype, run=0, sync=True, which=(True,) * 4):
    t = [torch.full((n + 3,), 7.0, dtype=dtype, device=DEV) for _ in range(4)]
    p = [ctypes.c_void_p(a.data_ptr()) if w else None for a, w in zip(t, which)]
    sim.particles_device(*p, n, run=run, sync=sync)
    for a, w in zip(t, which):
        assert (a[n if w else 0:] == 7.0).all()  # nothing past the run, nothing unasked
    return [a[:n].cpu().numpy().astype(np.float64) for a in t]


def case(n, precision, seed):
    cfg, _ = presets.landau_small(n=32, ppc=4, precision=precision, seed=seed)
    rng = np.random.default_rng(seed)
    cfg.capacity = n
    return cfg, (rng.uniform(0, cfg.lx, n), rng.uniform(0, cfg.ly, n), rng.normal(size=n),
                 rng.normal(size=n))


@pytest.mark.parametrize("precision,dtype", [(_lib.PIC_FP32, torch.float32),
                                             (_lib.PIC_FP64, torch.float64)])
@pytest.mark.parametrize("n", [1, 255, 65_536, 65_537, 1_048_577])
def test_device_equals_host(n, precision, dtype):
    print(f"n={n} {dtype}", flush=True)
    cfg, parts = case(n, precision, n)
    with Simulation(cfg) as sim:
        sim.set_particles(*parts)
        for steps in (0, 5):  # synchronous velocities, then staggered ones
            sim.step(steps)
            for sync in (True, False):
                want = sim.particles(sync=sync)
                got = device_out(sim, n, dtype, sync=sync)
                assert all(np.array_equal(g, w) for g, w in zip(got, want))
            if steps == 0:
                for w, p in zip(want, parts):
                    assert np.array_equal(w, p.astype(np.float32) if dtype == torch.float32 else p)
        some = device_out(sim, n, dtype, which=(False, True, False, True))
        full = sim.particles()
        assert np.array_equal(some[1], full[1]) and np.array_equal(some[3], full[3])


def test_reading_leaves_the_run():
    """Outputs between the steps of a sort cycle (their records use the sort's target buffer)
    against the same steps without them; in a batch, run by run."""
    runs = [case(n, _lib.PIC_FP32, n) for n in (70_000, 3_000, 90_001)]
    ends = []
    for read in (False, True):
        with Batch([c for c, _ in runs]) as b:
            for k, (_, p) in enumerate(runs):
                b.set_particles(*p, run=k)
            for _ in range(9):
                b.step(1)
                if read:
                    for k, (_, p) in enumerate(runs):
                        device_out(b, p[0].size, torch.float32, run=k)
                        b.grid("phi", run=k)
            ends.append([b.particles(run=k, sync=False) for k in range(3)] +
                        [b.diagnostics(0, 9, run=k) for k in range(3)])
    for a, b in zip(*ends):
        assert all(np.array_equal(u, v) for u, v in zip(a, b))
