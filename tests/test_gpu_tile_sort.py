"""The tile sort where its kernel changes: counts around a chunk of 4096 particles and around the
64 and 512 of a wave and a pass, one tile holding everything, up to 4096 tiles (the counters of
all waves in LDS), and sorts by extrapolated positions.  The sort is stable, so running with it
before every step gives what a run without any drift from its tiles gives: particles in id order
equal those of a run that sorts once, bit for bit, and the charge is the same words (the field
energies of all steps are equal)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Simulation, _lib  # noqa: E402


def run(cfg, parts, tiling, nsteps):
    with Simulation(cfg) as sim:
        sim.set_tuning(*tiling)
        sim.set_particles(*parts)
        sim.step(nsteps)
        sim.sync()
        return ([np.array(a) for a in sim.particles(sync=False)],
                sim.diagnostics(0, nsteps)[:, _lib.PIC_DIAG_FIELD_ENERGY])


@pytest.mark.parametrize("prec", [_lib.PIC_FP32, _lib.PIC_FP64])
@pytest.mark.parametrize("nx,ny,tile,n,spread", [
    (16, 16, 8, 1, 1.0), (64, 64, 8, 63, 1.0), (64, 64, 8, 513, 1.0), (64, 64, 16, 4095, 1.0),
    (64, 64, 16, 4097, 0.02), (128, 64, 4, 20_000, 1.0), (256, 256, 4, 70_001, 1.0)])
def test_sort_every_step(nx, ny, tile, n, spread, prec):
    print(f"{nx}x{ny} tile {tile} n={n} spread {spread} prec {prec}", flush=True)
    rng = np.random.default_rng(nx + ny + n)
    lx, ly = 6.0, 3.0
    cfg = _lib.default_config(nx=nx, ny=ny, lx=lx, ly=ly, dt=0.05, qm=-1.0, precision=prec,
                              capacity=n)
    parts = (rng.uniform(0, lx, n) * spread, rng.uniform(0, ly, n) * spread,
             rng.normal(size=n), rng.normal(size=n))
    got, energy = run(cfg, parts, (tile, 2, 1, 1), 3)
    want, energy_once = run(cfg, parts, (tile, 2, 1, 8), 3)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    assert np.array_equal(energy, energy_once)
