"""pic_get_grid of the potential: the largest transform length along x (where phi beside Ex and Ey
would not fit a workgroup's LDS), a small run beside a large one in a batch, and no effect on the
run.  FP64 transforms of at most 22 stages each way keep phi within 1e-12 of its largest value
(44 stages of a few roundings of 2^-53)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib  # noqa: E402
from test_gpu_default_tuning import case  # noqa: E402


def phi_ref(oracle, sim, cfg, run=0):
    return oracle.poisson(sim.grid("rho", run), cfg.lx, cfg.ly)


@pytest.mark.parametrize("precision", [_lib.PIC_FP32, _lib.PIC_FP64])
@pytest.mark.parametrize("nx,ny", [(2048, 4), (2048, 64), (64, 2048), (2048, 2048)])
def test_phi_of_long_grids(oracle, nx, ny, precision):
    print(f"{nx}x{ny} precision {precision}", flush=True)
    cfg, parts = case(nx, ny, 60_000, precision, 1e-3, nx + ny)
    with Simulation(cfg) as sim:
        sim.set_particles(*parts)
        sim.step(3)
        ref = phi_ref(oracle, sim, cfg)
        phi = sim.grid("phi")
        assert np.abs(phi - ref).max() <= 1e-12 * np.abs(ref).max()


def test_phi_in_a_batch_and_beside_the_steps(oracle):
    runs = [case(2048, 8, 20_000, _lib.PIC_FP32, 1e-3, 1), case(16, 32, 5000, _lib.PIC_FP32, 1e-3, 2)]
    out = []
    for look in (False, True):
        with Batch([c for c, _ in runs]) as b:
            for k, (_, p) in enumerate(runs):
                b.set_particles(*p, run=k)
            b.step(4)
            if look:
                for k, (cfg, _) in enumerate(runs):
                    ref = phi_ref(oracle, b, cfg, k)
                    assert np.abs(b.grid("phi", k) - ref).max() <= 1e-12 * np.abs(ref).max()
            b.step(4)
            out.append([b.particles(run=k) + (b.diagnostics(0, 8, k),) for k in range(2)])
    for a, c in zip(*out):
        assert all(np.array_equal(u, v) for u, v in zip(a, c))
