"""Small grids, at the shapes where the one-workgroup Poisson solve changes its LDS layout
(padded and plain rows, long thin grids, the largest and smallest it takes, one above it): phi
against numpy's FFT (bar: the field's 1e-12), and whole engine steps under the default tiling,
with the end-of-step work folded into the field passes (graphs) and in kernels of its own
(eager), against the oracle's FP32 mirror bit for bit and between the two."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402

DEV = "cuda:0"
SHAPES = [(4, 4), (4, 8), (8, 8), (64, 64), (32, 128), (128, 32), (8, 512), (512, 8), (4, 1024),
          (1024, 4), (64, 128)]


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_phi(nx, ny):
    lx, ly = 7.0, 3.0
    rho = np.random.default_rng(nx + 5 * ny).normal(size=(nx, ny))
    kx = 2 * np.pi / lx * np.fft.fftfreq(nx, 1 / nx)
    ky = 2 * np.pi / ly * np.fft.fftfreq(ny, 1 / ny)
    k2 = kx[:, None] ** 2 + ky[None, :] ** 2
    k2[0, 0] = 1.0
    ph = np.fft.fft2(rho) / k2
    ph[0, 0] = 0.0
    want = np.fft.ifft2(ph).real
    t = torch.from_numpy(rho).to(DEV)
    phi = torch.full((nx, ny), float("nan"), dtype=torch.float64, device=DEV)
    g = _lib.pic_grid(nx, ny, lx, ly)
    check(lib.pic_op_poisson(ctypes.c_void_p(t.data_ptr()), ctypes.c_void_p(phi.data_ptr()),
                             ctypes.byref(g), None))
    assert np.abs(phi.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()


def case(nx, ny, n, precision, seed):
    rng = np.random.default_rng(seed)
    cfg = _lib.default_config(nx=nx, ny=ny, lx=9.0, ly=6.0, dt=0.02, qm=-1.0,
                              precision=precision, seed=seed, capacity=n)
    return cfg, (rng.uniform(0, 9.0, n), rng.uniform(0, 6.0, n), rng.normal(size=n),
                 rng.normal(size=n))


def run(cfg, parts, steps, graphs):
    with Simulation(cfg) as sim:
        sim.use_graphs(graphs)
        sim.set_particles(*parts)
        sim.step(steps)
        sim.sync()
        return sim.particles(), sim.diagnostics(0, steps)


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_steps_match_the_mirror(oracle, nx, ny):
    steps, n = 19, 5000  # two captured sequences of 8, then 3 eager steps
    print(f"{nx}x{ny}", flush=True)
    cfg, parts = case(nx, ny, n, _lib.PIC_FP32, nx * 3 + ny)
    (p, d), (pe, de) = run(cfg, parts, steps, True), run(cfg, parts, steps, False)
    ref = [a.astype(np.float32) for a in parts]
    dr = oracle.run_f32(*ref, nx, ny, 9.0, 6.0, cfg.dt, cfg.qm, -(9.0 * 6.0) / n, steps)
    for a, b, r in zip(p, pe, ref):
        assert np.array_equal(a, r) and np.array_equal(a, b)
    assert np.array_equal(d, de)
    assert np.abs(d[:, 0] - dr[:, 0]).max() <= 1e-12 * np.abs(dr[:, 0]).max()
    assert np.array_equal(d[:, 5], np.full(steps, n))


@pytest.mark.parametrize("precision", [_lib.PIC_FP32, _lib.PIC_FP64])
def test_batches_of_small_and_mixed_grids(precision):
    """Batches of small grids, alone and with a larger one: each run equals itself alone."""
    small = [case(nx, ny, n, precision, n) for nx, ny, n in
             ((32, 32, 4001), (64, 64, 20_000), (16, 8, 700))]
    mixed = small[:2] + [case(128, 64, 9000, precision, 9)]
    alone = {}
    for runs in (small, mixed):
        with Batch([c for c, _ in runs]) as b:
            for k, (_, p) in enumerate(runs):
                b.set_particles(*p, run=k)
            b.step(17)
            got = [(b.particles(run=k), b.diagnostics(0, 17, run=k)) for k in range(len(runs))]
        for (cfg, parts), (p, d) in zip(runs, got):
            key = (cfg.nx, cfg.ny)
            if key not in alone:
                alone[key] = run(cfg, parts, 17, True)
            pa, da = alone[key]
            assert all(np.array_equal(a, w) for a, w in zip(p, pa))
            assert np.abs(d[:, 0] - da[:, 0]).max() <= 1e-13 * np.abs(da[:, 0]).max()
