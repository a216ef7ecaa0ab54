"""pic_op_poisson at the smallest and largest grid sides and long thin grids (row groups and
column rows of every length class), against numpy's FFT; the density is read only.  Bar: the
field's 1e-12 of the largest value (an FP64 transform of 2^22 points is off by ~1e-15)."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402

DEV = "cuda:0"


@pytest.mark.parametrize("nx,ny", [(4, 4), (8, 4), (4, 2048), (2048, 4), (16, 1024), (256, 512),
                                   (2048, 2048)])
def test_phi(nx, ny):
    print(f"poisson {nx}x{ny}", flush=True)
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
    for _ in range(2):
        check(lib.pic_op_poisson(ctypes.c_void_p(t.data_ptr()), ctypes.c_void_p(phi.data_ptr()),
                                 ctypes.byref(g), None))
        torch.cuda.synchronize()
        assert np.abs(phi.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()
    assert np.array_equal(t.cpu().numpy(), rho)
