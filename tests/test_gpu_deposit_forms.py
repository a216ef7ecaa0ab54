"""pic_op_deposit at the edges of its three forms (global atomics, a whole grid in LDS,
positions grouped by tile): counts around each line of the choice, grids longer than wide,
everything in one cell, positions on and outside the box's edges.  The sums are integers, so
the result equals the oracle's fixed-point deposit bit for bit."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402

DEV = "cuda:0"


def deposit(fn, x, y, prec, nx, ny, lx, ly, qp):
    rho = torch.full((nx * ny,), float("nan"), dtype=torch.float64, device=DEV)
    g = _lib.pic_grid(nx, ny, lx, ly)
    tx, ty = torch.from_numpy(x).to(DEV), torch.from_numpy(y).to(DEV)
    check(fn(ctypes.c_void_p(tx.data_ptr()), ctypes.c_void_p(ty.data_ptr()), x.size, prec,
             ctypes.byref(g), qp, ctypes.c_void_p(rho.data_ptr()), None))
    torch.cuda.synchronize()
    return rho.cpu().numpy().reshape(nx, ny)


@pytest.mark.parametrize("dtype,prec", [(np.float32, _lib.PIC_FP32), (np.float64, _lib.PIC_FP64)])
@pytest.mark.parametrize("nx,ny,n,where", [
    (4, 4, 127, "box"), (4, 4, 128, "box"), (32, 16, 5001, "cell"), (64, 64, 40_000, "box"),
    (128, 128, 140_001, "box"), (4, 2048, 70_000, "box"), (16, 2048, 300_001, "box"),
    (2048, 16, 300_001, "box"), (256, 128, 262_143, "box"), (256, 128, 262_144, "cell"),
    (512, 512, 131_072, "box"), (512, 512, 1_048_577, "box"), (1024, 512, 600_000, "strip"),
    (1024, 2048, 1_100_000, "box")])
def test_forms_match_the_fixed_point_deposit(oracle, dtype, prec, nx, ny, n, where):
    print(f"{dtype.__name__} {nx}x{ny} n={n} {where}", flush=True)
    rng = np.random.default_rng(nx + ny + n)
    lx, ly = 12.0, 5.0
    if where == "cell":
        x, y = (np.full(n, (k - 0.75) / k * v).astype(dtype) for k, v in ((nx, lx), (ny, ly)))
    else:
        x, y = rng.uniform(0, lx, n).astype(dtype), rng.uniform(0, ly, n).astype(dtype)
        if where == "strip":
            y[:] = y % (ly / ny * 3)
        # edges: zero, the last value below the box length, cell corners
        x[:4] = [0, np.nextafter(dtype(lx), dtype(0)), lx / nx, 0]
        y[:4] = [0, np.nextafter(dtype(ly), dtype(0)), 0, ly / ny]
    qp = -lx * ly / n
    want = oracle.fixed_to_rho(oracle.deposit_fixed(x, y, nx, ny, lx, ly), nx, ny, lx, ly, qp)
    assert np.array_equal(deposit(lib.pic_op_deposit, x, y, prec, nx, ny, lx, ly, qp), want)
    if nx * ny <= 1 << 20:
        assert np.array_equal(deposit(lib.pic_op_deposit_noalloc, x, y, prec, nx, ny, lx, ly, qp),
                              want)
