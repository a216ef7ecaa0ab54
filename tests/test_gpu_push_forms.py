"""pic_op_gather_push with the field in LDS, packed, and read from the node arrays: particle
counts around the lines of the choice, grids at the LDS limit and longer than wide, positions
in the last cells (the padded row and column) and at the box's edges.  The three give the same
values, so FP32 results equal the oracle's mirror bit for bit."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402

DEV = "cuda:0"


def dptr(t):
    return ctypes.c_void_p(t.data_ptr())


def push(parts, ex, ey, prec, nx, ny, lx, ly, dt, qm, c):
    t = [torch.from_numpy(a.copy()).to(DEV) for a in (*parts, ex, ey)]
    ke = torch.zeros(1, dtype=torch.float64, device=DEV)
    g = _lib.pic_grid(nx, ny, lx, ly)
    check(lib.pic_op_gather_push(*(dptr(a) for a in t[:4]), parts[0].size, prec, dptr(t[4]),
                                 dptr(t[5]), ctypes.byref(g), dt, qm, c, dptr(ke), None))
    torch.cuda.synchronize()
    return [a.cpu().numpy() for a in t[:4]], float(ke.item())


@pytest.mark.parametrize("dtype,prec", [(np.float32, _lib.PIC_FP32), (np.float64, _lib.PIC_FP64)])
@pytest.mark.parametrize("nx,ny,big", [
    (32, 16, 1_048_576), (64, 64, 1_100_003), (4, 1024, 1_048_577), (256, 512, 1_600_001),
    (1024, 16, 1_572_864)])
def test_forms_agree(nx, ny, big, dtype, prec):
    """A large call (LDS or packed) against the same particles in calls of 4096 (node arrays)."""
    print(f"{dtype.__name__} {nx}x{ny} n={big}", flush=True)
    rng = np.random.default_rng(nx * ny + big)
    lx, ly, dt, qm, c = 12.0, 5.0, 0.05, -1.0, 1.0
    x, y = rng.uniform(0, lx, big).astype(dtype), rng.uniform(0, ly, big).astype(dtype)
    x[: big // 4] = (lx - lx / nx * rng.uniform(0, 1, big // 4)).astype(dtype) % dtype(lx)
    y[big // 8: big // 4] = (ly * (1 - 1e-7)) if dtype is np.float64 else np.nextafter(
        np.float32(ly), np.float32(0))
    x[:2], y[:2] = 0, 0
    vx, vy = rng.normal(size=big).astype(dtype), rng.normal(size=big).astype(dtype)
    ex, ey = rng.normal(size=nx * ny), rng.normal(size=nx * ny)
    got, ke = push((x, y, vx, vy), ex, ey, prec, nx, ny, lx, ly, dt, qm, c)
    ke_small = 0.0
    for a in (0, big // 8, big // 4 - 2048, big - 4096):
        sl = slice(a, a + 4096)
        want, k = push([v[sl] for v in (x, y, vx, vy)], ex, ey, prec, nx, ny, lx, ly, dt, qm, c)
        for g, w in zip(got, want):
            assert np.array_equal(g[sl], w)
        ke_small += k
    assert ke > ke_small > 0.0
