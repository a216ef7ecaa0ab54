"""pic_op_gather_push with interleaved node rows: the grids either side of the packed form
(small, beyond the L2, one row or column of cells wrapping far) and a state large enough for
the rows on a middle grid.  Every form gives the same values per particle, so a large call
equals the same particles pushed 4096 at a time from the node arrays, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from test_gpu_push_forms import push  # noqa: E402


@pytest.mark.parametrize("dtype,prec,nx,ny,n", [
    (np.float32, _lib.PIC_FP32, 128, 128, 1_048_577),   # rows: a small part of the L2
    (np.float32, _lib.PIC_FP32, 128, 128, 1_048_575),   # packed: one particle short
    (np.float64, _lib.PIC_FP64, 256, 128, 1_100_003),
    (np.float32, _lib.PIC_FP32, 1024, 1024, 1_048_576),  # rows: beyond the L2
    (np.float64, _lib.PIC_FP64, 4, 2048, 1_300_001),
    (np.float32, _lib.PIC_FP32, 256, 512, 6_291_457),    # rows: a large state
])
def test_rows_agree(dtype, prec, nx, ny, n):
    print(f"{dtype.__name__} {nx}x{ny} n={n}", flush=True)
    rng = np.random.default_rng(nx + ny + n)
    lx, ly, dt, qm, c = 12.0, 5.0, 0.05, -1.0, 1.0
    x, y = rng.uniform(0, lx, n).astype(dtype), rng.uniform(0, ly, n).astype(dtype)
    x[:4096] = (lx - lx / nx * rng.uniform(0, 1, 4096)).astype(dtype) % dtype(lx)
    y[2048:6144] = (ly - ly / ny * rng.uniform(0, 1, 4096)).astype(dtype) % dtype(ly)
    x[:2], y[:2] = 0, 0
    vx, vy = rng.normal(size=n).astype(dtype), rng.normal(size=n).astype(dtype)
    ex, ey = rng.normal(size=nx * ny), rng.normal(size=nx * ny)
    got, _ = push((x, y, vx, vy), ex, ey, prec, nx, ny, lx, ly, dt, qm, c)
    for a in (0, 2048, n // 2, n - 4096):
        sl = slice(a, a + 4096)
        want, _ = push([v[sl] for v in (x, y, vx, vy)], ex, ey, prec, nx, ny, lx, ly, dt, qm, c)
        for g, w in zip(got, want):
            assert np.array_equal(g[sl], w)
