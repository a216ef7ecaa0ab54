"""pic_op_gather_push over the orders that particles lie in (random, in cell order, near it, gathered in
a part of the grid), on grids where the form goes by that order and on those where it does not,
against the oracle's mirror, bit for bit, and the kinetic energy, whose terms are positive, to n
2^-53 (either side sums in FP64)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from test_gpu_push_forms import push  # noqa: E402

F32, F64 = np.float32, np.float64


def positions(order, nx, ny, lx, ly, n, dtype, rng):
    x, y = rng.uniform(0, lx, n), rng.uniform(0, ly, n)
    if order == "cloud":
        x = (lx * (0.9 + 0.03 * rng.normal(size=n))) % lx
        y = (ly * (0.1 + 0.03 * rng.normal(size=n))) % ly
    if order in ("sorted", "near"):
        o = np.argsort((x * (nx / lx)).astype(int) * ny + (y * (ny / ly)).astype(int))
        x, y = x[o], y[o]
    if order == "near":
        x = (x + 10 * lx / nx * rng.normal(size=n)) % lx
        y = (y + 10 * ly / ny * rng.normal(size=n)) % ly
    x, y = x.astype(dtype), y.astype(dtype)
    x[x >= lx] = 0
    y[y >= ly] = 0
    x[-3:], y[-3:] = 0, np.nextafter(dtype(ly), dtype(0))
    return x, y


@pytest.mark.parametrize("dtype,nx,ny,n", [
    (F32, 64, 64, 300_001), (F64, 64, 64, 270_000),          # in LDS
    (F32, 32, 16, 4097), (F64, 512, 512, 100_001),           # node arrays
    (F32, 512, 512, 600_001), (F64, 256, 256, 700_003),      # packed
    (F32, 128, 128, 1_100_001), (F64, 128, 128, 1_048_577),  # rows
    (F32, 1024, 1024, 600_001), (F32, 1024, 1024, 1_048_577), (F32, 512, 2048, 3_200_003),
    (F64, 1024, 1024, 600_001), (F64, 2048, 512, 1_048_577), (F32, 1024, 1024, 4_194_305)])
def test_orders_against_the_mirror(oracle, dtype, nx, ny, n):
    lx, ly, dt, qm, c = 12.0, 5.0, 0.05, -1.0, 1.0
    prec = _lib.PIC_FP32 if dtype is F32 else _lib.PIC_FP64
    rng = np.random.default_rng(nx + ny + n)
    ex, ey = rng.normal(size=nx * ny), rng.normal(size=nx * ny)
    for order in ("random", "sorted", "near", "cloud"):
        print(f"{dtype.__name__} {nx}x{ny} n={n} {order}", flush=True)
        x, y = positions(order, nx, ny, lx, ly, n, dtype, rng)
        vx, vy = rng.normal(size=n).astype(dtype), rng.normal(size=n).astype(dtype)
        got, ke = push((x, y, vx, vy), ex, ey, prec, nx, ny, lx, ly, dt, qm, c)
        e = ex.reshape(nx, ny), ey.reshape(nx, ny)
        ref = [a.copy() for a in (x, y, vx, vy)]
        if dtype is F32:
            ke_ref = oracle.push_f32(*ref, *e, lx, ly, dt, qm, c)
        else:
            ke_ref = oracle.push_f64(*ref, *e, lx, ly, dt, qm, c, quantized=1)
        for g, r in zip(got, ref):
            assert np.array_equal(g, r)
        assert abs(ke - ke_ref) <= n * 2.0 ** -53 * ke_ref
