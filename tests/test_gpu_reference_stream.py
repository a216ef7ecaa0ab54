"""pic_op_mcc_reference where the parallel resolution of the injected stream can go wrong:
streams of one uniform, at the edges of a thread's 16 positions and of a workgroup's 4096,
with a scan over more chunks than the scan's threads, exactly as long as what is drawn, and
one uniform short (refused).  The oracle walks the stream particle by particle."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from pic_amd._lib import lib  # noqa: E402

DEV = "cuda:0"


def hp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def gpu(vx, vy, prob, u):
    tv = [torch.from_numpy(a.copy()).to(DEV) for a in (vx, vy)]
    tu = torch.from_numpy(u).to(DEV)
    used = ctypes.c_int64(-1)
    rc = lib.pic_op_mcc_reference(*(ctypes.c_void_p(t.data_ptr()) for t in tv), vx.size, prob,
                                  ctypes.c_void_p(tu.data_ptr()), u.size, ctypes.byref(used),
                                  None)
    torch.cuda.synchronize()
    return rc, tv[0].cpu().numpy(), tv[1].cpu().numpy(), used.value


@pytest.mark.parametrize("n,prob", [(1, 0.0), (1, 1.0), (15, 0.5), (16, 0.0), (17, 0.5),
                                    (585, 1.0), (586, 0.9), (4095, 0.0), (4096, 0.0),
                                    (4097, 0.0), (4097, 0.3), (30_000, 0.14), (700_000, 0.22)])
def test_stream_lengths(oracle, n, prob):
    print(f"n={n} prob={prob}", flush=True)
    rng = np.random.default_rng(n)
    u = rng.uniform(size=7 * n + 3)
    vx, vy = rng.normal(size=n), rng.normal(size=n)
    ovx, ovy = vx.copy(), vy.copy()
    want = oracle.or_mcc_reference(n, hp(ovx), hp(ovy), prob, hp(u), u.size)
    for cut in (u.size, want):  # a longer stream, and one that is used up exactly
        rc, gx, gy, used = gpu(vx, vy, prob, u[:cut].copy())
        assert rc == _lib.PIC_OK and used == want
        assert np.array_equal(gx, ovx) and np.array_equal(gy, ovy)
    if want > 1:
        rc, gx, gy, _ = gpu(vx, vy, prob, u[: want - 1].copy())
        assert rc == _lib.PIC_ERR_ARG
        assert np.array_equal(gx, vx) and np.array_equal(gy, vy)


def test_many_chunks(oracle):
    """3,000,000 particles with few hits: more than 256 x 2 chunks for the one-workgroup scan."""
    n, prob = 3_000_000, 0.05
    rng = np.random.default_rng(11)
    u = rng.uniform(size=2 * n)
    vx, vy = rng.normal(size=n), rng.normal(size=n)
    ovx, ovy = vx.copy(), vy.copy()
    want = oracle.or_mcc_reference(n, hp(ovx), hp(ovy), prob, hp(u), u.size)
    rc, gx, gy, used = gpu(vx, vy, prob, u)
    assert rc == _lib.PIC_OK and used == want
    assert np.array_equal(gx, ovx) and np.array_equal(gy, ovy)
