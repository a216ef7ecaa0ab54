"""The operators' kept memory shared by threads and streams: several threads call operators of
different sizes at once, each on a stream of its own, some of the calls refused or ending early, and
every result equals the one of the same call alone."""
import ctypes
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from pic_amd._lib import lib  # noqa: E402

DEV = "cuda:0"


def dptr(t):
    return ctypes.c_void_p(t.data_ptr())


def ok(rc):
    assert rc == _lib.PIC_OK, lib.pic_last_error()


class Work:
    """Inputs and outputs of one thread; sizes and data by its seed."""

    def __init__(self, seed):
        self.n, self.side = 20_000 + 70_001 * seed, (64, 128, 256, 512)[seed % 4]
        self.cells = 300 + 1000 * seed
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        rand = lambda dtype: torch.rand(self.n, generator=g, device=DEV, dtype=dtype)
        self.prec = _lib.PIC_FP64 if seed % 2 else _lib.PIC_FP32
        dtype = torch.float64 if seed % 2 else torch.float32
        self.x, self.y, self.vx, self.vy = (rand(dtype) for _ in range(4))
        self.keys = (rand(torch.float64) * self.cells).to(torch.int32)
        self.bad = self.keys.clone()
        self.bad[self.n // 2] = self.cells
        self.u = torch.rand(8 * self.n, generator=g, device=DEV, dtype=torch.float64)
        G = self.side * self.side
        self.rho, self.phi, self.ex, self.ey = (torch.zeros(G, dtype=torch.float64, device=DEV)
                                                for _ in range(4))
        self.ke = torch.zeros(1, dtype=torch.float64, device=DEV)
        self.perm = torch.empty(self.n, dtype=torch.int32, device=DEV)
        self.counts = torch.empty(self.cells, dtype=torch.int32, device=DEV)
        self.offsets = torch.empty(self.cells + 1, dtype=torch.int32, device=DEV)
        self.grid = _lib.pic_grid(self.side, self.side, 1.0, 1.0)

    def calls(self, stream, refuse=False):
        """One round of calls on `stream` (all synchronous); a copy of every output."""
        s, g, n = ctypes.c_void_p(stream), ctypes.byref(self.grid), self.n
        used = ctypes.c_int64()
        with torch.cuda.stream(torch.cuda.ExternalStream(stream) if stream else
                               torch.cuda.default_stream()):
            x, y, vx, vy = (t.clone() for t in (self.x, self.y, self.vx, self.vy))
            wx, wy = self.u[:n].clone(), self.u[n:2 * n].clone()
            if refuse:
                assert lib.pic_op_sort(dptr(self.bad), n, self.cells, dptr(self.perm),
                                       dptr(self.counts), dptr(self.offsets), s) == _lib.PIC_ERR_ARG
                # a stream too short: the call ends with its memory still taken
                assert lib.pic_op_mcc_reference(dptr(wx), dptr(wy), n, 0.5, dptr(self.u), n // 2,
                                                ctypes.byref(used), s) == _lib.PIC_ERR_ARG
            ok(lib.pic_op_sort(dptr(self.keys), n, self.cells, dptr(self.perm), dptr(self.counts),
                               dptr(self.offsets), s))
            ok(lib.pic_op_deposit(dptr(x), dptr(y), n, self.prec, g, -1.0 / n, dptr(self.rho), s))
            ok(lib.pic_op_poisson(dptr(self.rho), dptr(self.phi), g, s))
            ok(lib.pic_op_efield(dptr(self.phi), dptr(self.ex), dptr(self.ey), g, s))
            ok(lib.pic_op_gather_push(dptr(x), dptr(y), dptr(vx), dptr(vy), n, self.prec,
                                      dptr(self.ex), dptr(self.ey), g, 0.01, -1.0, 1.0,
                                      dptr(self.ke), s))
            ok(lib.pic_op_mcc_reference(dptr(wx), dptr(wy), n, 0.5, dptr(self.u), self.u.numel(),
                                        ctypes.byref(used), s))
            out = [t.cpu().numpy() for t in (x, y, vx, vy, wx, wy, self.perm, self.counts,
                                             self.offsets, self.rho, self.phi, self.ke)]
        return out + [used.value]


def test_threads_and_streams():
    work = [Work(k) for k in range(5)]
    torch.cuda.synchronize()
    want = [w.calls(0) for w in work]
    streams = [torch.cuda.Stream() for _ in work]
    failures = []

    def run(k):
        try:
            for i in range(12):
                got = work[k].calls(streams[k].cuda_stream, refuse=(i + k) % 3 == 0)
                for a, b in zip(got, want[k]):
                    assert np.array_equal(a, b)
        except BaseException as e:  # noqa: BLE001  (reported by the main thread)
            failures.append((k, repr(e)))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(90)
    assert not any(t.is_alive() for t in threads) and not failures, failures


def test_calls_after_one_that_ended_early():
    w = Work(1)
    torch.cuda.synchronize()
    want = w.calls(0)
    for _ in range(3):
        for a, b in zip(w.calls(0, refuse=True), want):
            assert np.array_equal(a, b)
