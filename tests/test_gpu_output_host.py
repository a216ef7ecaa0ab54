"""Particles out to host arrays around the sizes where the copies change form (all arrays in one, each
by itself, in pieces): every form equals the output to device arrays, into all arrays or some of
them, and writes nothing past the run."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import Simulation, _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402
from test_gpu_output_forms import case, device_out  # noqa: E402


def host_out(sim, n, sync, which=(True,) * 4):
    a = [np.full(n + 3, 7.0) for _ in range(4)]
    dp = ctypes.POINTER(ctypes.c_double)
    check(lib.pic_get_particles(sim._ctx, 0, *(v.ctypes.data_as(dp) if w else None
                                               for v, w in zip(a, which)), n, int(sync)))
    for v, w in zip(a, which):
        assert (v[n if w else 0:] == 7.0).all()
    return [v[:n] for v in a]


@pytest.mark.parametrize("precision,dtype,sizes", [
    (_lib.PIC_FP32, torch.float32, (1, 32_768, 32_769, 1_048_576, 2_097_153)),
    (_lib.PIC_FP64, torch.float64, (1, 16_384, 16_385, 300_001))])
def test_host_equals_device(precision, dtype, sizes):
    for n in sizes:
        print(f"n={n} {dtype}", flush=True)
        cfg, parts = case(n, precision, n)
        with Simulation(cfg) as sim:
            sim.set_particles(*parts)
            sim.step(5)
            for sync in (True, False):
                want = device_out(sim, n, dtype, sync=sync)
                assert all(np.array_equal(g, w) for g, w in zip(host_out(sim, n, sync), want))
            for which in ((False, True, False, True), (True, False, False, False),
                          (False, False, True, True)):
                got = host_out(sim, n, False, which)
                for g, w, k in zip(got, want, which):
                    assert not k or np.array_equal(g, w)
