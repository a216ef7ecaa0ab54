"""Push windows that leave the fused sort's counters no room beside the kernel's own sums (FP32
windows of 101 nodes, 163,224 B of the 163,840 a workgroup can have, on 16 tiles): the sort runs
as separate kernels, and the trajectory is the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Simulation, _lib  # noqa: E402
from test_gpu_default_tuning import case, run  # noqa: E402


@pytest.mark.parametrize("n,tile,halo,fused", [(256, 64, 18, False), (128, 32, 34, False),
                                               (256, 64, 17, True), (128, 32, 33, True)])
def test_largest_windows(n, tile, halo, fused):
    cfg, parts = case(n, n, 50_000, _lib.PIC_FP32, 0.05, n)
    tuning = dict(tile=tile, halo=halo, splits=1, sort_every=4)
    with Simulation(cfg) as sim:
        sim.set_particles(*parts)
        sim.set_tuning(**tuning)
        assert sim.sort_fused() == fused
    _, got = run(cfg, parts, tuning, 9)
    _, ref = run(cfg, parts, dict(tile=8, halo=2, splits=1, sort_every=1), 9)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)
