"""A tuning that is refused leaves the run as it was: the tuning in force, the particles and the
steps that follow, in one run and in a batch (where one run's grid refuses for all)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Batch, Simulation, _lib  # noqa: E402
from test_gpu_default_tuning import case  # noqa: E402


def refuse(sim, code, **tuning):
    with pytest.raises(_lib.PicError) as e:
        sim.set_tuning(**tuning)
    assert e.value.code == code


@pytest.mark.parametrize("precision,tuning", [
    (_lib.PIC_FP64, dict(tile=32, halo=20, sort_every=2)),   # window of 73 nodes
    (_lib.PIC_FP32, dict(tile=64, halo=19, sort_every=2)),   # 103
])
@pytest.mark.parametrize("before", [None, dict(tile=16, halo=4, splits=2, sort_every=4)])
def test_run_goes_on(precision, tuning, before):
    cfg, parts = case(256, 256, 90_000, precision, 0.05, 5)
    out = []
    for refused in (False, True):
        with Simulation(cfg) as sim:
            if before:
                sim.set_tuning(**before)
            sim.set_particles(*parts)
            sim.step(5)
            t = sim.tuning()
            if refused:
                refuse(sim, _lib.PIC_ERR_INVALID_CONFIG, **tuning)
                assert sim.tuning() == t
            sim.step(13)
            sim.sync()
            out.append((sim.particles(sync=False), sim.diagnostics(0, 18), sim.num_particles()))
    for a, b in zip(out[0][0], out[1][0]):
        assert np.array_equal(a, b)
    assert np.array_equal(out[0][1], out[1][1]) and out[0][2] == out[1][2]


def test_batch_goes_on():
    runs = [case(256, 256, 60_000, _lib.PIC_FP32, 0.05, 6), case(64, 64, 9000, _lib.PIC_FP32, 0.05, 7)]
    out = []
    for refused in (False, True):
        with Batch([c for c, _ in runs]) as b:
            for k, (_, p) in enumerate(runs):
                b.set_particles(*p, run=k)
            b.step(3)
            if refused:
                refuse(b, _lib.PIC_ERR_INVALID_CONFIG, tile=32, halo=60)   # 256^2 alone refuses
                refuse(b, _lib.PIC_ERR_ARG, tile=64)                       # above 64^2's half
            b.step(10)
            b.sync()
            out.append([v for k in range(2) for v in b.particles(run=k, sync=False)])
    for a, c in zip(*out):
        assert np.array_equal(a, c)
