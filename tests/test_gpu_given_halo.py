"""A halo given without a tile: the default tile is halved until the caller's window fits the LDS,
so every halo that 16-cell tiles take is accepted, at creation and by set_tuning, and changes no
trajectory.  (160 KB hold a window of 101 nodes a side in FP32, 71 in FP64.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pic_amd import Simulation, _lib  # noqa: E402
from test_gpu_default_tuning import case, run  # noqa: E402

WIN = {_lib.PIC_FP32: 101, _lib.PIC_FP64: 71}


@pytest.mark.parametrize("precision,n,halo,want", [
    (_lib.PIC_FP32, 1024, 18, 64), (_lib.PIC_FP32, 1024, 19, 32), (_lib.PIC_FP32, 1024, 24, 32),
    (_lib.PIC_FP32, 1024, 42, 16), (_lib.PIC_FP32, 512, 34, 32), (_lib.PIC_FP32, 512, 36, 16),
    (_lib.PIC_FP64, 512, 19, 32), (_lib.PIC_FP64, 512, 20, 16), (_lib.PIC_FP64, 512, 27, 16),
    (_lib.PIC_FP64, 1024, 24, 16), (_lib.PIC_FP32, 64, 40, None)])
def test_accepted_and_same_trajectory(precision, n, halo, want):
    print(f"{n}^2 precision {precision} halo {halo}", flush=True)
    cfg, parts = case(n, n, 120_000, precision, 0.05, n + halo)
    _, ref = run(cfg, parts, dict(tile=8 if n < 1024 else 16, halo=2, splits=1, sort_every=1), 5)
    cfg.halo = halo
    t, got = run(cfg, parts, None, 5)
    cfg.halo = 0
    s, got2 = run(cfg, parts, dict(halo=halo), 5)
    for q in (t, s):
        assert want is None or q["tile"] == want, q
        assert q["halo"] == min(halo, (n - q["tile"] - 1) // 2)
        assert q["tile"] + 2 * q["halo"] + 1 <= WIN[precision]
    for a, b, r in zip(got, got2, ref):
        assert np.array_equal(a, r) and np.array_equal(b, r)


@pytest.mark.parametrize("precision,halo", [(_lib.PIC_FP32, 43), (_lib.PIC_FP64, 28)])
def test_refused_halos_stay_refused(precision, halo):
    """A window that 16-cell tiles do not fit either (512^2: 103 nodes FP32, 73 FP64)."""
    cfg, _ = case(512, 512, 1000, precision, 0.05, 1)
    cfg.capacity = 4_000_000  # no smaller tiles by the particle count
    cfg.halo = halo
    with pytest.raises(_lib.PicError) as e:
        Simulation(cfg)
    assert e.value.code == _lib.PIC_ERR_INVALID_CONFIG
