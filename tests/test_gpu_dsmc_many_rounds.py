"""DSMC passes of several rounds per cell, at both thread counts of the kernel (the choice is by
the number of cells) and either side of its line: cells of two and three particles, cells whose
rounds hold more pairs than are dealt at once, and cells that need one round, bit for bit against
the oracle over two passes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_collide import run_dsmc_op  # noqa: E402


@pytest.mark.parametrize("ncells,background,big,coeff", [
    (1, 0, (2051,), 5e-3),
    (70, 200, (2, 3, 2600, 64, 65, 1025), 4e-3),
    (32_768, 30_000, (700, 2300, 130), 3e-3),     # the last count at 256 threads
    (32_769, 30_000, (700, 2300, 130), 3e-3),     # the first at 128
    (70_001, 120_000, (2, 3, 2600, 64, 65, 1025), 4e-3),
])
def test_rounds_against_oracle(oracle, ncells, background, big, coeff):
    print(f"{ncells} cells, {background} particles + cells of {big}", flush=True)
    rng = np.random.default_rng(ncells + background)
    cnt = np.bincount(rng.integers(0, ncells, background), minlength=ncells)
    at = np.linspace(0, ncells - 1, len(big)).astype(int)
    cnt[at] = big
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    m = int(off[-1])
    vx, vy = (rng.normal(size=m).astype(np.float32) for _ in range(2))
    gmax = np.full(ncells, 4.0, np.float32)
    assert 0.5 * max(big) * (max(big) - 1) * coeff * 4.0 > 4 * (max(big) // 2)
    rvx, rvy, rg = vx.copy(), vy.copy(), gmax.copy()
    for step in (5, 6):
        vx, vy, gmax, got = run_dsmc_op(off, vx, vy, gmax, coeff, 31, step)
        want = oracle.or_dsmc_step_f32(ncells, oracle.p(off), oracle.p(rvx), oracle.p(rvy),
                                       oracle.p(rg), coeff, 31, step)
        assert got == want > 0
        assert np.array_equal(vx, rvx) and np.array_equal(vy, rvy) and np.array_equal(gmax, rg)
