"""The MCC null-collision test as a comparison of random words, from a probability that no word
passes to one that every word does, with particle counts around the shares of a workgroup.
Whole steps against the oracle, which compares uniforms: bit for bit, with the counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_collide_engine import engine_run, mcc_case, oracle_run  # noqa: E402


@pytest.mark.parametrize("factor", [1e-12, 1e-4, 1.0, 50.0, 1000.0])
@pytest.mark.parametrize("n", [1, 257, 32768])
def test_against_oracle(oracle, n, factor):
    cfg, parts = mcc_case()
    parts = [p[:n] for p in parts]
    cfg.mcc_ng *= factor  # nu_max dt = 0.1 at factor 1
    cfg.capacity = 4 * n + 64
    print(f"n={n} nu_max dt={0.1 * factor:g}", flush=True)
    want, counts = oracle_run(oracle, cfg, parts, 2)
    out = engine_run(cfg, parts, 2)
    for g, w in zip(out[0], want):
        assert np.array_equal(g, w)
    assert np.array_equal(out[1], counts)
    if factor == 1000.0:
        assert counts.sum() >= 2 * n  # every particle, every step
