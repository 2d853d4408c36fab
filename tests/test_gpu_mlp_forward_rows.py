"""The surrogate's forward kernel at the edges of its tiles (32 rows) and of the padding (128 rows):
against the oracle with BF16 operands, with the tolerance of test_gpu_surrogate.py, and the loss that
loss_grad returns for the same rows against the outputs (bitwise the same forward, sums in FP64)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-mlp-forward-rows]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 128, 129, 511, 513, 1025])
def test_forward_of_ragged_rows(n):
    from cnt_film_monte_carlo_amd import surrogate as S
    from oracle import mlp_oracle as MO
    say(f"forward of {n} rows")
    s = S.RateSurrogate()
    p = S.init_params(3)
    s.set_params(p)
    rng = np.random.default_rng(n)
    m = max(n, 32)
    f = s.features(*S.sample_geometries(rng, m, s.domain), rng.integers(0, 3, m),
                   rng.integers(0, 3, m), rng.uniform(150, 400, m))[:n]
    t = rng.normal(0, 1, n).astype(np.float32)
    y = s.forward(f)
    yo, _ = MO.forward(p.astype(np.float64), f.astype(np.float64), bf=True)
    assert np.abs(y - yo).max() <= 2e-3
    loss, _ = s.loss_grad(f, t)
    e = (y - t).astype(np.float32).astype(np.float64)
    assert loss == pytest.approx(float((e * e).mean()), rel=1e-12)
    s.close()
