"""The surrogate's training kernels at the edges of their tiles (32 rows), splits (512 rows) and row
blocks: gradients against the oracle, with the tolerance of test_gpu_surrogate.py, and a training
run against the same steps made one by one (bitwise: the same kernels' sums in the same order)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-train-step]", *a, file=sys.stderr, flush=True)


def _data(S, s, rng, n):
    g = S.sample_geometries(rng, n, s.domain)
    f = s.features(*g, rng.integers(0, 3, n), rng.integers(0, 3, n), rng.uniform(150, 400, n))
    return f, rng.normal(0, 1, n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 33, 128, 129, 511, 513, 640, 4099])
def test_loss_grad_ragged_rows(n):
    from cnt_film_monte_carlo_amd import surrogate as S
    from oracle import mlp_oracle as MO
    say(f"loss_grad of {n} rows")
    s = S.RateSurrogate()
    p = S.init_params(3)
    s.set_params(p)
    rng = np.random.default_rng(n)
    f, t = _data(S, s, rng, max(n, 32))
    f, t = f[:n], t[:n]
    loss, g = s.loss_grad(f, t)
    lo, go = MO.loss_grad(p.astype(np.float64), f.astype(np.float64), t.astype(np.float64), bf=True)
    assert loss == pytest.approx(lo, rel=2e-3)
    for name, off, shape in MO.LAYOUT:
        k = int(np.prod(shape))
        a, b = g[off:off + k], go[off:off + k]
        assert np.linalg.norm(a - b) <= 2e-3 * np.linalg.norm(b) + 1e-7, name
    # y of the same rows, through the forward kernel
    np.testing.assert_array_equal(loss, s.loss_grad(f, t)[0])
    s.close()


def _shuffles(n, seed, epochs):
    """Fisher-Yates with splitmix64, the order carried over from epoch to epoch."""
    mask = (1 << 64) - 1
    state = seed ^ 0x9E3779B97F4A7C15
    order = list(range(n))
    for _ in range(epochs):
        for i in range(n - 1, 0, -1):
            state = (state + 0x9E3779B97F4A7C15) & mask
            z = ((state ^ (state >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            j = (z ^ (z >> 31)) % (i + 1)
            order[i], order[j] = order[j], order[i]
        yield list(order)


@pytest.mark.parametrize("n,batch,epochs", [(128, 128, 3), (700, 256, 11), (1300, 640, 2)])
def test_training_equals_its_steps(n, batch, epochs):
    from cnt_film_monte_carlo_amd import surrogate as S
    say(f"train {n} rows, batch {batch}, {epochs} epochs against its steps")
    s, q = S.RateSurrogate(), S.RateSurrogate()
    rng = np.random.default_rng(9)
    f, t = _data(S, s, rng, n)
    p = S.init_params(4)
    s.set_params(p)
    q.set_params(p)
    lr, lr_min, seed = 3e-3, 1e-5, 77
    losses, _ = s.train(f, t, epochs, batch=batch, lr=lr, lr_min=lr_min, seed=seed)
    it, per = 0, n // batch
    for ep, order in enumerate(_shuffles(n, seed, epochs)):
        total = 0.0
        for b in range(per):
            rows = np.array(order[b * batch:(b + 1) * batch])
            loss, g = q.loss_grad(f[rows], t[rows])
            rate = lr_min + 0.5 * (lr - lr_min) * (1.0 + np.cos(np.pi * it / (epochs * per)))
            it += 1
            q.adam_step(g, rate, step=it)
            total += loss
        assert losses[ep] == pytest.approx(total / per, rel=1e-12)
    assert np.array_equal(s.get_params(), q.get_params())
    s.close()
    q.close()
