"""A surrogate call whose workspace does not fit the device fails and leaves the handle usable: smaller
calls after it give the results of those before it."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-surrogate-alloc]", *a, file=sys.stderr, flush=True)


@pytest.fixture()
def s():
    from cnt_film_monte_carlo_amd import surrogate as S
    q = S.RateSurrogate.load()
    yield q
    q.close()


def test_rates_after_a_call_that_does_not_fit(s):
    from cnt_film_monte_carlo_amd import surrogate as S
    g = S.sample_geometries(np.random.default_rng(1), 100, s.domain)
    before = s.rates(*g, 0, 1, 300.0)[:2]
    one, out = np.zeros(1), np.zeros(1)
    p = [v.ctypes.data_as(C.POINTER(C.c_double)) for v in (one, one, one, one, out)]
    say("2^40 geometries: 32 TiB of them on the device")
    # refused before anything is read from the arrays
    rc = s.lib.kmc_mlp_rates(s.h, 1 << 40, *p[:4], 0, 1, 300.0, p[4], None, None)
    assert rc < 0
    after = s.rates(*g, 0, 1, 300.0)[:2]
    for a, b in zip(before, after):
        assert np.array_equal(a, b)


def test_training_calls_after_a_batch_that_does_not_fit(s):
    from cnt_film_monte_carlo_amd import surrogate as S
    rng = np.random.default_rng(2)
    f = s.features(*S.sample_geometries(rng, 300, s.domain), 0, 1, 300.0)
    t = rng.normal(size=300).astype(np.float32)
    before = s.loss_grad(f, t)
    fp, tp = (v.ctypes.data_as(C.POINTER(C.c_float)) for v in (f, t))
    say("a batch of 2^30 rows: 2 TiB of activations on the device")
    rc = s.lib.kmc_mlp_train(s.h, 1 << 30, fp, tp, 1, 1 << 30, 1e-3, 1e-5, 1, None, None)
    assert rc < 0
    after = s.loss_grad(f, t)
    assert before[0] == after[0] and np.array_equal(before[1], after[1])
