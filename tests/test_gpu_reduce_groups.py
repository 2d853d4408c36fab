"""The record reduction with eight records in flight per thread: batches around its groups of 2,048
excitons, bins that all, some or none of the excitons have reached, against sums of the records read
back (relative 1e-12: another order of additions); and the time of bins that nobody has reached."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-reduce-groups]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def film(kmc, nw):
    w = nw.film_small()
    ctx = nw.make_context(w, nw.build_network(w), seed=3)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    dwell = 1.0 / float(np.mean(ctx.get_csr()["gamma"]))
    yield ctx, dwell
    ctx.close()


@pytest.mark.parametrize("n_exc,n_batches", [(1, 1), (2047, 1), (2048, 1), (2049, 1), (4097, 1),
                                             (6143, 3), (6144, 3), (14_000, 3), (14_000, 7)])
def test_sums_of_records(film, n_exc, n_batches):
    say(f"{n_exc} excitons in {n_batches} batches")
    ctx, dwell = film
    ctx.inject(n_exc)
    bins = 6
    ctx.set_samples(bins, 3 * dwell)
    ctx.run(2)   # the later bins are reached by some of the excitons only
    for _ in range(2):
        s = ctx.get_samples()
        made = np.arange(bins)[:, None] < s["n_recorded"][None, :]
        got, _ = ctx.reduce_samples(n_batches)
        for b in range(n_batches):
            lo, hi = b * n_exc // n_batches, (b + 1) * n_exc // n_batches
            for k in range(bins):
                m = made[k, lo:hi]
                d = s["disp"][k, lo:hi][m]
                want = [m.sum(), *(d * d).sum(0), s["drains"][k, lo:hi][m].sum()]
                np.testing.assert_allclose(got[k, b], want, rtol=1e-12, atol=0)
        ctx.run(1 << 40, t_max=4 * dwell)   # now all are
    assert made.all() and not got[:, :, 0].min() == 0


def test_unreached_bins_cost_little(film):
    ctx, dwell = film
    ctx.inject(1_000_000)
    ctx.set_samples(64, dwell)
    none = min(ctx.reduce_samples(32)[1] for _ in range(8))
    ctx.run(1 << 40, t_max=2 * dwell)
    every = min(ctx.reduce_samples(32)[1] for _ in range(8))
    say(f"64 bins of 1 M excitons: none reached {none:.3f} ms, all {every:.3f} ms")
    assert none <= 0.5 * every
