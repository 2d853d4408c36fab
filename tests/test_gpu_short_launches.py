"""Launches of a hop or a few with few excitons: the row-of-lanes kernel's fixed costs (the count of
excitons that can still move, the window of departure counts, a batch of 16 hops) against launches
without them, and the edges of window and batch against the oracle."""
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-short-launches]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def film(kmc, nw):
    w = nw.film_small()
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=61)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    yield ctx
    ctx.close()


def _hop_us(ctx, excitons, hops, count, t_step=np.inf):
    """Best hop-kernel time of a call of so many hops, or up to the next of a row of times."""
    ctx.inject(excitons)
    best = np.inf
    for k in range(40):
        ctx.run(hops, t_max=(k + 1) * t_step, count_sites=count)
        best = min(best, 1e3 * ctx.hop_time())
    return best


def test_many_waves_ending_together(film):
    line = 128 * torch.cuda.get_device_properties(0).multi_processor_count
    rows, lanes = (_hop_us(film, e, 1, False) for e in (line, line + 1))
    say(f"one hop of {line} excitons {rows:.1f} us, of one more {lanes:.1f} us")
    assert rows <= 3 * lanes
    assert film.run_stats() == (1, line + 1)


@pytest.mark.parametrize("n_exc,hops,t_step", [(1, 1, np.inf), (200, 1 << 40, 5e-9)])
def test_window_of_a_short_launch(kmc, nw, n_exc, hops, t_step):
    """Departure counts of a hop or a few on a film of far more lines than a window holds."""
    w = nw.film_large()
    w.net.n_tubes = 1500
    ctx = nw.make_context(w, nw.build_network(w), seed=5)
    ctx.set_rate_table(*nw.forster_tables(3))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    with_counts, without = (_hop_us(ctx, n_exc, hops, c, t_step) for c in (True, False))
    say(f"{n_exc} excitons on {ctx.n_sites} sites, {hops} hops or {t_step} s, with counts "
        f"{with_counts:.1f} us, without {without:.1f} us")
    ctx.close()
    assert with_counts <= 3 * without


@pytest.mark.parametrize("n_exc,hops", [(1, 1), (2, 3), (5, 1), (9, 2), (300, 1), (4100, 2), (16400, 5)])
def test_short_launches_match_oracle(kmc, orc, film, nw, n_exc, hops):
    """Windows of 4 lines per thread and hop, from 256 lines up to the film's."""
    say(f"{n_exc} excitons, calls of {hops} hops")
    ctx = film
    ctx.inject(n_exc)
    csr = ctx.get_csr()
    flags = nw.build_network(nw.film_small())["flags"]
    ox = orc.Excitons(csr, flags, seed=61, n_excitons=n_exc)
    for _ in range(3):
        ctx.run(hops)
        ox.run(hops)
    g = ctx.get_excitons()
    for k, o in (("site", ox.site), ("hops", ox.hops), ("hash", ox.hash), ("drains", ox.drains),
                 ("disp", ox.dsp)):
        assert np.array_equal(g[k], o), k
    assert np.array_equal(ctx.get_hop_counts(), ox.site_count)


def test_a_hop_costs_less_than_a_batch(film):
    one, batch = (_hop_us(film, 64, h, False) for h in (1, 16))
    say(f"64 excitons: one hop {one:.1f} us, a batch of 16 {batch:.1f} us")
    assert one <= 0.7 * batch


@pytest.mark.parametrize("n_exc", [1, 6, 1030, 20000])
@pytest.mark.parametrize("dwells", [0.3, 2.0, 4.5, 9.0])
def test_short_times_match_oracle(kmc, orc, film, nw, n_exc, dwells):
    """Runs up to times about as long as the first batch's four hops, with records and trace."""
    say(f"{n_exc} excitons up to {dwells} dwells at a time")
    ctx = film
    ctx.inject(n_exc)
    csr = ctx.get_csr()
    ox = orc.Excitons(csr, nw.build_network(nw.film_small())["flags"], seed=61, n_excitons=n_exc)
    step = dwells / float(np.mean(csr["gamma"]))
    nt = min(n_exc, 50)
    for q in (ctx, ox):
        q.set_samples(5, 4 * step)
        q.set_trace(nt, 200)
    for k in range(4):
        ctx.run(1 << 40, t_max=(k + 1) * step)
        ox.run(1 << 40, t_max=(k + 1) * step)
    g = ctx.get_excitons()
    for k, o in (("site", ox.site), ("hops", ox.hops), ("hash", ox.hash), ("drains", ox.drains),
                 ("disp", ox.dsp)):
        assert np.array_equal(g[k], o), k
    np.testing.assert_allclose(g["t_next"], ox.t_next, rtol=1e-12, atol=0)
    assert np.array_equal(ctx.get_hop_counts(), ox.site_count)
    s = ctx.get_samples()
    assert np.array_equal(s["n_recorded"], ox.k_rec)
    made = np.arange(5)[:, None] < ox.k_rec[None, :]
    assert np.array_equal(s["disp"][made], ox.rec_disp[made])
    tr = ctx.get_trace()
    n_hops = np.minimum(ox.hops[:nt].astype(np.int64), 200)
    assert np.array_equal(tr["n_hops"], n_hops)
    kept = np.arange(200)[None, :] < n_hops[:, None]
    assert np.array_equal(tr["sites"][kept], ox.tr_site[:nt][kept])
