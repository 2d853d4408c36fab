"""The hop kernel of launches with few excitons (a row of 16 lanes per exciton, 16 hops to a
batch) against the oracle where it can go wrong: excitons and hops around a wave's four and a
batch's sixteen, runs that end within a batch, and the line between it and the kernel for many
excitons.  Bar: everything bitwise, times 1e-12 relative."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T_REL = 1e-12


def say(*a):
    print("[gpu-hop-rows]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def film(kmc, nw):
    w = nw.film_small()
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=61)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    csr = ctx.get_csr()
    yield dict(w=w, net=net, ctx=ctx, csr=csr)
    ctx.close()


def _check(ctx, ox, bins):
    g = ctx.get_excitons()
    for k, o in (("site", ox.site), ("hops", ox.hops), ("hash", ox.hash), ("drains", ox.drains),
                 ("disp", ox.dsp)):
        assert np.array_equal(g[k], o), k
    np.testing.assert_allclose(g["t_next"], ox.t_next, rtol=T_REL, atol=0)
    assert np.array_equal(ctx.get_hop_counts(), ox.site_count)
    s = ctx.get_samples()
    assert np.array_equal(s["n_recorded"], ox.k_rec)
    valid = np.arange(bins)[:, None] < ox.k_rec[None, :]
    assert np.array_equal(s["disp"][valid], ox.rec_disp[valid])
    assert np.array_equal(s["drains"][valid], ox.rec_drain[valid])


# 32,768 excitons are the most that a 256-CU device gives a row of lanes each; one more takes the
# kernel with a lane per exciton
@pytest.mark.parametrize("E,H", [(1, 1), (3, 15), (4, 16), (5, 17), (67, 333), (1025, 31),
                                 (32768, 40), (32769, 40)])
def test_hop_budget(kmc, orc, film, E, H):
    say(f"{E} excitons x {H} hops, in two calls")
    c = film["ctx"]
    c.inject(E)
    ox = orc.Excitons(film["csr"], film["net"]["flags"], seed=61, n_excitons=E)
    T = float(np.median(ox.t_next)) * H / 4
    c.set_samples(7, T)
    ox.set_samples(7, T)
    for h in (H // 3, H - H // 3):
        c.run(h)
        ox.run(h)
    _check(c, ox, 7)


@pytest.mark.parametrize("E", [6, 2047, 32769])
def test_time_cap_and_trace(kmc, orc, film, E):
    """Excitons stop at t_max in the middle of a batch, whose later hops are dropped; the trace
    holds the hops made."""
    say(f"{E} excitons up to a time, traced")
    c = film["ctx"]
    c.inject(E)
    ox = orc.Excitons(film["csr"], film["net"]["flags"], seed=61, n_excitons=E)
    T = float(np.median(ox.t_next)) * 6
    nt = min(E, 300)
    for q in (c, ox):
        q.set_samples(9, T)
        q.set_trace(nt, 64)
    for f in (0.31, 1.0):
        c.run(1_000_000, t_max=f * T)
        ox.run(1_000_000, t_max=f * T)
    _check(c, ox, 9)
    tr = c.get_trace()
    made = np.minimum(ox.hops[:nt].astype(np.int64), 64)
    assert np.array_equal(tr["n_hops"], made)
    kept = np.arange(64)[None, :] < made[:, None]
    assert np.array_equal(tr["sites"][kept], ox.tr_site[:nt][kept])
    np.testing.assert_allclose(tr["times"][kept], ox.tr_time[:nt][kept], rtol=T_REL, atol=0)


def test_members_of_an_ensemble_agree(kmc, nw, film):
    """A member's kmc_run (row per exciton) and its ensemble run (lane per exciton): same bits."""
    w, net = film["w"], film["net"]
    ctxs = []
    for seed in (61, 61, 62):
        ctx = nw.make_context(w, net, seed=seed)
        c = film["csr"]
        ctx.set_csr(c["row_ptr"], c["col"], c["cum"], c["disp"])
        ctx.inject(777)
        ctx.set_samples(5, 1e-7)
        ctxs.append(ctx)
    ctxs[0].run(500)
    ens = kmc.Ensemble(ctxs[1:])
    ens.run(500)
    ens.close()
    a, b = ctxs[0].get_excitons(), ctxs[1].get_excitons()
    for k in a:
        assert np.array_equal(a[k], b[k]), k
    assert np.array_equal(ctxs[0].get_hop_counts(), ctxs[1].get_hop_counts())
    assert np.array_equal(ctxs[0].get_samples()["disp"], ctxs[1].get_samples()["disp"])
    for ctx in ctxs:
        ctx.close()
