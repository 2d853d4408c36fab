"""Contact mode's repopulation of both contacts in one pass where it can go wrong: live counts at
and around a tile of 2,048 slots, empty and one-sided contacts, more new particles than kept ones,
and two sections (their closed ranges meet, so the contacts are cleared one after the other),
against the oracle bit for bit, with and without drift (times 1e-12 relative)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NM = 1e-9


@pytest.mark.parametrize("v", [0.0, 10.0])
@pytest.mark.parametrize("n_seg,c1,c2", [(4, 512, 512), (4, 511, 512), (4, 513, 512), (4, 1, 0),
                                         (4, 0, 1), (3, 4100, 2), (2, 300, 40), (2, 1024, 1024)])
def test_contact_repopulation_edges(kmc, orc, nw, n_seg, c1, c2, v):
    print(f"[gpu-contact-move] {n_seg} sections, {c1}/{c2}, v {v}", file=sys.stderr, flush=True)
    w = nw.film_small()
    net = nw.build_network(w)
    net["flags"] = np.zeros(net["n"], np.uint8)
    for side in ("left", "right"):      # no link across the film's y period (open axes)
        lk = net[side]
        far = (lk >= 0) & (np.abs(net["y"][np.maximum(lk, 0)] - net["y"]) > 0.25 * np.ptp(net["y"]))
        net[side] = np.where(far, -1, lk).astype(np.int32)
    tab = nw.forster_tables(1)
    ctx = kmc.Context(kmc.Config(cutoff=w.cutoff, min_distance=0.4 * NM, seed=41))
    ctx.set_sites(net["x"], net["y"], net["z"], net["ox"], net["oy"], net["oz"], net["left"],
                  net["right"], net["chirality"], net["flags"])
    ctx.set_rate_table(*tab)
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    if v > 0.0:
        ctx.set_velocity(v)
    cap, dt, steps = 24000, 2e-8, 6
    ctx.contact_init(n_seg, c1, c2, cap)
    pop, cur, live = ctx.contact_run(dt, steps)
    onet = orc.Net(net, w.cutoff, 0.4 * NM)
    onet.set_table(*tab)
    ref = orc.contact(net, onet.csr(0), 41, n_seg, c1, c2, cap, dt, steps, velocity=v)
    assert np.array_equal(pop, ref["population"]) and np.array_equal(cur, ref["crossings"])
    assert np.array_equal(live, ref["n_live"])
    p = ctx.contact_particles()
    assert np.array_equal(p["id"], ref["id"]) and np.array_equal(p["site"], ref["site"])
    assert np.array_equal(p["hops"], ref["hops"])
    np.testing.assert_allclose(p["y"], ref["y"], rtol=1e-12, atol=0)
    np.testing.assert_allclose(p["t_next"], ref["t_next"], rtol=1e-12)
    assert ctx.contact_stats()[0] == ref["hops_made"]
    ctx.close()


@pytest.mark.parametrize("n_chir", [2, 3, 9, 16])
def test_contact_order_keys(kmc, orc, nw, n_chir):
    """The slots' order with one to four key bits for the chirality, 16 being the most a film has
    (one rate for all pairs, 15 nm cutoff): every particle as the oracle's."""
    print(f"[gpu-contact-move] {n_chir} chiralities", file=sys.stderr, flush=True)
    w = nw.film_small()
    net = nw.build_network(w)
    net["flags"] = np.zeros(net["n"], np.uint8)
    net["chirality"] = ((np.arange(net["n"]) // 20) % n_chir).astype(np.uint8)
    tab = ([0.0], [0.0], [0.0], [0.0], np.full(n_chir * n_chir, 1e12))
    ctx = kmc.Context(kmc.Config(cutoff=w.cutoff, min_distance=0.4 * NM, seed=43))
    ctx.set_sites(net["x"], net["y"], net["z"], net["ox"], net["oy"], net["oz"], net["left"],
                  net["right"], net["chirality"], net["flags"])
    ctx.set_rate_table(*tab)
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    ctx.contact_init(5, 900, 100, 8000)
    pop, cur, live = ctx.contact_run(2e-12, 4)
    onet = orc.Net(net, w.cutoff, 0.4 * NM)
    onet.set_table(*[np.asarray(t, float) for t in tab])
    ref = orc.contact(net, onet.csr(0), 43, 5, 900, 100, 8000, 2e-12, 4)
    assert np.array_equal(pop, ref["population"]) and np.array_equal(cur, ref["crossings"])
    assert np.array_equal(live, ref["n_live"]) and ref["hops_made"] > 1000
    p = ctx.contact_particles()
    for k in ("id", "site", "hops"):
        assert np.array_equal(p[k], ref[k]), k
    ctx.close()
