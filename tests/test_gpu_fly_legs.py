"""Flights along tubes where their legs can go wrong: tubes of one site (no links), of two sites
(both headings end on the same segment), rings of two (left and right the same site) and of three,
sites with one link only in one direction, drains on the way, flights of many segments, exciton
numbers around a wave, and runs that stop and go on in the middle of a segment.  Against the
oracle: sites, hashes, hops, drains, headings, displacements, departure counts bit for bit; times,
offsets and records as the device's logarithm allows (1e-12 relative, 1e-11 v t for offsets)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
T_REL = 1e-12


def _cut(net):
    left, right = net["left"].copy(), net["right"].copy()
    n = net["n"]
    for s in range(0, n, 20):           # tubes of 20 sites, by kind
        kind = (s // 20) % 5
        idx = np.arange(s, min(s + 20, n))
        if kind == 1:                   # no links
            left[idx], right[idx] = -1, -1
        elif kind in (2, 3):            # pairs: open, or closed into a ring of two
            a, b = idx[0::2], idx[1::2]
            right[a], left[b] = b, a
            left[a], right[b] = (-1, -1) if kind == 2 else (b, a)
        elif kind == 4:                 # a ring of three, and a one-way link into it
            right[idx[:3]], left[idx[:3]] = np.roll(idx[:3], -1), np.roll(idx[:3], 1)
            left[idx[3]], right[idx[3]] = idx[0], -1
            left[idx[4]] = -1
    return left, right


@pytest.mark.parametrize("v,E", [(1.0, 63), (30.0, 65), (200.0, 257), (1000.0, 1)])
def test_flight_legs(kmc, orc, nw, v, E):
    print(f"[gpu-fly-legs] v {v} m/s, {E} excitons", file=sys.stderr, flush=True)
    w = nw.film_small()
    net = nw.build_network(w)
    net["left"], net["right"] = _cut(net)
    ctx = nw.make_context(w, net, seed=5)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    ctx.set_velocity(v)
    o = orc.Excitons(ctx.get_csr(), net["flags"], 5, E, velocity=v,
                     links=(net["left"], net["right"]))
    t_s = 2e-8
    ctx.inject(E)
    ctx.set_samples(13, t_s)
    o.set_samples(13, t_s)
    for hops in (17, 400):              # the second run goes on in the middle of segments
        ctx.run(hops)
        o.run(hops)
    st, fl, smp = ctx.get_excitons(), ctx.get_flight(), ctx.get_samples()
    assert np.array_equal(st["site"], o.site) and np.array_equal(st["hash"], o.hash)
    assert np.array_equal(st["hops"], o.hops) and np.array_equal(st["drains"], o.drains)
    assert np.array_equal(st["disp"], o.dsp) and np.array_equal(fl["heading"], o.heading)
    assert np.array_equal(ctx.get_hop_counts(), o.site_count)
    assert np.array_equal(smp["n_recorded"], o.k_rec) and o.k_rec.max() > 0
    np.testing.assert_allclose(st["t_next"], o.t_next, rtol=T_REL, atol=0)
    np.testing.assert_allclose(fl["t_last"], o.t_last, rtol=T_REL, atol=0)
    np.testing.assert_allclose(fl["offset"], o.s_off, rtol=T_REL, atol=1e-11 * v * t_s)
    np.testing.assert_allclose(smp["disp"], o.rec_disp, rtol=T_REL, atol=1e-11 * v * t_s)
    ctx.close()
