"""The hop kernel with a lane per exciton where the row-of-lanes kernel now takes the smaller launches
over: exciton numbers just above the line between them (128 per compute unit), with ragged ends,
idle and trapped lanes, rows over many lines, drains, times, records and a trace.  Against the
oracle: bitwise, times 1e-12 relative."""
import sys

import numpy as np
import pytest
import torch

from conftest import site_arrays

pytestmark = pytest.mark.gpu
NM = 1e-9
T_REL = 1e-12


def say(*a):
    print("[gpu-hop-lanes]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def line():
    return 128 * torch.cuda.get_device_properties(0).multi_processor_count


def _check(ctx, ox):
    g = ctx.get_excitons()
    for k, o in (("site", ox.site), ("hops", ox.hops), ("hash", ox.hash), ("drains", ox.drains),
                 ("disp", ox.dsp)):
        assert np.array_equal(g[k], o), k
    fin = np.isfinite(ox.t_next)
    assert np.array_equal(np.isfinite(g["t_next"]), fin)
    np.testing.assert_allclose(g["t_next"][fin], ox.t_next[fin], rtol=T_REL, atol=0)
    assert np.array_equal(ctx.get_hop_counts(), ox.site_count)


@pytest.fixture(scope="module")
def film(kmc, nw):
    w = nw.film_small()
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=47)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    yield dict(net=net, ctx=ctx, csr=ctx.get_csr())
    ctx.close()


@pytest.mark.parametrize("extra", [1, 63, 65, 257, 1023])
def test_ragged_exciton_counts(orc, film, line, extra):
    """The idle lanes of the last wave take part in every cooperative row load and count nothing; a
    budget of no hops changes nothing."""
    E, H = line + extra, 60
    say(f"{E} excitons x {H} hops")
    c = film["ctx"]
    c.inject(E)
    ox = orc.Excitons(film["csr"], film["net"]["flags"], seed=47, n_excitons=E)
    c.run(0)
    for h in (1, H - 1):
        c.run(h)
        ox.run(h)
    _check(c, ox)
    assert int(ox.site_count.sum()) == E * H


def test_times_records_and_trace(orc, film, line):
    """Runs up to times, the first below every first dwell, with records that fall due for excitons
    that make no hop, and a trace that goes on from run to run."""
    E = line + 130
    say(f"{E} excitons up to four times")
    c = film["ctx"]
    c.inject(E)
    ox = orc.Excitons(film["csr"], film["net"]["flags"], seed=47, n_excitons=E)
    dwell = 1.0 / float(np.mean(film["csr"]["gamma"]))
    for q in (c, ox):
        q.set_samples(9, 12 * dwell)
        q.set_trace(900, 25)
    for t in (0.5 * float(np.min(ox.t_next)), dwell, 7 * dwell, 15 * dwell):
        c.run(1 << 40, t_max=t)
        ox.run(1 << 40, t_max=t)
    _check(c, ox)
    s = c.get_samples()
    assert np.array_equal(s["n_recorded"], ox.k_rec)
    made = np.arange(9)[:, None] < ox.k_rec[None, :]
    assert np.array_equal(s["disp"][made], ox.rec_disp[made])
    assert np.array_equal(s["drains"][made], ox.rec_drain[made])
    tr = c.get_trace()
    n_hops = np.minimum(ox.hops[:900].astype(np.int64), 25)
    assert np.array_equal(tr["n_hops"], n_hops)
    kept = np.arange(25)[None, :] < n_hops[:, None]
    assert np.array_equal(tr["sites"][kept], ox.tr_site[:900][kept])
    np.testing.assert_allclose(tr["times"][kept], ox.tr_time[:900][kept], rtol=T_REL, atol=0)


@pytest.mark.parametrize("excitons", [2000, None])
def test_wide_rows_drains_and_dead_sites(kmc, orc, nw, line, excitons):
    """A 6 x 6 x 6 grid of segments 4 nm apart, 50 to 187 neighbours each (rows over 5 to 18 lines),
    sources on one face, drains on the other, and a few sites without rates, a source
    among them: excitons trapped from the start, on the way and after a drain.  The same through the
    kernel of the smaller launches."""
    rng = np.random.default_rng(17)
    g = np.arange(6) * 4 * NM
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    ori = rng.normal(size=pos.shape)
    ori /= np.linalg.norm(ori, axis=1, keepdims=True)
    flags = np.zeros(len(pos), np.uint8)
    flags[pos[:, 0] == 0] = 1
    flags[pos[:, 0] == g[-1]] |= 2
    net = site_arrays(pos, ori, flags=flags)
    ctx = kmc.Context(kmc.Config(cutoff=15 * NM, seed=5))
    ctx.set_sites(net["x"], net["y"], net["z"], net["ox"], net["oy"], net["oz"], flags=flags)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    c = ctx.get_csr()
    deg = np.diff(c["row_ptr"])
    assert deg.min() > 8 and deg.max() > 150
    for s in range(3, len(pos), 97):
        c["cum"][c["row_ptr"][s]:c["row_ptr"][s + 1]] = 0.0
    dead = np.arange(3, len(pos), 97)
    assert flags[dead].any()
    ctx.set_csr(c["row_ptr"], c["col"], c["cum"], c["disp"])
    csr = ctx.get_csr()
    E = excitons or line + 77
    say(f"{E} excitons, rows of {deg.min()} to {deg.max()}, {len(dead)} dead sites")
    ctx.inject(E)
    ox = orc.Excitons(csr, flags, seed=5, n_excitons=E)
    ctx.set_samples(5, 1e-9)
    ox.set_samples(5, 1e-9)
    ctx.set_hop_schedule(40)
    for h in (90, 30):
        ctx.run(h)
        ox.run(h)
    _check(ctx, ox)
    assert int(ox.drains.sum()) > 0 and not np.isfinite(ox.t_next).all()
    s = ctx.get_samples()
    assert np.array_equal(s["n_recorded"], ox.k_rec)
    made = np.arange(5)[:, None] < ox.k_rec[None, :]
    assert np.array_equal(s["disp"][made], ox.rec_disp[made])
    ctx.close()
