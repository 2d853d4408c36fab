"""Runs in which most excitons are trapped, so that far fewer can move than a launch looks at:
sites without rates that absorb (a run bounded by its hops looks at every exciton), and excitons
re-injected on such sites before their clock passes t_max (a run bounded by a time looks at those
too).  Against the oracle, bitwise, times 1e-12 relative; and the hop kernels may take no longer
than where every exciton moves."""
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
NM = 1e-9
T_REL = 1e-12


def say(*a):
    print("[gpu-few-movable]", *a, file=sys.stderr, flush=True)


def _check(ctx, ox):
    g = ctx.get_excitons()
    for k, o in (("site", ox.site), ("hops", ox.hops), ("hash", ox.hash), ("drains", ox.drains),
                 ("disp", ox.dsp)):
        assert np.array_equal(g[k], o), k
    fin = np.isfinite(ox.t_next)
    assert np.array_equal(np.isfinite(g["t_next"]), fin)
    np.testing.assert_allclose(g["t_next"][fin], ox.t_next[fin], rtol=T_REL, atol=0)
    assert np.array_equal(ctx.get_hop_counts(), ox.site_count)


def _film(kmc, dead, lost):
    """200 sites on a line.  Sites 0..99 are sources: the first `dead` have no rates, the next
    `lost` lead to a drain, the others into a ring of ten sites."""
    n = 200
    pos = np.zeros((n, 3))
    pos[:, 1] = 10 * NM * np.arange(n)
    flags = np.zeros(n, np.uint8)
    flags[:100] = kmc.SITE_SOURCE
    flags[100:110] = kmc.SITE_DRAIN
    to = np.full(n, -1)
    to[dead:dead + lost] = 100 + np.arange(lost) % 10
    to[dead + lost:100] = 110
    to[100:110] = 110
    to[110:120] = 110 + (np.arange(10) + 1) % 10
    has = to >= 0
    row_ptr = np.concatenate([[0], np.cumsum(has)]).astype(np.int64)
    col = to[has].astype(np.int32)
    cum = np.full(col.size, 1e12)
    disp = (pos[col] - pos[has]).astype(np.float32)
    ctx = kmc.Context(kmc.Config(cutoff=15 * NM, seed=23))
    o = np.zeros(n)
    ctx.set_sites(*pos.T.copy(), o, o + 1.0, o, flags=flags)
    ctx.set_csr(row_ptr, col, cum, disp)
    return ctx, ctx.get_csr(), flags



@pytest.mark.parametrize("t_max", [np.inf, 1e-6])
@pytest.mark.parametrize("dead,lost", [(98, 0), (49, 49)])
def test_most_excitons_trapped(kmc, orc, dead, lost, t_max):
    E = 320 * torch.cuda.get_device_properties(0).multi_processor_count
    hops = 2000
    say(f"{E} excitons, {dead} dead and {lost} lost sources of 100, t_max {t_max}")
    ctx, csr, flags = _film(kmc, dead, lost)
    ctx.inject(E)
    ox = orc.Excitons(csr, flags, seed=23, n_excitons=E)
    ctx.set_samples(6, 2e-9)
    ox.set_samples(6, 2e-9)
    ctx.set_hop_schedule(300)
    for h in (hops // 4, hops - hops // 4):
        ctx.run(h, t_max=t_max)
        ox.run(h, t_max=t_max)
    _check(ctx, ox)
    s = ctx.get_samples()
    assert np.array_equal(s["n_recorded"], ox.k_rec)
    made = np.arange(6)[:, None] < ox.k_rec[None, :]
    assert np.array_equal(s["disp"][made], ox.rec_disp[made])
    assert np.array_equal(s["drains"][made], ox.rec_drain[made])
    ctx.close()


@pytest.mark.parametrize("t_max", [np.inf, 1e-6])
def test_trapped_excitons_cost_nothing(kmc, t_max):
    E = 320 * torch.cuda.get_device_properties(0).multi_processor_count
    ms = {}
    for name, dead, lost in (("few move", 49, 49), ("all move", 0, 0)):
        ctx, _, _ = _film(kmc, dead, lost)
        ms[name] = np.inf
        for _ in range(4):
            ctx.inject(E)
            ctx.run(2000, t_max=t_max)
            ms[name] = min(ms[name], ctx.hop_time())
        ctx.close()
    say(f"t_max {t_max}: hop kernels {ms}")
    assert ms["few move"] <= 1.5 * ms["all move"]
