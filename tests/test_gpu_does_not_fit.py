"""A sampling grid, a trace or a list of geometries that does not fit the device is refused and leaves
nothing half made: the run after it equals the oracle's."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-does-not-fit]", *a, file=sys.stderr, flush=True)


def test_grid_and_trace(kmc, orc, nw):
    w = nw.film_small()
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=8)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    E = 700
    ctx.inject(E)
    o = orc.Excitons(ctx.get_csr(), net["flags"], seed=8, n_excitons=E)
    ctx.set_samples(4, 1e-8)
    ctx.set_trace(10, 50)
    say("a grid of 2^31 - 1 bins: 11 TiB a component")
    with pytest.raises(kmc.KmcError) as e:
        ctx.set_samples((1 << 31) - 1, 1e-8)
    assert e.value.code == kmc.ERR_ALLOC
    say("a trace of 2^36 hops for 500 excitons: 128 TiB of sites")
    with pytest.raises(kmc.KmcError) as e:
        ctx.set_trace(500, 1 << 36)
    assert e.value.code == kmc.ERR_ALLOC
    ctx.run(300)
    o.run(300)
    g = ctx.get_excitons()
    assert np.array_equal(g["hash"], o.hash) and np.array_equal(g["hops"], o.hops)
    assert np.array_equal(g["disp"], o.dsp)
    for call, args in ((ctx.lib.kmc_get_samples, 3), (ctx.lib.kmc_get_trace, 3)):
        assert call(ctx.h, *[None] * args) == kmc.ERR_STATE
    ctx.close()


def test_geometries():
    from cnt_film_monte_carlo_amd import exciton as X
    d = X.CntModel(4, 2, 3)
    t = X.Transfer(d, d, 300.0)
    g = [np.array([v]) for v in (0.3, 2e-9, 1e-9, -1e-9)]
    before = t.rates(*g)
    p = [v.ctypes.data_as(C.POINTER(C.c_double)) for v in (*g, np.zeros(1))]
    say("2^40 geometries: 32 TiB of them on the device")
    assert t.lib.kmc_transfer_rates(t.h, 1 << 40, *p, None) < 0   # before it reads the arrays
    assert np.array_equal(t.rates(*g), before)
    t.close()
