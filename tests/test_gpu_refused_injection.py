"""An injection with drift that the film's links refuse leaves no half-made excitons behind: the calls
that need excitons refuse too, and the next injection makes a run equal to the oracle's."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_refused_injection_leaves_no_excitons(kmc, orc, nw):
    print("[gpu-refused-injection]", file=sys.stderr, flush=True)
    w = nw.film_small()
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=8)
    ctx.set_velocity(100.0)

    def sites(x):
        ctx.set_sites(x, net["y"], net["z"], net["ox"], net["oy"], net["oz"], net["left"],
                      net["right"], net["chirality"], net["flags"])
        ctx.set_rate_table(*nw.forster_tables(1))
        ctx.build_cells()
        ctx.build_rates(kmc.RATE_TABLE)

    i = int(np.flatnonzero(net["right"] >= 0)[7])
    j = int(net["right"][i])
    x, y, z = (net[k].copy() for k in ("x", "y", "z"))
    for a, k in ((x, "x"), (y, "y"), (z, "z")):
        a[j] = net[k][i]                     # two linked sites in one place
    net_y, net_z = net["y"], net["z"]
    net["y"], net["z"] = y, z
    sites(x)
    with pytest.raises(kmc.KmcError) as e:
        ctx.inject(500)
    assert e.value.code == kmc.ERR_GEOMETRY and f"sites {i} and {j} coincide" in str(e.value)
    with pytest.raises(kmc.KmcError) as e:
        ctx.run(10)
    assert e.value.code == kmc.ERR_STATE
    assert ctx.lib.kmc_get_excitons(ctx.h, *[None] * 6) == kmc.ERR_STATE
    assert ctx.lib.kmc_set_samples(ctx.h, 4, 1e-9) == kmc.ERR_STATE
    net["y"], net["z"] = net_y, net_z
    sites(net["x"])
    ctx.inject(300)
    o = orc.Excitons(ctx.get_csr(), net["flags"], 8, 300, velocity=100.0,
                     links=(net["left"], net["right"]))
    ctx.run(200)
    o.run(200)
    st = ctx.get_excitons()
    assert np.array_equal(st["hash"], o.hash) and np.array_equal(st["hops"], o.hops)
    ctx.close()
