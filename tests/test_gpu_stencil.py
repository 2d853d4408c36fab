"""The pair search (a lane per stencil cell) at small cell grids against the oracle's CSR: one, two
and three cells along an axis, periodic or open, where stencils wrap, drop cells or drop duplicates.
Bitwise."""
import sys

import numpy as np
import pytest

from conftest import site_arrays

pytestmark = pytest.mark.gpu
NM = 1e-9


def say(*a):
    print("[gpu-stencil]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("mask", [0, 1, 2, 5, 7])
@pytest.mark.parametrize("edge", [4.1, 6.4, 9.9])   # 2, 3 and 4 cells of 2 nm and more per period
@pytest.mark.parametrize("n", [1, 3, 257])
def test_small_grids(kmc, orc, nw, mask, edge, n):
    say(f"{n} sites, box {edge} nm, periodic mask {mask}")
    rng = np.random.default_rng(n + mask)
    pos = rng.uniform(0, edge * NM, (n, 3)) * 0.999
    pos[:, 2] *= 0.3 if not mask & 4 else 1.0     # one cell along an open z
    a = rng.uniform(0, 2 * np.pi, n)
    ori = np.stack([np.cos(a), np.sin(a), np.zeros(n)], 1)
    net = site_arrays(pos, ori, chir=rng.integers(0, 2, n))
    per = edge * NM
    ctx = kmc.Context(kmc.Config(cutoff=2 * NM, min_distance=0.1 * NM, periodic_mask=mask,
                                 period_len=(per, per, per), seed=1))
    ctx.set_sites(net["x"], net["y"], net["z"], net["ox"], net["oy"], net["oz"],
                  chirality=net["chirality"], flags=net["flags"])
    tab = nw.forster_tables(2)
    ctx.set_rate_table(*tab)
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    onet = orc.Net(net, 2 * NM, 0.1 * NM, mask, (0, 0, 0), (per, per, per))
    onet.set_table(*tab)
    g, o = ctx.get_csr(), onet.csr(0)
    for k in ("row_ptr", "col", "cum", "disp"):
        assert np.array_equal(g[k], o[k]), k
    ctx.close()
