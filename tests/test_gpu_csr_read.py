"""The CSR read back on both sides of the sizes where it is unpacked on the host (32,768 sites;
65,536 pairs, 16,384 for columns or displacements alone), whole and array by array, against the
oracle's: bitwise."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NM = 1e-9


def say(*a):
    print("[gpu-csr-read]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("n_tubes", [3, 130, 180, 490, 600, 1900])
def test_every_array_alone(kmc, orc, nw, n_tubes):
    w = nw.film_small()
    w.net.n_tubes = n_tubes
    w.net.box_hi = (n_tubes * 2 * NM, 500 * NM, 50 * NM)
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=3)
    tables = nw.forster_tables(1)
    ctx.set_rate_table(*tables)
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    onet = orc.Net(net, w.cutoff, 0.4 * NM, kmc.PERIODIC_Y, period_lo=(0.0, w.period_y[0], 0.0),
                   period_len=(0.0, w.period_y[1], 0.0))
    onet.set_table(*tables)
    want = onet.csr(0)
    n, nnz = ctx.n_sites, ctx.nnz
    say(f"{n} sites, {nnz} pairs")
    got = ctx.get_csr()
    for k in ("row_ptr", "col", "cum", "disp"):
        assert np.array_equal(got[k], want[k]), k
    ends = want["row_ptr"][1:]
    gamma = np.where(np.diff(want["row_ptr"]) > 0, want["cum"][np.maximum(ends - 1, 0)], 0.0)
    assert np.array_equal(got["gamma"], gamma)
    arrays = {"row_ptr": (np.zeros(n + 1, np.int64), kmc._I64), "col": (np.zeros(nnz, np.int32), kmc._I32),
              "cum": (np.zeros(nnz), kmc._D), "disp": (np.zeros((nnz, 3), np.float32), kmc._F),
              "gamma": (np.zeros(n), kmc._D)}
    order = list(arrays)
    for k, (a, ct) in arrays.items():
        ptrs = [a.ctypes.data_as(ct) if q == k else None for q in order]
        assert ctx.lib.kmc_get_csr(ctx.h, *ptrs) == 0
        assert np.array_equal(a, got[k]), k
    ctx.close()
