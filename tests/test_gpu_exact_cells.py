"""The exact rate's sums over pairs of unit cells about the tube's centre against the oracle's
literal first_order: tubes of one cell, odd and even numbers of cells, donors around a multiple of
a chunk's 64 atoms.  Tolerance 1e-9 relative, as for the ten-cell tubes (another order of sums)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-exact-cells]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("donor,acceptor", [((4, 2, 1), (4, 2, 1)), ((4, 2, 2), (4, 2, 3)),
                                            ((4, 2, 7), (4, 2, 2)), ((4, 2, 5), (4, 2, 10)),
                                            ((4, 2, 10), (5, 4, 5))])
def test_cells_match_literal_first_order(orc, donor, acceptor):
    from cnt_film_monte_carlo_amd import exciton as X
    say(f"first_order {donor} -> {acceptor} (n, m, cells)")
    d, a = X.CntModel(*donor), X.CntModel(*acceptor)
    wide = 0.2 * X.EV   # a broadening that matches states of tubes of different lengths
    t = X.Transfer(d, a, 300.0, broadening=wide)
    assert t.info.n_terms > 0
    rng = np.random.default_rng(8)
    n = 5
    th = np.concatenate([[0.0], rng.uniform(0, np.pi, n - 1)])
    z, s1, s2 = rng.uniform(1.5e-9, 8e-9, n), rng.uniform(-4e-9, 4e-9, n), rng.uniform(-4e-9, 4e-9, n)
    got = t.rates(th, z, s1, s2)
    td, ta = orc.tube_from_model(d), orc.tube_from_model(a)
    for k in range(n):
        ref, _ = orc.first_order(td, ta, 300.0, wide, z[k], s1[k], s2[k], th[k])
        assert got[k] == pytest.approx(ref, rel=1e-9, abs=1e-300), (k, got[k], ref)
    # a launch of one workgroup per geometry carries the same bits
    rep = 4200 // n + 1
    whole = t.rates(np.tile(th, rep), np.tile(z, rep), np.tile(s1, rep), np.tile(s2, rep))
    assert np.array_equal(whole[:n], got) and np.array_equal(whole[-n:], got)
    t.close()
