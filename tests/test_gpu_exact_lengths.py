"""The exact rate for acceptors of every number of cells around the lengths whose cell loop is
unrolled (up to 17 cells), even and odd, against the oracle's literal first_order.  Tolerance 1e-9
relative, as for the ten-cell tubes (another order of sums)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-exact-lengths]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("cells", [4, 5, 6, 8, 9, 11, 12, 13, 14, 15, 16, 17, 18, 19])
def test_every_length_matches_literal_first_order(orc, cells):
    from cnt_film_monte_carlo_amd import exciton as X
    d = a = X.CntModel(4, 2, cells)
    wide = 0.2 * X.EV
    t = X.Transfer(d, a, 300.0, broadening=wide)
    say(f"first_order (4,2) of {cells} cells, {t.info.n_terms} terms")
    assert t.info.n_terms > 0
    rng = np.random.default_rng(cells)
    n = 3
    th = np.concatenate([[0.0], rng.uniform(0, np.pi, n - 1)])
    z, s1, s2 = rng.uniform(1.5e-9, 8e-9, n), rng.uniform(-4e-9, 4e-9, n), rng.uniform(-4e-9, 4e-9, n)
    got = t.rates(th, z, s1, s2)
    td, ta = orc.tube_from_model(d), orc.tube_from_model(a)
    for k in range(n):
        ref, _ = orc.first_order(td, ta, 300.0, wide, z[k], s1[k], s2[k], th[k])
        assert got[k] == pytest.approx(ref, rel=1e-9, abs=1e-300), (k, got[k], ref)
    t.close()
