"""A new injection and a new sampling grid start from zero in the buffers of the run before (the
same sizes keep the same buffers): counts, records, recorded bins, for sizes that leave every
remainder of 16 bytes.  Whole numbers and zeros: exact."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,bins", [(1, 1), (2, 3), (3, 1), (5, 7), (257, 1), (1023, 5)])
def test_buffers_start_from_zero(kmc, nw, E, bins):
    print(f"[gpu-clear] {E} excitons, {bins} bins", file=sys.stderr, flush=True)
    w = nw.film_small()
    ctx = nw.make_context(w, nw.build_network(w), seed=3)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    ctx.inject(E)
    ctx.set_samples(bins, 1e-9)
    ctx.run(400)
    first = ctx.get_excitons()
    assert ctx.get_hop_counts().sum() == 400 * E and ctx.get_samples()["n_recorded"].max() > 0
    ctx.set_samples(bins, 1e-9)          # the grid anew, over the records of the run
    smp = ctx.get_samples()
    assert not smp["n_recorded"].any() and not smp["disp"].any() and not smp["drains"].any()
    ctx.inject(E)
    assert not ctx.get_hop_counts().any()
    ctx.set_samples(bins, 1e-9)
    ctx.run(400)
    again = ctx.get_excitons()
    for k in ("site", "hash", "hops", "drains", "disp", "t_next"):
        assert np.array_equal(first[k], again[k]), k
    assert ctx.get_hop_counts().sum() == 400 * E
    ctx.close()
