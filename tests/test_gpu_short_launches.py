"""Launches of a hop or a few with few excitons: the row-of-lanes kernel's fixed costs (the count of
excitons that can still move) against the lane-per-exciton kernel that one more exciton takes."""
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-short-launches]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def film(kmc, nw):
    w = nw.film_small()
    net = nw.build_network(w)
    ctx = nw.make_context(w, net, seed=61)
    ctx.set_rate_table(*nw.forster_tables(1))
    ctx.build_cells()
    ctx.build_rates(kmc.RATE_TABLE)
    yield ctx
    ctx.close()


def _hop_us(ctx, excitons, hops, count):
    ctx.inject(excitons)
    best = np.inf
    for _ in range(12):
        ctx.run(hops, count_sites=count)
        best = min(best, 1e3 * ctx.hop_time())
    return best


def test_many_waves_ending_together(film):
    line = 128 * torch.cuda.get_device_properties(0).multi_processor_count
    rows, lanes = (_hop_us(film, e, 1, False) for e in (line, line + 1))
    say(f"one hop of {line} excitons {rows:.1f} us, of one more {lanes:.1f} us")
    assert rows <= 3 * lanes
    assert film.run_stats() == (1, line + 1)
