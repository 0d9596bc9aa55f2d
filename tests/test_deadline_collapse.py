"""A pair level that collapses into the expansion of position k-4, under a
deadline: a trunk cut short is rolled back in all four of its sums."""
import pytest

import cuts_amd as F
from cuts_amd import workloads as W


@pytest.mark.gpu
def test_counts_of_the_roots_done(ctx):
    g = F.Graph.chung_lu(36692, 183831, 2.1, 1400, 11)
    dg = ctx.upload(g)
    p = F.Plan(W.query_graph(W.C4_2PEND))
    whole = ctx.match(dg, p)
    for kw in (dict(time_limit_ms=1e6), dict(time_limit_ms=1e6, trunks=37), dict(time_limit_ms=1e6, budget=1 << 20)):
        r = ctx.match(dg, p, **kw)
        assert (r.count, r.level_sizes, r.complete) == (whole.count, whole.level_sizes, True)
    cut = 0
    for ms in (0.05, 0.3, 0.6, 1.2, 2.4):
        r = ctx.match(dg, p, time_limit_ms=ms, trunks=64)
        if r.complete:
            assert (r.count, r.level_sizes) == (whole.count, whole.level_sizes)
            continue
        cut += 1
        if r.roots_done == 0:
            assert r.count == 0
            continue
        # level 0 counts the roots there are, the others what the finished trunks took
        part = ctx.match(dg, p, roots=(0, r.last_root + 1, 1))
        assert part.level_sizes[0] == r.roots_done
        assert (r.count, r.level_sizes[1:]) == (part.count, part.level_sizes[1:]), ms
    assert cut
