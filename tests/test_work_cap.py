"""A work cap tested on the device, without the readback of each level's work.

A capped run returns what the run with every level's readback returns (the
same decision, work, counts and level sizes), for caps around the whole work
and inside it, on a first run and on runs whose level sizes are remembered.
"""
import numpy as np
import pytest

import cuts_amd as F
from test_tail import CASES

SHAPES = {n: CASES[n] for n in ("path4 from its end", "triangle, leaf", "owners not adjacent",
                                "5-cycle, chord, two tails", "4-cycle, tail of two")}
SHAPES["4-clique"] = ([(a, b) for a in range(4) for b in range(a)], [0, 1, 2, 3])
SHAPES["5-cycle"] = ([(i, (i + 1) % 5) for i in range(5)], [0, 1, 2, 3, 4])


def graph(n, m, seed):
    rng = np.random.default_rng(seed)
    e = rng.integers(0, n, (m, 2))
    e = e[e[:, 0] != e[:, 1]]
    return F.Graph.from_edges(n, [(int(a), int(b)) for a, b in np.unique(np.sort(e, axis=1), axis=0)])


def outcome(r):
    return (r.work_capped, r.work, r.count, list(r.level_sizes), r.complete, r.roots_done, r.last_root)


@pytest.mark.gpu
@pytest.mark.parametrize("flags", [0, F.FLAG_NO_TWO_HOP | F.FLAG_NO_ARC_COMMON, F.FLAG_NO_PAIR | F.FLAG_NO_CHAIN])
@pytest.mark.parametrize("name", SHAPES)
def test_capped_runs_equal_runs_with_readbacks(name, flags):
    edges, order = SHAPES[name]
    k = len(order)
    ctx = F.Context()
    for n, m in ((60, 300), (4000, 12000)):  # one planning block; level 1 over more than one
        dg = ctx.upload(graph(n, m, seed=k))
        plan = F.Plan(F.Graph.from_edges(k, edges), order)
        total = ctx.match(dg, plan, flags=flags | F.FLAG_SYNC_LEVELS).work
        caps = sorted({1, total // 50, total // 5, total // 2, total * 9 // 10, total - 1, total, total + 1} - {0, -1})
        for cap in caps:
            for kw in ({}, {"roots": (0, n, 3)}, {"trunks": 3}):
                want = outcome(ctx.match(dg, plan, flags=flags | F.FLAG_SYNC_LEVELS, max_work=cap, **kw))
                for _ in range(3):
                    assert outcome(ctx.match(dg, plan, flags=flags, max_work=cap, **kw)) == want, (cap, total, kw)
        want = outcome(ctx.match(dg, plan, flags=flags))
        assert want[1] == total and not want[0]
        for cap in caps:  # level sizes remembered from the run before
            got = ctx.match(dg, plan, flags=flags, max_work=cap)
            assert got.work_capped == (cap < total)
            assert cap < total or outcome(got) == want


@pytest.mark.gpu
def test_remembered_sizes_with_a_smaller_budget():
    """A level that a remembered size lets run without its readback, in rows
    that a smaller budget makes too few: the run is repeated, not cut short."""
    edges, order = SHAPES["5-cycle, chord, two tails"]
    dg = F.Context().upload(graph(4000, 12000, seed=7))
    plan = F.Plan(F.Graph.from_edges(len(order), edges), order)
    for flags in (0, F.FLAG_NO_PAIR | F.FLAG_NO_CHAIN):
        want = outcome(dg.ctx.match(dg, plan, flags=flags | F.FLAG_SYNC_LEVELS))
        for budget in (0, 2048, 0, 2048):
            assert outcome(dg.ctx.match(dg, plan, flags=flags, budget=budget)) == want


@pytest.mark.gpu
@pytest.mark.parametrize("flags", [0, F.FLAG_NO_PAIR | F.FLAG_NO_CHAIN])
@pytest.mark.parametrize("name", SHAPES)
def test_the_cap_in_every_trunk(name, flags):
    """The cap a candidate below, at and above the work of each number of
    trunks: the run ends at the last level of one trunk, or in the next."""
    edges, order = SHAPES[name]
    dg = F.Context().upload(graph(60, 300, seed=len(order)))
    plan = F.Plan(F.Graph.from_edges(len(order), edges), order)
    for trunks in (2, 5):
        size = -(-60 // trunks)
        ends = [dg.ctx.match(dg, plan, flags=flags | F.FLAG_SYNC_LEVELS, roots=(0, size * t, 1)).work
                for t in range(1, trunks + 1)]
        for cap in sorted({e + d for e in ends for d in (-1, 0, 1)} - {-1, 0}):
            runs = [dg.ctx.match(dg, plan, flags=flags | f, max_work=cap, trunks=trunks) for f in (F.FLAG_SYNC_LEVELS, 0, 0)]
            want, *got = [outcome(r) + (r.chunks,) for r in runs]
            assert got == [want, want], (cap, ends, trunks)
