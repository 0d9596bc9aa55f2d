"""The last two positions counted from whole prefixes (positions 0..k-3).

A pair of leaves of which one hangs on position k-3 itself has
|A| * |B| - |A & B| completions per row of level k-3; a position k-2 joined
to two older positions followed by a leaf on one of them has
|A & B| * (|C| - 1); a 2-edge tail on position k-3 takes the chain's closed
form with an intersection per prefix vertex.  Where an index holds |N(u) & N(w)| the expansion of
position k-3 counts them, else stored rows do and the intersections are
walked.  Counts equal the oracle's, level sizes and merge-model bytes the CPU
trie walk's, in every mode that changes the route.
"""
import numpy as np
import pytest

import cuts_amd as F
import oracle

# name -> (edges, order); the order puts the leaf's owner at position k-3
CASES = {
    "path3": ([(0, 1), (0, 2)], [0, 1, 2]),
    "path4, inner first": ([(0, 1), (1, 2), (2, 3)], [1, 2, 0, 3]),
    "path4, from one side": ([(0, 1), (1, 2), (2, 3)], [2, 1, 0, 3]),
    "two leaves on the newest": ([(0, 1), (1, 2), (1, 3)], [0, 1, 2, 3]),
    "owners not adjacent": ([(0, 1), (1, 2), (0, 3), (2, 4)], [0, 1, 2, 3, 4]),
    "triangle, a leaf each": ([(0, 1), (1, 2), (2, 0), (1, 3), (2, 4)], [0, 1, 2, 3, 4]),
    "5-cycle, chord, two tails": ([(0, 1), (1, 2), (2, 3), (3, 4), (4, 0), (0, 2), (3, 5), (4, 6)],
                                  [0, 2, 1, 3, 4, 5, 6]),
    "diamond, leaf": ([(0, 1), (0, 2), (1, 2), (1, 3), (2, 3), (1, 4)], [0, 1, 2, 3, 4]),
    "triangle, leaf": ([(0, 1), (1, 2), (2, 0), (0, 3)], [0, 1, 2, 3]),
    "path3 from its end": ([(0, 1), (1, 2)], [0, 1, 2]),
    "path4 from its end": ([(0, 1), (1, 2), (2, 3)], [0, 1, 2, 3]),
    "triangle, tail of two on the newest": ([(0, 1), (1, 2), (2, 0), (2, 3), (3, 4)], [0, 1, 2, 3, 4]),
    "4-cycle, tail of two": ([(0, 1), (1, 2), (2, 3), (3, 0), (3, 4), (4, 5)], [0, 1, 2, 3, 4, 5]),
    "5-cycle, chord, tail of two": ([(0, 1), (1, 2), (2, 3), (3, 4), (4, 0), (0, 2), (4, 5), (5, 6)],
                                    [0, 1, 2, 3, 4, 5, 6]),
    "4-cycle, leaf": ([(0, 1), (1, 2), (2, 3), (3, 0), (0, 4)], [0, 1, 2, 3, 4]),
}
FLAGS = [0, F.FLAG_NO_BITMAP, F.FLAG_NO_TWO_HOP, F.FLAG_NO_TWO_HOP | F.FLAG_NO_BITMAP,
         F.FLAG_NO_TWO_HOP | F.FLAG_NO_ARC_COMMON, F.FLAG_NO_PAIR, F.FLAG_NO_CHAIN]


def tail_kind(k, edges, order):
    at = {v: i for i, v in enumerate(order)}
    back = [set() for _ in range(k)]
    for a, b in edges:
        i, j = at[a], at[b]
        back[max(i, j)].add(min(i, j))
    if back[k - 1] == {k - 2}:
        return 3 if back[k - 2] == {k - 3} else 0
    if len(back[k - 1]) != 1:
        return 0
    (c,) = back[k - 1]
    if len(back[k - 2]) == 1:
        return 1 if k - 3 in back[k - 2] | back[k - 1] else 0
    return 2 if len(back[k - 2]) == 2 and c in back[k - 2] else 0


def test_cases_cover_every_kind():
    kinds = [tail_kind(len(o), e, o) for e, o in CASES.values()]
    assert 0 not in kinds and kinds.count(1) >= 6 and kinds.count(2) >= 2 and kinds.count(3) >= 5


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("hubs", [False, True])
def test_counts_sizes_and_bytes(ctx, monkeypatch, name, hubs):
    """hubs: no two-hop index but hub rows for a dozen vertices, the index
    that graphs too large for the other one have."""
    if hubs:
        monkeypatch.setenv("CUTS_H2_MAX_WEDGES", "0")
        monkeypatch.setenv("CUTS_H2_HUB_MIN_DEG", "8")
        monkeypatch.setenv("CUTS_H2_HUB_ROWS", "12")
    edges, order = CASES[name]
    k = len(order)
    g = F.Graph.chung_lu(97, 330, 2.3, 0, 40 + k)
    og = oracle.OGraph.from_view(g.view())
    qa = oracle.qmatrix(k, oracle.undirected(edges))
    want = oracle.count(og, qa)
    p = F.Plan(F.Graph.from_edges(k, edges), order)
    cpu = oracle.trie_cpu(og, qa, p.order, nthreads=4)
    assert cpu.count == want
    sizes = [cpu.level[i] for i in range(k)]
    dg = ctx.upload(g)
    assert (dg.info()["hub_rows"] > 0) == hubs
    for flags in FLAGS:
        for extra in (0, F.FLAG_SYNC_LEVELS, F.FLAG_PROFILE, F.FLAG_NO_FUSE):
            r = ctx.match(dg, p, flags=flags | extra)
            assert (r.count, r.level_sizes) == (want, sizes), (flags, extra)
            if extra == F.FLAG_PROFILE:
                assert sum(r.merge_bytes.values()) == cpu.bytes, flags
        # a repeated query's chained levels, small buffers, trunks, a root sample
        assert ctx.match(dg, p, flags=flags).count == want
        assert ctx.match(dg, p, flags=flags, budget=2048).count == want
        assert ctx.match(dg, p, flags=flags, trunks=7).count == want
        assert ctx.match(dg, p, flags=flags, noalloc=True).count == want
        halves = [ctx.match(dg, p, flags=flags, roots=(i, g.V, 2)) for i in (0, 1)]
        assert sum(h.count for h in halves) == want
        assert [sum(h.level_sizes[i] for h in halves) for i in range(k)] == sizes


@pytest.mark.gpu
def test_thresholds_above_two_and_a_deadline(ctx):
    """Query self-loops raise a leaf's threshold past what the indexes serve;
    a run under a deadline counts the roots that it finished."""
    g = F.Graph.chung_lu(300, 1500, 2.2, 0, 5)
    og = oracle.OGraph.from_view(g.view())
    arcs = [(0, 1), (1, 2), (2, 0), (1, 3), (2, 4)]
    for loops in ([(4, 4)], [(3, 3), (4, 4)]):
        both = [a for e in arcs for a in (e, e[::-1])] + loops
        a = np.asarray(both, dtype=np.uint32)
        q = F.Graph.from_arcs(5, a[:, 0], a[:, 1])
        want = oracle.count(og, oracle.qmatrix(5, both))
        p = F.Plan(q, [0, 1, 2, 3, 4])
        dg = ctx.upload(g)
        for flags in FLAGS:
            assert ctx.match(dg, p, flags=flags).count == want, (loops, flags)
            assert ctx.match(dg, p, flags=flags, time_limit_ms=1e6, trunks=9).count == want


@pytest.mark.gpu
@pytest.mark.parametrize("queue", ["level", "persistent"])
def test_batch_counts_them_too(ctx, queue):
    """The batched queue, with its flushes cut into items of one candidate, of
    a few, and not at all."""
    g = F.Graph.chung_lu(160, 700, 2.2, 0, 12)
    og = oracle.OGraph.from_view(g.view())
    plans, want = [], []
    for edges, order in CASES.values():
        k = len(order)
        plans.append(F.Plan(F.Graph.from_edges(k, edges), order))
        want.append(oracle.count(og, oracle.qmatrix(k, oracle.undirected(edges))))
    dg = ctx.upload(g)
    single = [ctx.match(dg, p) for p in plans]
    assert [r.count for r in single] == want
    for kw in (dict(), dict(item_work=1), dict(item_work=50, vchunk=9), dict(item_work=1 << 20)):
        for flags in (0, F.FLAG_NO_TWO_HOP, F.FLAG_NO_PAIR, F.FLAG_NO_CHAIN, F.FLAG_NO_BITMAP):
            b = F.Batch(ctx, dg, plans, queue=queue, flags=flags, arena_bytes=1 << 28, **kw)
            for _ in range(2):
                r = b.run()
                assert r.counts == want, (kw, flags)
                assert r.level_sizes == [s.level_sizes for s in single], (kw, flags)
