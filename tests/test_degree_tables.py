"""The degree and chain tables that a run builds on first use: runs that read
them at once, on the same stream and from concurrent matchers, with thresholds
met by all, some and none of the vertices."""
import numpy as np
import pytest

import cuts_amd as F
import oracle

SHAPES = {
    "path4 from its end": ([(0, 1), (1, 2), (2, 3)], [0, 1, 2, 3]),
    "tail of two under a 4-star": ([(0, 1), (0, 2), (0, 3), (1, 4), (4, 5)], [0, 2, 3, 1, 4, 5]),
    "triangle, tail of two on the newest": ([(0, 1), (1, 2), (2, 0), (2, 3), (3, 4)], [0, 1, 2, 3, 4]),
    "triangle, a leaf each": ([(0, 1), (1, 2), (2, 0), (1, 3), (2, 4)], [0, 1, 2, 3, 4]),
}


def graph(V, seed):
    """Lists on both sides of a wave's 64 entries."""
    rng = np.random.default_rng(seed)
    e = [rng.integers(V, size=(2 * V, 2))]
    for i, d in enumerate((63, 64, 65, 128)):
        e.append(np.stack([np.full(d, i), rng.permutation(V)[:d]], 1))
    e = np.concatenate(e)
    return F.Graph.from_edges(V, e[e[:, 0] != e[:, 1]])


def loops(edges, k, heavy):
    """Arcs of the query with a self-loop on vertex k-1, which raises its threshold."""
    return [a for e in edges for a in (e, e[::-1])] + ([(k - 1, k - 1)] if heavy else [])


@pytest.mark.gpu
@pytest.mark.parametrize("heavy", [False, True])
@pytest.mark.parametrize("name", SHAPES)
def test_first_use(ctx, name, heavy):
    edges, order = SHAPES[name]
    k = len(order)
    arcs = np.asarray(loops(edges, k, heavy), dtype=np.uint32)
    q = F.Graph.from_arcs(k, arcs[:, 0], arcs[:, 1])
    g = graph(151, k + heavy)
    want = oracle.count(oracle.OGraph.from_view(g.view()), oracle.qmatrix(k, arcs.tolist()))
    for entry in (dict(), dict(noalloc=True), dict(flags=F.FLAG_NO_TWO_HOP)):
        dg = ctx.upload(g)  # a graph that holds no tables yet
        for _ in range(2):
            assert ctx.match(dg, F.Plan(q, order), **entry).count == want, entry
    dg = ctx.upload(g)
    results, _ = ctx.match_many(dg, [F.Plan(q, order) for _ in range(16)], workers=8)
    assert [r.count for r in results] == [want] * 16
    assert F.Batch(ctx, ctx.upload(g), [F.Plan(q, order)], arena_bytes=1 << 28).run().counts == [want]
