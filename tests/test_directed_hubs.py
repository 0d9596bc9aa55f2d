"""Hub bitmaps of directed graphs' out-lists and in-lists: graphs with long
lists on both sides, on one, and on none, counts equal to the oracle's with
and without the bitmaps; a query self-loop, whose threshold the constraints
of its position do not imply."""
import numpy as np
import pytest

import cuts_amd as F
import oracle

QUERIES = {
    "two paths": (4, [(0, 1), (0, 2), (1, 3), (2, 3)]),
    "two paths back": (4, [(1, 0), (2, 0), (3, 1), (3, 2)]),
    "feed-forward, closed": (5, [(0, 1), (0, 2), (1, 2), (2, 3), (1, 4), (3, 4)]),
    "both ways": (4, [(0, 1), (1, 0), (1, 2), (2, 0), (2, 3), (0, 3)]),
    "loop on the last": (4, [(0, 1), (0, 2), (1, 3), (2, 3), (3, 3)]),
}


def graph(seed, out_hubs, in_hubs):
    rng = np.random.default_rng(seed)
    V = 210
    e = [rng.integers(V, size=(420, 2))]
    for i in range(out_hubs):
        t = rng.permutation(V)[:90]
        e.append(np.stack([np.full(len(t), i), t], 1))
    for i in range(in_hubs):
        t = rng.permutation(V)[:90]
        e.append(np.stack([t, np.full(len(t), 20 + i)], 1))
    e = np.concatenate(e)
    loops = np.stack([np.arange(0, 40, 3)] * 2, 1)
    e = np.concatenate([e[e[:, 0] != e[:, 1]], loops])
    return F.Graph.from_arcs(V, e[:, 0], e[:, 1])


@pytest.mark.gpu
@pytest.mark.parametrize("out_hubs,in_hubs", [(3, 3), (4, 0), (0, 4), (0, 0)])
def test_counts(ctx, out_hubs, in_hubs):
    g = graph(10 * out_hubs + in_hubs, out_hubs, in_hubs)
    v = g.view()
    assert not v["symmetric"]
    assert (np.diff(v["out_off"].astype(np.int64)).max() >= 32) == (out_hubs > 0)
    assert (np.diff(v["in_off"].astype(np.int64)).max() >= 32) == (in_hubs > 0)
    og = oracle.OGraph.from_view(v)
    dg = ctx.upload(g)
    plans, wants = [], []
    for name, (k, arcs) in QUERIES.items():
        a = np.asarray(arcs, dtype=np.uint32)
        p = F.Plan(F.Graph.from_arcs(k, a[:, 0], a[:, 1]))
        want = oracle.count(og, oracle.qmatrix(k, arcs))
        cpu = oracle.trie_cpu(og, oracle.qmatrix(k, arcs), p.order, nthreads=4)
        for flags in (0, F.FLAG_NO_BITMAP, F.FLAG_SYNC_LEVELS, F.FLAG_PROFILE):
            r = ctx.match(dg, p, flags=flags)
            assert r.count == want, (name, flags)
            assert r.level_sizes == [cpu.level[i] for i in range(k)], (name, flags)
        rows = ctx.match(dg, p, write=True, emb_cap=max(want, 1)).rows
        assert len(rows) == want and len({tuple(x) for x in rows.tolist()}) == want, name
        plans.append(p)
        wants.append(want)
    assert F.Batch(ctx, dg, plans, arena_bytes=1 << 28).run().counts == wants
