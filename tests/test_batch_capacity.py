"""The batch queue's capacity counts flushes of up to 256 rows of whole
level-0 items: finer items, and the flushes that come of them, take no run's
capacity away."""
import pytest

import cuts_amd as F
import oracle

SHAPES = {"4-cycle": (4, [(0, 1), (1, 2), (2, 3), (3, 0)]), "4-clique": (4, [(a, b) for a in range(4) for b in range(a)])}


@pytest.mark.gpu
@pytest.mark.parametrize("queue", ["level", "persistent"])
@pytest.mark.parametrize("name", SHAPES)
def test_least_capacity_is_that_of_uncut_items(ctx, name, queue):
    k, edges = SHAPES[name]
    g = F.Graph.chung_lu(4000, 12000, 2.4, 0, 2)
    dg = ctx.upload(g)
    plans = [F.Plan(F.Graph.from_edges(k, edges))]
    want = oracle.count(oracle.OGraph.from_view(g.view()), oracle.qmatrix(k, oracle.undirected(edges)))

    def run(cap, work):
        # item_work of 2^20: a flush is one item; level 0 is 16 items of 256 roots either way
        b = F.Batch(ctx, dg, plans, queue=queue, queue_cap=cap, item_work=work, vchunk=256, arena_bytes=1 << 28)
        return [b.run().counts for _ in range(2)]

    def fits(cap, work):
        try:
            return run(cap, work) == [[want]] * 2
        except F.CutsError as e:
            assert e.code == -5 and "work queue full" in str(e)
            return False

    lo, hi = 16, 1 << 15
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if fits(mid, 1 << 20) else (mid, hi)
    assert not fits(hi - 1, 1 << 20) and fits(hi, 1 << 20)
    assert not fits(hi - 1, 16384)
    # flushes at 16,384 candidates are a few more than those of full stages alone
    cap = hi + hi // 100 + 4
    assert fits(cap, 16384), cap


@pytest.mark.gpu
@pytest.mark.parametrize("queue", ["level", "persistent"])
def test_level_0_in_whole_items(ctx, queue):
    """The 4-clique's run with one level-0 item flushes 171 times at its
    largest level; items of 512 roots cut into items of 2,048 candidates flush
    204 times."""
    g = F.Graph.chung_lu(4000, 12000, 2.4, 0, 2)
    dg = ctx.upload(g)
    k, edges = SHAPES["4-clique"]
    p = F.Plan(F.Graph.from_edges(k, edges))
    want = ctx.match(dg, p)
    b = F.Batch(ctx, dg, [p], queue=queue, queue_cap=171, arena_bytes=1 << 28)
    for _ in range(3):
        r = b.run()
        assert (r.counts, r.level_sizes) == ([want.count], [want.level_sizes])
    with pytest.raises(F.CutsError):
        F.Batch(ctx, dg, [p], queue=queue, queue_cap=170, arena_bytes=1 << 28).run()
