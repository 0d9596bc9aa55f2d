"""Routes of the last two positions and of the last written level that other
tests do not take: a chain on position k-3 with thresholds that no index serves,
written embeddings under a work cap, and memory that passes between graphs on
several threads."""
import threading

import numpy as np
import pytest

import cuts_amd as F
import oracle
from test_tail import CASES, FLAGS, tail_kind
from test_work_cap import outcome

CHAINS = [n for n, (e, o) in CASES.items() if tail_kind(len(o), e, o) == 3]


@pytest.mark.gpu
@pytest.mark.parametrize("hubs", [False, True])
@pytest.mark.parametrize("name", CHAINS)
def test_chain_thresholds_above_two(ctx, monkeypatch, name, hubs):
    """A query self-loop raises its vertex's threshold by one: the last vertex's
    to 2, the one before it to 3, past what the index holds."""
    if hubs:
        monkeypatch.setenv("CUTS_H2_MAX_WEDGES", "0")
        monkeypatch.setenv("CUTS_H2_HUB_MIN_DEG", "8")
        monkeypatch.setenv("CUTS_H2_HUB_ROWS", "12")
    edges, order = CASES[name]
    k = len(order)
    g = F.Graph.chung_lu(97, 330, 2.3, 0, 60 + k)
    og = oracle.OGraph.from_view(g.view())
    dg = ctx.upload(g)
    last, before = order[-1], order[-2]
    for loops in ([last], [before], [last, before], [last, before, order[-3]]):
        arcs = [a for e in edges for a in (e, e[::-1])] + [(v, v) for v in loops]
        a = np.asarray(arcs, dtype=np.uint32)
        p = F.Plan(F.Graph.from_arcs(k, a[:, 0], a[:, 1]), order)
        want = oracle.count(og, oracle.qmatrix(k, arcs))
        sizes = ctx.match(dg, p, flags=F.FLAG_NO_SHORTCUT).level_sizes
        assert sizes[-1] == want
        for flags in FLAGS:
            for extra in (0, F.FLAG_SYNC_LEVELS, F.FLAG_PROFILE):
                r = ctx.match(dg, p, flags=flags | extra)
                assert (r.count, r.level_sizes) == (want, sizes), (loops, flags, extra)
            for kw in (dict(budget=2048), dict(trunks=5), dict(noalloc=True), dict(time_limit_ms=1e6, trunks=4)):
                r = ctx.match(dg, p, flags=flags, **kw)
                assert (r.count, r.level_sizes) == (want, sizes), (loops, flags, kw)


@pytest.mark.gpu
@pytest.mark.parametrize("page", [50, 1 << 16])
@pytest.mark.parametrize("name", ["triangle, leaf", "path4 from its end", "4-cycle, leaf"])
def test_written_rows_under_a_cap(name, page):
    """The same decision, work and counts as with every level read back; all
    rows of a run that its cap leaves whole, on a first run and on later ones."""
    edges, order = CASES[name]
    k = len(order)
    ctx = F.Context()
    for n, m, st in ((60, 150, 1), (3000, 9000, 1), (3000, 9000, 16)):  # last levels of one planning block and of more
        g = F.Graph.chung_lu(n, m, 2.4, 40, k)
        dg = ctx.upload(g)
        p = F.Plan(F.Graph.from_edges(k, edges), order)
        kw = dict(write=True, emb_cap=page, roots=(st - 1, n, st))
        whole = ctx.match(dg, p, flags=F.FLAG_SYNC_LEVELS, **kw)
        rows = {tuple(x) for x in whole.rows.tolist()}
        assert len(rows) == min(page, whole.count)
        total = whole.work
        for cap in sorted({1, total // 20, total // 2, total - 1, total, total + 1} - {0}):
            want = outcome(ctx.match(dg, p, flags=F.FLAG_SYNC_LEVELS, max_work=cap, **kw))
            for _ in range(3):
                r = ctx.match(dg, p, max_work=cap, **kw)
                assert outcome(r) == want, (n, cap, total)
                if not r.work_capped:
                    got = {tuple(x) for x in r.rows.tolist()}
                    assert len(got) == len(rows) and (got == rows or page < whole.count)


@pytest.mark.gpu
def test_memory_between_graphs_on_several_threads():
    """Contexts that upload, match, release and trim beside one that matches
    many queries: every count is the one of a graph of its own."""
    graphs = [F.Graph.chung_lu(3000 + 900 * i, 14000 + 3000 * i, 2.2, 700, i) for i in range(4)]
    shapes = [CASES[n] for n in ("triangle, leaf", "5-cycle, chord, tail of two", "owners not adjacent")]

    def plans():
        return [F.Plan(F.Graph.from_edges(len(o), e), o) for e, o in shapes]

    ctx = F.Context()
    want = []
    for g in graphs:
        dg = ctx.upload(g)
        want.append([ctx.match(dg, p, roots=(3, g.V, 16)).count for p in plans()])
    errors = []

    def work(t):
        try:
            c, ps = F.Context(), plans()
            for i in range(10):
                j = (t + i) % len(graphs)
                dg = c.upload(graphs[j])
                got = [c.match(dg, p, roots=(3, graphs[j].V, 16), budget=1 << (16 + 4 * (i % 3))).count for p in ps]
                assert got == want[j], (t, i)
                del dg
                if i % 4 == 3:
                    c.trim()
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    dg, ps = ctx.upload(graphs[0]), plans() * 6
    for _ in range(6):
        results, _ = ctx.match_many(dg, ps, roots=[(3, graphs[0].V, 16)] * len(ps), workers=6)
        assert [r.count for r in results] == want[0] * 6
    for t in threads:
        t.join()
    assert not errors, errors[0]
