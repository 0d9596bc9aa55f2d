"""The work that a user of the matcher has it do, as cases that can be timed.

A case names its sizes only; `prepare` makes the data graph, queries and handles of a seed, `run` is
one pass through the public entry points.  Data graphs are those of `cuts_amd.workloads` (Chung-Lu
and R-MAT generators) with seeds of their own, in the sizes of that module and below.

Kinds of passes:
  count    one query after the other, whole counts (`Context.match`)
  sample   one query on a residue class of the data vertices for order position 0
  walks    a list of random-walk queries, each on its admitted root sample, one after the other
  many     the same list handed to concurrent streams (`Context.match_many`)
  batch    random-walk queries matched together by the device work queue (`Batch.run`)
  directed a query with directed arcs on a directed graph: every level expanded, none in closed form
  listing  all embeddings around one data vertex, written to the caller's rows
  cold     a data graph uploaded, its first query matched, the graph released
  predict  table sizes predicted for prefix sets of many queries (`Mpnn.forward`)
  gradient loss and gradient of one training batch of that network (`Mpnn.gradient`)
"""
from functools import lru_cache

import numpy as np
import torch

import cuts_amd
from cuts_amd import learned as LN
from cuts_amd import workloads as W

SHAPES = {"tri_tail": [W.TRI_TAIL2], "c4_pend": [W.C4_2PEND], "k4e_tail": [W.K4E_TAIL2],
          "c4_pend+k4e_tail": [W.C4_2PEND, W.K4E_TAIL2], "c5_chord": [W.C5CHORD_2TAIL]}
# two directed triangles sharing an arc's head, closed by a second path
DIRECTED_ARCS = [(0, 1), (0, 2), (1, 2), (2, 3), (1, 4), (3, 4)]
# sizes of walk queries and the most work one may take (candidates examined, trie rows)
WALK_WORK, WALK_ROWS = 1 << 27, 1 << 20


def listed():
    chung4k = dict(graph="chung_lu", n=4096, m=32768, gamma=2.3, max_deg=0)
    chung37k = dict(graph="chung_lu", n=36692, m=183831, gamma=2.1, max_deg=1400)
    return [
        # an interactive look at one vertex: few rows, all latency
        dict(name="listing_4k", kind="listing", page=1 << 14, **chung4k),
        # one small pattern on a small graph, the shortest whole count
        dict(name="tri_tail_4k", kind="count", shapes="tri_tail", **chung4k),
        # two 6-vertex patterns on a graph of the size of an e-mail network, whole counts
        dict(name="two_shapes_37k", kind="count", shapes="c4_pend+k4e_tail", **chung37k),
        # a 7-vertex pattern on the largest graph, on a sample of the roots, in the default order
        dict(name="c5_chord_rmat20", kind="sample", shapes="c5_chord", graph="rmat", scale=20, stride=128),
        # queries of 6 to 10 vertices arriving one at a time
        dict(name="walks_rmat18", kind="walks", graph="rmat", scale=18, queries=15, kmin=6, kmax=10),
        # the same kind of queries as a throughput job
        dict(name="many_rmat18", kind="many", graph="rmat", scale=18, queries=30, kmin=6, kmax=10, workers=4),
        # many queries against one resident graph in one graph launch
        dict(name="batch_37k", kind="batch", queries=45, kmin=4, kmax=12, queue="level", **chung37k),
        # citation- or call-graph like data: directed arcs
        dict(name="directed_37k", kind="directed", stride=1, both=0.25, **chung37k),
        # the command line's life: load, one query, done -- with the two-hop index of mid-size graphs
        dict(name="cold_37k", kind="cold", shapes="k4e_tail", stride=1, **chung37k),
        # and with the hub rows of graphs too large for that index
        dict(name="cold_rmat18", kind="cold", shapes="c5_chord", graph="rmat", scale=18, stride=256),
        # the sizes that pick the orders of a few dozen queries
        dict(name="predict_12k", kind="predict", samples=12000, kmin=6, kmax=10),
        # one batch of the order network's training
        dict(name="gradient_2k", kind="gradient", samples=2048, kmin=5, kmax=10),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    def chung():
        n = _log(rng, 1000, 36000)
        return dict(graph="chung_lu", n=n, m=int(n * rng.uniform(4.0, 7.0)), gamma=round(rng.uniform(2.1, 2.6), 2),
                    max_deg=rng.choice([0, 1400]) if n < 8000 else 1400)

    def rmat(lo, hi):
        return dict(graph="rmat", scale=rng.randint(lo, hi))

    kind = rng.choice(["listing", "count", "sample", "walks", "many", "batch", "directed", "cold", "predict", "gradient"])
    c = dict(kind=kind)
    if kind == "listing":
        c.update(chung())
        c.update(n=min(c["n"], 4096), m=min(c["m"], 28000), page=_log(rng, 1 << 9, 1 << 14))
    elif kind == "count":
        c.update(chung(), shapes=rng.choice(["tri_tail", "c4_pend", "k4e_tail"]))
    elif kind == "sample":
        c.update(rmat(14, 18), shapes=rng.choice(["c5_chord", "tri_tail"]))
        c.update(stride=1 << (c["scale"] - rng.randint(9, 11)))
    elif kind in ("walks", "many"):
        c.update(rmat(14, 17), queries=rng.randint(4, 15), kmin=rng.randint(4, 7), kmax=rng.randint(7, 9))
        if kind == "many":
            c.update(workers=rng.choice([2, 3, 4]))
    elif kind == "batch":
        c.update(chung(), queries=rng.randint(6, 40), kmin=rng.randint(4, 6), kmax=rng.randint(6, 11),
                 queue=rng.choice(["level", "level", "persistent"]))
    elif kind == "directed":
        c.update(chung(), stride=rng.randint(1, 4), both=round(rng.uniform(0.0, 0.5), 2))
    elif kind == "cold":
        c.update(chung() if rng.random() < 0.5 else rmat(13, 17))
        if c["graph"] == "rmat":
            c.update(shapes="c5_chord", stride=1 << (c["scale"] - 10))
        else:
            c.update(shapes=rng.choice(["tri_tail", "k4e_tail"]), stride=1)
    else:
        c.update(samples=_log(rng, 60, 14000) if kind == "predict" else _log(rng, 100, 4096),
                 kmin=rng.randint(3, 6), kmax=rng.randint(7, 12))
    return c


# ------------------------------------------------------------------ inputs
@lru_cache(maxsize=6)
def _chung_lu(n, m, gamma, max_deg, seed):
    return cuts_amd.Graph.chung_lu(n, m, gamma, max_deg, seed)


@lru_cache(maxsize=6)
def _rmat(scale, seed):
    return cuts_amd.Graph.rmat(scale, 16, 0.57, 0.19, 0.19, seed)


def _graph(case, seed):
    if case["graph"] == "rmat":
        return _rmat(case["scale"], 1000 + seed)
    return _chung_lu(case["n"], case["m"], case["gamma"], case["max_deg"], 1000 + seed)


def _directed(g, both, seed):
    """Every edge of g as one arc of random direction, `both` of them as two."""
    v = g.view()
    src = np.repeat(np.arange(v["V"], dtype=np.uint32), np.diff(v["out_off"].astype(np.int64)))
    dst = v["out_adj"]
    half = src < dst
    src, dst = src[half], dst[half]
    rng = np.random.default_rng(seed)
    flip = rng.random(len(src)) < 0.5
    s, d = np.where(flip, dst, src), np.where(flip, src, dst)
    two = rng.random(len(src)) < both
    return cuts_amd.Graph.from_arcs(v["V"], np.concatenate([s, d[two]]), np.concatenate([d, s[two]]))


def _samples(case, seed):
    """Prefix sets of random connected query graphs: (k, adjacency masks, set), as the order search asks for."""
    rng = np.random.default_rng(seed)
    out = []
    while len(out) < case["samples"]:
        k = int(rng.integers(case["kmin"], case["kmax"] + 1))
        adj = [0] * k

        def join(a, b):
            adj[a] |= 1 << b
            adj[b] |= 1 << a

        for v in range(1, k):
            join(v, int(rng.integers(v)))
        for _ in range(int(rng.integers(0, k + 1))):
            a, b = (int(t) for t in rng.integers(k, size=2))
            if a != b:
                join(a, b)
        # sets grown from a random vertex, one vertex at a time: the prefixes of random connected orders
        for _ in range(4):
            sm = 1 << int(rng.integers(k))
            while True:
                out.append((k, adj, sm))
                near = 0
                for v in range(k):
                    if sm >> v & 1:
                        near |= adj[v]
                near &= ~sm
                if not near:
                    break
                free = [v for v in range(k) if near >> v & 1]
                sm |= 1 << free[int(rng.integers(len(free)))]
    return out[:case["samples"]]


def _network_inputs(case, seed):
    gfeat = LN.graph_features(_chung_lu(4096, 32768, 2.3, 0, 1000 + seed))
    x, adj, meta = LN.encode(_samples(case, seed), gfeat)
    # targets in the range of log(1 + table size) / 10
    t = np.random.default_rng(seed + 7).uniform(0.0, 2.5, len(meta)).astype(np.float32)
    return LN.init_params(seed), x, adj, meta, t


def prepare(case, seed):
    kind = case["kind"]
    ctx = cuts_amd.Context(0)
    s = dict(kind=kind, ctx=ctx)
    if kind in ("predict", "gradient"):
        params, x, adj, meta, t = _network_inputs(case, seed)
        s.update(net=LN.Mpnn(ctx, params=params), x=x, adj=adj, meta=meta, t=t)
        return s
    g = _graph(case, seed)
    if kind == "directed":
        g = _directed(g, case["both"], seed)
        arcs = np.asarray(DIRECTED_ARCS, dtype=np.uint32)
        s["plans"] = [cuts_amd.Plan(cuts_amd.Graph.from_arcs(5, arcs[:, 0], arcs[:, 1]))]
        s["roots"] = [W.root_sample(g.V, case["stride"])]
    elif kind == "listing":
        v = g.view()
        deg = np.diff(v["out_off"].astype(np.int64))
        # an anchor among the upper half of the degrees whose triangles with a pendant fit the page: its
        # neighbour pairs and a third neighbour bound them
        few = max(int(case["page"] ** (1 / 3)), 3)
        near = np.flatnonzero((deg <= few) & (deg >= np.median(deg)))
        anchor = int(np.random.default_rng(seed).choice(near if len(near) else np.flatnonzero(deg <= few)))
        s["plans"] = [cuts_amd.Plan(W.query_graph(W.Shape("triangle+pendant", 4, ((0, 1), (1, 2), (2, 0), (0, 3)))))]
        s["roots"] = [(anchor, anchor + 1, 1)]
    elif kind in ("walks", "many", "batch"):
        pass
    else:
        s["plans"] = [cuts_amd.Plan(W.query_graph(q)) for q in SHAPES[case["shapes"]]]
        s["roots"] = [W.root_sample(g.V, case["stride"]) if "stride" in case else None] * len(s["plans"])
    if kind == "cold":
        s["graph"] = g
        return s
    dg = s["dg"] = ctx.upload(g)
    if kind in ("walks", "many", "batch"):
        queries, _ = W.admit(ctx, dg, g, case["queries"], seed=seed, max_work=WALK_WORK, max_rows=WALK_ROWS,
                             kmin=case["kmin"], kmax=case["kmax"], max_tries_per_k=60)
        s["plans"] = [cuts_amd.Plan(cuts_amd.Graph.from_edges(q["k"], q["edges"])) for q in queries]
        s["roots"] = [tuple(q["roots"]) for q in queries]
        if kind == "many":
            s["workers"] = case["workers"]
        if kind == "batch":
            s["batch"] = cuts_amd.Batch(ctx, dg, s["plans"], roots=s["roots"], queue=case["queue"])
    if kind == "listing":
        s["rows"] = cuts_amd.pinned_array((case["page"], 4))
    if kind in ("walks", "many", "batch"):
        s["queries"] = case["queries"]
    return s


# ------------------------------------------------------------------ passes
def _matched(counts, level_sizes, rows=None):
    """Counts and level sizes, one row per query asked for (a set may hold fewer than its quota)."""
    c = np.zeros(rows or len(counts), dtype=np.uint64)
    s = np.zeros((len(c), cuts_amd.MAX_QUERY), dtype=np.uint64)
    for i, (n, sizes) in enumerate(zip(counts, level_sizes)):
        c[i] = n
        s[i, :len(sizes)] = sizes
    return {"counts": c, "level_sizes": s}


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "predict":
        return state["net"].forward(state["x"], state["adj"], state["meta"])
    if kind == "gradient":
        loss, grad = state["net"].gradient(state["x"], state["adj"], state["meta"], state["t"])
        return {"loss": loss, "gradient": grad}
    if kind == "batch":
        r = state["batch"].run()
        return _matched(r.counts, r.level_sizes, state["queries"])
    if kind == "many":
        results, _ = ctx.match_many(state["dg"], state["plans"], roots=state["roots"], workers=state["workers"])
    elif kind == "listing":
        # rows come in no fixed order: a program that shows or compares them sorts them (a page at most)
        r = ctx.match(state["dg"], state["plans"][0], roots=state["roots"][0], write=True, rows_out=state["rows"])
        rows = r.rows.astype(np.int64)
        key = (rows[:, 0] << 48) | (rows[:, 1] << 32) | (rows[:, 2] << 16) | rows[:, 3]
        key.sort()
        page = np.full(len(state["rows"]), -1, dtype=np.int64)
        page[:len(key)] = key
        return {"counts": np.asarray([r.count], dtype=np.uint64), "rows": page}
    else:
        dg = ctx.upload(state["graph"]) if kind == "cold" else state["dg"]
        results = [ctx.match(dg, p, roots=rt) for p, rt in zip(state["plans"], state["roots"])]
    return _matched([r.count for r in results], [r.level_sizes for r in results], state.get("queries"))


# ------------------------------------------------------------- what it takes
def _arcs(case):
    """Arcs of the data graph, and its vertices (R-MAT: after duplicates and loops are dropped, about 14 of 16)."""
    if case["graph"] == "rmat":
        return int(28 * 2 ** case["scale"]), 2 ** case["scale"]
    return 2 * case["m"], case["n"]


def _params():
    h, f = LN.HIDDEN, LN.FEATS
    return 2 * f * h + h + 2 * (2 * h * h + h) + 2 * h * h + h + h + 1


def work(case):
    kind = case["kind"]
    if kind in ("predict", "gradient"):
        n, h, f = case["samples"], LN.HIDDEN, LN.FEATS
        k = 0.5 * (case["kmin"] + case["kmax"])
        flops = n * (k * 2 * (2 * f * h + 4 * h * h) + 2 * (2 * h * h + h))
        nbytes = n * (LN.NODES * (4 * f + 2) + 4 + 4) + 2 * _params()
        if kind == "gradient":
            # input gradients and weight gradients cost what the forward products cost, each
            return {"bytes": nbytes + 4 * n + 4 * _params(), "flops": 3 * flops}
        return {"bytes": nbytes, "flops": flops}
    arcs, V = _arcs(case)
    if kind == "directed":
        arcs = int(2 * case["m"] * (1 + case["both"]))  # out-lists and in-lists
    if kind == "listing":
        # the lists of an average vertex's neighbours, and the rows written
        d = arcs / V
        return {"bytes": 4 * d * d + 8 * d + 16 * d * d, "flops": 0}
    # offsets, lists and degrees once; the level sizes of every query
    return {"bytes": 4 * (V + 1) + 4 * arcs + 8 * V + 128 * case.get("queries", 1), "flops": 0}


# ------------------------------------------------------- the network, in 64 bits
def _network(w, x, adj, meta):
    """The network's output for every sample, as float64; w: the flat weights, rounded to bfloat16."""
    n, nodes, f = x.shape
    h = LN.HIDDEN
    k = torch.from_numpy((meta & 0xFF).astype(np.int64))
    sets = torch.from_numpy((meta >> 16).astype(np.int64))
    bit = torch.arange(nodes)
    live = (bit[None, :] < k[:, None]).double()
    near = ((torch.from_numpy(adj.astype(np.int64))[:, :, None] >> bit) & 1).double() * live[:, None, :]
    inset = ((sets[:, None] >> bit) & 1).double() * live
    at = 0

    def take(*shape):
        nonlocal at
        m = int(np.prod(shape))
        at += m
        return w[at - m:at].reshape(*shape)

    a = torch.from_numpy(x).double() * live[:, :, None]
    for fan in (f, h, h):
        ws, wn, b = take(fan, h), take(fan, h), take(h)
        a = torch.relu(b + a @ ws + torch.bmm(near, a) @ wn) * live[:, :, None]
    pooled = torch.cat([(a * inset[:, :, None]).sum(1), a.sum(1) / k[:, None].double()], 1)
    wr, br, wo, bo = take(2 * h, h), take(h), take(h), take(1)
    return torch.relu(br + pooled @ wr) @ wo + bo


def exact(case, seed):
    if case["kind"] not in ("predict", "gradient"):
        return None  # whole numbers: they stay equal
    params, x, adj, meta, t = _network_inputs(case, seed)
    w = torch.from_numpy(params).bfloat16().double()
    if case["kind"] == "predict":
        with torch.no_grad():
            return _network(w, x, adj, meta)
    w.requires_grad_()
    loss = ((_network(w, x, adj, meta) - torch.from_numpy(t).double()) ** 2).mean()
    loss.backward()
    return {"loss": loss.detach(), "gradient": w.grad}
