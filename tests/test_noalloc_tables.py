"""A no-allocation run on a few roots builds no table of the whole graph in
its scratch, which it would build again on every call."""
import time

import numpy as np
import pytest

import cuts_amd as F


@pytest.mark.gpu
def test_few_roots(ctx):
    g = F.Graph.rmat(19, 16, 0.57, 0.19, 0.19, 5)
    v = g.view()
    a = int(np.flatnonzero(np.diff(v["out_off"].astype(np.int64)) == 6)[0])
    dg = ctx.upload(g)
    p = F.Plan(F.Graph.from_edges(4, [(0, 1), (1, 2), (2, 3)]), [0, 1, 2, 3])
    roots = (a, a + 1, 1)

    def run(flags):
        ts = []
        for _ in range(20):
            t = time.perf_counter()
            r = ctx.match(dg, p, noalloc=True, roots=roots, flags=flags)
            ts.append(time.perf_counter() - t)
        return np.median(ts[2:]), (r.count, r.level_sizes)

    t, got = run(0)
    t_off, want = run(F.FLAG_NO_CHAIN)  # needs no table
    assert got == want
    print(f"{1e6 * t:.0f} {1e6 * t_off:.0f} us")
    assert t <= 2 * t_off  # 6 times with the tables built
    r = ctx.match(dg, p, roots=roots)  # leaves its tables with the graph
    assert (r.count, r.level_sizes) == want
    assert run(0)[1] == want
    whole = ctx.match(dg, p)
    got = ctx.match(dg, p, noalloc=True)
    assert (got.count, got.level_sizes) == (whole.count, whole.level_sizes)
