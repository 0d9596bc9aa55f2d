"""A run that its work cap ends costs no more than the same run with every
level's work read back: without remembered level sizes, and after a whole run
has left them."""
import time

import numpy as np
import pytest

import cuts_amd as F
from test_tail import CASES

SHAPES = {n: CASES[n] for n in ("triangle, leaf", "owners not adjacent", "5-cycle, chord, two tails")}
SHAPES["4-clique"] = ([(a, b) for a in range(4) for b in range(a)], [0, 1, 2, 3])


def plan(name):
    edges, order = SHAPES[name]
    return F.Plan(F.Graph.from_edges(len(order), edges), order)


@pytest.mark.gpu
@pytest.mark.parametrize("hints", [False, True])
@pytest.mark.parametrize("name", SHAPES)
def test_ended_by_the_cap(name, hints):
    """Medians of 25 runs in turn; a fifth more covers their spread (the run
    repeated after its cap took 1.4 to 2.1 times the readbacks' time)."""
    dg = F.Context().upload(F.Graph.chung_lu(4096, 32768, 2.3, 0, 3))
    ctx, roots = dg.ctx, (7, 4096, 64)
    for cap in (1 << 8, 1 << 10, 1 << 12, 1 << 14):
        plans = [plan(name) for _ in range(28)]
        times = {0: [], F.FLAG_SYNC_LEVELS: []}
        for p in plans:
            if hints:
                for flags in times:
                    ctx.match(dg, p, flags=flags, roots=roots)
            got = {}
            for flags in times:
                t = time.perf_counter()
                r = ctx.match(dg, p, flags=flags, roots=roots, max_work=cap)
                times[flags].append(time.perf_counter() - t)
                got[flags] = (r.work_capped, r.work, r.count, r.level_sizes, r.complete, r.roots_done, r.last_root)
            if not hints:
                assert got[0] == got[F.FLAG_SYNC_LEVELS]
        capped = got[0][0]
        spec, sync = (np.median(t[3:]) for t in times.values())
        print(name, hints, cap, capped, f"{1e6 * spec:.0f} {1e6 * sync:.0f} us", flush=True)
        assert spec <= 1.2 * sync, (cap, spec, sync)
