"""What an upload says of a directed graph's hub bitmaps: the rows of both
sides."""
import numpy as np
import pytest

import cuts_amd as F


@pytest.mark.gpu
@pytest.mark.parametrize("out_hubs,in_hubs", [(0, 0), (2, 0), (0, 3), (4, 5)])
def test_rows_of_both_sides(ctx, out_hubs, in_hubs):
    rng = np.random.default_rng(out_hubs + 7 * in_hubs)
    V = 300
    e = [np.stack([np.arange(V - 1), np.arange(1, V)], 1)]
    for i in range(out_hubs):
        e.append(np.stack([np.full(50, i), 100 + rng.permutation(V - 100)[:50]], 1))
    for i in range(in_hubs):
        e.append(np.stack([100 + rng.permutation(V - 100)[:50], np.full(50, 20 + i)], 1))
    e = np.concatenate(e)
    info = ctx.upload(F.Graph.from_arcs(V, e[:, 0], e[:, 1])).info()
    assert info["hubs"] == out_hubs + in_hubs
    assert info["hub_min_deg"] == (32 if info["hubs"] else 0)
