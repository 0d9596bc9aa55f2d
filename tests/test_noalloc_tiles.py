"""The no-allocation entry point on a level of more work than its scratch has
room to index at once: a last pair counted from whole prefixes over 4.8e10
candidates, whose tile index alone would be 256 MB.  The level goes out in
parts, as it did when its rows were stored."""
import numpy as np
import pytest

import cuts_amd as F


@pytest.mark.gpu
def test_level_of_more_tiles_than_the_scratch(ctx):
    D = 240_000
    star = np.stack([np.zeros(D, np.int64), np.arange(1, D + 1)], 1)
    more = [[i, D + 3 * (i - 1) + j] for i in (1, 2, 3) for j in (1, 2, 3)]
    dg = ctx.upload(F.Graph.from_edges(D + 10, np.concatenate([star, np.asarray(more)])))
    p = F.Plan(F.Graph.from_edges(5, [(0, 1), (1, 2), (2, 3), (2, 4)]), [0, 1, 2, 3, 4])
    want = ctx.match(dg, p)
    # position 2 on the centre (from one of the 3 hubs, whose other neighbours are 3 leaves) or on a hub
    # (from one of the centre's other D - 1 neighbours), then an ordered pair of its other neighbours
    assert want.count == 3 * 3 * (D - 1) * (D - 2) + 3 * (D - 1) * 3 * 2
    got = ctx.match(dg, p, noalloc=True)
    assert (got.count, got.level_sizes) == (want.count, want.level_sizes)
