"""Common-neighbour rows built at upload (csrc/index.hip) at the edges of their
tiles: vertex counts around 64 rows and 256 vertices, enough groups of rows for
the XCD-wise order, lists on both sides of one thread's longest (64), and a
list near 2^16; and the per-arc table that is filled from them.  Whole counts,
equal to the matrix product's."""
import numpy as np
import pytest

import cuts_amd as F

sp = pytest.importorskip("scipy.sparse")


def graph(V, seed, long_lists=()):
    """A sparse random graph in which vertex i has about long_lists[i] neighbours."""
    rng = np.random.default_rng(seed)
    m = 3 * V
    e = [rng.integers(V, size=(m, 2))]
    for i, d in enumerate(long_lists):
        others = rng.permutation(V)[:min(d, V)]
        e.append(np.stack([np.full(len(others), i), others], 1))
    e = np.concatenate(e)
    e = e[e[:, 0] != e[:, 1]]
    g = F.Graph.from_edges(V, e)
    v = g.view()
    A = sp.csr_matrix((np.ones(len(v["out_adj"]), np.int64), v["out_adj"].astype(np.int64), v["out_off"].astype(np.int64)),
                      shape=(V, V))
    return g, A


def check_arcs(dg, g, A, C):
    v = g.view()
    src = np.repeat(np.arange(v["V"]), np.diff(v["out_off"].astype(np.int64)))
    assert np.array_equal(dg.arc_common(), np.asarray(C[src, v["out_adj"].astype(np.int64)]).ravel())


SIZES = [(3, (2,)), (63, (62,)), (64, (63, 40)), (65, (64, 63)), (255, (66, 65, 64)), (257, (256, 63)),
         (2047, (1500, 65, 64, 63)), (2113, (2000, 700, 128, 129))]


@pytest.mark.gpu
@pytest.mark.parametrize("V,long_lists", SIZES)
def test_two_hop_index(ctx, V, long_lists):
    g, A = graph(V, V, long_lists)
    C = (A @ A).tolil()
    C.setdiag(0)
    C = C.tocsr()
    C.eliminate_zeros()
    C.sort_indices()
    dg = ctx.upload(g)
    off, v, c = dg.two_hop()
    assert np.array_equal(off.astype(np.int64), C.indptr)
    assert np.array_equal(v.astype(np.int64), C.indices)
    assert np.array_equal(c.astype(np.int64), C.data)
    check_arcs(dg, g, A, C)


@pytest.mark.gpu
@pytest.mark.parametrize("V,long_lists", SIZES)
@pytest.mark.parametrize("rows", [1, 65, 4096])
def test_hub_rows(ctx, monkeypatch, V, long_lists, rows):
    monkeypatch.setenv("CUTS_H2_MAX_WEDGES", "0")
    monkeypatch.setenv("CUTS_H2_HUB_MIN_DEG", "1")
    monkeypatch.setenv("CUTS_H2_HUB_ROWS", str(rows))
    g, A = graph(V, V, long_lists)
    C = np.asarray((A @ A).todense())
    np.fill_diagonal(C, 0)
    dg = ctx.upload(g)
    rid, got = dg.hub_rows()
    assert len(got) == min(rows, int((np.diff(A.indptr) > 0).sum()))
    for u in np.flatnonzero(rid >= 0):
        assert np.array_equal(got[rid[u]], C[u]), u
    check_arcs(dg, g, A, sp.csr_matrix(C))


@pytest.mark.gpu
def test_longest_list_and_reused_memory(ctx, monkeypatch):
    """A list of 65,535 entries (counts of 16 bits); graphs uploaded after it
    is gone, whose arrays may take its memory."""
    monkeypatch.setenv("CUTS_H2_MAX_WEDGES", "0")
    monkeypatch.setenv("CUTS_H2_HUB_MIN_DEG", "1000")
    V = 65600
    both = np.concatenate([np.stack([np.full(65535, c), np.arange(2, 65537)], 1) for c in (0, 1)])
    dg = ctx.upload(F.Graph.from_edges(V, both))
    rid, rows = dg.hub_rows()
    assert rid[0] >= 0 and rid[1] >= 0 and rows[rid[0]][1] == 65535 and rows[rid[1]][0] == 65535
    assert not rows[rid[0]][2:].any() and rows[rid[0]][0] == 0
    del dg, rows
    for seed in range(3):
        g, A = graph(3000 - 500 * seed, seed, (1200, 1100))
        dg = ctx.upload(g)
        rid, rows = dg.hub_rows()
        C = np.asarray((A @ A).todense())
        np.fill_diagonal(C, 0)
        for u in np.flatnonzero(rid >= 0):
            assert np.array_equal(rows[rid[u]], C[u])
        del dg
