"""The network's forward and backward kernels at the sizes where their tiles
end: one sample, counts around the samples of a block and of a full grid, and
query sizes 1 to 16 (the 16 rows of a product), against the FP64 reference."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from cuts_amd import learned as LN  # noqa: E402
from oracle import mpnn_ref  # noqa: E402


def batch(n, kmin, kmax, seed):
    rng = np.random.default_rng(seed)
    x = np.zeros((n, LN.NODES, LN.FEATS), np.float32)
    adj = np.zeros((n, LN.NODES), np.uint16)
    meta = np.zeros(n, np.uint32)
    for i in range(n):
        k = int(rng.integers(kmin, kmax + 1))
        x[i, :k] = rng.uniform(0.0, 1.0, (k, LN.FEATS))
        a = np.triu(rng.random((k, k)) < 0.4, 1)
        a |= a.T
        adj[i, :k] = (a << np.arange(k)).sum(1)
        meta[i] = k | (int(rng.integers(1 << k)) << 16)
    return x, adj, meta, rng.uniform(0.0, 2.5, n).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("n,kmin,kmax", [(1, 1, 1), (1, 16, 16), (3, 1, 16), (4, 5, 9), (5, 15, 16), (7, 1, 4),
                                         (8, 8, 8), (9, 1, 16), (1023, 2, 12), (1025, 1, 16), (2051, 4, 10)])
def test_tiles_match_the_reference(ctx, n, kmin, kmax):
    """Sums of at most 2,051 samples' products of 128 FP32 terms each: the
    error of a random walk of that length stays below 2e-5 of the result's
    norm (2^-24 sqrt(2051 * 128) = 3e-5 in the worst case of one sign)."""
    x, adj, meta, t = batch(n, kmin, kmax, 100 + n)
    p = mpnn_ref.bf16_round(LN.init_params(n))
    net = LN.Mpnn(ctx, p)
    loss, grad, y = mpnn_ref.loss_and_grad(p, x, adj, meta, t)
    got = net.forward(x, adj, meta)
    assert np.linalg.norm(got - y) <= 2e-5 * max(np.linalg.norm(y), 1e-3)
    gl, gg = net.gradient(x, adj, meta, t)
    assert abs(gl - loss) <= 2e-5 * max(abs(loss), 1e-6)
    assert np.linalg.norm(gg - grad) <= 2e-5 * max(np.linalg.norm(grad), 1e-6)
    again = net.gradient(x, adj, meta, t)
    assert again[0] == gl and np.array_equal(again[1], gg)
