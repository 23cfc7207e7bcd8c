"""One sparse contraction at the edges of the form that keeps its forests in LDS
(up to 18000 vertices) and of its final sort (1024 candidates), against the
oracle: sizes on both sides of each, trees (every edge may be needed), equal keys
and contraction to two vertices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _edges(rng, n, m, w):
    """A random tree on all vertices and random edges up to m."""
    perm = rng.permutation(n)
    par = perm[(rng.random(n - 1) * np.arange(1, n)).astype(np.int64)]
    u = np.concatenate([perm[1:], rng.integers(0, n, m - (n - 1))])
    v = np.concatenate([par, rng.integers(0, n, m - (n - 1))])
    v = np.where(u == v, (v + 1) % n, v)
    ww = rng.integers(1, w + 1, m) if w < 2**39 else np.full(m, w)
    return np.stack([np.minimum(u, v), np.maximum(u, v), ww], 1).astype(np.uint64)[rng.permutation(m)]


@pytest.mark.parametrize("n,m,tgt,w", [
    (2, 1, 1, 9), (2, 5, 2, 9), (700, 1023, 2, 50), (700, 1024, 2, 50), (700, 1025, 2, 50), (1025, 1024, 1, 9),
    (1026, 1025, 1, 9), (17999, 40000, 12729, 100), (18000, 40001, 12730, 100), (18001, 40001, 12730, 100),
    (18000, 17999, 2, 7), (18001, 18000, 2, 7), (2049, 300000, 1450, 1), (2049, 300000, 2, 2**40 - 1)])
def test_contraction_edges(ctx, orc, n, m, tgt, w):
    E = _edges(np.random.default_rng(n + m), n, m, w)
    print(f"sparse contract n={n} m={m} tgt={tgt} w={w}", flush=True)
    assert np.array_equal(ctx.sparse_contract(E, n, tgt, 17, 3, 5), orc.sparse_contract(n, E, tgt, 17, 3, 5))
