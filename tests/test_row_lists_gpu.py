"""Sparse nodes handed to the dense engine as row lists (128 or more nodes of 129
to 2048 vertices with short rows) against the same trials on the summed matrix:
raw cuts are equal.  Sizes at the edges of the row pieces and of the range;
graphs whose merges follow one heavy vertex (a row of thousands of entries with
parallel edges), whose PR pass pairs vertices up until the row pool overflows,
plain random ones, disconnected ones; 32- and 64-bit entries; the last length that
goes as lists and the first that does not."""
import numpy as np
import pytest
from graphgen import dense

pytestmark = pytest.mark.gpu

TRIALS = 130


def _graph(kind, n, m, wmax):
    rng = np.random.default_rng(n * 31 + m + wmax % 97)
    path = np.stack([np.arange(n - 1), np.arange(1, n)], 1)
    k = m - (n - 1)
    if kind == "hub":  # most edges end at vertex n / 3, several times each
        hub = n // 3
        u = rng.integers(0, n, k)
        v = np.where(rng.random(k) < 0.9, hub, rng.integers(0, n, k))
    elif kind == "pairs":
        u = rng.integers(0, n // 2, k) * 2
        v = np.where(rng.random(k) < 0.8, u + 1, rng.integers(0, n, k))
    else:
        u, v = rng.integers(0, n, k), rng.integers(0, n, k)
    v = np.where(u == v, (v + 1) % n, v)
    if kind == "split":  # two components
        cut = n // 2
        u, v = np.where((u < cut) == (v < cut), u, v), v
        v = np.where(u == v, np.where(v + 1 == cut, 0, np.where(v + 1 == n, cut, v + 1)), v)
        path = path[path[:, 1] != cut]
    e = np.concatenate([path, np.stack([u, v], 1)])
    w = rng.integers(1, wmax + 1, len(e))
    w[0] = 1  # a light end of the path: a low bound, so the PR pass has work
    if kind == "pairs":
        w[len(path):] += wmax
    e = np.concatenate([e, w[:, None]], 1).astype(np.uint64)
    sw = rng.random(len(e)) < 0.4
    e[sw, 0], e[sw, 1] = e[sw, 1].copy(), e[sw, 0].copy()
    return e[rng.permutation(len(e))]


@pytest.mark.parametrize("n,m", [(129, 400), (130, 420), (255, 1500), (257, 1600), (400, 4000), (400, 4001), (511, 6000),
                                 (513, 6000), (1023, 20000), (1025, 26000), (2047, 100000), (2048, 60000)])
@pytest.mark.parametrize("kind", ["random", "hub", "pairs", "split"])
@pytest.mark.parametrize("wmax", [5, 2**33])
def test_lists_equal_matrix(ctx, n, m, kind, wmax):
    e = _graph(kind, n, m, wmax)
    print(f"row lists {kind} n={n} m={len(e)} wmax={wmax}", flush=True)
    assert int(e[:, :2].max()) == n - 1 and (e[:, 0] != e[:, 1]).all()
    canon = np.stack([np.minimum(e[:, 0], e[:, 1]), np.maximum(e[:, 0], e[:, 1]), e[:, 2]], 1)
    raw_s, _ = ctx.ks_sparse(e, n, 6, 1, TRIALS)
    raw_d, _ = ctx.ks_dense(dense(n, canon), 6, 1, TRIALS)
    assert list(raw_s) == list(raw_d)
