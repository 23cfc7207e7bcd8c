"""Edge-list connected components at the sizes where the giant component's maps
change form (one exact map up to 2^20 vertices, two coarse ones above, groups of
more than 32 vertices, the queued run pass above 2^22), around the one and a half
edges a vertex from which the maps are used and the three quarters from which an
unordered list is sampled, with sorted and shuffled lists, odd lengths, a list
that starts on an odd 8-byte boundary, and small blocks without a giant component.
Labels equal scipy's components as minimum ids."""
import numpy as np
import pytest
from scipy.sparse import coo_matrix
from scipy.sparse.csgraph import connected_components

import cac

pytestmark = pytest.mark.gpu


def _edges(rng, n, m, order):
    e = _blocks(rng, n, m) if order == "blocks" else _giant(rng, n, m)
    return e[np.argsort(e[:, 0] * n + e[:, 1])] if order == "sorted" else e[rng.permutation(m)]


def _blocks(rng, n, m):
    u = rng.integers(0, n, m)
    e = np.stack([u, np.minimum(u // 16 * 16 + rng.integers(0, 16, m), n - 1)], axis=1)
    return np.sort(e, axis=1)


def _giant(rng, n, m):
    """A random part over every other block of 40 vertices (one giant component
    and stragglers, so groups are whole, mixed and outside), short paths beside it
    and edges from the last vertices."""
    blocks = n // 80
    a = rng.integers(0, blocks, (m // 2, 2)) * 80 + rng.integers(0, 40, (m // 2, 2))
    s = rng.integers(0, n - 3, m // 4)
    b = np.stack([s, s + rng.integers(1, 3, m // 4)], axis=1)
    e = np.concatenate([a, b, [[n - 1, n - 2], [n - 2, 0], [n - 1, n - 1]]])
    e = np.concatenate([e, np.stack([np.full(m - len(e), n // 3), rng.integers(0, n, m - len(e))], axis=1)])
    return np.sort(e, axis=1)


def _want(n, e):
    k, comp = connected_components(coo_matrix((np.ones(len(e), np.int8), (e[:, 0], e[:, 1])), shape=(n, n)),
                                   directed=False)
    first = np.full(k, n, np.int64)
    np.minimum.at(first, comp, np.arange(n))
    return first[comp], k


SIZES = [(5000, (1 << 18) + 1), ((1 << 18) + 1, 3 << 16), ((1 << 18) + 1, (3 << 17) - 1), ((1 << 18) + 1, 3 << 17),
         ((1 << 20) - 1, (3 << 19) + 1), (1 << 20, (3 << 19) + 1), ((1 << 20) + 1, (3 << 19) + 3),
         ((1 << 21) + 77, (3 << 20) + 201), ((1 << 22) + 5, (3 << 21) + 15), ((1 << 24) + 3, (3 << 23) + 9)]


@pytest.mark.parametrize("n,m", SIZES)
@pytest.mark.parametrize("order", ["sorted", "shuffled", "blocks"])
def test_cc_map_forms(ctx, n, m, order):
    if n > 1 << 23 and order == "shuffled":
        pytest.skip("the run pass of this size is the one above 2^22")
    rng = np.random.default_rng(n)
    print(f"cc maps n {n} m {m} {order}", flush=True)
    e = _edges(rng, n, m, order)
    assert len(e) == m and e.max() < n
    want, k = _want(n, e)
    print(f"  {k} components", flush=True)
    de, dl = ctx.alloc((m + 1) * 8), ctx.alloc(n * 4)
    try:
        de.upload(np.concatenate([[[0, 0]], e]).astype(np.uint32))
        for skip, mode in ((0, cac.LABEL_MIN_ID), (1, cac.LABEL_MIN_ID), (1, cac.LABEL_RANK)):
            # skip 0 counts the leading loop as an edge: an even length, 16-byte aligned
            count = ctx.cc_dev(de.ptr + 8 * skip, m + 1 - skip, n, dl.ptr, mode)
            assert count == k
            lab = dl.download(np.uint32, n)
            if mode == cac.LABEL_MIN_ID:
                assert np.array_equal(lab, want)
            else:
                roots = np.flatnonzero(want == np.arange(n))
                assert np.array_equal(roots[lab], want)
        if n <= cac.CC_STATIC_MAX_N:
            assert ctx.cc_static_dev(de.ptr + 8, m, n, dl.ptr) == k
            assert np.array_equal(dl.download(np.uint32, n), want)
    finally:
        de.free()
        dl.free()
