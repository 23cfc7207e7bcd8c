"""Edge lists of fewer than one and a half edges a vertex above 2^22 vertices, where a
list in no order is hooked past the giant component's bitmap and an ordered one is
not: on both sides of 2^22 vertices, of three quarters and of one and a half edges a
vertex, sorted, shuffled, and with an ordered head and a shuffled tail.  Labels equal
scipy's components as minimum ids."""
import numpy as np
import pytest
from scipy.sparse import coo_matrix
from scipy.sparse.csgraph import connected_components

import cac

pytestmark = pytest.mark.gpu


def _want(n, e):
    k, comp = connected_components(coo_matrix((np.ones(len(e), np.int8), (e[:, 0], e[:, 1])), shape=(n, n)),
                                   directed=False)
    first = np.full(k, n, np.int64)
    np.minimum.at(first, comp, np.arange(n))
    return first[comp], k


@pytest.mark.parametrize("n,m", [(1 << 22, (3 << 21) - 1), ((1 << 22) + 1, 2621441), ((1 << 22) + 1, 3145727),
                                 ((1 << 22) + 65, 3145793), ((1 << 22) + 2, (3 << 21) - 9)])
@pytest.mark.parametrize("order", ["sorted", "shuffled", "mixed"])
def test_cc_sparse_lists(ctx, n, m, order):
    rng = np.random.default_rng(n + m)
    # random edges among the even vertices below 7n/8, short paths beside them
    a = rng.integers(0, n // 16 * 7, (m * 3 // 4, 2)) * 2
    s = rng.integers(0, n - 2, m - len(a))
    e = np.sort(np.concatenate([a, np.stack([s, s + 1 + s % 2], axis=1)]), axis=1)
    e = e[np.argsort(e[:, 0] * n + e[:, 1])] if order != "shuffled" else e[rng.permutation(m)]
    if order == "mixed":
        e[m // 2:] = e[m // 2:][rng.permutation(m - m // 2)]
    print(f"cc sparse n {n} m {m} {order}", flush=True)
    want, k = _want(n, e)
    de = ctx.alloc(8 * m)
    dl = ctx.alloc(4 * n)
    try:
        de.upload(e.astype(np.uint32))
        count = ctx.cc_dev(de.ptr, m, n, dl.ptr, cac.LABEL_MIN_ID)
        assert count == k
        assert np.array_equal(dl.download(np.uint32, n), want)
        count = ctx.cc_static_dev(de.ptr, m, n, dl.ptr, cac.LABEL_MIN_ID)
        assert count == k
        assert np.array_equal(dl.download(np.uint32, n), want)
    finally:
        de.free()
        dl.free()
