"""Connected components of small graphs, which run in one workgroup, at the edges
of its range: vertex counts around whole 64s and 32768, edge counts around 32768,
paths, stars, random lists, loops, no edges, and out-of-range ids.  Labels equal
the union-find oracle below, as minimum ids and as ranks, for host arrays and for
device buffers; just past the range the general sequence gives the same."""
import numpy as np
import pytest

import cac

pytestmark = pytest.mark.gpu


def _want(n, e):
    par = list(range(n))

    def find(x):
        while par[x] != x:
            par[x] = par[par[x]]
            x = par[x]
        return x

    for u, v in e.tolist():
        a, b = find(u), find(v)
        if a != b:
            par[max(a, b)] = min(a, b)
    return np.array([find(v) for v in range(n)], np.int64)


def _edges(kind, n, m):
    rng = np.random.default_rng(n * 7 + m)
    if kind == "path":  # from the far end: every link joins two long chains or a chain and a vertex
        u = np.arange(n - 1)[rng.permutation(n - 1)][:m] if n > 1 else np.zeros(0, np.int64)
        return np.stack([u + 1, u], axis=1)
    if kind == "star":
        return np.stack([rng.integers(0, n, m), np.full(m, n - 1)], axis=1)
    return rng.integers(0, n, (m, 2))


@pytest.mark.parametrize("n,m", [(1, 0), (1, 3), (2, 1), (63, 40), (64, 64), (65, 200), (1000, 0), (4097, 3001),
                                 (32767, 20000), (32768, 32768), (32769, 32768), (32768, 32769), (500, 32768)])
@pytest.mark.parametrize("kind", ["random", "path", "star"])
def test_small_cc(ctx, n, m, kind):
    e = _edges(kind, n, m)
    m = len(e)
    want = _want(n, e)
    roots = np.flatnonzero(want == np.arange(n))
    print(f"small cc n {n} m {m} {kind}: {len(roots)} components", flush=True)
    de, dl = ctx.alloc(max(m, 1) * 8), ctx.alloc(n * 4)
    try:
        de.upload(e.astype(np.uint32) if m else np.zeros((1, 2), np.uint32))
        for mode in (cac.LABEL_MIN_ID, cac.LABEL_RANK):
            lab, count = ctx.cc(e.astype(np.uint32), n, mode)
            assert count == len(roots)
            assert ctx.cc_dev(de.ptr, m, n, dl.ptr, mode) == len(roots)
            for got in (lab, dl.download(np.uint32, n)):
                assert np.array_equal(roots[got] if mode == cac.LABEL_RANK else got, want)
    finally:
        de.free()
        dl.free()


@pytest.mark.parametrize("n,m", [(1, 1), (64, 100), (32768, 32768), (32769, 100)])
def test_small_cc_bad_ids(ctx, n, m):
    e = np.zeros((m, 2), np.uint32)
    for at, end, val in ((0, 0, n), (m - 1, 1, 0xFFFFFFFF)):
        bad = e.copy()
        bad[at, end] = val
        with pytest.raises(cac.CacError):
            ctx.cc(bad, n, cac.LABEL_MIN_ID)
    lab, count = ctx.cc(e, n, cac.LABEL_MIN_ID)
    assert count == n and np.array_equal(lab, np.arange(n))
