"""Square-root trials in 32-bit arithmetic on the packed graph (at most 2^16
vertices, total weight below 2^31) and the general form on either side of those
limits: raw cuts equal the oracle's, exact integers.  Small targets make the
trials' cuts differ, so a wrong draw, label or survivor shows."""
import numpy as np
import pytest

import cac

pytestmark = pytest.mark.gpu


def _graph(rng, n, m, w):
    """A path through all vertices and random edges, loops and repeats among them."""
    u = np.concatenate([np.arange(n - 1), rng.integers(0, n, max(m - n + 1, 0))])
    v = np.concatenate([np.arange(1, n), rng.integers(0, n, max(m - n + 1, 0))])
    return np.stack([u, v, w(len(u))], axis=1).astype(np.uint64)


def _check(ctx, orc, n, e, t, trials, differ=True, dpr=0):
    raw = ctx.sqrt_cut_trials(e, n, t, 7, 2, trials)
    want = [orc.sqrt_trial(n, e, t, 7, 2 + i, dpr) for i in range(trials)]
    print(f"packed n {n} m {len(e)} t {t}: {len(set(want))} different cuts", flush=True)
    assert raw.tolist() == want
    assert not differ or len(set(want)) > 1


@pytest.mark.parametrize("n,m,t", [(7, 9, 2), (50, 97, 5), (1001, 4099, 9), (1024, 16384, 12), (4097, 16387, 6),
                                   (32768, 250001, 5), (65535, 500003, 5), (65536, 700002, 5), (65537, 400001, 5)])
@pytest.mark.parametrize("weights", ["one", "mixed"])
def test_packed_sizes(ctx, orc, n, m, t, weights):
    rng = np.random.default_rng(n + m)
    e = _graph(rng, n, m, (lambda k: np.full(k, 9)) if weights == "one" else (lambda k: rng.integers(0, 60, k)))
    e[: n - 1, 2] = np.maximum(e[: n - 1, 2], 1)  # the path keeps it connected
    if weights == "one":
        e = e[e[:, 0] != e[:, 1]]  # one weight and no loop: draws by division
    _check(ctx, orc, n, e, t, 6, differ=n > 60)


@pytest.mark.parametrize("total", [2**31 - 1, 2**31, 2**31 + 1])
@pytest.mark.parametrize("n,m", [(500, 3000), (3001, 9001)])
def test_packed_weight_limit(ctx, orc, n, m, total):
    """Total weights just below the limit run packed, at and above it in 64 bits."""
    rng = np.random.default_rng(n)
    e = _graph(rng, n, m, lambda k: rng.integers(1, 2**31 // (2 * m), k))
    e[:, 2] = e[:, 2] * np.uint64(total // int(e[:, 2].sum()))
    e[-1, 2] += np.uint64(total - int(e[:, 2].sum()))
    assert int(e[:, 2].sum()) == total
    _check(ctx, orc, n, e, 15, 6)


def test_packed_high_concurrency_rule(orc):
    rng = np.random.default_rng(5)
    n = 3000
    e = _graph(rng, n, 12001, lambda k: rng.integers(1, 40, k))
    with cac.Context(0) as c:
        c.set_sampling_rule(cac.SAMPLE_HC)
        _check(c, orc, n, e, 20, 6, dpr=cac.hc_draws(n))


def test_packed_disconnected_is_zero(ctx, orc):
    rng = np.random.default_rng(6)
    n = 2002
    e = _graph(rng, 1001, 4000, lambda k: rng.integers(1, 40, k))
    f = e.copy()
    f[:, :2] += np.uint64(1001)
    _check(ctx, orc, n, np.concatenate([e, f]), 2, 3, differ=False)
    assert ctx.sqrt_cut_trials(np.concatenate([e, f]), n, 2, 7, 2, 3).max() >= 0


def test_packed_and_general_graphs_in_one_batch(ctx, orc):
    """Graphs above 2^16 vertices, heavy graphs and packed ones share a chunk."""
    rng = np.random.default_rng(8)
    sizes = [(300, 1500, 50), (70001, 150000, 50), (2000, 9000, 2**22), (65536, 140000, 30), (9, 14, 3)]
    lists = [_graph(rng, n, m, lambda k, w=w: rng.integers(1, w, k)) for n, m, w in sizes]
    descs = np.zeros(len(sizes), dtype=cac.GRAPH_DESC)
    off = 0
    for d, (n, _, _), e in zip(descs, sizes, lists):
        d["edge_offset"], d["m"], d["n"], d["trials"] = off, len(e), n, 3
        off += len(e)
    cuts, trials = ctx.mincut_batch(np.concatenate(lists), descs, 0.95, 11)
    for c, (n, _, _), e in zip(cuts, sizes, lists):
        t = cac.intermediate_size(n, len(e))
        assert c == min(orc.sqrt_trial(n, e, t, 11, i) for i in range(3))
