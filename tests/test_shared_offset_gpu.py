"""Batches whose graphs take parts of one edge list from the same offset (growing
prefixes of it): each graph's flag, total weight and packed form belong to its own
edges, so every cut equals the oracle's for that prefix alone, in either order."""
import numpy as np
import pytest

import cac

pytestmark = pytest.mark.gpu


def _ring(rng, n, chords, wide=1):
    """A heavy cycle through n vertices and light chords (trials' cuts differ);
    the chords after the first hundred weigh `wide` times as much."""
    e = [(i, (i + 1) % n, int(rng.integers(10**5, 2 * 10**5))) for i in range(n)]
    for k, (a, b) in enumerate(rng.integers(0, n, size=(chords, 2))):
        e.append((a, b, int(rng.integers(1, 10**4)) * (wide if k >= 100 else 1)))
    return np.array(e, dtype=np.uint64)


def _check(ctx, orc, e, parts, trials=2):
    """parts: (m, n) per graph, all from the first edge."""
    descs = np.array([(0, m, n, trials) for m, n in parts], dtype=cac.GRAPH_DESC)
    seen = set()
    for seed in range(3):
        cuts, _ = ctx.mincut_batch(e, descs, 0.95, seed)
        want = [min(orc.sqrt_trial(n, e[:m], cac.intermediate_size(n, m), seed, i) for i in range(trials))
                for m, n in parts]
        assert cuts.tolist() == want, (seed, parts)
        seen.update(want)
    assert len(seen) > 1


def _orders(*parts):
    return [list(parts), list(parts)[::-1]]


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("n", [333, 700, 2501])
def test_prefixes_with_mixed_weights(ctx, orc, n, order):
    e = _ring(np.random.default_rng(n), n, 5 * n)
    _check(ctx, orc, e, _orders((n, n), (n + 137, n), (3 * n, n), (len(e), n))[order])


@pytest.mark.parametrize("order", [0, 1])
def test_prefix_of_one_weight(ctx, orc, order):
    """The prefix needs no weight prefix, the whole list does."""
    e = _ring(np.random.default_rng(1), 600, 2000)
    e[:600, 2] = 150000
    _check(ctx, orc, e, _orders((600, 600), (len(e), 600))[order])


@pytest.mark.parametrize("order", [0, 1])
def test_prefixes_on_both_sides_of_32_bits(ctx, orc, order):
    """The prefix's total weight is below 2^31, the whole list's is not."""
    n = 900
    e = _ring(np.random.default_rng(2), n, 2000, wide=2**10)
    assert int(e[: n + 100, 2].sum()) < 2**31 <= int(e[:, 2].sum())
    _check(ctx, orc, e, _orders((n + 100, n), (len(e), n))[order])


@pytest.mark.parametrize("order", [0, 1])
def test_one_list_as_two_vertex_counts(ctx, orc, order):
    """The same edges with and without isolated vertices past 2^16: one packed, one not."""
    n = 400
    e = _ring(np.random.default_rng(3), n, 900)
    _check(ctx, orc, e, _orders((len(e), n), (len(e), 70001))[order], trials=1)


@pytest.mark.parametrize("order", [0, 1])
def test_prefixes_in_the_wide_form(orc, order):
    """Every trial sampled by grid-wide kernels: a round-0 prefix per graph."""
    n = 701
    e = _ring(np.random.default_rng(4), n, 5 * n)
    with cac.Context(0) as c:
        c.tune_set(cac.TUNE_WIDE_SAMPLING, 0, 1)
        _check(c, orc, e, _orders((n + 137, n), (3 * n, n), (len(e), n))[order])
