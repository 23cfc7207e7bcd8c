"""The approximate cut's linking passes: edge groups of 1 to 64 (about m / n, a power
of two), a partial last group, first disconnected levels on both sides of the four
that run side by side, weights of 0, several steps of the grid, and the form that
runs one level at a time (forests above 2^30 bytes for four).  Level and trial count
equal the oracle's exactly."""
import numpy as np
import pytest

import cac

pytestmark = pytest.mark.gpu
F32_95 = float(np.float32(0.95))


def _graph(n, m, wmax):
    """A path through all vertices and random edges, loops and weights of 0 among them."""
    rng = np.random.default_rng(n + m)
    u = np.concatenate([np.arange(n - 1), rng.integers(0, n, m - n + 1)])
    v = np.concatenate([np.arange(1, n), rng.integers(0, n, m - n + 1)])
    e = np.stack([u, v, rng.integers(0 if wmax > 1 else 1, wmax + 1, m)], axis=1).astype(np.int64)
    e[: n - 1, 2] = np.maximum(e[: n - 1, 2], 1)
    return e


def _check(ctx, orc, n, e, p, level=None):
    want = orc.approx_cut(n, e, p, 7)
    print(f"approx n {n} m {len(e)} level {want[0].bit_length() - 1}", flush=True)
    assert level is None or want[0] == 1 << level
    assert ctx.approx_cut(e, n, p, 7) == want


@pytest.mark.parametrize("n,m,wmax,level", [(300, 307, 200, 1), (300, 307, 3000, 5), (257, 1100, 30, 4),
                                            (400, 2051, 200, 7), (50, 2003, 1, 4), (50, 2003, 3, 5), (50, 2003, 30, 8),
                                            (30, 6007, 3000, 17), (1000, 40013, 1, 3), (1000, 40013, 3, 4),
                                            (700, 140009, 30, 10)])
def test_approx_groups(ctx, orc, n, m, wmax, level):
    _check(ctx, orc, n, _graph(n, m, wmax), F32_95, level)


def test_approx_many_edges(ctx, orc):
    """More edges a pass than the grid has threads."""
    _check(ctx, orc, 20000, _graph(20000, 2300007, 1), F32_95)


def test_approx_one_level_at_a_time(ctx, orc):
    n, p = 1530000, 1 - 1e-12  # 44 copies: four forests would take 1.08 GB
    assert 16 * n * orc.approx_trials(p) > 1 << 30
    e = np.stack([np.arange(n - 1), np.arange(1, n), np.full(n - 1, 64)], axis=1).astype(np.int64)
    _check(ctx, orc, n, e, p, 3)
