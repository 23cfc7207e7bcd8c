"""Square-root trials whose contracted graph is left as row lists (129 to 2048
super-vertices, at least twice as many vertices, most surviving edges at one
super-vertex), and the matrix form on either side of those limits and where the
lists exceed their room: raw cuts equal the oracle's.  Ring lattices with random
chords and two communities with a weak link between them.  Above 2^16 vertices and
in the wide form the lists come from the matrix, up to 4096 super-vertices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(rng, kind, n, d, weights):
    v = np.repeat(np.arange(n), d)
    u = (v + np.tile(np.arange(1, d + 1), n)) % n
    if kind == "ring":
        far = rng.random(len(u)) < 0.3
        u = np.where(far, rng.integers(0, n, len(u)), u)
    else:  # two random communities, d + 3 edges between them
        half = n // 2
        u = np.where(v < half, rng.integers(0, half, len(v)), rng.integers(half, n, len(v)))
        cross = np.stack([rng.integers(0, half, d + 3), rng.integers(half, n, d + 3)], 1)
        u, v = np.concatenate([u, cross[:, 0]]), np.concatenate([v, cross[:, 1]])
    u = np.where(u == v, np.where(v > 0, v - 1, 1), u)
    w = np.full(len(u), 3) if weights == "one" else rng.integers(1, 9, len(u))
    return np.stack([u, v, w], axis=1).astype(np.uint64)


@pytest.mark.parametrize("n,d,t", [(257, 6, 129), (258, 6, 129), (3000, 8, 128), (3000, 8, 129), (3000, 3, 700),
                                   (5000, 12, 500), (9000, 8, 2047), (9000, 8, 2048), (9000, 8, 2049),
                                   (4095, 8, 2048), (60000, 6, 900)])
@pytest.mark.parametrize("kind", ["ring", "two"])
@pytest.mark.parametrize("weights", ["one", "mixed"])
def test_trial_lists(ctx, orc, n, d, t, kind, weights):
    e = _graph(np.random.default_rng(n + t), kind, n, d, weights)
    raw = ctx.sqrt_cut_trials(e, n, t, 7, 2, 4)
    want = [orc.sqrt_trial(n, e, t, 7, 2 + i, 0) for i in range(4)]
    print(f"trial lists {kind} {weights} n {n} m {len(e)} t {t}: cuts {sorted(set(want))}", flush=True)
    assert raw.tolist() == want


@pytest.mark.parametrize("n,d,t", [(65537, 3, 128), (65537, 3, 129), (70001, 3, 2049), (70001, 4, 4096),
                                   (70001, 4, 4097), (150000, 7, 1100), (70001, 1, 1000)])
@pytest.mark.parametrize("kind", ["ring", "two"])
@pytest.mark.parametrize("scale", [1, 2**20])
def test_lists_from_matrix(ctx, orc, n, d, t, kind, scale):
    e = _graph(np.random.default_rng(n + t), kind, n, d, "mixed")
    e[:, 2] *= np.uint64(scale)  # 2^20: a total of 2^31 or more keeps 64-bit matrices
    raw = ctx.sqrt_cut_trials(e, n, t, 7, 2, 2)
    want = [orc.sqrt_trial(n, e, t, 7, 2 + i, 0) for i in range(2)]
    print(f"lists from matrix {kind} {scale} n {n} m {len(e)} t {t}: cuts {sorted(set(want))}", flush=True)
    assert raw.tolist() == want
