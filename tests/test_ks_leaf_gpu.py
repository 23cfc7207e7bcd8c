"""The Karger-Stein base case (at most 128 vertices) on the device against the
oracle, exact integers: sizes around one and two vertices per lane, 32- and
64-bit entries, shapes whose phases contract everything, a few or one pair."""
import numpy as np
import pytest
from graphgen import dense, erdos_renyi

import cac

pytestmark = pytest.mark.gpu


def _graph(rng, shape, n, wmax):
    w = lambda k: rng.integers(1, wmax + 1, k)
    iu, ju = np.triu_indices(n, 1)
    if shape == "complete":
        keep = np.ones(len(iu), bool)
    elif shape == "cycle":  # every phase ends on a vertex of degree 2
        keep = (ju == iu + 1) | ((iu == 0) & (ju == n - 1))
    elif shape == "blocks":  # two complete halves and one light edge: a cut far below every degree
        h = n // 2
        keep = ((iu < h) == (ju < h))
    else:
        return dense(n, erdos_renyi(rng, n, min(1.0, 6.0 / n), wmax=wmax))
    A = np.zeros((n, n), np.int64)
    A[iu[keep], ju[keep]] = w(int(keep.sum()))
    if shape == "blocks":
        A[0, n - 1] = 1
    return A + A.T


@pytest.mark.parametrize("wmax", [1, 1000, 1 << 40])
@pytest.mark.parametrize("shape", ["complete", "cycle", "blocks", "sparse"])
@pytest.mark.parametrize("n", [3, 17, 63, 64, 65, 127, 128])
def test_leaf_equals_oracle(ctx, orc, n, shape, wmax):
    if shape == "sparse" and n < 17:
        n += 4
    rng = np.random.default_rng(n * 7 + len(shape))
    A = _graph(rng, shape, n, wmax)
    print(f"leaf n {n} {shape} wmax {wmax}", flush=True)
    raw, mn = ctx.ks_dense(A, 1, 0, 1)
    assert raw.tolist() == [orc.ks_trial(A, 1, 0)]
    assert mn == min(orc.stoer_wagner(A), int(A.sum(1).min()))
