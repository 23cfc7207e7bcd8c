"""A server whose whole budget is what one group of queries is admitted with runs
that group, whatever its graphs weigh, with the cuts of the oracle's trials."""
import numpy as np
import pytest

import cac

pytestmark = pytest.mark.gpu
F32_95 = float(np.float32(0.95))


def _queries(wmax):
    """Graphs of 90 vertices (no Karger-Stein levels to leave room) to 6000, one
    trial or a few."""
    out = []
    for i, (n, d, trials) in enumerate([(90, 40.0, 1), (400, 12.0, 2), (1500, 30.0, 3), (6000, 9.0, 2)]):
        e = cac.gen_gnp(n, d, 31, i, wmax=wmax)
        out.append((n, e, 50 + i, trials))
    return out


@pytest.mark.parametrize("wmax", [100, 2**30])
@pytest.mark.parametrize("alone", [False, True])
def test_budget_of_exactly_the_admitted_bytes(orc, wmax, alone):
    qs = _queries(wmax)
    for group in ([[q] for q in qs] if alone else [qs]):
        recs = [cac.Server.query(cac.QUERY_MINCUT, e, n, F32_95, sd, trials=T) for n, e, sd, T in group]
        with cac.Server(0, workers=1, hbm_budget=4 << 30, max_batch=16) as srv:
            need = 0
            for r in recs:
                srv.replay([r], np.zeros(1))
                need = max(need, srv.stats()[0])
        with cac.Server(0, workers=1, hbm_budget=need, max_batch=16) as srv:
            res = srv.replay(recs, np.zeros(len(recs)))
            assert srv.stats()[0] <= need
        for r, (n, e, sd, T) in zip(res, group):
            assert r["status"] == 0
            e3 = np.stack([e["u"], e["v"], e["w"]], axis=1).astype(np.uint64)
            want = min(orc.sqrt_trial(n, e3, int(r["t"]), sd, i) for i in range(T))
            assert r["cut"] == want, (n, wmax, r["cut"], want)


@pytest.mark.parametrize("n,d", [(3000, 4.0), (150001, 4.0), (400000, 1.4), (1050000, 3.2)])
def test_cc_query_fits_its_edges_labels_and_bitmap(orc, n, d):
    """A components query takes its upload, its endpoints, its labels and, from 2^18
    edges, a bit per vertex; the coarse map of the giant component takes no more."""
    e = cac.gen_gnp(n, d, 3, 1, wmax=9)
    m = len(e)
    up = lambda x: (x + 255) // 256 * 256  # noqa: E731
    bitmap = up((n + 63) // 64 * 8) if m >= 1 << 18 else 0
    need = up(16 * m) + up(8 * m) + up(4 * n) + 256 + bitmap + 4096
    lab = np.zeros(n, dtype=np.uint32)
    with cac.Server(0, workers=1, hbm_budget=need, max_batch=4) as srv:
        res = srv.replay([cac.Server.query(cac.QUERY_CC, e, n, labels=lab)], np.zeros(1))
        assert res[0]["status"] == 0
        assert srv.stats()[0] == need
    want, nc = orc.cc(np.stack([e["u"], e["v"]], 1).astype(np.uint32), n)
    assert res[0]["ncomp"] == nc and np.array_equal(lab, want)
