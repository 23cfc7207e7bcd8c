"""The workloads that the framework's performance is measured on.

Every case is one call (or one burst of calls) through the public entry points of
the ctypes mirror (comm-avoiding-cuts-cc_amd/cac.py), over the ranges a user of
the command lines, of the batched entry point and of the serving loop meets:
connected components on edge lists and on a CSR, dense and sparse Karger-Stein,
the square-root min cut of one graph and of a batch, the approximate cut, and a
burst of served queries.  Inputs are random graphs made from the seed; results
are whole numbers (labels, component counts, cuts, trial counts).
"""
import importlib
import math

import numpy as np
import torch

cac = importlib.import_module("comm-avoiding-cuts-cc_amd.cac")

P = float(np.float32(0.95))       # the command lines parse their probability as a float
P_KS = float(np.float32(0.90))    # karger_stein's fixed probability


def listed():
    return [
        # parallel_cc on a small graph: host arrays in and out, latency only
        dict(name="cc_host_small", kind="cc_host", n=2000, m=3000, rank=True),
        # an edge list in file order (no order at all), sizes that divide nothing
        dict(name="cc_list_random", kind="cc_list", n=10000019, m=24000041, graph="uniform", rank=True),
        # the benchmark's R-MAT graph as a sorted edge list resident in HBM
        dict(name="cc_list_rmat", kind="cc_list", n=1 << 24, m=1 << 28, graph="rmat", rank=False),
        # the same graph held as a symmetric CSR: the headline workload
        dict(name="cc_csr_rmat", kind="cc_csr", n=1 << 24, m=1 << 28, graph="rmat", rank=False),
        # a mid-sized dense matrix with weights that need 64-bit sums
        dict(name="ks_dense_700_heavy", kind="ks_dense", n=700, wmax=1 << 36, trials=49),
        # the dense Karger-Stein benchmark: complete graph, weights U[1, 42]
        dict(name="ks_dense_8192", kind="ks_dense", n=8192, wmax=42, trials=169),
        # square_root on G(1000, 0.05): the smallest min-cut solve in use
        dict(name="mincut_er1000", kind="mincut_er", n=1000, p=0.05, wmax=100),
        # square_root on the reference's Watts-Strogatz experiment
        dict(name="mincut_ws32k", kind="mincut_ws", n=32000, d=16),
        # karger_stein (sparse recursion) on the same family
        dict(name="karger_stein_ws48k", kind="karger_stein", n=48000, d=16),
        # a batch of planted-cut graphs of uneven size, two or more trials each
        dict(name="mincut_batch_768", kind="batch", count=768, nmin=256, nmax=65536, hard=False),
        # approx_cut on a few Watts-Strogatz graphs
        dict(name="approx_ws32k", kind="approx", n=32000, d=16, graphs=3),
        # a burst of mixed queries on the serving loop, uploads included
        dict(name="serve_burst_48", kind="serve", count=48, nmin=1000, nmax=300000),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cc_host", "cc_list", "cc_list", "cc_csr", "ks_dense", "ks_dense", "mincut_er", "mincut_ws",
                       "karger_stein", "batch", "approx", "serve"])
    if kind == "cc_host":
        n = _log_uniform(rng, 300, 200000)
        return dict(kind=kind, n=n, m=int(n * rng.uniform(0.5, 3)), rank=rng.random() < 0.5)
    if kind in ("cc_list", "cc_csr"):
        graph = rng.choice(["rmat", "uniform"])
        m = _log_uniform(rng, 1 << 18, 1 << 28)
        deg = rng.uniform(0.6, 4) if graph == "uniform" else rng.uniform(8, 32)
        n = min((1 << 24) + 1001, max(1024, int(m / deg)))
        if graph == "rmat":
            n = 1 << max(10, min(24, n.bit_length()))
        return dict(kind=kind, n=n, m=m, graph=graph, rank=rng.random() < 0.5)
    if kind == "ks_dense":
        n = _log_uniform(rng, 150, 8192)
        # from the trials of one solve (p = 0.95) to log2(n)^2
        trials = rng.randint(cac.ks_trials(n, P), int(math.log2(n) ** 2))
        return dict(kind=kind, n=n, wmax=rng.choice([42, 100, 1000, 1 << 20, 1 << 36]), trials=trials)
    if kind == "mincut_er":
        n = _log_uniform(rng, 200, 4000)
        return dict(kind=kind, n=n, p=round(rng.uniform(3, 6) * math.log(n) / n, 4), wmax=rng.choice([50, 100, 1 << 30]))
    if kind == "mincut_ws":
        return dict(kind=kind, n=_log_uniform(rng, 1000, 64000), d=rng.randint(6, 16))
    if kind == "karger_stein":
        return dict(kind=kind, n=_log_uniform(rng, 3000, 64000), d=rng.randint(6, 16))
    if kind == "batch":
        return dict(kind=kind, count=_log_uniform(rng, 16, 768), nmin=256, nmax=_log_uniform(rng, 2048, 65536),
                    hard=rng.random() < 0.3)
    if kind == "approx":
        return dict(kind=kind, n=_log_uniform(rng, 1000, 96000), d=rng.randint(6, 16), graphs=rng.randint(2, 4))
    return dict(kind="serve", count=_log_uniform(rng, 8, 64), nmin=1000, nmax=_log_uniform(rng, 10000, 300000))


# ---- inputs --------------------------------------------------------------------
_held = {}


def _handle(kind):
    """The context (or server) a program holds while it does one kind of work.  A
    context keeps its grown device buffers, so the one held for the previous kind
    of work is closed first."""
    if kind not in _held:
        for h in _held.values():
            h.close()
        _held.clear()
        torch.cuda.empty_cache()
        _held[kind] = cac.Server(0, workers=4, hbm_budget=160 << 30, max_batch=64) if kind == "serve" \
            else cac.Context(0)
    return _held[kind]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _edge_keys(case, seed):
    """Undirected edges as u << 32 | v (u < v) on the GPU: an R-MAT list is sorted
    and without duplicates (at most m edges), a uniform one in random order."""
    g = _gen(seed)
    n, m = case["n"], case["m"]
    if case.get("graph", "uniform") == "uniform":
        e = torch.randint(0, n, (m, 2), generator=g, device="cuda")
        return (e.amin(1) << 32) | e.amax(1)
    u = torch.zeros(m, dtype=torch.int32, device="cuda")
    v = torch.zeros(m, dtype=torch.int32, device="cuda")
    for _ in range(n.bit_length() - 1):  # quadrants (0.45, 0.22, 0.22, 0.11)
        x = torch.rand(m, generator=g, device="cuda")
        u.mul_(2).add_(x >= 0.67)
        v.mul_(2).add_(((x >= 0.45) & (x < 0.67)) | (x >= 0.89))
    lo, hi = torch.minimum(u, v).long(), torch.maximum(u, v)
    del u, v, x
    keys = (lo << 32) | hi
    del lo, hi
    keys = keys[(keys >> 32) != (keys & 0xFFFFFFFF)]
    return torch.unique_consecutive(keys.sort().values)


def _edges_dev(case, seed):
    """(u, v) pairs of 32-bit ids on the GPU."""
    k = _edge_keys(case, seed)
    out = torch.empty((len(k), 2), dtype=torch.int32, device="cuda")
    out[:, 0] = k >> 32
    out[:, 1] = k & 0xFFFFFFFF
    return out


def _ws(seed, n, d, lo=64, hi=1023):
    """A Watts-Strogatz graph whose edges all weigh the same."""
    w = int(np.random.default_rng(seed).integers(lo, hi + 1))
    return cac.gen_ws(n, d, seed, 0.3, w)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case, seed=seed, h=_handle(kind))
    n = case.get("n", 0)
    if kind == "cc_host":
        s["edges"] = _edges_dev(case, seed).cpu().numpy().view(np.uint32)
    elif kind in ("cc_list", "cc_csr"):
        e = _edges_dev(case, seed)
        s["m"] = len(e)
        s["labels"] = torch.empty(n, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        if kind == "cc_list":
            s["edges"] = e
        else:
            s["offsets"] = torch.empty(n + 1, dtype=torch.int32, device="cuda")
            s["cols"] = torch.empty(2 * len(e), dtype=torch.int32, device="cuda")
            s["h"].csr_build_dev(e.data_ptr(), len(e), n, s["offsets"].data_ptr(), s["cols"].data_ptr())
    elif kind == "ks_dense":
        a = torch.randint(1, case["wmax"] + 1, (n, n), generator=_gen(seed), device="cuda").triu_(1)
        s["adj"] = a + a.T
    elif kind == "mincut_er":
        rng = np.random.default_rng(seed)
        u, v = np.triu_indices(n, 1)
        keep = rng.random(len(u)) < case["p"]
        keep |= v == u + 1  # a path through all vertices: connected
        s["edges"] = np.empty(int(keep.sum()), dtype=cac.EDGE)
        s["edges"]["u"], s["edges"]["v"] = u[keep], v[keep]
        s["edges"]["w"] = rng.integers(1, case["wmax"] + 1, int(keep.sum()))
    elif kind in ("mincut_ws", "karger_stein"):
        s["edges"] = _ws(seed, n, case["d"])
    elif kind == "approx":
        s["graphs"] = [_ws(seed * 8 + i, n + i, case["d"], 1, 20000) for i in range(case["graphs"])]
    elif kind == "batch":
        first = (seed % 1000003) * 1024  # the generator numbers its graphs
        gen = cac.gen_planted_hard if case["hard"] else cac.gen_planted
        descs, edges, _ = gen(first, case["count"], seed, case["nmin"], case["nmax"])
        for d in descs:
            d["trials"] = max(2, cac.ks_trials(cac.intermediate_size(int(d["n"]), int(d["m"])), P))
        s["descs"] = descs
        s["edges"] = torch.from_numpy(edges.view(np.int64)).cuda()
    else:
        rng = np.random.default_rng(case["count"])  # the queries' sizes and kinds belong to the case
        s["queries"], labels = [], []
        for i in range(case["count"]):
            nq = int(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]))))
            e = cac.gen_gnp(nq, float(rng.uniform(8, 64)), seed, i, 100)
            if rng.random() < 0.7:
                labels.append(np.zeros(nq, dtype=np.uint32))
                s["queries"].append(cac.Server.query(cac.QUERY_CC, e, nq, labels=labels[-1]))
            else:
                t = min(cac.intermediate_size(nq, len(e)), 4096)
                s["queries"].append(cac.Server.query(cac.QUERY_MINCUT, e, nq, P, seed=i,
                                                     trials=max(2, cac.ks_trials(t, P))))
        s["labels"] = labels
        s["arrivals"] = np.zeros(case["count"])
    torch.cuda.synchronize()
    return s


def run(s):
    h, case, kind = s["h"], s["case"], s["kind"]
    n, seed = case.get("n", 0), s["seed"] & 0x7FFFFFFF
    if kind == "cc_host":
        labels, count = h.cc(s["edges"], n, cac.LABEL_RANK if case["rank"] else cac.LABEL_MIN_ID)
        return dict(labels=labels, count=count)
    if kind == "cc_list":
        count = h.cc_dev(s["edges"].data_ptr(), s["m"], n, s["labels"].data_ptr(),
                         cac.LABEL_RANK if case["rank"] else cac.LABEL_MIN_ID)
        return dict(labels=s["labels"], count=count)
    if kind == "cc_csr":
        count = h.cc_csr_dev(s["offsets"].data_ptr(), s["cols"].data_ptr(), n, s["labels"].data_ptr(),
                             cac.LABEL_RANK if case["rank"] else cac.LABEL_MIN_ID)
        return dict(labels=s["labels"], count=count)
    if kind == "ks_dense":
        raw, cut = h.ks_dense_dev(s["adj"].data_ptr(), n, seed, 0, case["trials"])
        return dict(raw=raw, cut=cut)
    if kind in ("mincut_er", "mincut_ws"):
        cut, trials = h.mincut(s["edges"], n, P, seed)
        return dict(cut=cut, trials=trials)
    if kind == "karger_stein":
        cut, trials = h.karger_stein(s["edges"], n, P_KS, seed)
        return dict(cut=cut, trials=trials)
    if kind == "batch":
        cuts, trials = h.mincut_batch_dev(s["edges"].data_ptr(), s["descs"], P, seed)
        return dict(cuts=cuts, trials=trials)
    if kind == "approx":
        got = [h.approx_cut(e, n + i, P, seed) for i, e in enumerate(s["graphs"])]
        return dict(approx=np.array([a for a, _ in got]), trials=np.array([t for _, t in got]))
    r = h.replay(s["queries"], s["arrivals"])
    return dict(status=r["status"], ncomp=r["ncomp"], cut=r["cut"], t=r["t"], trials=r["trials"],
                labels=np.concatenate(s["labels"]) if s["labels"] else np.zeros(0, np.uint32))


# ---- the work a pass cannot do without -----------------------------------------
def _ks_bytes(n, word=8):
    """One dense Karger-Stein trial: every child reads its parent's matrix and
    writes its own, leaves of 128 vertices are read once."""
    total, nodes, s = 0, 1, n
    while s > 128:
        t = max(int(math.ceil(s / math.sqrt(2.0))) + 1, 128)
        nodes *= 2
        total += nodes * word * (s * s + t * t)
        s = t
    return total + nodes * word * s * s


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind in ("cc_host", "cc_list"):
        return dict(bytes=8 * case["m"] + 12 * n, flops=0)
    if kind == "cc_csr":
        # the offsets, each vertex's first neighbour and parent, the labels: a graph
        # with one large component needs no more of its adjacency read
        return dict(bytes=16 * n, flops=0)
    if kind == "ks_dense":
        return dict(bytes=8 * n * n + case["trials"] * _ks_bytes(n), flops=0)
    if kind in ("mincut_er", "mincut_ws"):
        m = int(n * n / 2 * case["p"]) if kind == "mincut_er" else n * case["d"]
        t, trials = cac.intermediate_size(n, m), cac.sqrt_trials(n, m, P)
        return dict(bytes=trials * (16 * m + 8 * t * t), flops=0)
    if kind == "karger_stein":
        m = n * case["d"]
        return dict(bytes=cac.ks_trials(n, P_KS) * 2 * 40 * m, flops=0)
    if kind == "batch":
        lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
        mean = (case["nmax"] - case["nmin"]) / (hi - lo)
        return dict(bytes=case["count"] * 5 * 16 * 8 * mean, flops=0)
    if kind == "approx":
        return dict(bytes=case["graphs"] * 16 * n * case["d"], flops=0)
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return dict(bytes=case["count"] * 16 * 18 * (case["nmax"] - case["nmin"]) / (hi - lo), flops=0)


# ---- connected components in plain torch ---------------------------------------
def _components(u, v, n):
    """Minimum vertex id of every vertex's component, 64-bit, by hooking roots to
    the smallest neighbouring root and pointer jumping."""
    lab = torch.arange(n, device=u.device)
    while True:
        lu, lv = lab[u], lab[v]
        out = lu != lv
        if not bool(out.any()):
            return lab
        u, v, lu, lv = u[out], v[out], lu[out], lv[out]
        lab.scatter_reduce_(0, torch.maximum(lu, lv), torch.minimum(lu, lv), "amin")
        while True:
            up = lab[lab]
            if torch.equal(up, lab):
                break
            lab = up


def exact(case, seed):
    if case["kind"] not in ("cc_host", "cc_list", "cc_csr"):
        return None  # cuts are minima over random trials: whole numbers of the program's own draws
    k = _edge_keys(case, seed)
    lab = _components(k >> 32, k & 0xFFFFFFFF, case["n"])
    roots = lab == torch.arange(case["n"], device=lab.device)
    if case["rank"]:
        lab = (torch.cumsum(roots, 0) - 1)[lab]
    return dict(labels=lab, count=int(roots.sum()))
