"""Workloads whose time per call is measured, through the public entry points.

listed() names them, draw() gives more of the same ranges, prepare() makes
what a program holds before the call (a resident graph, an engine, queries,
training rows), run() is one call, work() is the traffic and arithmetic it
cannot do without, exact() is a 64-bit reference where floats are computed.

Graphs are of the kinds the framework is used on: Chung-Lu power-law graphs
(the serving graphs), R-MAT graphs (hub-heavy, kept sets below half the graph)
and graphs of overlapping dense communities on a sparse background (social
and collaboration networks, where searches finish with a proof).
"""

import ctypes as C
import os

import numpy as np
import torch

from scs_amd import graphgen, scs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"


def listed():
    return [
        # core numbers of a CSR already on the GPU (a caller that cannot
        # allocate, or re-peels a changing graph): the serving graph's size
        dict(name="core_large", kind="core", graph="chung_lu", n=500_000, m=8_000_000, beta=2.2),
        # a program's start: host CSR in, resident graph with core numbers out
        dict(name="graph_create", kind="create", graph="chung_lu", n=100_000, m=1_500_000,
             beta=2.3),
        # per-query preprocessing with everything copied out: a client that
        # wants the local graphs themselves
        dict(name="prep_probe", kind="probe", graph="chung_lu", n=4_000, m=88_000, beta=2.5,
             queries=8),
        # admission of a full batch on the serving graph (most queries keep
        # most of it)
        dict(name="prep_serving", kind="prep", graph="chung_lu", n=500_000, m=8_000_000, beta=2.2,
             queries=64),
        # admission of a full batch where every query gets its own compacted
        # CSR (hub-heavy graph, kept sets below half of it)
        dict(name="prep_local", kind="prep", graph="rmat", n=1 << 17, m=10 << 17, beta=0.0,
             queries=64),
        # greedy lower bounds on the GPU, a few queries of a small graph
        dict(name="heuristic_small", kind="heuristic", graph="chung_lu", n=4_000, m=88_000,
             beta=2.5, queries=8),
        # a full batch on a large one
        dict(name="heuristic_large", kind="heuristic", graph="chung_lu", n=100_000, m=1_500_000,
             beta=2.3, queries=64),
        # eight queries one after another, each to its proven optimum: latency
        dict(name="search_one", kind="search", graph="communities", n=2_000, queries=8, batch=1,
             learned=0, budget=200_000),
        # a batch of queries, each to its proven optimum
        dict(name="search_batch", kind="search", graph="communities", n=20_000, queries=64,
             batch=64, learned=1, budget=200_000),
        # searches that no budget lets finish, on kept sets of most of a large
        # graph: a batch of its stream, each query searched to its node budget
        dict(name="search_serving", kind="search", graph="chung_lu", n=50_000, m=750_000,
             beta=2.3, queries=64, batch=64, learned=1, budget=16),
        # two epochs of mini-batch training of the branching model
        dict(name="mlp_train", kind="train", rows=32_768, batch=2_048, epochs=2),
        # scoring many candidates with the engine's inference routine
        dict(name="mlp_infer", kind="infer", rows=200_000),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["core", "create", "probe", "prep", "prep", "heuristic", "heuristic", "search",
                       "search", "train", "infer"])
    if kind in ("train", "infer"):
        rows = _log(rng, 500, 32_768) if kind == "train" else _log(rng, 100, 200_000)
        if kind == "infer":
            return dict(kind=kind, rows=rows)
        return dict(kind=kind, rows=rows, batch=_log(rng, 256, 4_096), epochs=rng.randint(1, 2))
    if kind == "search":
        queries = _log(rng, 1, 64)
        return dict(kind=kind, graph="communities", n=_log(rng, 500, 20_000), queries=queries,
                    batch=1 if queries <= 8 and rng.random() < 0.5 else queries,
                    learned=rng.randint(0, 1), budget=200_000)
    top = {"core": 500_000, "create": 100_000, "probe": 8_000, "prep": 300_000,
           "heuristic": 100_000}[kind]
    n = _log(rng, 1_000, top)
    case = dict(kind=kind, graph="chung_lu", n=n, m=int(n * rng.uniform(6, 15)),
                beta=round(rng.uniform(2.2, 2.6), 3))
    if kind in ("prep", "heuristic") and rng.random() < 0.4:
        scale = rng.randint(11, 17)
        case.update(graph="rmat", n=1 << scale, m=rng.randint(6, 10) << scale, beta=0.0)
    if kind in ("probe", "prep", "heuristic"):
        case["queries"] = rng.randint(1, 8) if kind == "probe" else _log(rng, 1, 64)
    return case


# --- graphs -----------------------------------------------------------------

def _csr(n, u, v):
    """Simple symmetric CSR of the pairs, built on the GPU: (off, adj)."""
    keep = u != v
    u, v = u[keep], v[keep]
    key = torch.unique(torch.cat([u * n + v, v * n + u]))
    off = torch.zeros(n + 1, dtype=torch.int64, device=u.device)
    off[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return off, (key % n).to(torch.int32)


def _chung_lu(n, m, beta, seed):
    """Expected degrees (i + i0) ** (-1 / (beta - 1)), the largest about
    n / 25 (2 % to 25 % of the vertices in the workloads of this framework)."""
    alpha = 1.0 / (beta - 1.0)
    idx = np.arange(n, dtype=np.float64)
    dmax = max(3.0 * 2 * m / n, n / 25.0)
    lo, hi = 1e-9, 1e12
    for _ in range(100):
        mid = (lo * hi) ** 0.5
        if dmax * np.sum((mid / (idx + mid)) ** alpha) < 2 * m:
            lo = mid
        else:
            hi = mid
    w = (hi / (idx + hi)) ** alpha
    cdf = torch.from_numpy(np.cumsum(w) / np.sum(w)).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = torch.rand(2, m, generator=g, device=DEV, dtype=torch.float64)
    uv = torch.searchsorted(cdf, r, right=True).clamp_(max=n - 1)
    return _csr(n, uv[0], uv[1])


def _rmat(n, m, seed):
    scale = n.bit_length() - 1
    a, b, c = 0.57, 0.19, 0.19
    g = torch.Generator(device=DEV).manual_seed(seed)
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros_like(u)
    for level in range(scale):
        r = torch.rand(m, generator=g, device=DEV)
        bit = 1 << (scale - 1 - level)
        u += (r >= a + b).long() * bit
        v += (((r >= a) & (r < a + b)) | (r >= a + b + c)).long() * bit
    return _csr(n, u, v)


def _communities(n, seed):
    """Overlapping communities of 6 to 24 vertices, 60 % of their pairs
    joined, and one random edge a vertex."""
    rng = np.random.default_rng(seed)
    us, vs, total = [rng.integers(0, n, n)], [rng.integers(0, n, n)], 0
    while total < 1.3 * n:
        size = int(rng.integers(6, 25))
        members = rng.integers(0, n, size)
        i, j = np.triu_indices(size, 1)
        pick = rng.random(i.size) < 0.6
        us.append(members[i[pick]])
        vs.append(members[j[pick]])
        total += size
    return _csr(n, torch.from_numpy(np.concatenate(us)).to(DEV),
                torch.from_numpy(np.concatenate(vs)).to(DEV))


def _graph(case, seed):
    if case["graph"] == "rmat":
        return _rmat(case["n"], case["m"], seed)
    if case["graph"] == "communities":
        return _communities(case["n"], seed)
    return _chung_lu(case["n"], case["m"], case["beta"], seed)


# A query program keeps its graph and engine and only its queries change: the
# last one of each is held, and a case with another graph or engine replaces it.
_HELD = {}


def _resident(case):
    key = tuple(case.get(k) for k in ("graph", "n", "m", "beta"))
    if _HELD.get("graph_key") != key:
        _HELD.clear()
        off, adj = (t.cpu().numpy() for t in _graph(case, 7))
        G = scs.Graph.from_csr(off, adj)
        _HELD.update(graph_key=key, graph=G, core=G.core().astype(np.int64))
    return _HELD["graph"], _HELD["core"]


def _engine(case, **kw):
    G, core = _resident(case)
    key = tuple(sorted(kw.items())) + (case.get("learned", 0),)
    if _HELD.get("engine_key") != key:
        _HELD.pop("engine", None)
        E = scs.Engine(G, **kw)
        if case.get("learned"):
            E.set_model(scs.Model.load(os.path.join(ROOT, "models", "branching_c1.npz")), True)
        _HELD.update(engine_key=key, engine=E)
    return _HELD["engine"], core


def _queries(case, core, seed):
    """(l, h, q, heuristic flag, dominating-set limit) of the stream that
    belongs to the kind of graph."""
    count = case["queries"]
    if case["graph"] == "communities":  # windows inside a community
        kw = dict(core_min=5, l_lo=3, l_hi=7, dh_lo=1, dh_hi=3)
    elif case["graph"] == "rmat":
        kw = dict(core_min=1, l_lo=10, l_hi=60, dh_lo=10, dh_hi=100)
    elif case["n"] >= 250_000:  # the serving stream
        kw = dict(core_min=1, l_lo=5, l_hi=50, dh_lo=5, dh_hi=150, heu=(0, 1),
                  limit_doms=(4, 8, 16))
    else:
        kw = dict(core_min=min(8, int(core.max())), l_lo=5, l_hi=40, dh_lo=5, dh_hi=60)
    return [(x.l, x.h, x.q, x.heu, x.limit_doms)
            for x in graphgen.make_queries(core, count, seed, **kw)]


def _ubd(kl, h):
    """Diameter bound of a subgraph of at most h vertices and min degree kl."""
    if kl <= 1:
        return h - 1
    for d in range(1, h + 1):
        least = kl + d if d <= 2 else kl + d + 1 + (d // 3) * (kl - 2)
        if least > h:
            return d - 1
    return h - 1


def _bounds(qs, core, seed):
    """q, lower bound and depth bound as admission has them: a query without
    the heuristic starts from 0, one with it from 40 % to 95 % of its upper
    bound."""
    rng = np.random.default_rng(seed)
    q, kl, ubd = [], [], []
    for (l, h, v, heu, _) in qs:
        ku = min(int(core[v]), h - 1)
        k = min(int(ku * rng.uniform(0.4, 0.95)), ku - 1) if heu and ku > 1 else 0
        q.append(v)
        kl.append(k)
        ubd.append(_ubd(k, h))
    return tuple(np.array(x, np.uint32) for x in (q, kl, ubd))


# --- model rows ---------------------------------------------------------------

def _rows(n, seed):
    """Candidate rows as search traces give them (dC, dR, distance, core,
    slack, score) and labels a branching order can learn."""
    rng = np.random.default_rng(seed)
    X = np.stack([rng.integers(0, 20, n), rng.integers(0, 200, n), rng.integers(1, 6, n),
                  rng.integers(1, 60, n), rng.integers(1, 30, n), rng.random(n) * 4],
                 axis=1).astype(np.float32)
    y = (3 * X[:, 0] + X[:, 3] - 5 * X[:, 2] + rng.normal(0, 10, n) > 40).astype(np.float32)
    return X, y


def _norm(X):
    mean, std = np.zeros(8), np.ones(8)
    mean[:6], std[:6] = X.astype(np.float64).mean(0), X.astype(np.float64).std(0)
    return mean, 1.0 / np.maximum(std, 1e-6)


def _model(seed, X):
    d = scs.model_init(seed).to_arrays()
    d["mean"], d["scale"] = (a.astype(np.float32) for a in _norm(X))
    rng = np.random.default_rng(seed)
    d["b1"], d["b2"] = (rng.normal(0, 0.1, 64).astype(np.float32) for _ in range(2))
    return scs.Model.from_arrays(d)


# --- the cases ----------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("core", "create"):
        _HELD.clear()
        off, adj = _graph(case, seed)
        if kind == "create":
            return dict(case=case, off=off.cpu().numpy(), adj=adj.cpu().numpy())
        return dict(case=case, off=off, adj=adj,
                    core=torch.zeros(case["n"], dtype=torch.int32, device=DEV))
    if kind in ("probe", "prep"):
        E, core = _engine(case, limit_queries=64, waves_per_cu=1,
                          mem_budget=(1 << 30) if kind == "probe" else (16 << 30))
        q, kl, ubd = _bounds(_queries(case, core, seed), core, seed)
        st = dict(case=case, E=E, q=q, kl=kl, ubd=ubd)
        if kind == "probe":
            n, k, nnz = case["n"], len(q), E.graph.nnz
            st.update(K=np.zeros(k, np.uint32), nnz=np.zeros(k, np.uint64),
                      kept=np.zeros((k, n), np.uint32), loff=np.zeros((k, n + 1), np.uint32),
                      dist=np.zeros((k, n), np.uint32), ladj=np.zeros((k, nnz), np.uint32))
        return st
    if kind == "heuristic":
        G, core = _resident(case)
        return dict(case=case, G=G, qs=[x[:3] for x in _queries(case, core, seed)])
    if kind == "search":
        E, core = _engine(case, limit_queries=64, node_budget=case["budget"],
                          heuristic_threads=12, mem_budget=8 << 30)
        return dict(case=case, E=E, qs=_queries(case, core, seed))
    _HELD.clear()
    X, y = _rows(case["rows"], seed)
    if kind == "infer":
        return dict(case=case, X=X, model=_model(seed, X))
    return dict(case=case, X=X, y=y, seed=seed, start=scs.model_init(seed).to_arrays())


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "core":
        f = scs.lib().scs_core_numbers_noalloc
        f.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p, C.c_void_p]
        rc = f(s["off"].data_ptr(), s["adj"].data_ptr(), case["n"], s["core"].data_ptr(),
               torch.cuda.current_stream().cuda_stream)
        if rc:
            raise scs.SCSError(rc, "scs_core_numbers_noalloc")
        return s["core"]
    if kind == "create":
        G = scs.Graph.from_csr(s["off"], s["adj"])
        out = G.core()
        G.close()
        return out.astype(np.int64)
    if kind == "prep":
        K, nnz = s["E"].prep_many(s["q"], s["kl"], s["ubd"])
        return K.astype(np.int64), nnz.astype(np.int64)
    if kind == "probe":
        f = scs.lib().scs_prep_probe_many
        f.argtypes = [C.c_void_p, C.c_uint32] + [C.c_void_p] * 8 + [C.c_uint32, C.c_void_p,
                                                                     C.c_uint64]
        p = {k: s[k].ctypes.data for k in ("q", "kl", "ubd", "K", "nnz", "kept", "loff", "dist",
                                           "ladj")}
        rc = f(s["E"]._h, len(s["q"]), p["q"], p["kl"], p["ubd"], p["K"], p["nnz"], p["kept"],
               p["loff"], p["dist"], case["n"], p["ladj"], s["ladj"].shape[1])
        if rc:
            raise scs.SCSError(rc, "scs_prep_probe_many")
        return {"K": s["K"].view(np.int32), "nnz": s["nnz"].view(np.int64),
                **{k: s[k].view(np.int32) for k in ("kept", "loff", "dist", "ladj")}}
    if kind == "heuristic":
        got = scs.heuristic_gpu(s["G"], s["qs"])
        sets = np.full((len(got), 200), -1, np.int64)
        for i, (_, H) in enumerate(got):
            sets[i, :len(H)] = H
        return np.array([k for k, _ in got]), np.array([len(H) for _, H in got]), sets
    if kind == "search":
        # which of several optimal communities is returned, and through how
        # many nodes, depends on the order in which waves take tasks
        res, qs, b = [], s["qs"], case["batch"]
        for i in range(0, len(qs), b):
            res += s["E"].run(qs[i:i + b])
        out = {k: np.array([getattr(r, k) for r in res], np.int64)
               for k in ("kl", "heu_kl", "ku", "kept")}
        if case["graph"] == "communities":
            out["proven"] = np.array([r.status != "CAPPED" for r in res], np.int64)
        return out
    if kind == "infer":
        return scs.mlp_infer(s["model"], s["X"])
    m = scs.Model.from_arrays(s["start"])
    loss = scs.mlp_train(m, s["X"], s["y"], epochs=case["epochs"], batch=case["batch"], lr=2e-3,
                         pos_weight=2.0, seed=s["seed"])
    return {"loss": loss, **{k: v for k, v in m.to_arrays().items()}}


def _size(case):
    """Vertices and adjacency entries (about; duplicates are merged)."""
    if case["graph"] == "communities":
        return case["n"], 14 * case["n"]
    return case["n"], int((1.6 if case["graph"] == "rmat" else 1.9) * case["m"])


def work(case):
    kind = case["kind"]
    if kind == "infer":
        return dict(bytes=28 * case["rows"], flops=2 * (6 * 64 + 64 * 64 + 64) * case["rows"])
    if kind == "train":
        steps = case["epochs"] * max(1, case["rows"] // min(case["batch"], case["rows"]))
        rows = steps * min(case["batch"], case["rows"])
        return dict(bytes=28 * rows + steps * 7 * 4 * 4737,
                    flops=6 * (6 * 64 + 64 * 64 + 64) * rows)
    n, nnz = _size(case)
    if kind in ("core", "create"):
        return dict(bytes=8 * n + 4 * nnz + 4 * n, flops=0)
    q = case["queries"]
    if kind == "probe":  # the graph once, each query's local graph once
        return dict(bytes=12 * n + 4 * nnz + q * (16 * n + 4 * nnz), flops=0)
    if kind == "prep":  # the graph once, each query's distances
        return dict(bytes=12 * n + 4 * nnz + q * 4 * n, flops=0)
    # the graph once, an answer a query
    return dict(bytes=12 * n + 4 * nnz + q * 400, flops=0)


def exact(case, seed):
    """The inference scores in 64 bits, on the weights as they are given."""
    if case["kind"] != "infer":
        return None
    X, _ = _rows(case["rows"], seed)
    d = {k: np.asarray(v, np.float64) for k, v in _model(seed, X).to_arrays().items()}
    x = (X.astype(np.float64) - d["mean"][:6]) * d["scale"][:6]
    h = np.maximum(x @ d["w1"][:6] + d["b1"], 0)
    h = np.maximum(h @ d["w2"] + d["b2"], 0)
    return h @ d["w3"] + d["b3"]
