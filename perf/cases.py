"""The work that a user of this framework has it do, as cases that can be timed.

Every kind goes through the package's public entry points:

  search   `Index.search` (host arrays in and out), `Index.search_async` (device
           tensors) or a replayed `Index.capture`, over an index built here
  coded    the engine's search with the sign-code pre-filter
  select   `select_nearest`: seeds against a catalogue or an entry pool, and the
           exact neighbours of a query block over a whole corpus (ground truth)
  graph    `build_graph`: sweep, prune, reverse
  codes    `build_codes`
  offline  the offline builder's stages on the device: candidates from a graph,
           mutual ranks, prune, reverse, in-degree floor, degree fill

Rows are drawn from a low-dimensional latent space plus a little noise, which is
how embeddings of text and images lie (an intrinsic dimension of a few tens in
hundreds or thousands of coordinates).  Rows are normalised for ip; for l2 their
lengths spread by about a quarter.  The searches' knobs are those of accurate
search (recall near 1), where branches that race for the shared claims still
return the same neighbours.
"""
from __future__ import annotations

import math

import torch

import swann_amd
from swann_amd import _engine, offline
from swann_amd._select import select_nearest
from swann_amd.build import add_reverse, build_graph, knn_candidates, robust_prune
from swann_amd.codes import build_codes

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16}
LATENT = 24
NOISE = 0.05


def listed():
    return [
        # one query of a chat or web service, numpy in and out: pure latency
        dict(name="search-one", kind="search", call="host", n=50_000, d=768, dtype="f32",
             metric="ip", degree=64, nq=1, branches=32, queue=32, stop_eps=0.3, team=16),
        # a serving loop that replays a captured search of a few wide queries
        dict(name="search-captured", kind="search", call="graph", n=60_000, d=4096, dtype="f16",
             metric="ip", degree=64, nq=8, branches=128, queue=24, stop_eps=0.3, team=32),
        # a batch from a request queue over an fp32 l2 corpus
        dict(name="search-batch", kind="search", call="device", n=150_000, d=960, dtype="f32",
             metric="l2", degree=64, nq=500, branches=32, queue=12, stop_eps=0.2, team=16),
        # offline evaluation or a join: thousands of queries at wide search knobs
        dict(name="search-bulk", kind="search", call="device", n=200_000, d=1536, dtype="f16",
             metric="ip", degree=64, nq=4096, branches=64, queue=44, stop_eps=0.3, team=16),
        # the same corpus through the sign-code pre-filter
        dict(name="search-coded", kind="coded", n=200_000, d=1536, dtype="f16", metric="ip",
             degree=64, nq=1000, branches=32, queue=24, stop_eps=0.3, team=16),
        # seeds of a batch against a large entry pool
        dict(name="select-pool", kind="select", nq=2000, P=131_072, d=1024, E=32, metric="ip"),
        # exact neighbours of a block of queries over a whole corpus (ground truth)
        dict(name="select-exact", kind="select", nq=1024, P=400_003, d=768, E=10, metric="l2"),
        # an fp16 corpus indexed with the sizes the benchmark uses
        dict(name="graph-f16", kind="graph", n=100_000, d=1536, dtype="f16", metric="ip",
             degree=64, candidates=128),
        # an fp32 l2 corpus indexed with Index.build's defaults
        dict(name="graph-f32", kind="graph", n=100_000, d=960, dtype="f32", metric="l2",
             degree=96, candidates=128),
        # a small corpus of word vectors whose width is not a multiple of eight
        dict(name="graph-ragged", kind="graph", n=20_011, d=100, dtype="f32", metric="ip",
             degree=48, candidates=64),
        # sign codes of a corpus before it is served with the pre-filter
        dict(name="codes", kind="codes", n=400_000, d=1536, dtype="f16"),
        # a graph rebuilt offline from another graph, with every extra on
        dict(name="offline", kind="offline", n=60_000, d=768, dtype="f32", metric="ip",
             degree=64, width=96, mutual=8, min_in=8, fill="bridge"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi, odd=0.25):
    """A width: mostly a multiple of eight, as padded corpora have, else any."""
    d = _log(rng, lo, hi)
    return d if rng.random() < odd else max(8, d // 8 * 8)


def draw(rng):
    kind = rng.choice(["search", "search", "search", "coded", "select", "select", "graph",
                       "graph", "codes", "offline"])
    if kind == "select":
        # at least a few hundred entries come back, so that one pair of equally
        # near rows is a small share of them (search-one and the captured search
        # hold the selection of one and of eight queries)
        c = dict(kind=kind, nq=_log(rng, 10, 4096), P=_log(rng, 512, 500_000),
                 d=_dim(rng, 32, 4096), E=_log(rng, 10, 128), metric=rng.choice(["ip", "l2"]))
        c["E"] = max(c["E"], 640 // c["nq"])
        while c["nq"] * c["P"] * c["d"] > 2000 * 131_072 * 1024 or c["P"] * c["d"] > 1 << 30:
            c["nq"], c["P"], c["d"] = (max(64, c["nq"] * 3 // 4) if c["nq"] > 64 else c["nq"],
                                       max(512, c["P"] * 3 // 4), max(32, c["d"] * 3 // 4))
        c["d"] = max(8, c["d"] // 8 * 8) if rng.random() < 0.75 else c["d"]
        return c
    dtype = rng.choice(["f32", "f16"])
    if kind == "codes":
        n, d = _log(rng, 1_000, 400_000), _dim(rng, 32, 1536)
        return dict(kind=kind, n=n, d=d, dtype="f16" if dtype == "f16" else "f32")
    metric = "ip" if kind == "coded" else rng.choice(["ip", "l2"])
    if kind == "graph":
        d = _dim(rng, 64, 1536)
        n = _log(rng, 5_000, 100_000 if d % 8 == 0 else 20_011)
        if d % 8:
            d = min(d, 201)
        return dict(kind=kind, n=n, d=d, dtype=dtype, metric=metric,
                    degree=rng.choice([32, 48, 64, 96]),
                    candidates=rng.choice([96, 100, 128]))
    if kind == "offline":
        return dict(kind=kind, n=_log(rng, 5_000, 60_000), d=_dim(rng, 64, 768), dtype=dtype,
                    metric=metric, degree=rng.choice([32, 48, 64]), width=96,
                    mutual=rng.choice([4, 8, 16]), min_in=rng.choice([4, 8]),
                    fill=rng.choice(["near", "far", "bridge"]))
    plain = kind == "search"
    d = _dim(rng, 96 if plain else 256, 1536)
    nq = _log(rng, 1, 4096) if plain else _log(rng, 100, 1000)
    return dict(kind=kind, n=_log(rng, 20_000, 150_000 if d % 8 == 0 else 30_000), d=d,
                dtype=dtype, metric=metric, degree=64, nq=nq, branches=rng.choice([32, 64]),
                queue=rng.choice([32, 44]), stop_eps=0.3, team=rng.choice([8, 16, 32]),
                **({"call": rng.choice(["host", "device"] + ["graph"] * (nq <= 64))}
                   if plain else {}))


# ---- inputs ---------------------------------------------------------------
def _rows(g, basis, m, metric, dtype):
    d = basis.shape[1]
    out = torch.empty((m, d), dtype=dtype, device=DEVICE)
    for a in range(0, m, 65536):
        b = min(m, a + 65536)
        x = torch.randn((b - a, LATENT), generator=g, device=DEVICE) @ basis
        x += NOISE * torch.randn((b - a, d), generator=g, device=DEVICE)
        if metric == "ip":
            x /= x.norm(dim=1, keepdim=True)
        out[a:b] = x
    return out


def _inputs(c, seed, m_rows, m_queries):
    """(rows, fp32 queries) of the case's width, type and metric, from the seed."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    basis = torch.randn((LATENT, c["d"]), generator=g, device=DEVICE) / LATENT ** 0.5
    X = _rows(g, basis, m_rows, c.get("metric", "ip"), DTYPES[c.get("dtype", "f32")])
    return X, _rows(g, basis, m_queries, c.get("metric", "ip"), torch.float32)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "select":
        V, Q = _inputs(c, seed, c["P"], c["nq"])
        return dict(case=c, Q=Q, V=V)
    if kind in ("graph", "codes"):
        return dict(case=c, X=_inputs(c, seed, c["n"], 1)[0])
    if kind == "offline":
        # the graph to start from: another builder's kNN lists
        X, _ = _inputs(c, seed, c["n"], 1)
        return dict(case=c, X=X, Gc=knn_candidates(X, c["width"], metric=c["metric"])[0])
    X, Q = _inputs(c, seed, c["n"], c["nq"])
    index = swann_amd.Index.build(X, metric=c["metric"], degree=c["degree"])
    knobs = dict(branches=c["branches"], queue=c["queue"], stop_eps=c["stop_eps"],
                 team=c["team"])
    state = dict(case=c, index=index, Q=Q, knobs=knobs)
    if kind == "coded":
        state["codes"] = (*build_codes(X), 0.2)      # load_codes' margin
    elif c["call"] == "host":
        state["Q"] = Q.cpu().numpy()
    elif c["call"] == "graph":
        state["captured"] = index.capture(c["nq"], k=10, **knobs)
    return state


# ---- one pass -------------------------------------------------------------
def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "select":
        return select_nearest(state["Q"], state["V"], c["E"],
                              metric=swann_amd.index.METRICS[c["metric"]])
    if kind == "graph":
        return build_graph(state["X"], metric=c["metric"], degree=c["degree"],
                           candidates=c["candidates"])
    if kind == "codes":
        return build_codes(state["X"])
    if kind == "offline":
        return _offline(state["X"], state["Gc"], c)
    if kind == "coded":
        return _coded(state["index"], state["Q"], state["codes"], c)
    if c["call"] == "host":
        return state["index"].search(state["Q"], k=10, **state["knobs"])
    if c["call"] == "graph":
        return state["captured"].run(state["Q"])
    ids, dist, _, overflow = state["index"].search_async(state["Q"], k=10, **state["knobs"])
    return ids, dist, overflow


def _coded(index, Q, codes, c):
    """Seeds from the index's catalogue, then the engine's search with codes."""
    ids = select_nearest(Q, index._cat, c["branches"])
    seeds = index.catalogue[ids].to(torch.int32)
    ids, dist, _ = _engine.search(index.X, index.G, Q, seeds, k=10, L=c["queue"], B=64,
                                  team_size=c["team"], stop_eps=c["stop_eps"],
                                  shared_cache=True, shared_bound=True, exclusive=True,
                                  elide_visited=True, codes=codes)
    return ids, dist


def _offline(X, Gc, c):
    cand, dist = offline.candidates_from_graph(X, Gc, c["width"], metric=c["metric"])
    protect = offline.mutual_rank(cand, c["mutual"])
    G = robust_prune(X, cand, dist, c["degree"], metric=c["metric"], protect=protect)
    G = add_reverse(X, G, c["degree"], metric=c["metric"])
    G = offline.enforce_min_in(X, G, cand, c["min_in"], metric=c["metric"], rounds=6)
    return dist, offline.fill_degree(G, cand, rule=c["fill"])


# ---- what a pass cannot do without -----------------------------------------
def work(case):
    c, kind, d = case, case["kind"], case["d"]
    size = 2 if c.get("dtype") == "f16" else 4
    if kind == "select":
        return dict(bytes=4 * (c["nq"] + c["P"]) * d + 8 * c["nq"] * c["E"],
                    flops=2 * c["nq"] * c["P"] * d)
    n = c["n"]
    if kind == "codes":
        return dict(bytes=n * (d * size + d / 8 + 4), flops=4 * n * d)
    if kind == "graph":
        # every pair once, then two Grams of at most 128 rows a node
        return dict(bytes=n * (d * size + 4 * c["degree"]),
                    flops=n * n * d + 2 * n * 128 * 128 * d)
    if kind == "offline":
        return dict(bytes=n * (d * size + 8 * c["width"] + 4 * c["degree"]),
                    flops=2 * n * c["width"] * d + n * (c["width"] ** 2 + 128 ** 2) * d)
    # rows a branch scores, about (the kernels' own counters over these ranges:
    # 300 to 700); the codes leave about one in three
    rows = c["nq"] * c["branches"] * (200 + 7 * c["queue"]) // (3 if kind == "coded" else 1)
    return dict(bytes=rows * d * size + c["nq"] * (4 * d + 80),
                flops=2 * rows * d + 2 * c["nq"] * min(4096, n) * d)


def tolerance(case):
    if case["kind"] == "select":
        return {"differ": 0.004}       # swapped neighbours a rounding apart
    if case["kind"] == "codes":
        return {"rel": 1e-6, "differ": 1e-5}
    if case["kind"] in ("graph", "offline"):
        # one near-tie that falls the other way shifts the rest of its row: the
        # prune's Gram in another order of sums changes up to 6e-5 of the edges
        return {"rel": 1e-6, "differ": 0.0005}
    # branches race for the shared claims: now and then another row ends a list
    return {"rel": 5e-3, "max": 0.5, "differ": 0.005}


# ---- the same in 64 bits ----------------------------------------------------
def exact(case, seed):
    c = case
    if c["kind"] == "codes":
        X = _inputs(c, seed, c["n"], 1)[0]
        mu = torch.zeros(c["d"], dtype=torch.float64, device=DEVICE)
        for x in X.split(65536):
            mu += x.double().sum(0)
        mu = (mu / c["n"]).float()
        alpha = torch.cat([(x.double() - mu.double()).abs().mean(1) for x in X.split(65536)])
        return None, alpha, mu.double()
    if c["kind"] == "offline":
        s = prepare(c, seed)
        X, Gc, out = s["X"], s["Gc"].long(), []
        for a in range(0, c["n"], 512):
            x, y = X[a:a + 512].double(), X[Gc[a:a + 512]].double()
            out.append(1 - (y * x[:, None]).sum(2) if c["metric"] == "ip" else
                       ((y - x[:, None]) ** 2).sum(2))
        return torch.cat(out).sort(1).values, None
    # rows chosen by a search, a selection or a prune are whole numbers, and an
    # approximate search's distances are those of the rows it chose
    return None
