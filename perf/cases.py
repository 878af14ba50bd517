"""Calls of this library as a program makes them, to be timed.

A case is one call (or, for the serving loop, one burst of requests) through the public Python
binding of libsvdb.so on a store that already holds its rows:

  kd       kdtree_nearest: one query, k = 1, Euclidean over the first `kd` coordinates — the
           reference server's own /nearest request
  compare  one cosine_similarity / euclidean_distance / dot_product call — a /compare request
  pairs    svdb_pair_metrics over `nq` pairs of stored rows — a batched /compare
  host     svdb_search with query rows, ids and scores in host memory — a /nearest request or a
           batch body, metric per query where `metric` is "mixed"
  device   svdb_search_device with queries, ids and scores resident in HBM — bulk jobs
  serve    a burst of `nq` requests through the serving loop: sizes log-uniform in 1..512, k in
           {1, 10, 100}, all metrics, one request in twenty an update of a row

torch is imported before the library is loaded, so both use one HIP runtime and torch tensors can
be handed to svdb_search_device.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "simple-vector-db_amd"))
import svdb  # noqa: E402

METRICS = ("l2", "cos", "dot")
ELEMENT_BYTES = {"fp64": 8, "auto": 2, "bf16": 2, "fp8": 1}  # of the rows a first pass has to read


def listed():
    return [
        # The reference server's default request: one point, k = 1, kd dimension 3, on the small
        # store of the benchmark's kd-tree leg (10,000 x 128 uniform rows): launch latency.
        dict(name="kd_one_10k", kind="kd", rows=10_000, dim=128, kd=3, data="uniform"),
        # One /compare/cosine request: two 128-wide rows, a float back.
        dict(name="compare_one", kind="compare", dim=128, metric="cos", data="uniform"),
        # A batched /compare: a million random pairs of stored rows.
        dict(name="pairs_1m", kind="pairs", rows=500_000, dim=128, nq=1_000_000, metric="cos",
             data="mixture"),
        # /nearest?number=10 with one query on a million-row store.
        dict(name="host_one_1m", kind="host", rows=1_000_000, dim=128, nq=1, k=10, metric="l2",
             precision="auto", data="mixture"),
        # A batch body: 64 queries, cosine.
        dict(name="host_64_cos", kind="host", rows=500_000, dim=128, nq=64, k=10, metric="cos",
             precision="auto", data="mixture"),
        # A ragged batch over rows of an odd width, all three metrics in one call, k = 100.
        dict(name="host_101_mixed_k100", kind="host", rows=200_003, dim=200, nq=101, k=100,
             metric="mixed", precision="auto", data="gauss"),
        # The bulk job of the benchmark: 16,384 resident queries, top-10 Euclidean, BF16 first pass.
        dict(name="device_16k_bf16", kind="device", rows=2_000_000, dim=128, nq=16_384, k=10,
             metric="l2", precision="auto", data="mixture"),
        # The plain FP64 scan in batches of 1,024 over N(0, 1) rows.
        dict(name="device_1k_fp64", kind="device", rows=500_000, dim=128, nq=1_024, k=10,
             metric="dot", precision="fp64", data="gauss"),
        # The plain FP64 scan at a ragged width (not a multiple of 32) and a small ragged batch.
        dict(name="device_77_fp64_d100", kind="device", rows=300_001, dim=100, nq=77, k=100,
             metric="l2", precision="fp64", data="gauss"),
        # Text embeddings, 768 wide, FP8 first pass, top-100 in batches of 4,096.
        dict(name="device_4k_fp8_768", kind="device", rows=150_000, dim=768, nq=4_096, k=100,
             metric="dot", precision="fp8", data="mixture1"),
        # 1,536-wide embeddings answered through the BF16 first pass, a small batch body.
        dict(name="host_32_bf16_1536", kind="host", rows=60_000, dim=1_536, nq=32, k=10,
             metric="cos", precision="bf16", data="mixture1"),
        # A burst on the serving loop.
        dict(name="serve_64", kind="serve", rows=1_000_000, dim=128, nq=64, data="gauss"),
    ]


def _log(rng, lo, hi):
    """A whole number whose logarithm is uniform over lo..hi."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("kd", "compare", "pairs", "host", "host", "host", "bulk", "bulk", "fp64",
                       "fp64", "fp8", "wide", "serve"))
    metric = rng.choice(METRICS)
    k = rng.choice((1, 10, 10, 100, _log(rng, 1, 128)))
    if kind == "kd":
        dim = _log(rng, 3, 256)
        return dict(kind="kd", rows=_log(rng, 200, 50_000), dim=dim,
                    kd=min(dim, rng.choice((3, 3, 8, dim))), data="uniform")
    if kind == "compare":
        return dict(kind="compare", dim=_log(rng, 3, 1_536), metric=metric, data="uniform")
    if kind == "pairs":
        return dict(kind="pairs", rows=_log(rng, 5_000, 500_000), dim=_log(rng, 16, 128),
                    nq=_log(rng, 1, 1_000_000), metric=metric, data="mixture")
    if kind == "host":
        dim = rng.choice((128, 128, _log(rng, 16, 256)))
        return dict(kind="host", rows=_log(rng, 5_000, 128_000_000 // max(dim, 128)), dim=dim,
                    nq=_log(rng, 1, 512), k=k, metric=rng.choice((metric, "mixed")),
                    precision="auto", data=rng.choice(("mixture", "gauss")))
    if kind == "bulk":
        dim = rng.choice((128, 128, _log(rng, 24, 256)))
        return dict(kind="device", rows=_log(rng, 50_000, 256_000_000 // max(dim, 128)), dim=dim,
                    nq=_log(rng, 512, 16_384 * 128 // max(dim, 128)), k=k, metric=metric,
                    precision="auto", data="mixture")
    if kind == "fp64":
        dim = rng.choice((128, 96, 256, _log(rng, 16, 256)))
        return dict(kind="device", rows=_log(rng, 5_000, 64_000_000 // max(dim, 128)), dim=dim,
                    nq=_log(rng, 1, 1_024), k=k, metric=metric, precision="fp64", data="gauss")
    if kind == "fp8":
        dim = rng.choice((768, 1_536, _log(rng, 260, 1_536)))
        return dict(kind="device", rows=_log(rng, 20_000, 110_000_000 // max(dim, 768)), dim=dim,
                    nq=_log(rng, 64, 4_096), k=rng.choice((10, 100)), metric=metric,
                    precision="fp8", data="mixture1")
    if kind == "wide":
        dim = rng.choice((768, 1_536, _log(rng, 260, 1_536)))
        return dict(kind="host", rows=_log(rng, 10_000, 92_000_000 // max(dim, 768)), dim=dim,
                    nq=_log(rng, 1, 256), k=k, metric=metric, precision="bf16", data="mixture1")
    return dict(kind="serve", rows=_log(rng, 100_000, 1_000_000), dim=128, nq=_log(rng, 8, 64),
                data=rng.choice(("mixture", "gauss")))


# ---- inputs -------------------------------------------------------------------------------------


def _generator(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 8 + part)
    return g


def _points(kind, n, dim, seed, part):
    """n x dim doubles on the GPU: uniform on [-1, 1], N(0, 1), or a mixture of 1,024 clusters
    (sigma 0.05 about centres on the unit sphere, norms LogNormal(0, 0.5), or (0, 1) for
    "mixture1")."""
    g = _generator(seed, part)
    new = dict(generator=g, device="cuda", dtype=torch.float64)
    if kind == "uniform":
        return torch.rand(n, dim, **new) * 2 - 1
    if kind == "gauss":
        return torch.randn(n, dim, **new)
    centres = torch.randn(1024, dim, generator=_generator(seed, 7), device="cuda",
                          dtype=torch.float64)
    centres /= centres.norm(dim=1, keepdim=True)
    x = torch.randn(n, dim, **new).mul_(0.05)
    x += centres[torch.randint(0, 1024, (n,), generator=g, device="cuda")]
    s = 1.0 if kind == "mixture1" else 0.5
    x *= torch.exp(s * torch.randn(n, 1, **new)) / x.norm(dim=1, keepdim=True)
    return x


def _metrics(case):
    if case["metric"] != "mixed":
        return case["metric"]
    return [METRICS[i % 3] for i in range(case["nq"])]


def _plan(case, seed):
    """The requests of one burst: ("search", first pool row, queries, k, metric) or ("update", row,
    pool row).  Sizes, k and metrics go with the number of requests, which rows are meant with the
    seed.  The rows an update changes are set back at the end of the burst."""
    shape, rng = random.Random(case["nq"]), random.Random(seed)
    plan = []
    for i in range(case["nq"]):
        if i % 20 == 10:
            plan.append(("update", rng.randrange(case["rows"]), rng.randrange(4096)))
        else:
            n = _log(shape, 1, 512)
            plan.append(("search", rng.randrange(4096 - n + 1), n, shape.choice((1, 10, 100)),
                         shape.choice(METRICS)))
    return plan


def _inputs(case, seed):
    """The rows and the queries (on the GPU)."""
    kind = case["kind"]
    if kind == "compare":
        return None, _points(case["data"], 2, case["dim"], seed, 1)
    rows = _points(case["data"], case["rows"], case["dim"], seed, 0)
    if kind == "pairs":
        return rows, torch.randint(0, case["rows"], (2, case["nq"]),
                                   generator=_generator(seed, 1), device="cuda")
    n = {"kd": 1, "serve": 4096}.get(kind) or case["nq"]
    return rows, _points(case["data"], n, case["kd"] if kind == "kd" else case["dim"], seed, 1)


def prepare(case, seed):
    kind = case["kind"]
    rows, queries = _inputs(case, seed)
    if kind == "compare":
        a, b = queries.cpu().numpy()
        return dict(case=case, a=a, b=b)
    host = rows.cpu().numpy()
    del rows
    db = svdb.Database(kd_dimension=case.get("kd", 3))
    db.bulk_insert(host)
    state = dict(case=case, db=db)
    if kind == "kd":
        state["q"] = queries[0].cpu().numpy()
    elif kind == "pairs":
        state["ab"] = queries.cpu().numpy().astype(np.uint64)
    elif kind == "host":
        state["q"] = queries.cpu().numpy()
        state["metrics"] = _metrics(case)
    elif kind == "device":
        if case["precision"] == "fp8":
            db.enable_shadow("fp8")
            db.set_shortlist(128)
        state["q"] = queries
        state["ids"] = torch.empty(case["nq"], case["k"], dtype=torch.int64, device="cuda")
        state["scores"] = torch.empty(case["nq"], case["k"], dtype=torch.float64, device="cuda")
    else:
        state["pool"] = queries.cpu().numpy()
        state["plan"] = _plan(case, seed)
        state["old"] = {p[1]: host[p[1]].copy() for p in state["plan"] if p[0] == "update"}
        state["server"] = svdb.Server(db)
    del queries, host
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return state


# ---- a pass -------------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "kd":
        return state["db"].kd_nearest(state["q"])
    if kind == "compare":
        return svdb.legacy_metric(state["a"], state["b"], case["metric"])
    if kind == "pairs":
        return state["db"].pair_metrics(state["ab"][0], state["ab"][1], case["metric"])
    if kind == "host":
        ids, scores = state["db"].search(state["q"], case["k"], state["metrics"],
                                         case["precision"])
        return ids.view(np.int64), scores
    if kind == "device":
        q = state["q"]
        state["db"].search_device(q.data_ptr(), case["nq"], case["dim"], case["k"],
                                  case["metric"], case["precision"], state["ids"].data_ptr(),
                                  state["scores"].data_ptr())
        return state["ids"], state["scores"]
    server, pool = state["server"], state["pool"]
    tickets = []
    for p in state["plan"]:
        if p[0] == "search":
            tickets.append(server.submit_search(pool[p[1]:p[1] + p[2]], p[3], p[4]))
        else:
            tickets.append(server.submit_update(p[1], pool[p[2]]))
    back = [server.submit_update(row, old) for row, old in state["old"].items()]
    ids, scores = [], []
    for p, t in zip(state["plan"], tickets):
        rc, i, s, _ = server.wait(t)
        if rc != 0:
            raise RuntimeError("request failed: %d" % rc)
        if p[0] == "search":
            ids.append(i.view(np.int64).ravel())
            scores.append(s.ravel())
    for t in back:
        server.wait(t)
    return np.concatenate(ids), np.concatenate(scores)


def work(case):
    kind, dim = case["kind"], case["dim"]
    if kind == "kd":
        return dict(bytes=8 * case["kd"] * (case["rows"] + 1) + 8, flops=3 * case["rows"] * case["kd"])
    if kind == "compare":
        return dict(bytes=16 * dim + 4, flops=6 * dim)
    if kind == "pairs":
        return dict(bytes=case["nq"] * (16 * dim + 24), flops=6 * dim * case["nq"])
    if kind == "serve":
        searches = [p for p in _plan(case, 0) if p[0] == "search"]
        nq, out = sum(p[2] for p in searches), sum(p[2] * p[3] for p in searches)
        each = ELEMENT_BYTES["auto"]
    else:
        nq, out, each = case["nq"], case["nq"] * case["k"], ELEMENT_BYTES[case["precision"]]
    return dict(bytes=case["rows"] * dim * each + nq * dim * 8 + 16 * out,
                flops=2 * case["rows"] * dim * nq)


# ---- the same in plain torch, 64 bits ----------------------------------------------------------


def _best_scores(X, Q, k, metric):
    """The k best scores of each query.  Euclidean: the nearest by |x|^2 - 2 q.x, with 32 to
    spare, then sqrt(sum (x - q)^2) of those."""
    k = min(k, X.shape[0])
    if metric == "cos":
        xn = X.norm(dim=1)
    elif metric == "l2":
        x2 = X.square().sum(1)
    got = []
    step = max(1, 100_000_000 // X.shape[0])
    for i in range(0, Q.shape[0], step):
        q = Q[i:i + step]
        s = q @ X.T
        if metric == "cos":
            s /= xn
            s /= q.norm(dim=1, keepdim=True)
        elif metric == "l2":
            s.mul_(-2).add_(x2)
            near = s.topk(min(k + 32, X.shape[0]), dim=1, largest=False).indices
            part = [(X[near[j:j + 64]] - q[j:j + 64, None]).square().sum(2).sqrt()
                    for j in range(0, q.shape[0], 64)]
            got.append(torch.cat(part).sort(dim=1).values[:, :k])
            continue
        got.append(s.topk(k, dim=1).values)
    return torch.cat(got)


def _pair_values(a, b, metric):
    if metric == "l2":
        return (a - b).square().sum(-1).sqrt()
    dot = (a * b).sum(-1)
    return dot if metric == "dot" else dot / (a.norm(dim=-1) * b.norm(dim=-1))


def exact(case, seed):
    """What run() returns, ids left out."""
    kind = case["kind"]
    if kind == "kd":
        return None
    X, Q = _inputs(case, seed)
    if kind == "compare":
        return float(_pair_values(Q[0], Q[1], case["metric"]))
    if kind == "pairs":
        return torch.cat([_pair_values(X[ab[0]], X[ab[1]], case["metric"])
                          for ab in Q.split(100_000, dim=1)])
    if kind == "serve":
        got = []
        for p in _plan(case, seed):
            if p[0] == "update":
                X[p[1]] = Q[p[2]]
            else:
                got.append(_best_scores(X, Q[p[1]:p[1] + p[2]], p[3], p[4]).ravel())
        return None, torch.cat(got)
    metrics = _metrics(case)
    if not isinstance(metrics, str):
        out = torch.empty(case["nq"], case["k"], dtype=torch.float64, device="cuda")
        for m in METRICS:
            at = [i for i, v in enumerate(metrics) if v == m]
            if at:
                out[at] = _best_scores(X, Q[at], case["k"], m)
        return None, out
    return None, _best_scores(X, Q, case["k"], metrics)
