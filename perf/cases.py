"""The calls whose speed this repository is measured by, made as a user's
program makes them: the public entry points of gem_amd on seeded graphs of the
shapes of gem_amd.workloads, from one small query to a batch on the 2^22
vertex R-MAT graph.

A case names a path ("path"), a graph and the queries.  Graphs:
  er    Erdos-Renyi: `vertices`, `edges`, `labels` uniform labels
  rmat  R-MAT: 2^`scale` vertices of average degree `degree`, `labels` labels,
        Zipf distributed when `zipf`, else uniform
Queries are random-walk subgraphs of `size` vertices (`size_min` to `size_max`
in a batch, spread evenly), of average degree >= 3 when `dense`.

Paths:
  match     one query through the plain pipeline (filter, tables, GEM order,
            edge-at-a-time join): what the reference runs per query
  prepare   filter and edge tables of one query
  embed     the plain pipeline returning the embeddings themselves, at most `capacity`
  batch     match_batch: many queries, GEM's orders, exact counts per level
  learned   match_batch_learned with a shipped order model, restarts and the
            committed tuning: the benchmark's path
  relaxed   every relaxed query of one query at a threshold
  stream    match_batch with the graph in host memory and streamed tables
  rank      the order model's scores of one query's candidate orders
  gradient  loss and gradient of the order model over a training set
"""
import math
import os

import numpy as np
import torch

from gem_amd import GEM_MAX_QE, GEM_MAX_QV, GemContext, Graph, Query
from gem_amd.autotune import apply, load_tuning
from gem_amd.learned import OrderModel, match_batch_learned
from gem_amd.workloads import CAP

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FEATURES, HIDDEN = 272, 128  # the order model: 272 -> 128 -> 128 -> 1


def listed():
    return [
        # The smallest call: one 5-vertex query on the 10,000-vertex
        # Erdos-Renyi graph, the interactive use; latency and launches.
        dict(name="match_er10k", path="match", graph="er", vertices=10000, edges=50000, labels=8, size=5, dense=False),
        # One 8-vertex dense query on a power-law graph by the plain pipeline:
        # large intermediate levels, expand and select steps.
        dict(name="match_rmat18", path="match", graph="rmat", scale=18, degree=16.0, labels=64, zipf=False, size=8,
             dense=True),
        # What every query on a large graph pays before its join: candidates
        # and edge tables of a 16-vertex query on the benchmark's graph.
        dict(name="prepare_rmat22", path="prepare", graph="rmat", scale=22, degree=16.0, labels=32, zipf=True,
             size=16, dense=False),
        # The embeddings themselves (enumeration): about a million rows.
        dict(name="embed_er20k", path="embed", graph="er", vertices=20011, edges=119999, labels=3, size=5,
             dense=False, capacity=4 << 20),
        # The 20 queries of the small workload as one batch, exact.
        dict(name="batch_er10k", path="batch", graph="er", vertices=10000, edges=50000, labels=8, queries=20,
             size_min=5, size_max=5),
        # Exact counting of many mid-size queries on a power-law graph.
        dict(name="batch_rmat18", path="batch", graph="rmat", scale=18, degree=16.0, labels=64, zipf=False,
             queries=24, size_min=4, size_max=9),
        # The learned-order workload's graph shape, its query sizes.
        dict(name="learned_rmat20", path="learned", graph="rmat", scale=20, degree=16.0, labels=16, zipf=True,
             model="rmat20", queries=16, size_min=3, size_max=24),
        # The benchmark's graph, sizes and model, a part of its 512 queries.
        dict(name="learned_rmat22", path="learned", graph="rmat", scale=22, degree=16.0, labels=32, zipf=True,
             model="rmat22", queries=12, size_min=3, size_max=32),
        # The reference's -t 1: a query with every spanning edge set that
        # leaves out one edge.
        dict(name="relaxed_rmat17", path="relaxed", graph="rmat", scale=17, degree=16.0, labels=64, zipf=False,
             size=7, dense=True, threshold=1),
        # Out of core: graph in host memory, edge tables streamed through a
        # small device cache, sparse queries of up to 12 vertices, degree 64.
        dict(name="stream_rmat18", path="stream", graph="rmat", scale=18, degree=64.0, labels=64, zipf=True,
             queries=5, size_min=3, size_max=12, cache_mb=128),
        # The order model scoring one query's 8 candidates.
        dict(name="rank_8", path="rank", tuples=8),
        # One training step's loss and gradient over the larger shipped
        # model's 20,480 tuples.
        dict(name="gradient_20480", path="gradient", tuples=20480),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["match", "prepare", "embed", "batch", "batch", "learned", "relaxed", "stream", "rank",
                       "gradient"])
    if path in ("rank", "gradient"):
        return dict(path=path, tuples=_log_int(rng, 1, 64) if path == "rank" else _log_int(rng, 256, 20480))
    if path == "embed":
        n = _log_int(rng, 2000, 20000)
        return dict(path=path, graph="er", vertices=n, edges=int(n * rng.uniform(4, 6)), labels=rng.randint(3, 6),
                    size=rng.randint(3, 5), dense=False, capacity=4 << 20)
    if path in ("match", "batch") and rng.random() < 0.4:
        n = _log_int(rng, 1000, 20000)
        g = dict(graph="er", vertices=n, edges=int(n * rng.uniform(4, 6)), labels=rng.randint(6, 12))
    elif path == "learned":
        g = dict(graph="rmat", scale=rng.randint(16, 20), degree=16.0, labels=rng.randint(16, 32), zipf=True)
    elif path == "stream":
        g = dict(graph="rmat", scale=rng.randint(15, 17), degree=round(rng.uniform(32, 64), 2), labels=64, zipf=True)
    else:
        top = {"match": 18, "prepare": 21, "batch": 18, "relaxed": 17}[path]
        g = dict(graph="rmat", scale=rng.randint(13, top), degree=round(rng.uniform(8, 16), 2),
                 labels=rng.randint(64, 100), zipf=False)
    c = dict(path=path, **g)
    if path == "match":
        c.update(size=rng.randint(3, 8), dense=rng.random() < 0.5 and g["graph"] == "rmat")
    elif path == "prepare":
        c.update(size=rng.randint(4, 32), dense=False)
    elif path == "batch":
        lo = rng.randint(3, 5)
        c.update(queries=rng.randint(1, 24), size_min=lo, size_max=rng.randint(lo, 8 if g["graph"] == "rmat" else 6))
    elif path == "learned":
        c.update(model="rmat20" if c["scale"] <= 20 else "rmat22", queries=rng.randint(4, 12), size_min=3,
                 size_max=rng.randint(8, 24))
    elif path == "relaxed":
        c.update(size=rng.randint(5, 7), dense=True, threshold=1)
    elif path == "stream":
        c.update(queries=rng.randint(1, 5), size_min=3, size_max=rng.randint(6, 12), cache_mb=128)
    return c


# ------------------------------------------------------------------ inputs
def _graph(case, seed):
    if case["graph"] == "er":
        return Graph.erdos_renyi(case["vertices"], case["edges"], case["labels"], seed)
    return Graph.rmat(case["scale"], case["degree"], case["labels"], seed, zipf=case["zipf"])


def _queries(case, g, seed):
    """The case's queries: (size, dense) each, the first random walks that fit."""
    n = case.get("queries", 1)
    lo, hi = case.get("size_min", case.get("size")), case.get("size_max", case.get("size"))
    sizes = [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)]
    out, walk = [], 0
    for k in sizes:
        while True:
            q = Query.random_walk(g, k, seed * 100000 + walk)
            walk += 1
            if q.num_e >= 2 and (not case.get("dense") or q.dense) and (case["path"] != "stream" or not q.dense):
                out.append(q)
                break
            if walk > 50000:
                raise RuntimeError("no random walk gives such a query")
    return out


def _tuples(case, seed):
    """Features as the planner quantises them (16 log2(1 + x) for counts and
    estimates, 16 x for small numbers, zero past the query's last level) and
    labels as the trainer standardises them."""
    rng = np.random.default_rng(seed)
    n, levels, per = case["tuples"], 32, 8
    f = np.zeros((n, FEATURES), np.int32)
    size = rng.integers(4, levels + 1, n)
    lv = np.zeros((n, levels, per), np.float64)
    lv[:, :, 0] = 16 * rng.uniform(4, 18, (n, levels))
    lv[:, :, 1] = 16 * rng.integers(1, 4, (n, levels))
    lv[:, :, 2] = 16 * rng.integers(0, 4, (n, levels))
    lv[:, :, 3] = 16 * rng.uniform(0, 8, (n, levels))
    lv[:, :, 4] = lv[:, :, 3] + 16 * rng.uniform(0, 3, (n, levels))
    lv[:, :, 5] = 16 * rng.uniform(0, 40, (n, levels))
    lv[:, :, 6] = 16 * rng.integers(1, 8, (n, levels))
    lv[:, :, 7] = 16 * rng.uniform(14, 20, (n, levels))
    lv[np.arange(levels)[None, :] >= size[:, None]] = 0
    f[:, :levels * per] = np.rint(lv).reshape(n, levels * per)
    f[:, levels * per:levels * per + 11] = np.rint(16 * rng.uniform(1, 24, (n, 11)))
    y = rng.standard_normal(n).astype(np.float32)
    return f, y


def _weights(seed):
    """He-uniform weights and small biases, flat: W1 b1 W2 b2 W3 b3."""
    rng = np.random.default_rng(seed + 7919)
    part = []
    for fan_in, fan_out in ((FEATURES, HIDDEN), (HIDDEN, HIDDEN), (HIDDEN, 1)):
        lim = math.sqrt(6.0 / fan_in)
        part += [rng.uniform(-lim, lim, fan_in * fan_out), rng.uniform(-0.05, 0.05, fan_out)]
    return np.concatenate(part).astype(np.float32)


def prepare(case, seed):
    path = case["path"]
    ctx = GemContext(0)
    s = dict(path=path, ctx=ctx)
    if path in ("rank", "gradient"):
        s["feats"], s["labels"] = _tuples(case, seed)
        s["model"] = OrderModel(ctx, seed=seed)
        s["model"].set_params(_weights(seed))
        return s
    g = _graph(case, seed)
    if path == "stream":
        ctx.set_graph_residency(True)
        ctx.set_table_stream(case["cache_mb"] << 20, 1 << 20)
    ctx.load_data(g)
    qs = _queries(case, g, seed)
    s.update(graph=g, queries=qs, query=qs[0])
    if path == "match":
        ctx.set_work_limit(10 ** 9)
    elif path == "embed":
        s.update(order=ctx.match_full(qs[0])["order"], capacity=case["capacity"])
    elif path == "learned":
        cfg = load_tuning(os.path.join(ROOT, "gem_amd", "tuning", "rmat22.json"))
        apply(ctx, cfg)
        s["orders"] = int(cfg.get("max_orders", 8))
        s["model"] = OrderModel.load(ctx, os.path.join(ROOT, "gem_amd", "models", f"order_mlp_{case['model']}.npz"))
    elif path == "relaxed":
        s["threshold"] = case["threshold"]
    return s


# -------------------------------------------------------------------- pass
def _result(r):
    return [r["count"], int(r["saturated"]), int(r["work_limited"])]


def _fixed(rows, n):
    """Rows in an array of n rows (the queries of two seeds differ in their
    edges, their results' shapes do not)."""
    a = np.asarray(rows).astype(np.int64)
    out = np.full((n,) + a.shape[1:], -1, np.int64)
    out[:len(a)] = a
    return out


def run(s):
    path, ctx = s["path"], s["ctx"]
    if path == "rank":
        return s["model"].predict(s["feats"])
    if path == "gradient":
        loss, grad = s["model"].loss_grad(s["feats"], s["labels"])
        return dict(loss=np.float32(loss), grad=grad)
    if path == "match":
        r = ctx.match_full(s["query"], cap=CAP)
        return dict(result=np.array(_result(r) + [r["rows_processed"]]), order=_fixed(r["order"], GEM_MAX_QE))
    if path == "prepare":
        ncan, _ = ctx.filter(s["query"], want_lists=False)
        sizes = ctx.build_edge_tables()
        return dict(candidates=_fixed(ncan, GEM_MAX_QV), tables=_fixed(sizes, 2 * GEM_MAX_QE))
    if path == "embed":
        ctx.filter(s["query"], want_lists=False)
        ctx.build_edge_tables()
        r = ctx.join(s["order"], embeddings_capacity=s["capacity"])
        # the whole array of `capacity` rows that the embeddings are the head of
        return dict(count=r["count"], rows=r["embeddings"].base.view(np.int32))
    if path in ("batch", "stream"):
        res = ctx.match_batch(s["queries"], cap=CAP if path == "stream" else 0)
        out = dict(results=np.array([_result(r) for r in res]))
        if path == "batch":
            out["levels"] = np.concatenate([r["level_rows"] for r in res]).astype(np.int64)
        return out
    if path == "learned":
        res = match_batch_learned(ctx, s["queries"], s["model"], max_orders=s["orders"], cap=CAP,
                                  work_limit=10 ** 12, first_attempt=10 ** 8)
        return np.array([_result(r) for r in res])
    res = ctx.match_relaxed(s["query"], s["threshold"], cap=CAP)
    return _fixed([_result(r) for r in res], GEM_MAX_QE + 1)


# ------------------------------------------------------------ what it costs
def work(case):
    path = case["path"]
    if path in ("rank", "gradient"):
        n, p = case["tuples"], FEATURES * HIDDEN + HIDDEN * HIDDEN + HIDDEN
        if path == "rank":
            return dict(bytes=4 * n * FEATURES + 2 * p + 4 * n, flops=2 * n * p)
        # forward, the weight gradients, and the two inner layers' input gradients
        return dict(bytes=4 * n * FEATURES + 4 * n + 2 * p + 4 * p,
                    flops=2 * n * (2 * p + HIDDEN * HIDDEN + HIDDEN))
    # the graph once (offsets, labels, the adjacency of both directions) and a
    # bitmap word and a position per 64 vertices and query vertex
    if case["graph"] == "er":
        n, slots = case["vertices"], 2 * case["edges"]
    else:
        n = 2 ** case["scale"]
        slots = n * case["degree"] * 0.97
    nq = case.get("queries", 1)
    k = (case.get("size_min", case.get("size")) + case.get("size_max", case.get("size"))) / 2
    return dict(bytes=9 * n + 4 * slots + nq * k * (n / 64) * 12, flops=0)


def exact(case, seed):
    """The order model in 64 bits on the weights as it holds them (bf16
    matrices, float biases).  Counts are whole numbers: none."""
    if case["path"] not in ("rank", "gradient"):
        return None
    f, y = _tuples(case, seed)
    flat = torch.from_numpy(_weights(seed))
    W, at = [], 0
    for fan_in, fan_out in ((FEATURES, HIDDEN), (HIDDEN, HIDDEN), (HIDDEN, 1)):
        w = flat[at:at + fan_in * fan_out].view(fan_in, fan_out).to(torch.bfloat16).double()
        at += fan_in * fan_out
        b = flat[at:at + fan_out].double()
        at += fan_out
        W += [w.requires_grad_(), b.requires_grad_()]
    x = torch.from_numpy(f).double() / 64.0
    h = torch.relu(x @ W[0] + W[1])
    h = torch.relu(h @ W[2] + W[3])
    out = (h @ W[4] + W[5]).reshape(-1)
    if case["path"] == "rank":
        return out.detach().numpy()
    loss = 0.5 * (out - torch.from_numpy(y).double()).square().mean()
    loss.backward()
    return dict(loss=loss.detach().numpy(), grad=torch.cat([w.grad.reshape(-1) for w in W]).numpy())
