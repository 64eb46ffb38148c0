"""What a program that uses this matcher has it do, as cases to be timed.

Every case goes through the public entry points (gpsm_amd.matcher.Context and
ResidentGraph, gpsm_amd.planner, and the C ABI where it has no Python
wrapper).  The paths, with what each stands for:

match    one query against a resident data graph: the reference's own call
         (one Match::match per query), counting or with the sorted tuple list.
batch    many queries in one call, with the heuristic or the learned join
         order, with plain launches or through the cached graphs.
filter   the candidate sets alone (queries whose embeddings are too many to
         enumerate still have them).
tables   the candidate-edge tables in the reference's layout.
build    a data graph put on the device from an edge list, CSR read back.
scan     the allocation-free exclusive scan on device buffers.
output   the end of the reference's pipeline: the directed, edge-labelled
         check of a tuple list and its text lines.
planner  the join-order network: forward, or loss and gradients.

Queries are random walks, cycles and cliques taken from the data graph; those
of a matching case are kept by the framework's own feasibility rule (the exact
join finishes within a budget of examined candidates).  Where the size of the
result follows from the query, the query is the case's own and the seed
renumbers the data graph's vertices (and the query's, where that leaves the
sizes alone): other inputs, results of the same shape, and hubs at any id.
"""
import ctypes as C
import math
from collections import OrderedDict

import numpy as np
import torch

from gpsm_amd import _lib
from gpsm_amd import graphs as G
from gpsm_amd import planner
from gpsm_amd import workloads
from gpsm_amd.matcher import Context

KINDS = {"tree": _lib.Q_WALK_TREE, "induced": _lib.Q_WALK_INDUCED, "half": _lib.Q_WALK_HALF,
         "cycle": _lib.Q_CYCLE, "clique": _lib.Q_CLIQUE}
ORDERS = {"heuristic": _lib.ORDER_HEURISTIC, "learned": _lib.ORDER_LEARNED}
F, H = _lib.FEAT, _lib.HIDDEN


def listed():
    return [
        # the smallest call: one 6-vertex walk query on a 10k-vertex graph, its
        # embeddings returned (about a thousand rows); latency of the pipeline
        _match("match_er10k_tuples", "er", 10_000, 40_000, 8, 0.0, 6, 6, "tree", budget=10_000, tuples=True,
               graph_seed=1),
        # a single query counted on the 1M-vertex power-law graph that a
        # service keeps resident: the ordinary request
        _match("match_cl1m_count", "chung_lu", 1_000_000, 8_000_000, 16, 1.0, 4, 6, "half", budget=1_000_000_000,
               graph_seed=2),
        # a query with many embeddings, all of them wanted, sorted
        _match("match_cl100k_tuples", "chung_lu", 100_000, 800_000, 16, 1.0, 4, 5, "tree", budget=3_000_000,
               tuples=True, graph_seed=77),
        # many small queries on a small graph: a launch-bound batch
        _batch("batch_cl3k", "chung_lu", 3_000, 12_000, 3, 0.0, 24, 3, 7, "half", budget=10_000_000),
        # the benchmark's mix of walk queries with the learned order
        {"name": "batch_cl1m_mix", "path": "mix", "queries": 245, "order": "learned"},
        # cycles and cliques on an R-MAT graph: every vertex has back edges
        _batch("batch_rmat18_shapes", "rmat", 1 << 18, 4_194_304, 32, 0.8, 32, 4, 6, "shapes", budget=500_000_000,
               graph_seed=5),
        # candidate sets of a query far too large to enumerate
        {"name": "filter_cl1m", "path": "filter", "graph": "chung_lu", "n": 1_000_000, "edges": 8_000_000,
         "labels": 16, "zipf": 1.0, "graph_seed": 2, "kmin": 14, "kmax": 14, "kind": "half"},
        # candidate-edge tables of an 8-vertex query, copied out
        {"name": "tables_cl100k", "path": "tables", "graph": "chung_lu", "n": 100_000, "edges": 800_000,
         "labels": 16, "zipf": 1.0, "graph_seed": 77, "kmin": 6, "kmax": 8, "kind": "half"},
        # a new data graph of the benchmark's size, from its edge list
        {"name": "build_cl1m", "path": "build", "graph": "chung_lu", "n": 1_000_000, "edges": 8_000_000,
         "labels": 16, "zipf": 1.0, "graph_seed": 2},
        # the largest arrays the allocation-free scan is meant for, odd length
        {"name": "scan_100m", "path": "scan", "values": 100_000_007},
        # half a million 5-vertex tuples checked and written as text
        {"name": "output_500k", "path": "output", "n": 50_000, "edges": 400_000, "rows": 500_000, "q": 5},
        # the planner's training mini-batch
        {"name": "planner_grad_256", "path": "planner", "samples": 256, "pass": "grad"},
    ]


def _match(name, graph, n, edges, labels, zipf, kmin, kmax, kind, budget, tuples=False, order="heuristic",
           graph_seed=0):
    return {"name": name, "path": "match", "graph": graph, "n": n, "edges": edges, "labels": labels, "zipf": zipf,
            "graph_seed": graph_seed, "kmin": kmin, "kmax": kmax, "kind": kind, "budget": budget, "tuples": tuples,
            "order": order}


def _batch(name, graph, n, edges, labels, zipf, queries, kmin, kmax, kind, budget, order="heuristic",
           use_graph=False, graph_seed=0):
    return {"name": name, "path": "batch", "graph": graph, "n": n, "edges": edges, "labels": labels, "zipf": zipf,
            "graph_seed": graph_seed, "queries": queries, "kmin": kmin, "kmax": kmax, "kind": kind,
            "budget": budget, "order": order, "use_graph": use_graph}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, lo, hi):
    kind = rng.choice(["er", "chung_lu", "chung_lu", "rmat"])
    n = _log(rng, lo, hi)
    if kind == "rmat":
        n = 1 << max(10, n.bit_length() - 1)
    return {"graph": kind, "n": n, "edges": int(n * rng.uniform(3, 12)), "labels": rng.randint(3, 32),
            "zipf": rng.choice([0.0, 0.8, 1.0]), "graph_seed": rng.randint(3, 1 << 20)}


def draw(rng):
    path = rng.choice(["match", "match", "batch", "batch", "batch", "filter", "tables", "build", "scan", "output",
                       "planner"])
    if path == "scan":
        return {"path": path, "values": _log(rng, 1000, 100_000_000)}
    if path == "planner":
        return {"path": path, "samples": _log(rng, 32, 65536), "pass": rng.choice(["forward", "grad"])}
    if path == "output":
        n = _log(rng, 2_000, 50_000)
        return {"path": path, "n": n, "edges": 8 * n, "rows": _log(rng, 1_000, 1_000_000), "q": rng.randint(2, 8)}
    if path == "build":
        c = _draw_graph(rng, 2_000, 600_000)
        return dict(c, path=path)
    if path == "filter":
        k = rng.randint(3, 32)
        return dict(_draw_graph(rng, 5_000, 600_000), path=path, kmin=k, kmax=k,
                    kind=rng.choice(["tree", "induced", "half"]))
    if path == "tables":
        kmin = rng.randint(3, 8)
        return dict(_draw_graph(rng, 2_000, 200_000), path=path, kmin=kmin, kmax=kmin + rng.randint(0, 3),
                    kind=rng.choice(["tree", "induced", "half"]))
    c = _draw_graph(rng, 2_000, 300_000)
    c.update(path=path, kmin=rng.randint(3, 4), kmax=rng.randint(4, 8),
             kind=rng.choice(["tree", "half", "induced", "shapes"]), order=rng.choice(["heuristic", "learned"]))
    if path == "match":
        c["tuples"] = rng.random() < 0.5
        c["budget"] = _log(rng, 10_000, 1_000_000 if c["tuples"] else 300_000_000)
    else:
        c["queries"] = _log(rng, 2, 128)
        c["budget"] = _log(rng, 100_000, 100_000_000)
        c["use_graph"] = rng.random() < 0.3
    return c


# --- what a program keeps: one context, its resident graphs, its planner -------

_CTX = None
_GRAPHS = OrderedDict()    # host CSRs
_RESIDENT = OrderedDict()  # data graphs on the device
_QUERIES = OrderedDict()   # cases' own queries


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = Context(0)
        planner.install(_CTX)
    return _CTX


def _kept(cache, key, make, most):
    if key in cache:
        cache.move_to_end(key)
    else:
        cache[key] = make()
        while len(cache) > most:
            cache.popitem(last=False)
    return cache[key]


def _spec(case, seed):
    gs = case.get("graph_seed", 0) or seed
    return (case["graph"], case["n"], case["edges"], case["labels"], case["zipf"], gs)


def _generate(spec):
    kind, n, m, labels, zipf, seed = spec
    if kind == "er":
        g = G.erdos_renyi(n, m, seed)
    elif kind == "rmat":
        g = G.rmat(n.bit_length() - 1, m, 0.57, 0.19, 0.19, seed)
    else:
        g = G.chung_lu(n, m, 2.1, seed)
    return G.set_labels(g, labels, zipf, seed)


def _graph(case, seed):
    spec = _spec(case, seed)
    return _kept(_GRAPHS, spec, lambda: _generate(spec), 4)


def _resident(case, seed):
    g = _graph(case, seed)
    return _kept(_RESIDENT, _spec(case, seed), lambda: _ctx().upload(g), 4)


def _draws(g, count, case, seed):
    kinds = ["cycle", "clique"] if case["kind"] == "shapes" else [case["kind"]]
    out = []
    for i, kind in enumerate(kinds):
        share = (count + len(kinds) - 1 - i) // len(kinds)
        kmax = min(case["kmax"], 6) if case["kind"] == "shapes" else case["kmax"]
        kmin = min(max(case["kmin"], 3), kmax)
        try:
            out.append(G.queries(g, share, kmin, kmax, KINDS[kind], seed + i, 0))
        except _lib.GpsmError:  # a graph without such a shape
            out.append(G.queries(g, share, 3, 4, KINDS["tree"], seed + i, 0))
    return [q for qs in zip(*out) for q in qs] + [q for qs in out for q in qs[min(map(len, out)):]]


def _feasible(rg, count, case, seed):
    """count queries whose exact join examines at most the budget; a query of
    a few vertices where the case's sizes have none."""
    kept, work = [], []
    for r in range(3):
        qs = _draws(rg.g, max(64, 3 * count), case, seed + 104729 * r)
        for q, x in zip(qs, rg.match_batch(qs, work_budget=case["budget"])):
            if x.status == 0:
                kept.append(q)
                work.append(x.join_work)
        if len(kept) >= count:
            break
    if not kept:
        kept, work = G.queries(rg.g, count, 2, 2, KINDS["tree"], seed, 0), [1] * count
    if case["path"] == "match":  # the one with the most work of its draws
        return [kept[max(range(len(kept)), key=lambda i: work[i])]]
    return [kept[i % len(kept)] for i in range(count)]


def _own_query(case, choose):
    """The query that belongs to the case, chosen on its data graph as generated."""
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    return _kept(_QUERIES, key, lambda: choose(_resident(case, 0)), 16)


def _renumbered_edges(case, rng):
    """The case's data graph with its vertices numbered at random."""
    g = _graph(case, 0)
    ids = rng.permutation(g.n).astype(np.uint32)
    src, dst = g.edges()
    labels = np.empty_like(g.labels)
    labels[ids] = g.labels
    return ids[src], ids[dst], labels


def _renumbered(case, rng):
    src, dst, labels = _renumbered_edges(case, rng)
    return _ctx().upload_edges(len(labels), src, dst, labels)


def prepare(case, seed):
    path = case["path"]
    rng = np.random.default_rng(seed)
    if path == "match":
        state = {"path": path, "tuples": case["tuples"], "order": ORDERS[case["order"]], "width": case["kmax"]}
        if not case["tuples"]:
            rg = _resident(case, seed)
            return dict(state, rg=rg, q=_feasible(rg, 1, case, seed)[0])
        q = _own_query(case, lambda rg: _feasible(rg, 1, case, case["graph_seed"])[0])
        ids = rng.permutation(q.n).astype(np.uint32)
        lab = np.empty_like(q.labels)
        lab[ids] = q.labels
        return dict(state, rg=_renumbered(case, rng), q=G.Query(lab, ids[q.src], ids[q.dst]))
    if path == "batch":
        rg = _resident(case, seed)
        return {"path": path, "rg": rg, "qs": _feasible(rg, case["queries"], case, seed), "width": case["kmax"],
                "order": ORDERS[case["order"]], "use_graph": case["use_graph"]}
    if path == "mix":
        # the stored queries of the benchmark graph, in an order of the seed
        mix = {"graph": "chung_lu", "n": 1_000_000, "edges": 8_000_000, "labels": 16, "zipf": 1.0, "graph_seed": 2}
        qs, _ = workloads.load_set("chunglu1m_mix4_32")
        pick = rng.permutation(len(qs))[:case["queries"]]
        return {"path": "batch", "rg": _resident(mix, seed), "qs": [qs[i] for i in pick], "width": 6,
                "order": ORDERS[case["order"]], "use_graph": False}
    if path == "filter":
        rg = _resident(case, seed)
        return {"path": path, "rg": rg, "q": _draws(rg.g, 1, case, seed)[0]}
    if path == "tables":
        q = _own_query(case, lambda rg: _draws(rg.g, 1, case, case["graph_seed"])[0])
        return {"path": path, "rg": _renumbered(case, rng), "q": q}
    if path == "build":
        src, dst, labels = _renumbered_edges(case, rng)
        order = rng.permutation(len(src)).astype(np.int64)
        flip = rng.random(len(src)) < 0.5
        a, b = src[order], dst[order]
        a, b = np.where(flip, b, a), np.where(flip, a, b)
        twice = len(a) // 50  # some edges are listed in both directions
        return {"path": path, "n": len(labels), "src": np.concatenate([a, b[:twice]]),
                "dst": np.concatenate([b, a[:twice]]), "labels": labels}
    if path == "scan":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randint(0, 1 << 16, (case["values"],), dtype=torch.int32, device="cuda", generator=gen)
        y = torch.empty_like(x)
        torch.cuda.synchronize()
        return {"path": path, "x": x, "y": y, "total": C.c_uint64()}
    if path == "output":
        return _prepare_output(case, rng, seed)
    m = planner.MLP(_ctx(), seed=seed)
    return {"path": path, "m": m, "pass": case["pass"], "x": _features(case, rng), "t": _targets(case, rng)}


def _features(case, rng):
    return rng.standard_normal((case["samples"], F)).astype(np.float32)


def _targets(case, rng):
    return (3 + rng.standard_normal(case["samples"])).astype(np.float32)


def _prepare_output(case, rng, seed):
    """A data graph with directed, labelled arcs (most edges in both
    directions, most of one label), a path query, and tuples that walk it."""
    n, q = case["n"], case["q"]
    g = G.set_labels(G.chung_lu(n, case["edges"], 2.1, seed), 4, 0.0, seed)
    src, dst = g.edges()
    both = rng.random(len(src)) < 0.9
    a = np.concatenate([src, dst[both]])
    b = np.concatenate([dst, src[both]])
    rg = _ctx().upload(g)
    rg.set_directed(a, b, (rng.random(len(a)) < 0.05).astype(np.uint32))
    deg = g.degree()
    t = np.empty((case["rows"], q), dtype=np.uint32)
    t[:, 0] = np.repeat(np.arange(n, dtype=np.uint32), deg)[rng.integers(0, g.adj, case["rows"])]
    for j in range(1, q):
        v = t[:, j - 1]
        t[:, j] = g.col[g.row_offset[v].astype(np.int64) + (rng.random(len(v)) * deg[v]).astype(np.int64)]
    query = G.path_query(q)
    arcs = [(j, j + 1, 0) for j in range(q - 1)]
    return {"path": "output", "rg": rg, "q": query, "arcs": arcs, "tuples": t,
            "text": np.zeros(case["rows"] * (16 * q + 1), dtype=np.uint8), "bytes": C.c_uint64()}


# --- one pass -------------------------------------------------------------------

def _table(rows, width, dtype):
    """Ragged per-query lists as one zero-padded array."""
    out = np.zeros((len(rows), width), dtype=dtype)
    for i, r in enumerate(rows):
        out[i, :len(r)] = r
    return out


def _results(rs, w):
    return {"count": np.array([r.count for r in rs], dtype=np.uint64).view(np.int64),
            "hash": np.array([r.hash for r in rs], dtype=np.uint64).view(np.int64),
            "status": np.array([r.status for r in rs], dtype=np.int64),
            "join_work": np.array([r.join_work for r in rs], dtype=np.int64),
            "order": _table([r.order for r in rs], w, np.int64),
            "cand": _table([r.cand for r in rs], w, np.int64),
            "level_rows": _table([r.level_rows for r in rs], w, np.int64),
            "level_work": _table([r.level_work for r in rs], w, np.int64)}


def run(state):
    path = state["path"]
    if path == "match":
        kw = {"want_tuples": True, "tuple_cap": 1 << 22} if state["tuples"] else {}
        r = state["rg"].match(state["q"], order_mode=state["order"], **kw)
        out = _results([r], state["width"])
        if state["tuples"]:
            out["tuples"] = r.tuples.view(np.int32)
        return out
    if path == "batch":
        rs = state["rg"].match_batch(state["qs"], order_mode=state["order"], use_graph=state["use_graph"])
        return _results(rs, state["width"])
    if path == "filter":
        bitmaps, counts = state["rg"].filter(state["q"])
        return {"bitmaps": bitmaps.view(np.int32), "counts": counts.view(np.int32)}
    if path == "tables":
        edges, tables = state["rg"].candidate_edges(state["q"])
        return {"edges": np.array(edges, dtype=np.int64),
                "ids": np.concatenate([t[0] for t in tables]).view(np.int32),
                "offsets": np.concatenate([t[1] for t in tables]).view(np.int32),
                "lists": np.concatenate([t[2] for t in tables]).view(np.int32)}
    if path == "build":
        rg = _ctx().upload_edges(state["n"], state["src"], state["dst"], state["labels"])
        out = {"row_offset": rg.g.row_offset.view(np.int32), "col": rg.g.col.view(np.int32),
               "hubs": np.array(rg.hubs(), dtype=np.int64)}
        rg.free()
        return out
    if path == "scan":
        x, y, total = state["x"], state["y"], state["total"]
        _lib.check(_lib.lib().gpsm_scan_u32_noalloc(_ctx().h, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()),
                                                    x.numel(), C.byref(total)), "gpsm_scan_u32_noalloc")
        return {"sums": y, "total": total.value}
    if path == "output":
        t, text, need = state["tuples"], state["text"], state["bytes"]
        keep = state["rg"].verify_directed(state["q"], state["arcs"], t)
        flags = keep.astype(np.uint8)
        _lib.check(_lib.lib().gpsm_format_tuples(_ctx().h, _lib.ptr(t), len(t), t.shape[1], _lib.ptr(flags),
                                                 _lib.ptr(text), text.size, C.byref(need)), "gpsm_format_tuples")
        return {"keep": flags, "text": text, "bytes": need.value}
    m = state["m"]
    if state["pass"] == "forward":
        return {"y": m.forward(state["x"])}
    loss, grad = m.grad(state["x"], state["t"])
    return {"loss": loss, "grad": grad}


# --- what a pass cannot do without ----------------------------------------------

def work(case):
    path = case["path"]
    if path == "scan":
        return {"bytes": 8 * case["values"] + 8, "flops": 0}
    if path == "planner":
        b = case["samples"]
        fwd = 2 * (F * H + H * H + H)
        params = 4 * _lib.N_PARAMS
        if case["pass"] == "forward":
            return {"bytes": 4 * b * (F + 1) + params, "flops": fwd * b}
        return {"bytes": 4 * b * (F + 1) + 2 * params, "flops": (fwd + 2 * (2 * H * H + H * F + H)) * b}
    if path == "output":
        # tuples and arcs read, flags and about 10 characters per value written
        return {"bytes": case["rows"] * (14 * case["q"] + 1) + 12 * 2 * case["edges"], "flops": 0}
    if path == "mix":
        n, m, q = 1_000_000, 8_000_000, 4 * case["queries"]
    else:
        n, m, q = case["n"], case["edges"], case.get("kmax", 0) * case.get("queries", 1)
    csr = 4 * (2 * n + 1) + 8 * m  # offsets, columns, labels
    if path == "build":
        return {"bytes": 8 * m + 4 * n + csr, "flops": 0}
    if path == "filter":
        return {"bytes": csr + q * ((n + 31) // 32) * 4, "flops": 0}
    rows = 3 * case["budget"] // 4 if case.get("tuples") else 0  # embeddings returned, about
    return {"bytes": csr + 1600 * case.get("queries", 1) + 4 * rows * case.get("kmax", 0), "flops": 0}


# --- the network in 64 bits -----------------------------------------------------

def exact(case, seed):
    """Forward, loss and gradients of the planner network in 64 bits for the
    same weights and inputs; every other path returns whole numbers."""
    if case["path"] != "planner":
        return None
    rng = np.random.default_rng(seed)
    x, t = _features(case, rng).astype(np.float64), _targets(case, rng).astype(np.float64)
    m = planner.MLP(_ctx(), seed=seed)
    p = m.get().astype(np.float64)  # the weights that prepare() starts from
    m.free()
    w1, b1, w2, b2, w3, b3 = np.split(p, np.cumsum([H * F, H, H * H, H, H]))
    w1, w2 = w1.reshape(H, F), w2.reshape(H, H)
    h1 = np.maximum(x @ w1.T + b1, 0)
    h2 = np.maximum(h1 @ w2.T + b2, 0)
    y = h2 @ w3 + b3
    if case["pass"] == "forward":
        return {"y": y}
    dy = (y - t) / len(t)
    d2 = (dy[:, None] * w3) * (h2 > 0)
    d1 = (d2 @ w2) * (h1 > 0)
    grad = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), h2.T @ dy, [dy.sum()]])
    return {"loss": float(0.5 * np.mean((y - t) ** 2)), "grad": grad}
