"""The timed work of the mining engine: what programs have it do, through the
public entry points of ``gpm_amd`` and ``cost_model``.

Kinds of case (``case["kind"]``):

  tc        triangle count of an oriented graph (``DeviceGraph.tc``)
  clique    k-clique counts (``clique`` for one k, ``clique_all`` for 3, 4, 5)
  learned   features, cost model and the cost-scheduled clique count of one
            graph, the whole learned path
  patterns  the fixed patterns P1 - P8 and Motif4 in one formulation
  match     batches of labeled queries against a resident graph
  prep      edge list to CSR to oriented DAG to host arrays
  setops    a batch of sorted-list pairs through one set primitive

Graphs are R-MAT (a, b, c, d = .57, .19, .19, .05), symmetrised, without
duplicates and self loops, or Erdos-Renyi with a fixed number of edges, drawn
from the seed alone.  ``n`` need not be a power of two (R-MAT samples past n
are dropped), and ``samples`` is the number of edge samples before duplicates
go.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gpm-artifact_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import gpm_amd as G  # noqa: E402
import workloads as W  # noqa: E402
from cost_model import CostModel  # noqa: E402

K = 1024


# ------------------------------------------------------------------- cases

def listed():
    return [
        # The reference's smallest real use: one edge-centric triangle count
        # of a small sparse graph, where launches and the host path count.
        {"name": "tc_edge_er16k", "kind": "tc", "graph": "er", "n": 16 * K, "samples": 128 * K, "variant": "edge"},
        # The default (vertex-centric) triangle count of a large power-law
        # graph, one million vertices.
        {"name": "tc_vertex_rmat20", "kind": "tc", "graph": "rmat", "n": 1024 * K, "samples": 16 * 1024 * K,
         "variant": "vertex"},
        # A 4-clique count of an ordinary graph of odd size.
        {"name": "clique4_rmat100k", "kind": "clique", "graph": "rmat", "n": 100003, "samples": 1100000, "k": 4,
         "policy": "degree"},
        # The benchmark's workload: 3-, 4- and 5-cliques of R-MAT scale 20 in
        # one pass over the roots.
        {"name": "clique_all_rmat20", "kind": "clique", "graph": "rmat", "n": 1024 * K, "samples": 16 * 1024 * K,
         "k": 0, "policy": "degree"},
        # Learned scheduling end to end: a program that has the two graphs
        # resident predicts root costs and counts 5-cliques by them.
        {"name": "learned5_rmat18", "kind": "learned", "graph": "rmat", "n": 256 * K, "samples": 16 * 256 * K, "k": 5},
        # Every fixed pattern by direct enumeration (the G2Miner solver).
        {"name": "patterns_direct_rmat9", "kind": "patterns", "graph": "rmat", "n": 512, "samples": 16 * 512,
         "pids": "P1 P2 P3 P4 P5 P6 P7 P8 Motif4", "form": "direct"},
        # Every fixed pattern by the counting formulation (PatternSolver), at
        # the scale where the bench compares the two formulations.
        {"name": "patterns_counting_rmat11", "kind": "patterns", "graph": "rmat", "n": 2 * K, "samples": 32 * K,
         "pids": "P1 P2 P3 P4 P5 P6 P7 P8 Motif4", "form": "counting"},
        # The motif census of a large graph.
        {"name": "motif4_rmat19", "kind": "patterns", "graph": "rmat", "n": 512 * K, "samples": 8192 * K,
         "pids": "Motif4", "form": "counting"},
        # The named queries (triangle, 4-cycle, diamond, three-star) with
        # random labels as one batch that is asked again and again.
        {"name": "match_named_rmat18", "kind": "match", "graph": "rmat", "n": 256 * K, "samples": 16 * 256 * K,
         "labels": 8, "queries": "named", "batches": 1, "count": 4, "policy": "degree"},
        # A query service on a graph of the size and label count of the
        # reference's protein network (9460 vertices, 37081 edges, 307
        # labels): batches of queries of 4 to 10 vertices cut out of the data
        # graph, each batch another one than the last.
        {"name": "match_service_9460", "kind": "match", "graph": "rmat", "n": 9460, "samples": 42000,
         "labels": 307, "queries": "sampled", "batches": 2, "count": 100, "policy": "learned"},
        # Preparation of a graph that comes as a host edge list: build, orient
        # and hand the DAG back.
        {"name": "prep_rmat17", "kind": "prep", "graph": "rmat", "n": 128 * K, "samples": 2048 * K},
        # The set primitives as a library: many pairs of sorted lists.
        {"name": "setops_isect_4k", "kind": "setops", "op": "isect", "variant": "merge", "pairs": 4096,
         "mean": 600, "span": 1 << 20},
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["tc", "tc", "clique", "clique", "clique", "learned", "patterns", "patterns", "match", "match",
                       "prep", "setops"])
    if kind == "tc":
        n = _between(rng, 5000, 900000)
        return {"kind": kind, "graph": rng.choice(["er", "rmat"]), "n": n, "samples": int(n * rng.uniform(3, 16)),
                "variant": rng.choice(["edge", "vertex"])}
    if kind == "clique":
        n = _between(rng, 3000, 800000)
        return {"kind": kind, "graph": "rmat", "n": n, "samples": int(n * rng.uniform(6, 16)),
                "k": rng.choice([0, 3, 4, 5]), "policy": rng.choice(["degree", "degree_split"])}
    if kind == "learned":
        n = _between(rng, 3000, 250000)
        return {"kind": kind, "graph": "rmat", "n": n, "samples": int(n * rng.uniform(6, 16)), "k": rng.choice([4, 5])}
    if kind == "patterns":
        if rng.random() < 0.4:
            n = _between(rng, 5000, 500000)
            return {"kind": kind, "graph": "rmat", "n": n, "samples": int(n * rng.uniform(5, 16)), "pids": "Motif4",
                    "form": "counting"}
        form = rng.choice(["direct", "counting", "prefilter"])
        n = _between(rng, 200, 500 if form == "direct" else 1900)
        pids = sorted(rng.sample(["P%d" % i for i in range(1, 9)], rng.randint(2, 5)))
        return {"kind": kind, "graph": "rmat", "n": n, "samples": int(n * rng.uniform(5, 15)),
                "pids": " ".join(pids), "form": form}
    if kind == "match":
        if rng.random() < 0.5:
            n = _between(rng, 4000, 250000)
            return {"kind": kind, "graph": "rmat", "n": n, "samples": int(n * rng.uniform(6, 16)), "labels": 8,
                    "queries": "named", "batches": 1, "count": 4, "policy": rng.choice(["degree", "learned"])}
        n = _between(rng, 3000, 16000)
        return {"kind": kind, "graph": "rmat", "n": n, "samples": int(n * rng.uniform(3, 6)),
                "labels": rng.randint(100, 307), "queries": "sampled", "batches": 2, "count": _between(rng, 8, 100),
                "policy": rng.choice(["degree", "learned"])}
    if kind == "prep":
        n = _between(rng, 3000, 130000)
        return {"kind": kind, "graph": rng.choice(["er", "rmat"]), "n": n, "samples": int(n * rng.uniform(4, 15))}
    return {"kind": "setops", "op": rng.choice(["isect_count", "isect", "diff_count", "diff", "fuse"]),
            "variant": rng.choice(["binary", "two_phase", "merge", "hash", "bitmap"]),
            "pairs": _between(rng, 50, 4000), "mean": _between(rng, 10, 500), "span": 1 << rng.randint(14, 20)}


# ------------------------------------------------------------------ inputs

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _edges(case, seed):
    """Edge list (two uint32 arrays on the host) of the case's graph."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(1000003 * seed + 17)
    n, m = case["n"], case["samples"]
    if case["graph"] == "er":
        pair = torch.zeros(0, dtype=torch.int64, device=dev)
        while len(pair) < m:  # distinct pairs without self loops, in random order
            u = torch.randint(0, n, (m + m // 4 + 64,), generator=gen, device=dev)
            v = torch.randint(0, n, (m + m // 4 + 64,), generator=gen, device=dev)
            u, v = torch.minimum(u, v), torch.maximum(u, v)
            pair = torch.unique(torch.cat([pair, (u * n + v)[u != v]]))
        pair = pair[torch.randperm(len(pair), generator=gen, device=dev)[:m]]
        src, dst = pair // n, pair % n
    else:
        src = torch.zeros(m, dtype=torch.int64, device=dev)
        dst = torch.zeros(m, dtype=torch.int64, device=dev)
        for _ in range(max(1, (n - 1).bit_length())):
            r = torch.rand(m, generator=gen, device=dev)
            src = 2 * src + (r >= 0.76)
            dst = 2 * dst + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        keep = (src < n) & (dst < n)
        src, dst = src[keep], dst[keep]
    to32 = lambda t: t.to(torch.int32).cpu().numpy().view(np.uint32)  # noqa: E731
    return to32(src), to32(dst)


def _queries(case, sym, labels, seed):
    if case["queries"] == "named":
        named = [q for name, q in W.named_queries(seed + 7) if name != "pyramid-6"]
        return [named[: case["count"]]]
    host = sym.to_host()
    return [W.sampled_queries(host, labels, case["count"], 31 * seed + b)
            for b in range(case["batches"])]


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "setops":
        rng = np.random.default_rng(seed)

        def one():
            size = min(case["span"] // 2, 2 * case["mean"], int(rng.lognormal(math.log(case["mean"]), 0.8)))
            return np.unique(rng.integers(0, case["span"], size, dtype=np.uint32))

        pairs = []
        for _ in range(case["pairs"]):
            a, b = one(), one()
            shared = a[rng.random(len(a)) < 0.3]  # lists of neighbours have entries in common
            pairs.append((a, np.union1d(b, shared).astype(np.uint32)))
        state["pairs"] = pairs
        # The program's own buffers for the lists of all pairs (A has at most
        # twice the mean a list, B twice that).
        room = {"isect": [2], "diff": [2], "fuse": [2, 2, 4]}.get(case["op"], [])
        state["lists"] = [np.zeros(r * case["mean"] * case["pairs"], np.uint32) for r in room]
        return state
    src, dst = _edges(case, seed)
    if kind == "prep":
        state["edges"] = (case["n"], src, dst)
        state["offsets"], state["adj"] = np.zeros(case["n"] + 1, np.uint32), np.zeros(case["samples"], np.uint32)
        return state
    labels = None
    if kind == "match":
        labels = np.random.default_rng(seed + 1).integers(0, case["labels"], case["n"]).astype(np.uint32)
    sym = G.DeviceGraph.build(case["n"], src, dst, labels=labels, n_labels=case.get("labels", 0))
    if kind in ("tc", "clique"):
        state["dag"] = sym.orient()
    elif kind == "learned":
        state["sym"], state["dag"] = sym, sym.orient()
        state["model"] = CostModel.load_default(5)
    else:
        state["sym"] = sym
        if kind == "match":
            state["queries"] = _queries(case, sym, labels, seed)
    return state


POLICY = {"degree": G.SCHED_DEGREE, "degree_split": G.SCHED_DEGREE_SPLIT, "learned": G.SCHED_LEARNED}
FORM = {"direct": G.FORM_G2MINER, "counting": G.FORM_PATTERN, "prefilter": G.FORM_BLOCK_PREFILTER}
SETOP = {"isect_count": G.SETOP_ISECT_COUNT, "isect": G.SETOP_ISECT, "diff_count": G.SETOP_DIFF_COUNT,
         "diff": G.SETOP_DIFF, "fuse": G.SETOP_FUSE}
SETV = {"binary": G.SETV_BINARY, "two_phase": G.SETV_TWO_PHASE, "merge": G.SETV_MERGE, "hash": G.SETV_HASH,
        "bitmap": G.SETV_BITMAP}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "tc":
        return state["dag"].tc(G.TC_EDGE if case["variant"] == "edge" else G.TC_VERTEX)
    if kind == "clique":
        if case["k"] == 0:
            return state["dag"].clique_all(POLICY[case["policy"]])
        return state["dag"].clique(case["k"], POLICY[case["policy"]])
    if kind == "learned":
        feat = G.vertex_features(state["sym"], state["dag"])
        log_cost = state["model"].predict_log(feat)
        cost = np.expm1(np.clip(log_cost, 0.0, 60.0)).astype(np.float32)
        return [feat, log_cost, state["dag"].clique(case["k"], policy=G.SCHED_LEARNED, cost=cost)]
    if kind == "patterns":
        out = []
        for pid in case["pids"].split():
            counts, scalar = state["sym"].pattern(pid, FORM[case["form"]])
            out.append(np.array(counts + [scalar], dtype=np.uint64).view(np.int64))
        return out
    if kind == "match":
        return [state["sym"].match_batch(batch, policy=POLICY[case["policy"]]).astype(np.int64)
                for batch in state["queries"]]
    if kind == "prep":
        with G.DeviceGraph.build(*state["edges"]) as sym, sym.orient() as dag:
            u32p = C.POINTER(C.c_uint32)
            status = G.lib().gpm_graph_copy_csr(dag.handle, state["offsets"].ctypes.data_as(u32p),
                                                state["adj"].ctypes.data_as(u32p))
        if status != G.GPM_OK:
            raise G.GpmError(status, "copying the DAG")
        return [state["offsets"].view(np.int32), state["adj"].view(np.int32)]
    counts, lists = G.setops(SETOP[case["op"]], SETV[case["variant"]], state["pairs"])
    if lists is not None:
        for part, buf in zip(zip(*lists) if case["op"] == "fuse" else [lists], state["lists"]):
            np.concatenate(part, out=buf[: sum(map(len, part))])
    return [counts.astype(np.int64)] + [buf.view(np.int32) for buf in state["lists"]]


# ---------------------------------------------------------- work and values

def work(case):
    """Each input read once and each output written once.  Edges count before
    duplicates go (R-MAT keeps 0.9 and more of them)."""
    if case["kind"] == "setops":
        lists = 4 * case["pairs"] * case["mean"] * 2 * 1.4  # mean of the length distribution
        return {"bytes": lists * 1.3 + 24 * case["pairs"], "flops": 0}
    n, m = case["n"], case["samples"]
    dag, sym = 4 * (n + 1) + 4 * m, 4 * (n + 1) + 8 * m
    if case["kind"] in ("tc", "clique"):
        return {"bytes": dag + 24, "flops": 0}
    if case["kind"] == "learned":
        # the features (16 bytes a vertex) go to the host and back, and the
        # predictions to the host
        return {"bytes": dag + 4 * (n + 1) + 36 * n, "flops": 2 * n * (4 * 64 + 64 * 64 + 64)}
    if case["kind"] == "prep":
        return {"bytes": 8 * m + dag, "flops": 0}
    if case["kind"] == "patterns":
        return {"bytes": sym + 48, "flops": 0}
    return {"bytes": sym + 4 * n + 8 * case["batches"] * case["count"], "flops": 0}


def exact(case, seed):
    """The learned path's features and predictions in 64 bits; every other
    output is a whole number."""
    if case["kind"] != "learned":
        return None
    n = case["n"]
    src, dst = (torch.from_numpy(e.astype(np.int64)) for e in _edges(case, seed))
    keep = src != dst
    src, dst = src[keep], dst[keep]
    key = torch.unique(torch.cat([src * n + dst, dst * n + src]))
    u, v = key // n, key % n
    deg = torch.bincount(u, minlength=n)
    up = (deg[v] > deg[u]) | ((deg[v] == deg[u]) & (v > u))
    du, dv = u[up], v[up]
    out_deg = torch.bincount(du, minlength=n)
    hop = torch.zeros(n, dtype=torch.float64).index_add_(0, du, out_deg[dv].double())
    feat = torch.stack([deg.double(), out_deg.double(), hop, torch.zeros(n, dtype=torch.float64)], dim=1)
    with np.load(os.path.join(PKG, "weights", "clique_k5.npz"), allow_pickle=False) as z:
        p = {k: torch.from_numpy(z[k].astype(np.float64)) for k in ("mean", "std", "w1", "b1", "w2", "b2", "w3", "b3")}
    x = (torch.log1p(feat) - p["mean"]) / p["std"]
    h = torch.relu(x @ p["w1"].T + p["b1"])
    h = torch.relu(h @ p["w2"].T + p["b2"])
    return [feat, (h @ p["w3"].T)[:, 0] + p["b3"][0], None]
