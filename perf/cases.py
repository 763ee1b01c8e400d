"""What a user of this solver has it do, as cases that can be timed.

Every case goes through the public Python entry points (vcgpu.py over the C
ABI): `solve_mvc`, `Context.solve` on a kept `GraphSet`, and `Server`.  The
graphs come from the repository's seeded generators (graphgen.py), in the
families and sizes of its benchmark and tests; a case's inputs depend on the
seed alone.

Only searches that finish are listed, so that every answer is the exact one:
a minimum cover size, or the yes/no of "is there a cover of size <= k?".
Those are what `run` returns.  The covers themselves are asked for and come
back as in a user's program, but a graph has many minimum covers and which
one a parallel search meets first is not determined, so covers (and node
counts) cannot be compared between two runs; their sizes are the returned
minima.  All answers are whole numbers, hence the tolerance "exact".
"""
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.getcwd(), "parallel-vertex-cover-algorithms-on-gpus_amd"))

import graphgen  # noqa: E402
import vcgpu  # noqa: E402

# A search that a case does not expect to be long is ended after this time
# (its graphs then report that they were not solved).
TIME_LIMIT_MS = 30000


def listed():
    return [
        # the smallest calls: small graphs handed over, bounded, uploaded,
        # solved and given back one after the other, as a program with a few
        # questions does it
        {"name": "calls_er_40", "kind": "call", "family": "er", "n": 40, "degree": 4.0, "graphs": 4},
        # the benchmark's small hard graphs, each on a kept set: a few
        # thousand tree nodes, where launch and hand-off latency count
        {"name": "mvc_reg3_120", "kind": "mvc", "family": "reg3", "n": 120, "degree": 3.0, "graphs": 4},
        # the benchmark's decision problem: no at opt - 1, yes at opt, on a
        # graph of some thousand vertices that is a chain of reductions
        {"name": "pvc_ba_2000", "kind": "pvc", "family": "ba", "n": 2000, "degree": 6.0, "graphs": 1},
        # the benchmark's plain graph: long searches that fill the chip
        {"name": "mvc_er_200", "kind": "mvc", "family": "er", "n": 200, "degree": 9.95, "graphs": 2},
        # dense graphs (the reference's cop_hat family is dense): long
        # adjacency lists, shallow trees of many branches
        {"name": "mvc_dense_250", "kind": "mvc", "family": "er", "n": 250, "degree": 124.5, "graphs": 3},
        # the reference's other mode (-v stackonly): a static split, no worklist
        {"name": "stackonly_er_90", "kind": "stackonly", "family": "er", "n": 90, "degree": 5.34, "graphs": 4},
        # a large sparse network, int16 node state in HBM
        {"name": "mvc_sparse_24000", "kind": "mvc", "family": "er", "n": 24001, "degree": 2.0, "graphs": 1},
        # the same beyond 32,767 vertices: int32 node state
        {"name": "mvc_sparse_40000", "kind": "mvc", "family": "er", "n": 40009, "degree": 2.0, "graphs": 1},
        # a small batch from a caller that cannot allocate device memory
        {"name": "batch_noalloc_61", "kind": "batch", "count": 61, "ask": "mvc", "entry": "noalloc"},
        # the batched workload: uneven graphs, one launch, covers wanted
        {"name": "batch_mvc_1024", "kind": "batch", "count": 1024, "ask": "mvc", "entry": "solve"},
        # the same as a decision ("is there a cover below the greedy one?"),
        # dispatched as a captured HIP graph
        {"name": "batch_pvc_graph_509", "kind": "batch", "count": 509, "ask": "pvc", "entry": "graph"},
        # a burst of requests into a continuous-batching server
        {"name": "served_256", "kind": "served", "count": 256},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["call", "reg3", "pvc", "er", "dense", "stackonly", "sparse", "sparse", "batch", "batch", "served"])
    if kind == "call":
        return {"kind": "call", "family": "er", "n": _log(rng, 20, 120), "degree": round(rng.uniform(1.5, 6.0), 2),
                "graphs": rng.randint(3, 6)}
    if kind == "reg3":
        return {"kind": "mvc", "family": "reg3", "n": 2 * rng.randint(25, 65), "degree": 3.0, "graphs": rng.randint(3, 6)}
    if kind == "pvc":
        return {"kind": "pvc", "family": "ba", "n": _log(rng, 200, 3000), "degree": float(rng.choice([4, 6])),
                "graphs": rng.randint(1, 3)}
    if kind == "er":
        return {"kind": "mvc", "family": "er", "n": rng.randint(60, 170), "degree": round(rng.uniform(3.0, 10.0), 2),
                "graphs": rng.randint(2, 4)}
    if kind == "dense":
        n = rng.randint(60, 250)
        return {"kind": "mvc", "family": "er", "n": n, "degree": round((n - 1) * rng.uniform(0.5, 0.9), 2),
                "graphs": rng.randint(2, 4)}
    if kind == "stackonly":
        return {"kind": "stackonly", "family": "er", "n": rng.randint(40, 100), "degree": round(rng.uniform(3.0, 6.0), 2),
                "graphs": rng.randint(3, 6)}
    if kind == "sparse":
        return {"kind": "mvc", "family": "er", "n": _log(rng, 1000, 40000), "degree": round(rng.uniform(1.2, 2.0), 2),
                "graphs": 1}
    if kind == "served":
        return {"kind": "served", "count": _log(rng, 16, 256)}
    return {"kind": "batch", "count": _log(rng, 8, 900), "ask": rng.choice(["mvc", "mvc", "pvc"]),
            "entry": rng.choice(["solve", "solve", "graph", "noalloc"])}


_context = None


def _ctx():
    """The program's one context on GPU 0 (its scratch is kept across solves)."""
    global _context
    if _context is None:
        _context = vcgpu.Context(0)
    return _context


def _sparse_er(n, m, seed):
    """m distinct uniform pairs: graphgen's pairwise draw needs n^2 memory."""
    rng = np.random.Generator(np.random.PCG64(seed))
    pairs = rng.integers(0, n, size=(2 * m + 64, 2))
    pairs = np.sort(pairs[pairs[:, 0] != pairs[:, 1]], axis=1)
    key, first = np.unique(pairs[:, 0] * n + pairs[:, 1], return_index=True)
    key = key[np.argsort(first)][:m]
    return np.stack([key // n, key % n], axis=1).astype(np.uint32)


def _graph(case, seed, i):
    """Graph i of a case: the case's family and mean degree, its size drawn
    from the upper tenth of the range up to the case's n."""
    rng = np.random.Generator(np.random.PCG64([seed, i]))
    family, degree = case["family"], case["degree"]
    n = case["n"] - int(rng.integers(case["n"] // 10 + 1))
    sub = int(rng.integers(1 << 31))
    if family == "reg3":
        n -= n & 1
        edges = graphgen.regular3_rewired(n, sub)
    elif family == "ba":
        edges = graphgen.barabasi_albert(n, round(degree / 2), sub)
    elif n >= 800:
        edges = _sparse_er(n, int(n * degree / 2), sub)
    else:
        edges = graphgen.erdos_renyi(n, degree / (case["n"] - 1), sub)
    return vcgpu.csr_from_edges(n, edges)


def _batch_graph(i, seed):
    """Graph i of the benchmark's batch distribution (half Erdos-Renyi with
    p ~ U[0.02, 0.15], half Barabasi-Albert with m in {2, 3, 4}), its
    Erdos-Renyi half up to 120 vertices, where every search finishes."""
    rng = np.random.Generator(np.random.PCG64([seed, i]))
    sub = int(rng.integers(1 << 31))
    if i % 2 == 0:
        n = int(rng.integers(40, 121))
        return vcgpu.csr_from_edges(n, graphgen.erdos_renyi(n, float(rng.uniform(0.02, 0.15)), sub))
    n = int(rng.integers(40, 401))
    return vcgpu.csr_from_edges(n, graphgen.barabasi_albert(n, int(rng.choice([2, 3, 4])), sub))


def _below_bound(g, u):
    """Is there a smaller cover than the greedy one?"""
    return vcgpu.Job(vcgpu.VC_PVC, max(u - 1, 0), u, 0)


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    params = vcgpu.Params(time_limit_ms=TIME_LIMIT_MS)
    state = {"ctx": ctx, "kind": kind, "params": params}
    if kind in ("batch", "served"):
        graphs = [_batch_graph(i, seed) for i in range(case["count"])]
        bounds = [vcgpu.upper_bound(g, seed=1)[0] for g in graphs]
        mvc = [vcgpu.Job(vcgpu.VC_MVC, 0, u, 0) for u in bounds]
        pvc = [_below_bound(g, u) for g, u in zip(graphs, bounds)]
        if kind == "served":
            # half the requests are decisions, in both families
            state["requests"] = [(g, (mvc, pvc)[(i >> 1) & 1][i]) for i, g in enumerate(graphs)]
            return state
        state["jobs"] = mvc if case["ask"] == "mvc" else pvc
        state["noalloc"] = case["entry"] == "noalloc"
        if case["entry"] == "graph":
            params.flags |= vcgpu.VC_FLAG_GRAPH
        state["set"] = ctx.upload(graphs)
        return state
    graphs = [_graph(case, seed, i) for i in range(case["graphs"])]
    if kind == "call":
        state["graphs"] = graphs
        return state
    if kind == "stackonly":
        params.version = vcgpu.VC_STACK_ONLY
        params.start_depth = 4
    state["asks"] = []  # (set, job): one launch each
    for g in graphs:
        u, _ = vcgpu.upper_bound(g, seed=1)
        kept, job = ctx.upload(g), vcgpu.Job(vcgpu.VC_MVC, 0, u, 0)
        if kind == "pvc":
            # the question's two sides: one below the minimum, and the minimum
            (r,), _, _ = ctx.solve(kept, job, params)
            state["asks"] += [(kept, vcgpu.Job(vcgpu.VC_PVC, k, u, 0)) for k in (max(r.minimum - 1, 0), r.minimum)]
        else:
            state["asks"].append((kept, job))
    return state


def run(state):
    ctx, kind, params = state["ctx"], state["kind"], state["params"]
    if kind == "call":
        got = [vcgpu.solve_mvc(ctx, g, params) for g in state["graphs"]]
        return {"answer": np.array([size for size, _, _, _ in got], np.int64),
                "solved": np.array([r.solved for _, _, r, _ in got], np.int64)}
    if kind == "served":
        server = vcgpu.Server(ctx, max_vertices=400, slots=512, arena_bytes=32 << 20, time_limit_ms=TIME_LIMIT_MS)
        try:
            tickets = [server.submit(g, job) for g, job in state["requests"]]
            got = [server.wait(t, TIME_LIMIT_MS)[0] for t in tickets]
        finally:
            server.stop()
        return _answers(got, [job for _, job in state["requests"]])
    if kind == "batch":
        got, _, _ = ctx.solve(state["set"], state["jobs"], params, raise_on_error=False, noalloc=state["noalloc"])
        return _answers(got, state["jobs"])
    got = [ctx.solve(kept, job, params, raise_on_error=False)[0][0] for kept, job in state["asks"]]
    out = _answers(got, [job for _, job in state["asks"]])
    if kind == "pvc":
        # k is the minimum or one less: a cover found has the minimum's size
        out["size"] = np.array([r.minimum for r in got], np.int64)
    return out


def _answers(results, jobs):
    """The minimum of each MVC job, the yes/no of each PVC job, and whether
    the search finished."""
    return {"answer": np.array([r.minimum if j.instance == vcgpu.VC_MVC else r.k_found
                                for r, j in zip(results, jobs)], np.int64),
            "solved": np.array([r.solved for r in results], np.int64)}


def _graph_bytes(n, m):
    """A graph's CSR arrays read once, its result record and its cover written once."""
    return 4 * (n + 1) + 8 * m + 4 * n + 32 + n


def work(case):
    """The search tree's work has no closed form; what no solver can do
    without is reading the graphs and writing the answers."""
    if case["kind"] in ("batch", "served"):
        # means of the distribution: 80 vertices at p = 0.085, 220 at m = 3
        each = (_graph_bytes(80, 270) + _graph_bytes(220, 650)) / 2
        return {"bytes": case["count"] * each, "flops": 0}
    asks = case["graphs"] * (2 if case["kind"] == "pvc" else 1)
    n = 0.95 * case["n"]
    return {"bytes": asks * _graph_bytes(n, n * case["degree"] / 2), "flops": 0}


def tolerance(case):
    return "exact"
