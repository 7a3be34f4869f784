"""What is timed: the calls a program makes to this library, over the sizes it makes them at.

Every case is one call through the Python binding (`sssp_amd`) or, for callers
that own their device arrays, through the C ABI that the binding exposes:

  kind      call
  solve     DeviceGraph.solve: one source, distances returned to the host
  bfs       DeviceGraph.bfs: one source, visited flags and levels returned
  batch     DeviceGraph.solve_batch: many sources on one graph
  pack      GraphPack.solve: many independent graphs, one source each
  wrapper   sssp_init_distances_* and sssp_bellman_ford_* on device arrays
  ingest    DeviceGraph from host arrays, one solve, and its release

Graphs: `rmat` (the library's generator, the shape of the reference's own
inputs), `skewed` (power-law endpoints with scrambled ids; V and E need not be
powers of two), `uniform` (u32 weights 1..255) and `grid` (four neighbours,
long paths).
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "parallel-task1_amd")
sys.path.insert(0, PKG)

import sssp_amd as S  # noqa: E402

F32_MAX = float(np.finfo(np.float32).max)
F64_MAX = float(np.finfo(np.float64).max)


def listed():
    return [
        # the smallest call: a graph that fits one workgroup's LDS; latency alone
        {"name": "solve_rmat11", "kind": "solve", "graph": "rmat", "scale": 11, "ef": 16,
         "schedule": "heuristic"},
        # a mid-size graph with odd counts, default schedule
        {"name": "solve_skewed_odd", "kind": "solve", "graph": "skewed", "V": 1234567,
         "E": 11111111, "schedule": "heuristic"},
        # long shortest paths: hundreds of relaxation rounds over little data each
        {"name": "solve_grid", "kind": "solve", "graph": "grid", "rows": 517, "cols": 389,
         "schedule": "heuristic"},
        # the 2^22-vertex R-MAT configuration with the trained round scheduler
        {"name": "solve_rmat22", "kind": "solve", "graph": "rmat", "scale": 22, "ef": 32,
         "schedule": "learned"},
        # the benchmark's graph: 537 M edges
        {"name": "solve_rmat25", "kind": "solve", "graph": "rmat", "scale": 25, "ef": 16,
         "schedule": "learned"},
        # integer weights on a graph without hubs
        {"name": "solve_uniform_u32", "kind": "solve", "graph": "uniform", "V": 6000000,
         "E": 96000000, "schedule": "learned"},
        # breadth-first search on the 2^22-vertex R-MAT graph
        {"name": "bfs_rmat22", "kind": "bfs", "graph": "rmat", "scale": 22, "ef": 32,
         "schedule": "learned"},
        # 256 sources on one graph
        {"name": "batch_rmat20_256", "kind": "batch", "graph": "rmat", "scale": 20, "ef": 16,
         "n": 256},
        # a thousand small graphs of mixed sizes, solved together
        {"name": "pack_1024", "kind": "pack", "n": 1024, "smin": 8, "smax": 14, "ef": 8},
        # the reference's device wrapper on the caller's arrays, edges in file order
        {"name": "wrapper_f32", "kind": "wrapper", "graph": "skewed", "V": 1048576,
         "E": 16777216, "dtype": "f32"},
        # its double instantiation, odd sizes
        {"name": "wrapper_f64", "kind": "wrapper", "graph": "skewed", "V": 300007,
         "E": 4100009, "dtype": "f64"},
        # a graph used once: upload, layout build, one solve
        {"name": "ingest_solve", "kind": "ingest", "graph": "skewed", "V": 1000003,
         "E": 16000001, "schedule": "heuristic"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve_rmat", "solve_rmat", "solve_skewed", "solve_grid", "solve_uniform",
                       "bfs", "batch", "pack", "wrapper", "ingest"])
    sched = rng.choice(["heuristic", "learned", "plain"])
    if kind in ("solve_rmat", "bfs"):
        scale = rng.randint(10, 23)
        ef = rng.randint(5, 48 if scale < 23 else 24)
        return {"kind": "bfs" if kind == "bfs" else "solve", "graph": "rmat", "scale": scale,
                "ef": ef, "schedule": sched}
    if kind == "solve_skewed":
        V = _log(rng, 1000, 12000000)
        return {"kind": "solve", "graph": "skewed", "V": V, "E": V * rng.randint(3, 16) + rng.randint(1, 999),
                "schedule": sched}
    if kind == "solve_grid":
        return {"kind": "solve", "graph": "grid", "rows": _log(rng, 20, 700),
                "cols": _log(rng, 20, 700), "schedule": sched}
    if kind == "solve_uniform":
        V = _log(rng, 5000, 8000000)
        return {"kind": "solve", "graph": "uniform", "V": V, "E": V * rng.randint(6, 16) + rng.randint(1, 999),
                "schedule": sched}
    if kind == "batch":
        scale = rng.randint(12, 19)
        return {"kind": "batch", "graph": "rmat", "scale": scale, "ef": rng.randint(6, 16),
                "n": rng.randint(2, 300 if scale < 18 else 180)}
    if kind == "pack":
        return {"kind": "pack", "n": _log(rng, 20, 1500), "smin": 8, "smax": rng.randint(10, 14),
                "ef": rng.randint(5, 12)}
    V = _log(rng, 2000, 2000000)
    E = V * rng.randint(4, 16) + rng.randint(1, 999)
    if kind == "wrapper":
        dtype = rng.choice(["f32", "f32", "f64", "u32"])
        return {"kind": "wrapper", "graph": "uniform" if dtype == "u32" else "skewed", "V": V,
                "E": E, "dtype": dtype}
    return {"kind": "ingest", "graph": "skewed", "V": V, "E": E, "schedule": "heuristic"}


# ---- inputs -----------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _edges(case, seed):
    """src, dst (int32) and weights on the GPU, and the vertex count."""
    kind = case["graph"]
    if kind == "rmat":  # bit-identical to DeviceGraph.rmat with these arguments
        s, t, w = S.rmat(case["scale"], case["ef"], seed=seed + 1, threads=64)
        return (torch.from_numpy(s).cuda(), torch.from_numpy(t).cuda(), torch.from_numpy(w).cuda(),
                1 << case["scale"])
    g = _gen(seed)
    if kind == "grid":
        R, C = case["rows"], case["cols"]
        ids = torch.arange(R * C, device="cuda", dtype=torch.int32).reshape(R, C)
        right = (ids[:, :-1].reshape(-1), ids[:, 1:].reshape(-1))
        down = (ids[:-1].reshape(-1), ids[1:].reshape(-1))
        src = torch.cat([right[0], right[1], down[0], down[1]])
        dst = torch.cat([right[1], right[0], down[1], down[0]])
        w = 0.1 + 0.9 * torch.rand(src.numel(), device="cuda", generator=g)
        return src, dst, w, R * C
    V, E = case["V"], case["E"]
    if kind == "uniform":
        src = torch.randint(0, V, (E,), device="cuda", generator=g, dtype=torch.int32)
        dst = torch.randint(0, V, (E,), device="cuda", generator=g, dtype=torch.int32)
        w = torch.randint(1, 256, (E,), device="cuda", generator=g, dtype=torch.int32)
        return src, dst, w, V

    def ends(power):  # skewed ranks, spread over the ids
        u = torch.rand(E, device="cuda", generator=g, dtype=torch.float64)
        r = (u.pow_(power) * V).long().clamp_(max=V - 1)
        return ((r * 2654435761 + 12345) % V).int()

    src, dst = ends(3), ends(2)
    w = torch.rand(E, device="cuda", generator=g)
    if case.get("dtype") == "f64":
        w = torch.rand(E, device="cuda", generator=g, dtype=torch.float64)
    return src, dst, w, V


def _rmat_source(case, rng):
    """A vertex with out-edges, hub or ordinary: the expected out-degree of an
    id with k one bits is E * 0.76^(scale - k) * 0.24^k."""
    scale = case["scale"]
    E = case["ef"] << scale
    top = 0
    while top < scale - 1 and E * 0.76 ** (scale - top - 1) * 0.24 ** (top + 1) >= 12:
        top += 1
    bits = rng.sample(range(1, scale), rng.randint(0, top)) if top else []
    return sum(1 << b for b in bits)


def _source(case, seed, src):
    rng = random.Random(seed * 7919 + 3)
    if case["graph"] == "rmat":
        return _rmat_source(case, rng)
    if case["graph"] == "grid":
        return rng.randrange(case["cols"])  # a vertex of the first row
    return int(src[rng.randrange(src.numel())].item())


def _pack_scales(case):
    """Every scale of the range in turn, in a shuffled order."""
    scales = case["smin"] + np.arange(case["n"]) % (case["smax"] - case["smin"] + 1)
    return np.random.default_rng(5).permutation(scales).astype(np.int32)


def _pack_inputs(case, seed):
    scales = _pack_scales(case)
    s, t, w, offs = S.rmat_many(scales, case["ef"], seed0=seed + 5)
    counts = (1 << scales).astype(np.int32)
    sources = np.minimum.reduceat(s, offs[:-1]).astype(np.int32)
    return s, t, w, offs, counts, sources


def _host(t):
    a = t.cpu().numpy()
    return a.view(np.uint32) if a.dtype == np.int32 else a


def _network(name):
    m = S.MLP(0)
    m.set_params(np.fromfile(os.path.join(PKG, "models", name), np.float32))
    return m


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pack":
        s, t, w, offs, counts, sources = _pack_inputs(case, seed)
        return {"kind": kind, "pack": S.GraphPack(s, t, w, offs, counts), "sources": sources}
    if kind == "wrapper":
        src, dst, w, V = _edges(case, seed)
        real = torch.float64 if case["dtype"] == "f64" else torch.float32
        dist = torch.empty(V, device="cuda", dtype=torch.int32 if case["dtype"] == "u32" else real)
        st = {"kind": kind, "src": src, "dst": dst, "w": w, "V": V, "dtype": case["dtype"],
              "dist": dist, "source": _source(case, seed, src)}
        torch.cuda.synchronize()
        return st
    if kind == "ingest":
        src, dst, w, V = _edges(case, seed)
        return {"kind": kind, "src": src.cpu().numpy(), "dst": dst.cpu().numpy(), "w": _host(w),
                "V": V, "source": _source(case, seed, src), "schedule": case["schedule"]}
    src = None
    if case["graph"] == "rmat":
        g = S.DeviceGraph.rmat(case["scale"], case["ef"], seed=seed + 1, threads=64)
    else:
        src, dst, w, V = _edges(case, seed)
        g = S.DeviceGraph(src.cpu().numpy(), dst.cpu().numpy(), _host(w), V)
    st = {"kind": kind, "graph": g}
    if kind == "batch":
        rng = random.Random(seed * 7919 + 3)
        st["sources"] = np.array([_rmat_source(case, rng) for _ in range(case["n"])], np.int32)
        return st
    st["source"] = _source(case, seed, src)
    st["schedule"] = case["schedule"]
    if case["schedule"] == "learned":
        if kind == "bfs":
            g.set_bfs_mlp(_network("scheduler_bfs_mlp.f32"))
        else:
            g.set_mlp(_network("scheduler_mlp.f32"))
    return st


# ---- one pass ---------------------------------------------------------------
def _check(rc):
    if rc != S.OK:
        raise S.SSSPError(rc, S.last_error())


def run(state):
    kind = state["kind"]
    if kind == "solve":
        d, st = state["graph"].solve(state["source"], state["schedule"])
        return {"distances": d, "reached": st["reached"]}
    if kind == "bfs":
        visited, levels, st = state["graph"].bfs(state["source"], state["schedule"])
        return {"visited": visited, "levels": levels, "reached": st["reached"]}
    if kind == "batch":
        d, _ = state["graph"].solve_batch(state["sources"])
        return {"distances": d}
    if kind == "pack":
        d, _ = state["pack"].solve(state["sources"])
        return {"distances": d}
    if kind == "wrapper":
        L, V, t = S.lib(), state["V"], state["dtype"]
        p = ctypes.c_void_p
        dist = p(state["dist"].data_ptr())
        _check(getattr(L, "sssp_init_distances_" + t)(dist, V, state["source"]))
        _check(getattr(L, "sssp_bellman_ford_" + t)(
            p(state["src"].data_ptr()), p(state["dst"].data_ptr()), p(state["w"].data_ptr()), V,
            state["src"].numel(), state["source"], dist, None))
        return {"distances": state["dist"]}
    with S.DeviceGraph(state["src"], state["dst"], state["w"], state["V"]) as g:
        d, st = g.solve(state["source"], state["schedule"])
    return {"distances": d, "reached": st["reached"]}


# ---- what a pass cannot do without ------------------------------------------
def _counts(case):
    if case["kind"] == "pack":
        V = int((1 << _pack_scales(case).astype(np.int64)).sum())
        return V, V * case["ef"]
    if case["graph"] == "rmat":
        return 1 << case["scale"], case["ef"] << case["scale"]
    if case["graph"] == "grid":
        R, C = case["rows"], case["cols"]
        return R * C, 2 * (R * (C - 1) + C * (R - 1))
    return case["V"], case["E"]


def work(case):
    """Each edge (two ids and a weight) read once, each result written once;
    one addition and one comparison per edge and source."""
    V, E = _counts(case)
    kind = case["kind"]
    n = case["n"] if kind == "batch" else 1
    edge, vertex = 12, 4 * n
    if kind == "bfs":
        edge, vertex = 8, 5
    if case.get("dtype") == "f64":
        edge, vertex = 16, 8
    return {"bytes": edge * E + vertex * V, "flops": 2 * E * n}


# ---- the same in 64 bits ------------------------------------------------------
def _bellman_ford64(src, dst, w, V, sources, unreached):
    d = torch.full((V,), math.inf, device="cuda", dtype=torch.float64)
    d[torch.as_tensor(sources, device="cuda", dtype=torch.int64)] = 0.0
    w = w.double()
    while True:
        cand = d[src] + w
        low = cand < d[dst]
        if not bool(low.any()):
            break
        d.scatter_reduce_(0, dst[low].long(), cand[low], "amin")
    return torch.where(torch.isinf(d), torch.full_like(d, unreached), d)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("bfs", "batch") or case.get("graph") == "uniform":
        return None  # whole numbers; or too many sources to solve this way
    if kind == "pack":
        s, t, w, offs, counts, sources = _pack_inputs(case, seed)
        base = np.concatenate([[0], np.cumsum(counts.astype(np.int64))])
        shift = np.repeat(base[:-1], np.diff(offs))
        d = _bellman_ford64(torch.from_numpy(s + shift).cuda(), torch.from_numpy(t + shift).cuda(),
                            torch.from_numpy(w).cuda(), int(base[-1]), base[:-1] + sources, F32_MAX)
        return {"distances": d}
    if _counts(case)[1] > 1 << 28:
        return None
    src, dst, w, V = _edges(case, seed)
    source = _source(case, seed, src)
    if kind == "wrapper":
        d = _bellman_ford64(src, dst, w, V, [source], F64_MAX if case["dtype"] == "f64" else F32_MAX)
        return {"distances": d}
    return {"distances": _bellman_ford64(src, dst, w, V, [source], F32_MAX), "reached": None}
