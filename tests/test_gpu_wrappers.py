"""GPU parity of the reference-shaped wrappers over caller-owned device arrays,
for the three weight types: init_distances_wrapper<W> and
bellman_ford_wrapper<W> (algorithm/sssp/gpu/bellman_ford.cu:38-144,
instantiated for float and double at :150-156; unsigned is the integer-weight
configuration). Results are compared bit for bit with the oracle's
cpu_bellman_ford restatement (sssp.hpp:3-71), itself pinned to the reference's
compiled code for float and double; unreached vertices must hold FLT_MAX,
DBL_MAX or 0xFFFFFFFF. The arrays are checked before any pass: bad ids and
negative or NaN weights give SSSP_ERR_ARG.
"""
import ctypes as C

import numpy as np
import pytest

import sssp_amd as S
from conftest import HipBuffer

DBL_MAX = np.finfo(np.float64).max
INF = {np.float32: S.F32_INF, np.float64: DBL_MAX, np.uint32: S.U32_INF}
SUFFIX = {np.float32: "f32", np.float64: "f64", np.uint32: "u32"}


def _graph(dtype):
    s, d, w32 = S.rmat(12, 16, seed=21, threads=64)
    rng = np.random.default_rng(5)
    if dtype == np.float32:
        w = w32
    elif dtype == np.float64:
        w = rng.random(len(s))  # full 53-bit doubles
        w[::97] = 0.0
    else:
        w = rng.integers(1, 256, len(s)).astype(np.uint32)
    return s, d, w, 1 << 12


def _bits(a):
    return a.view({4: np.uint32, 8: np.uint64}[a.itemsize])


def _run(lib, dtype, s, d, w, V, source):
    with HipBuffer(s) as ds, HipBuffer(d) as dd, HipBuffer(w) as dw, \
            HipBuffer(np.zeros(V, dtype)) as dist:
        k = SUFFIX[dtype]
        rc = getattr(lib, "sssp_init_distances_" + k)(dist.ptr, V, source)
        assert rc == S.OK, S.last_error()
        init = dist.get()
        passes = C.c_int32(0)
        rc = getattr(lib, "sssp_bellman_ford_" + k)(ds.ptr, dd.ptr, dw.ptr, V, len(s), source,
                                                     dist.ptr, C.byref(passes))
        assert rc == S.OK, S.last_error()
        return init, dist.get(), passes.value


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32], ids=["f32", "f64", "u32"])
def test_wrappers_match_oracle(gpu, lib, oracle, dtype):
    s, d, w, V = _graph(dtype)
    for source in (0, int(s[len(s) // 2])):
        print(f"wrapper {SUFFIX[dtype]} RMAT-12 ef16 source {source}", flush=True)
        init, got, passes = _run(lib, dtype, s, d, w, V, source)
        # init_distances_wrapper: the type's max everywhere but the source
        exp_init = np.full(V, INF[dtype], dtype)
        exp_init[source] = 0
        assert np.array_equal(_bits(init), _bits(exp_init))
        ref, ref_passes = oracle.bf(s, d, w, V, source)
        assert np.array_equal(_bits(got), _bits(ref))
        unreached = ref == INF[dtype]
        assert unreached.any() and (~unreached).sum() > 1
        assert np.all(_bits(got[unreached]) == _bits(np.array([INF[dtype]], dtype))[0])
        assert 1 <= passes <= V


@pytest.mark.gpu
def test_wrappers_reject_bad_arrays(gpu, lib):
    s, d, w, V = _graph(np.float32)
    bad_w = w.copy()
    bad_w[100] = -0.5
    nan_w = np.random.default_rng(1).random(len(s))
    nan_w[7] = np.nan
    bad_id = d.copy()
    bad_id[3] = V
    cases = [("f32 negative weight", np.float32, s, d, bad_w),
             ("f64 NaN weight", np.float64, s, d, nan_w),
             ("u32 id out of range", np.uint32, s, bad_id, np.ones(len(s), np.uint32))]
    for name, dtype, ss, dd_, ww in cases:
        print("wrapper rejects:", name, flush=True)
        with HipBuffer(ss) as a, HipBuffer(dd_) as b, HipBuffer(ww.astype(dtype)) as c, \
                HipBuffer(np.zeros(V, dtype)) as dist:
            k = SUFFIX[dtype]
            assert getattr(lib, "sssp_init_distances_" + k)(dist.ptr, V, 0) == S.OK
            rc = getattr(lib, "sssp_bellman_ford_" + k)(a.ptr, b.ptr, c.ptr, V, len(ss), 0,
                                                         dist.ptr, None)
            assert rc == S.ERR_ARG, name
            msg = S.last_error()
            assert ("weight" in msg) if "weight" in name else ("outside" in msg), msg
    with HipBuffer(s) as a, HipBuffer(bad_id) as b, HipBuffer(np.zeros(V, np.uint8)) as vis:
        assert lib.sssp_bfs_edges(a.ptr, b.ptr, V, len(s), vis.ptr, 0, None) == S.ERR_ARG


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32], ids=["f32", "f64", "u32"])
@pytest.mark.parametrize("V,E,shift", [(1, 3, 0), (65, (3 << 18) - 1, 0),
                                       (1, (3 << 18) + 3, 0), (65, 3 << 18, 1), (1 << 20, 3 << 20, 0), ((1 << 20) + 1, (3 << 20) + 2, 0),
                                       (3000000, 4000003, 1)])
def test_wrapper_change_bits(gpu, lib, oracle, dtype, V, E, shift):
    """The change bits of the wrappers' passes, on both sides of the edge count they
    start at: fewer vertices than a word,
    exactly as many as bits, one and many more (vertices share bits), edge
    counts off the vector width, arrays one element off their alignment; and
    a second call that goes on from distances the caller lowered. Bit
    equality with the oracle."""
    rng = np.random.default_rng(V + E)
    s = (rng.random(E) ** 2 * V).astype(np.int32)
    d = rng.integers(0, V, E).astype(np.int32)
    w = rng.integers(1, 256, E).astype(dtype) if dtype == np.uint32 else rng.random(E).astype(dtype)
    a, b = int(s[0]), int(s[-1])
    pad = [np.concatenate([x[:shift], x]) for x in (s, d, w)]
    k, size = SUFFIX[dtype], np.dtype(dtype).itemsize
    refs = [oracle.bf(s, d, w, V, x)[0] for x in (a, b)]
    with HipBuffer(pad[0]) as ds, HipBuffer(pad[1]) as dd, HipBuffer(pad[2]) as dw, \
            HipBuffer(np.zeros(V, dtype)) as dist:
        at = [C.c_void_p(C.cast(x.ptr, C.c_void_p).value + shift * n)
              for x, n in ((ds, 4), (dd, 4), (dw, size))]
        assert getattr(lib, "sssp_init_distances_" + k)(dist.ptr, V, a) == S.OK
        for source, ref in ((a, refs[0]), (b, np.minimum(*refs))):
            print(f"wrapper bits: {k} V {V} E {E} shift {shift} source {source}", flush=True)
            if source != a:
                one = C.c_void_p(C.cast(dist.ptr, C.c_void_p).value + source * size)
                assert getattr(lib, "sssp_init_distances_" + k)(one, 1, 0) == S.OK
            assert getattr(lib, "sssp_bellman_ford_" + k)(*at, V, E, source, dist.ptr,
                                                           None) == S.OK, S.last_error()
            assert np.array_equal(_bits(dist.get()), _bits(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("weights", ["random", "equal", "two", "mostly_zero"])
@pytest.mark.parametrize("ends", ["hubs", "even", "sparse"])
def test_wrapper_light_classes(gpu, lib, oracle, ends, weights):
    """Wrapper passes with a light class of a graph with hubs, of one without,
    and with none (few edges per vertex, equal weights, or too many of the
    lightest): bit equality with the oracle."""
    rng = np.random.default_rng(31)
    E = (3 << 18) + 5
    V = 200003 if ends == "sparse" else 40009
    s, d = ((rng.random(E) ** (4 if ends == "hubs" else 1) * V).astype(np.int32)
            for _ in range(2))
    w = {"random": rng.random(E), "equal": np.full(E, 0.25), "two": rng.integers(1, 3, E) / 4,
         "mostly_zero": np.where(rng.random(E) < 0.8, 0.0, rng.random(E))}[weights]
    w = w.astype(np.float32)
    source = int(s[0])
    print(f"wrapper light class: {ends}, {weights}", flush=True)
    _, got, passes = _run(lib, np.float32, s, d, w, V, source)
    assert np.array_equal(_bits(got), _bits(oracle.bf(s, d, w, V, source)[0]))
    assert 1 <= passes <= V


@pytest.mark.gpu
@pytest.mark.parametrize("order,V,E,routes", [
    ("random", 50000, (3 << 18) - 1, "0000"), ("random", 50000, 3 << 18, "1010"),
    ("random", 300000, 800000, "0000"), ("random", 50000, 15 << 17, "1110"),
    ("random", 70000, 45 << 16, "1111"), ("by_src", 50000, (15 << 17) - 1, "0000"),
    ("by_src", 50000, 15 << 17, "1010"), ("by_dst", 50000, 15 << 17, "1010"),
    ("by_src", 300000, (15 << 18) - 1, "0000"), ("by_dst", 300000, 15 << 18, "1010"),
    ("by_src", 300000, 15 << 19, "1111"), ("near", 300000, 15 << 19, "0000"),
    ("near_by_dst", 40000, 15 << 18, "0000"), ("near_shuffled", 70000, 15 << 18, "1111")])
def test_wrapper_route_follows_the_list(gpu, lib, oracle, order, V, E, routes):
    """Which passes a list gets (f32, f64, u32, hops; 1: over changed sources
    only), on both sides of every line: lists in random order, by source, by
    destination, and ordered ones between near ids, where the passes over every
    edge are the faster. Bit equality with the oracle on both routes."""
    rng = np.random.default_rng(E + V)
    s = rng.integers(0, V, E).astype(np.int32)
    if order.startswith("near"):
        d = np.clip(s + rng.integers(-200, 201, E), 0, V - 1).astype(np.int32)
        d[::100] = rng.integers(0, V, len(d[::100]))  # and a few far edges
    else:
        d = rng.integers(0, V, E).astype(np.int32)
    if not order.endswith(("random", "shuffled")):
        o = np.argsort(d if order.endswith("by_dst") else s, kind="stable")
        s, d = s[o], d[o]
    w = rng.integers(1, 256, E)
    source, route = int(s[E // 3]), C.c_int32(-1)
    ref = oracle.dijkstra(s, d, w.astype(np.uint32), V, source)
    far = ref == S.U32_INF
    with HipBuffer(s) as ds, HipBuffer(d) as dd:
        for k, dtype in enumerate((np.float32, np.float64, np.uint32)):
            print(f"wrapper route: {order} V {V} E {E} {SUFFIX[dtype]}", flush=True)
            _, got, passes = _run(lib, dtype, s, d, w.astype(dtype), V, source)
            assert lib.sssp_debug_wrapper_route(C.byref(route)) == S.OK
            # whole weights: distances stay exact in every type
            assert np.array_equal(got[~far], ref[~far].astype(dtype))
            assert np.all(got[far] == INF[dtype]) and 1 <= passes <= V
            assert route.value == int(routes[k]), SUFFIX[dtype]
        with HipBuffer(np.zeros(V, np.uint8)) as vis:
            print(f"wrapper route: {order} V {V} E {E} hops", flush=True)
            assert lib.sssp_bfs_edges(ds.ptr, dd.ptr, V, E, vis.ptr, source, None) == S.OK
            assert np.array_equal(vis.get(), (~far).astype(np.uint8))
        assert lib.sssp_debug_wrapper_route(C.byref(route)) == S.OK
        assert route.value == int(routes[3]), "hops"


@pytest.mark.gpu
@pytest.mark.parametrize("weights", ["random", "light_path", "heavy_path"])
def test_wrapper_passes_beyond_the_rings(gpu, lib, oracle, weights):
    """Passes over changed sources past number 64, where the light ones end and
    the rings of pass states wrap, several times over: a path of 300 hops, whose
    edges are light, heavy or mixed, in front of a random graph, listed in random
    order; f32, f64, u32 and hops. Bit equality with the oracle."""
    V, E, hops = 70000, 3000001, 300
    rng = np.random.default_rng(61)
    s, d = (rng.integers(hops, V, E).astype(np.int32) for _ in range(2))
    w = rng.integers(1, 256, E)
    at = rng.permutation(E)[:hops]
    s[at], d[at] = np.arange(hops), np.arange(1, hops + 1)
    if weights != "random":
        w[at] = 1 if weights == "light_path" else 255
    ref = oracle.dijkstra(s, d, w.astype(np.uint32), V, 0)
    far, route = ref == S.U32_INF, C.c_int32(0)
    for dtype in (np.float32, np.float64, np.uint32):
        print(f"wrapper past the rings: {weights} {SUFFIX[dtype]}", flush=True)
        _, got, passes = _run(lib, dtype, s, d, w.astype(dtype), V, 0)
        assert lib.sssp_debug_wrapper_route(C.byref(route)) == S.OK and route.value == 1
        assert np.array_equal(got[~far], ref[~far].astype(dtype))  # whole weights: exact
        assert np.all(got[far] == INF[dtype])
        # light passes follow a path of light edges for the first 64 passes at most
        assert hops - 64 <= passes <= V
    print(f"wrapper past the rings: {weights} hops", flush=True)
    with HipBuffer(s) as ds, HipBuffer(d) as dd, HipBuffer(np.zeros(V, np.uint8)) as vis:
        passes = C.c_int32(0)
        assert lib.sssp_bfs_edges(ds.ptr, dd.ptr, V, E, vis.ptr, 0, C.byref(passes)) == S.OK
        assert lib.sssp_debug_wrapper_route(C.byref(route)) == S.OK and route.value == 1
        assert np.array_equal(vis.get(), (~far).astype(np.uint8)) and passes.value >= hops
