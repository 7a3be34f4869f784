"""GPU parity: the HIP path (through the C ABI) against the CPU oracle.

Bar: bit-exact distances for f32 and u32 (the fixpoint of d[v] <= d[u] (+) w
is unique for w >= 0, so every schedule must land on the same bits as the
oracle's restatement of cpu_bellman_ford, sssp.hpp:3-71), plus the
shortest-path certificate (all edges satisfied, tight parent tree).
"""
import ctypes as C
import mmap

import numpy as np
import pytest

import sssp_amd as S
from conftest import bits, small_graphs

SCHEDS = ["plain", "heuristic", "learned", "push", "all", "pull"]


def _check_solution(g, oracle, src, dst, w, V, source, d, sched):
    ref = oracle.dijkstra(src, dst, w, V, source)
    assert np.array_equal(bits(d), bits(ref)), f"{sched}: distances differ from the oracle"
    ok, counts, par = g.certify(source)
    assert ok, f"{sched}: GPU certificate failed: {counts}"
    rc, oc = oracle.certify(src, dst, w, V, source, d, par)
    assert rc == 0, f"{sched}: oracle rejects the GPU parents/distances: {oc}"


@pytest.mark.gpu
def test_device_is_gfx950(gpu):
    info = S.device_info(0)
    print(info)
    assert info["arch"].startswith("gfx950")


@pytest.mark.gpu
@pytest.mark.parametrize("name,V,src,dst,w", small_graphs(), ids=[g[0] for g in small_graphs()])
def test_small_graphs_every_schedule(gpu, oracle, name, V, src, dst, w):
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        for sched in SCHEDS:
            d, st = g.solve(0, sched)
            _check_solution(g, oracle, src, dst, w, V, 0, d, sched)
        g.set_param("plain_kernel", 2)  # the plain pass over the blocked list too
        d, st = g.solve(0, "plain")
        _check_solution(g, oracle, src, dst, w, V, 0, d, "plain (blocked)")
    if name == "chain":
        assert np.array_equal(d, (np.arange(10) * np.float32(0.5)).astype(np.float32))
    if name == "disconnected":
        assert np.all(d[3:] == S.F32_INF)


@pytest.mark.gpu
def test_device_ingest_from_bin(gpu, oracle, tmp_path):
    """A graph streamed from the reference's binary file format equals the one
    built from the same arrays: layouts, and distances under every schedule."""
    src, dst, w = S.rmat(14, 16, seed=12, threads=8)
    V = 1 << 14
    p = tmp_path / "g.bin"
    S.save_bin(p, src, dst, w, V)
    with S.DeviceGraph.from_bin(p) as g1, S.DeviceGraph(src, dst, w, V) as g2:
        g1.set_param("plain_below_edges", 0)  # exercise the round engine
        g2.set_param("plain_below_edges", 0)  # exercise the round engine
        assert (g1.V, g1.E) == (V, len(src))
        L1, L2 = g1.layout(), g2.layout()
        for k in L1:
            assert np.array_equal(L1[k].view(np.uint8), L2[k].view(np.uint8)), k
        ref = oracle.dijkstra(src, dst, w, V, 3)
        for sched in SCHEDS:
            d, _ = g1.solve(3, sched)
            assert np.array_equal(bits(d), bits(ref)), sched
    su, tu, wu = S.er(1 << 12, 8, seed=5, weight_mode=1)
    pu = tmp_path / "u.bin"
    S.save_bin(pu, su, tu, wu, 1 << 12)
    with S.DeviceGraph.from_bin(pu, weight_dtype=np.uint32) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        d, _ = g.solve(0, "heuristic")
        assert np.array_equal(d, oracle.dijkstra(su, tu, wu, 1 << 12, 0))
    # several chunks (4 Mi records each) through the two pinned buffers
    s2, t2, w2 = S.rmat(20, 16, seed=13, threads=64)
    p2 = tmp_path / "big.bin"
    S.save_bin(p2, s2, t2, w2, 1 << 20)
    with S.DeviceGraph.from_bin(p2, csc=False) as g1, S.DeviceGraph(s2, t2, w2, 1 << 20, csc=False) as g2:
        g1.set_param("plain_below_edges", 0)  # exercise the round engine
        g2.set_param("plain_below_edges", 0)  # exercise the round engine
        a, _ = g1.solve(5, "plain")
        b, _ = g2.solve(5, "plain")
        assert np.array_equal(bits(a), bits(b))
        L1, L2 = g1.layout(csc=False), g2.layout(csc=False)
        assert np.array_equal(L1["el_dst"], L2["el_dst"])


@pytest.mark.gpu
@pytest.mark.parametrize("relabel", [True, False])
def test_layout_is_stable_sort(gpu, relabel):
    """The layouts are stable sorts of the edge list renamed into slots; slots
    rank the vertices by descending in- plus out-degree, then descending
    out-degree, then vertex id (the identity with relabel=False)."""
    src, dst, w = S.rmat(11, 16, seed=3, threads=4)
    V = 1 << 11
    with S.DeviceGraph(src, dst, w, V, relabel=relabel) as g:
        L = g.layout()
        order = g.vertex_order()
    if relabel:
        out = np.bincount(src, minlength=V)
        tot = out + np.bincount(dst, minlength=V)
        exp = np.empty(V, np.int32)
        exp[np.lexsort((np.arange(V), -out, -tot))] = np.arange(V, dtype=np.int32)
        assert np.array_equal(order, exp)
        assert not np.array_equal(order, np.arange(V))
    else:
        assert np.array_equal(order, np.arange(V))
    src, dst = order[src], order[dst]
    p = np.argsort(src, kind="stable")
    assert np.array_equal(L["el_src"], src[p])
    assert np.array_equal(L["el_dst"], dst[p])
    assert np.array_equal(bits(L["el_w"]), bits(w[p]))
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=V))])
    assert np.array_equal(L["row_ptr"], rp)
    q = np.argsort(dst, kind="stable")
    assert np.array_equal(L["csc_src"], src[q])
    assert np.array_equal(bits(L["csc_w"]), bits(w[q]))
    cp = np.concatenate([[0], np.cumsum(np.bincount(dst, minlength=V))])
    assert np.array_equal(L["col_ptr"], cp)


@pytest.mark.gpu
@pytest.mark.parametrize("relabel", [None, True], ids=["ids", "slots"])
@pytest.mark.parametrize("scale,ef,seed,threads", [(10, 16, 1, 64), (14, 16, 9, 64), (16, 16, 0, 1)])
def test_rmat_every_schedule_bit_exact(gpu, oracle, scale, ef, seed, threads, relabel):
    src, dst, w = S.rmat(scale, ef, seed=seed, threads=threads)
    V = 1 << scale
    sources = [0] + list(S.pick_sources(src, V, seed + 100, 3))
    with S.DeviceGraph(src, dst, w, V, relabel=relabel) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        for s in sources:
            ref, _ = oracle.bf(src, dst, w, V, s)
            for sched in SCHEDS:
                d, st = g.solve(s, sched)
                assert np.array_equal(bits(d), bits(ref)), (s, sched, st)
                assert st["reached"] == int((d != S.F32_INF).sum()), (s, sched, st)
            ok, counts, par = g.certify(s)
            assert ok, counts
            rc, oc = oracle.certify(src, dst, w, V, s, d, par)
            assert rc == 0, oc


@pytest.mark.gpu
@pytest.mark.parametrize("logV,deg", [(12, 16), (15, 8)])
def test_er_u32_bit_exact(gpu, oracle, logV, deg):
    V = 1 << logV
    src, dst, w = S.er(V, deg, seed=3, weight_mode=1)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        ref, _ = oracle.bf(src, dst, w, V, 0)
        dj = oracle.dijkstra(src, dst, w, V, 0)
        assert np.array_equal(ref, dj)
        for sched in SCHEDS:
            d, st = g.solve(0, sched)
            assert d.dtype == np.uint32
            assert np.array_equal(d, ref), sched
            assert st["reached"] == int((d != np.uint32(0xFFFFFFFF)).sum()), (sched, st)
        ok, counts, par = g.certify(0)
        assert ok, counts
        rc, oc = oracle.certify(src, dst, w, V, 0, d, par)
        assert rc == 0, oc


@pytest.mark.gpu
def test_edge_order_does_not_change_distances(gpu):
    src, dst, w = S.rmat(13, 16, seed=4, threads=8)
    V = 1 << 13
    perm = np.random.default_rng(0).permutation(len(src))
    with S.DeviceGraph(src, dst, w, V) as g1, S.DeviceGraph(src[perm], dst[perm], w[perm], V) as g2:
        g1.set_param("plain_below_edges", 0)  # exercise the round engine
        g2.set_param("plain_below_edges", 0)  # exercise the round engine
        for sched in ("plain", "heuristic"):
            a, _ = g1.solve(5, sched)
            b, _ = g2.solve(5, sched)
            assert np.array_equal(bits(a), bits(b))


@pytest.mark.gpu
def test_repeat_solves_reuse_graph(gpu, oracle):
    """Stamps and ticks carry across solves on one graph; results must not."""
    src, dst, w = S.rmat(12, 8, seed=7, threads=8)
    V = 1 << 12
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        for s in [0, 1, 2, 0, 3]:
            for sched in ("push", "all", "pull", "heuristic"):
                d, _ = g.solve(s, sched)
                ref = oracle.dijkstra(src, dst, w, V, s)
                assert np.array_equal(bits(d), bits(ref))


@pytest.mark.gpu
def test_verify_pass_and_trace(gpu):
    src, dst, w = S.rmat(12, 16, seed=2, threads=8)
    with S.DeviceGraph(src, dst, w, 1 << 12) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        g.set_param("trace_events", 1)
        d, st = g.solve(0, "heuristic")
        tr = g.trace()
        assert st["verify_passes"] >= 1
        assert tr["mode"][-1] == S.MODE_VERIFY
        assert len(tr["mode"]) == st["iterations"]
        assert st["t_solve_ms"] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("tail_edges,group", [(1 << 14, 4), (1 << 14, 1), (64, 4), (64, 3)])
def test_tail_rounds_bit_exact(gpu, oracle, tail_edges, group):
    """Tail rounds (push rounds queued without a decision or host round trip
    between them, entry lists built in one pass) land on the oracle's
    fixpoint: f32 R-MAT (several sources, heuristic and learned), u32 ER and
    BFS levels. A bound of 64 out-edges makes the frontier cross it again and
    again (tail runs that stop and resume); group 1 runs under trace_events
    (one round per host check, each timed)."""
    src, dst, w = S.rmat(16, 16, seed=13, threads=8)
    V = 1 << 16
    sources = [0] + list(S.pick_sources(src, V, 131, 3))
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        g.set_param("tail_edges", tail_edges)
        g.set_param("tail_group", group)
        g.set_param("trace_events", 1 if group == 1 else 0)
        tails = 0
        for s in sources:
            for sched in ("heuristic", "learned"):
                print(f"tail rounds: rmat16 f32 source {s} {sched} tail_edges {tail_edges} "
                      f"group {group}", flush=True)
                d, st = g.solve(int(s), sched)
                assert np.array_equal(bits(d), bits(oracle.dijkstra(src, dst, w, V, int(s)))), \
                    (s, sched)
                tr = g.trace()
                assert len(tr["mode"]) == st["iterations"]
                assert tr["mode"][-1] == S.MODE_VERIFY
                k = tr["mode"] == S.MODE_TAIL
                tails += int(k.sum())
                if group == 1 and k.any():
                    assert (tr["frontier"][k] > 0).all() and (tr["ms"][k] > 0).all()
                    assert (tr["frontier_edges"][k] <= tail_edges).all()
        assert tails > 0, "no tail rounds ran"
        ok, counts, par = g.certify(int(sources[-1]))
        assert ok, counts
        print(f"tail rounds: rmat16 BFS tail_edges {tail_edges} group {group}", flush=True)
        vis, lev, st = g.bfs(int(sources[1]), "heuristic")
        rvis, rlev, _ = oracle.bfs(src, dst, V, int(sources[1]))
        assert np.array_equal(lev, rlev) and np.array_equal(vis.view(np.uint8), rvis)
    V = 1 << 15
    src, dst, w = S.er(V, 8, seed=17, weight_mode=1)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)
        g.set_param("tail_edges", tail_edges)
        g.set_param("tail_group", group)
        print(f"tail rounds: er15 u32 tail_edges {tail_edges} group {group}", flush=True)
        d, st = g.solve(5, "heuristic")
        assert np.array_equal(d, oracle.dijkstra(src, dst, w, V, 5))


@pytest.mark.gpu
def test_push_rounds_with_frontier_bitmap(gpu, oracle):
    """Push rounds that mark their lowered vertices in a bitmap and queue them
    in one pass (push_bits_edges) land on the oracle's fixpoint: f32 R-MAT with
    the push-only, heuristic and learned schedules (tail rounds on and off),
    u32 ER, BFS levels."""
    src, dst, w = S.rmat(16, 16, seed=31, threads=8)
    V = 1 << 16
    sources = [0] + list(S.pick_sources(src, V, 311, 3))
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        g.set_param("push_bits_edges", 1)    # every push round
        for tail in (0, 1 << 14):
            g.set_param("tail_edges", tail)
            for s in sources:
                for sched in ("push", "heuristic", "learned"):
                    print(f"bitmap push rounds: rmat16 source {s} {sched} tail {tail}", flush=True)
                    d, st = g.solve(int(s), sched)
                    assert np.array_equal(bits(d), bits(oracle.dijkstra(src, dst, w, V, int(s)))), \
                        (s, sched, tail)
        ok, counts, par = g.certify(int(sources[-1]))
        assert ok, counts
        print("bitmap push rounds: rmat16 BFS", flush=True)
        vis, lev, _ = g.bfs(int(sources[1]), "push")
        rvis, rlev, _ = oracle.bfs(src, dst, V, int(sources[1]))
        assert np.array_equal(lev, rlev)
    V = 1 << 15
    src, dst, w = S.er(V, 8, seed=37, weight_mode=1)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)
        g.set_param("push_bits_edges", 1)
        print("bitmap push rounds: er15 u32", flush=True)
        for sched in ("push", "heuristic"):
            d, st = g.solve(9, sched)
            assert np.array_equal(d, oracle.dijkstra(src, dst, w, V, 9)), sched


@pytest.mark.gpu
@pytest.mark.parametrize("scale,ef,seed,threads", [(12, 16, 3, 64), (16, 16, 0, 1), (18, 8, 11, 7)])
def test_device_rmat_generator_matches_host(gpu, scale, ef, seed, threads):
    s, d, w = S.rmat(scale, ef, seed=seed, threads=threads)
    g, (ds, dd, dw) = S.DeviceGraph.rmat(scale, ef, seed=seed, threads=threads, download_edges=True)
    try:
        assert np.array_equal(ds, s) and np.array_equal(dd, d)
        assert np.array_equal(bits(dw), bits(w))
        L = g.layout()
    finally:
        g.close()
    with S.DeviceGraph(s, d, w, 1 << scale) as h:
        h.set_param("plain_below_edges", 0)  # exercise the round engine
        M = h.layout()
    for k in ("row_ptr", "el_src", "el_dst", "col_ptr", "csc_src"):
        assert np.array_equal(L[k], M[k]), k


# ---------------------------------------------------------------- batches
@pytest.mark.gpu
@pytest.mark.parametrize("policy", [1, 2, 3])
def test_batch_sources_match_single_solves(gpu, oracle, policy):
    src, dst, w = S.rmat(13, 16, seed=21, threads=16)
    V = 1 << 13
    sources = S.pick_sources(src, V, 21, 48)
    with S.DeviceGraph(src, dst, w, V, relabel=True) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        D, st = g.solve_batch(sources, policy=policy)
        assert D.shape == (48, V) and st["t_solve_ms"] > 0
        for i in (0, 7, 47):
            ref, _ = oracle.bf(src, dst, w, V, int(sources[i]))
            assert np.array_equal(bits(D[i]), bits(ref))
        for i in range(48):
            d, _ = g.solve(int(sources[i]), "push")
            assert np.array_equal(bits(D[i]), bits(d)), i
        # replay of the captured launch with other sources
        s2 = sources[::-1].copy()
        D2, _ = g.solve_batch(s2, policy=policy)
        assert np.array_equal(bits(D2[0]), bits(D[-1]))


@pytest.mark.gpu
def test_batch_captured_launch_replays(gpu, oracle):
    """Policy 3 runs each chunk of sources as captured hipGraph launches (change
    flags and pass base cleared by a kernel, init, runs of 32 passes reading
    their pass number from the device, transposed output). Three replays with
    other sources, eager solves between them: each bit-equal to the passes
    queued from the host and to policy 1 (a workgroup per source)."""
    src, dst, w = S.rmat(14, 16, seed=41, threads=16)
    V = 1 << 14
    with S.DeviceGraph(src, dst, w, V, relabel=True) as g:
        for k in range(3):
            sources = S.pick_sources(src, V, 41 + k, 64)
            print(f"captured batch replay {k}: 64 sources, RMAT-14", flush=True)
            g.set_param("batch_capture", 1)
            D, _ = g.solve_batch(sources, policy=3)
            assert g.get_param("multi_passes") >= 1
            d, _ = g.solve(int(sources[k]), "heuristic")
            assert np.array_equal(bits(D[k]), bits(d))
            g.set_param("batch_capture", 0)
            D0, _ = g.solve_batch(sources, policy=3)
            assert np.array_equal(bits(D), bits(D0))
            D1, _ = g.solve_batch(sources, policy=1)
            assert np.array_equal(bits(D), bits(D1))
        ref, _ = oracle.bf(src, dst, w, V, int(sources[5]))
        assert np.array_equal(bits(D[5]), bits(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [1, 2], ids=["edge_list", "blocked"])
def test_plain_solve_queued_and_traced(gpu, oracle, kernel):
    """The plain schedule queues its passes four at a time (change flags tested
    on the device); with trace_events each pass is launched alone between
    events. Same distances; the traced solve records one row per pass, the
    last one a pass that changed nothing; a pass cap below the fixpoint gives
    up and leaves the graph usable. Both plain pass kernels."""
    src, dst, w = S.rmat(15, 16, seed=42, threads=16)
    V = 1 << 15
    ref = oracle.dijkstra(src, dst, w, V, 7)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_kernel", kernel)
        assert g.get_param("plain_blocked") == (kernel == 2)
        d, st = g.solve(7, "plain")
        assert np.array_equal(bits(d), bits(ref))
        assert 2 <= st["iterations"] <= V + 1 and st["verify_passes"] == 1
        g.set_param("trace_events", 1)
        d2, st2 = g.solve(7, "plain")
        g.set_param("trace_events", 0)
        assert np.array_equal(bits(d2), bits(ref))
        tr = g.trace()
        assert len(tr["ms"]) == st2["iterations"] and np.all(tr["ms"] > 0)
        # a plain solve capped below its pass count gives up, then solves again
        g.set_param("max_rounds", 1)
        with pytest.raises(S.SSSPError) as e:
            g.solve(7, "plain")
        assert e.value.code == S.ERR_NOT_CONVERGED
        g.set_param("max_rounds", 100000)
        d3, _ = g.solve(7, "plain")
        assert np.array_equal(bits(d3), bits(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [1, 2], ids=["edge_list", "blocked"])
def test_plain_kernels_bit_exact(gpu, oracle, kernel):
    """The plain schedule on either pass kernel -- the XCD-partitioned edge
    list, or the destination-blocked list (block minima in LDS, atomicMin
    write-backs for blocks split over several tiles) -- ends on the oracle's
    fixpoint: f32 with vertex ids and with degree-ordered slots, u32, BFS
    levels, and a graph whose hub block is split, with tiles down to 256
    edges."""
    src, dst, w = S.rmat(14, 16, seed=9, threads=64)
    V = 1 << 14
    sources = [0] + list(S.pick_sources(src, V, 109, 3))
    for relabel in (None, True):
        with S.DeviceGraph(src, dst, w, V, relabel=relabel) as g:
            g.set_param("plain_kernel", kernel)
            for s in sources:
                print(f"plain kernel {kernel}: rmat14 relabel {relabel} source {s}", flush=True)
                ref, _ = oracle.bf(src, dst, w, V, s)
                d, st = g.solve(s, "plain")
                assert np.array_equal(bits(d), bits(ref)), (s, st)
                assert st["verify_passes"] == 1
                ok, counts, _ = g.certify(s, parents=False)
                assert ok, counts
    V = 1 << 15
    src, dst, wu = S.er(V, 8, seed=3, weight_mode=1)
    with S.DeviceGraph(src, dst, wu, V) as g:
        g.set_param("plain_kernel", kernel)
        print(f"plain kernel {kernel}: er15 u32", flush=True)
        d, _ = g.solve(0, "plain")
        assert np.array_equal(d, oracle.dijkstra(src, dst, wu, V, 0))
    scale = 17
    src, dst, w = S.rmat(scale, 16, seed=44, threads=16)
    V = 1 << scale
    assert np.bincount(dst >> 14).max() > (1 << 19)  # the hub block is split
    with S.DeviceGraph(src, dst, w, V, relabel=True) as g:
        g.set_param("plain_kernel", kernel)
        for cap in (256, 1 << 17):
            g.set_param("blk_tile_cap", cap)
            for s in (0, int(src[999])):
                print(f"plain kernel {kernel}: rmat17 split blocks, cap {cap}, source {s}", flush=True)
                d, _ = g.solve(s, "plain")
                assert np.array_equal(bits(d), bits(oracle.dijkstra(src, dst, w, V, s))), (cap, s)
                _, lev, _ = g.bfs(s, "plain")
                assert np.array_equal(lev, oracle.bfs(src, dst, V, s)[1]), (cap, s)


@pytest.mark.gpu
def test_blocked_list_wide_chunks(gpu, oracle):
    """The blocked list packs each source as a delta to the previous edge of
    its 256-edge chunk; a chunk with a gap of 2^18 or more keeps its sources
    whole. A sparse graph on 2^20 vertices (few in-edges per block, sources
    far apart) has such chunks next to packed ones; the plain blocked pass,
    the dense rounds and BFS stay exact on both."""
    V = 1 << 20
    rng = np.random.default_rng(5)
    n = 1500
    src = rng.integers(0, V, n).astype(np.int32)
    dst = rng.integers(0, V, n).astype(np.int32)
    hop = np.sort(rng.choice(V, 400, replace=False)).astype(np.int32)  # a long path
    src = np.concatenate([src, hop[:-1], np.full(300, 7, np.int32)])
    dst = np.concatenate([dst, hop[1:], rng.integers(0, 1 << 14, 300).astype(np.int32)])
    w = rng.random(len(src), dtype=np.float32)
    with S.DeviceGraph(src, dst, w, V, relabel=False) as g:
        nw = g.get_param("blk_wide_chunks")
        print(f"wide chunks: {nw} of {g.get_param('blk_tiles')} tiles", flush=True)
        assert nw > 0
        g.set_param("plain_kernel", 2)
        g.set_param("plain_below_edges", 0)
        g.set_param("dense_all_frac", 0.0)  # every all-edge round dense
        for s in (int(hop[0]), 7, int(src[3])):
            ref = oracle.dijkstra(src, dst, w, V, s)
            for sched in ("plain", "all", "heuristic", "learned"):
                d, _ = g.solve(s, sched)
                assert np.array_equal(bits(d), bits(ref)), (s, sched)
            _, lev, _ = g.bfs(s, "all")
            assert np.array_equal(lev, oracle.bfs(src, dst, V, s)[1]), s


@pytest.mark.gpu
def test_blocked_tiles_by_source_range(gpu, oracle):
    """Tiles cut by source range and dispatched range by range (blk_range_bits):
    the default for a graph without hubs from 2^22 vertices (8 ranges), off for
    R-MAT; any range size keeps the dense rounds and the plain blocked pass on
    the oracle's fixpoint, f32 and u32."""
    V = 1 << 20
    src, dst, w = S.er(V, 4, seed=6, weight_mode=0)
    wu = (np.arange(len(src)) % 255 + 1).astype(np.uint32)
    with S.DeviceGraph(src, dst, w, V) as g, S.DeviceGraph(src, dst, wu, V) as gu:
        assert g.get_param("blk_range_bits") == 0  # below 2^22 vertices
        ref = oracle.dijkstra(src, dst, w, V, 5)
        refu = oracle.dijkstra(src, dst, wu, V, 5)
        for h in (g, gu):
            h.set_param("plain_below_edges", 0)
            h.set_param("dense_all_frac", 0.0)  # every all-edge round dense
            h.set_param("plain_kernel", 2)
        for rb in (18, 19, 20, 0):
            print(f"source ranges of 2^{rb}", flush=True)
            for h in (g, gu):
                h.set_param("blk_range_bits", rb)
            assert g.get_param("blk_range_bits") == rb
            for sched in ("all", "plain", "heuristic"):
                d, _ = g.solve(5, sched)
                assert np.array_equal(bits(d), bits(ref)), (rb, sched)
            du, _ = gu.solve(5, "all")
            assert np.array_equal(du, refu), rb
        for bad in (5, 17, 32):
            with pytest.raises(S.SSSPError):
                g.set_param("blk_range_bits", bad)
    V = 1 << 22
    src, dst, w = S.er(V, 2, seed=7, weight_mode=0)
    with S.DeviceGraph(src, dst, w, V) as g:
        assert g.get_param("blk_range_bits") == 19  # 8 ranges of 2^19 vertices
        d, _ = g.solve(0, "plain")
        assert np.array_equal(bits(d), bits(oracle.dijkstra(src, dst, w, V, 0)))
    src, dst, w = S.rmat(16, 16, seed=1, threads=8)
    with S.DeviceGraph(src, dst, w, 1 << 16) as g:
        assert g.get_param("blk_range_bits") == 0


@pytest.mark.gpu
def test_plain_kernel_choice(gpu):
    """plain_kernel 0 picks the blocked pass once the blocked list has 64
    tiles or more (here forced by a small tile cap), else the edge-list
    pass; 1 and 2 force either; other values are rejected."""
    src, dst, w = S.rmat(14, 16, seed=9, threads=64)
    with S.DeviceGraph(src, dst, w, 1 << 14) as g:
        assert g.get_param("plain_kernel") == 0
        assert g.get_param("blk_tiles") < 64 and g.get_param("plain_blocked") == 0
        g.set_param("blk_tile_cap", 2048)
        assert g.get_param("blk_tiles") >= 64 and g.get_param("plain_blocked") == 1
        g.set_param("plain_kernel", 1)
        assert g.get_param("plain_blocked") == 0
        for bad in (-1, 3):
            with pytest.raises(S.SSSPError):
                g.set_param("plain_kernel", bad)


@pytest.mark.gpu
def test_blocked_tiles_any_cap_and_order(gpu, oracle):
    """The dense rounds' tile table rebuilt with other caps (edges per tile,
    down to 256: most blocks split over several workgroups) and dispatch
    orders: every dense round still ends on the oracle's fixpoint."""
    src, dst, w = S.rmat(14, 16, seed=43, threads=16)
    V = 1 << 14
    ref = oracle.dijkstra(src, dst, w, V, 3)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)
        g.set_param("dense_all_frac", 0.0)  # every all-edge round dense
        for cap, order in ((256, 0), (1024, 1), (4096, 2), (1 << 20, 3), (1 << 17, 0)):
            print(f"blocked tiles: cap {cap}, order {order}", flush=True)
            g.set_param("blk_tile_cap", cap)
            g.set_param("blk_tile_order", order)
            assert g.get_param("blk_tile_cap") == cap and g.get_param("blk_tile_order") == order
            for sched in ("all", "heuristic"):
                d, _ = g.solve(3, sched)
                assert np.array_equal(bits(d), bits(ref)), (cap, order, sched)
        for name, bad in (("blk_tile_cap", 1002), ("blk_tile_cap", 128), ("blk_tile_order", 4)):
            with pytest.raises(S.SSSPError):
                g.set_param(name, bad)


@pytest.mark.gpu
@pytest.mark.parametrize("V,E,relabel", [(1, 8192, False), (256, 8191, False), (257, 8193, False),
                                         (40000, 3, False), (65537, 16385, True),
                                         (70001, 100003, False)])
def test_layouts_at_the_edges_of_the_sort_tiles(gpu, oracle, V, E, relabel):
    """Edge counts around the sort's tiles of 8192, one digit against two and
    three, empty digits, and edges that pile up in one digit: solves over every
    layout the sorts build (out-edges, in-edges, blocked list, XCD groups,
    batch records) end on the oracle's fixpoint. Bit equality."""
    rng = np.random.default_rng(V + E)
    src = (rng.random(E) ** 4 * V).astype(np.int32)
    dst = np.where(rng.random(E) < 0.5, V - 1, rng.integers(0, V, E)).astype(np.int32)
    w = rng.random(E, dtype=np.float32)
    sources = [int(x) for x in src[:3]]
    refs = [oracle.dijkstra(src, dst, w, V, x) for x in sources]
    with S.DeviceGraph(src, dst, w, V, relabel=relabel) as g:
        g.set_param("plain_below_edges", 0)
        g.set_param("dense_all_frac", 0.0)
        for sched, kernel in (("push", 0), ("pull", 0), ("all", 0), ("plain", 1), ("plain", 2)):
            print(f"layouts: V {V} E {E} relabel {relabel}, {sched} {kernel}", flush=True)
            g.set_param("plain_kernel", kernel)
            d, _ = g.solve(sources[0], sched)
            assert np.array_equal(bits(d), bits(refs[0])), (sched, kernel)
        got = g.solve_batch(np.array(sources, np.int32), policy=3)[0]
        for x, ref in zip(got, refs):
            assert np.array_equal(bits(x), bits(ref))


def _local_graph(case, rng):
    """Edges between near ids, no hubs, fewer than 8 per vertex."""
    if case in ("grid", "grid_u32", "grid_zero"):
        r, c = 173, 97  # 16781 vertices: one past the first block's rows
        v = np.arange(r * c, dtype=np.int32).reshape(r, c)
        a = np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()])
        b = np.concatenate([v[:, 1:].ravel(), v[1:].ravel()])
        return r * c, np.concatenate([a, b]), np.concatenate([b, a])
    if case == "path":  # against the ids, then on with them: tiles wake each other
        a = np.arange(30000, 0, -1, dtype=np.int32)
        return 60002, np.concatenate([a, [0], np.arange(30001, 60001)]), np.concatenate(
            [a - 1, [30001], np.arange(30002, 60002)])
    if case == "one_edge":
        return 7, np.array([3]), np.array([5])
    if case == "tile_edges":  # one block: a tile of 8192 slots, and one of one chunk
        V, E, span = 3000, 8193, 80
    else:  # "band": near ids with far jumps, some of them over whole chunks of gaps
        V, E, span = 600000, 1200000, 900
    s = rng.integers(0, V, E)
    d = np.clip(s + rng.integers(-span, span + 1, E), 0, V - 1)
    if case == "band":
        d[::50] = rng.integers(0, V, len(d[::50]))
    return V, s, d


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["grid", "grid_u32", "grid_zero", "path", "one_edge",
                                  "tile_edges", "band"])
def test_local_passes_bit_exact(gpu, oracle, case):
    """Graphs of near ids (local passes: tiles relaxed several times a pass, and
    only when a source changed) end on the oracle's fixpoint, for weights,
    zero weights, u32 and hops, from sources in the first, a middle and the
    last block, twice each (no state outlives a solve). Bit equality."""
    rng = np.random.default_rng(23)
    V, src, dst = _local_graph(case, rng)
    src, dst = src.astype(np.int32), dst.astype(np.int32)
    w = rng.random(len(src), dtype=np.float32)
    if case == "grid_u32":
        w = rng.integers(1, 256, len(src)).astype(np.uint32)
    elif case == "grid_zero":
        w[rng.random(len(src)) < 0.5] = 0
    with S.DeviceGraph(src, dst, w, V) as g:
        for source in (int(src[0]), V // 2, V - 1):
            ref = oracle.dijkstra(src, dst, w, V, source)
            for sched in ("heuristic", "learned", "heuristic"):
                print(f"local passes: {case}, source {source}, {sched}", flush=True)
                d, st = g.solve(source, sched)
                assert np.array_equal(bits(d), bits(ref)), (case, source, sched)
            hops = oracle.dijkstra(src, dst, np.ones(len(src), np.uint32), V, source)
            lv = g.bfs(source, "heuristic")[1]
            assert np.array_equal(lv, hops)
        if case in ("grid", "path"):
            d, plain = g.solve(int(src[0]), "plain")
            st = g.solve(int(src[0]), "heuristic")[1]
            assert st["iterations"] * 2 < plain["iterations"]


@pytest.mark.gpu
@pytest.mark.parametrize("V,E,kind", [(1, 1, "f32"), (64, 255, "f32"), (65, 256, "u32"),
                                      (2000, 8192, "f32"), (1 << 15, 8193, "u32"),
                                      (2000, 16384, "relabel"), (2000, 16385, "f32"),
                                      (1 << 15, 32768, "f32"), (2000, 32769, "f32"),
                                      (1 << 15, 1 << 17, "f32"), (1 << 15, (1 << 17) + 1, "f32"),
                                      ((1 << 15) + 1, 1 << 17, "f32"), (1 << 15, 100003, "relabel"),
                                      (300, 70001, "ties"), (2001, 0, "f32")])
def test_graphs_solved_whole_in_lds(gpu, oracle, V, E, kind):
    """Both sides of the sizes up to which a single solve runs in one
    workgroup, chunk remainders, a relabelled graph, no edges, hops, and a
    round limit below what the solve needs. Bit equality with the oracle."""
    rng = np.random.default_rng(V + E)
    src = (rng.random(E) ** 2 * V).astype(np.int32)
    dst = rng.integers(0, V, E).astype(np.int32)
    w = rng.integers(1, 256, E).astype(np.uint32) if kind == "u32" else rng.random(E, np.float32)
    if kind == "ties":
        w = np.full(E, 0.5, np.float32)
    with S.DeviceGraph(src, dst, w, V, relabel=kind == "relabel") as g:
        for source in sorted({int(src[0]) if E else 0, V - 1}):
            ref = oracle.dijkstra(src, dst, w, V, source)
            hops = oracle.dijkstra(src, dst, np.ones(E, np.uint32), V, source)
            for sched in ("heuristic", "learned", "plain"):
                print(f"in LDS: V {V} E {E} {kind}, source {source}, {sched}", flush=True)
                d, st = g.solve(source, sched)
                assert np.array_equal(bits(d), bits(ref)), sched
                assert st["reached"] == (ref != S.U32_INF if kind == "u32"
                                         else ref != S.F32_INF).sum()
                assert st["iterations"] >= 1 and st["verify_passes"] == 1
            assert np.array_equal(g.bfs(source, "heuristic")[1], hops)
            assert np.array_equal(bits(g.solve(source)[0]), bits(g.distances()))
        if V == 64:
            path = S.DeviceGraph(np.arange(63, dtype=np.int32), np.arange(1, 64, dtype=np.int32),
                                 np.ones(63, np.float32), 64)
            with path:
                path.set_param("max_rounds", 1)
                with pytest.raises(S.SSSPError):
                    path.solve(0, "heuristic")
                path.set_param("max_rounds", 1000)
                assert path.solve(0, "heuristic")[0][63] == 63


@pytest.mark.gpu
def test_tile_order_by_count(gpu, oracle):
    """More tiles than run at once are dispatched largest first (the plain
    schedule's smallest first), fewer smallest first, unless the caller set an
    order; all end on the oracle's fixpoint."""
    src, dst, w = S.rmat(14, 16, seed=47, threads=16)
    V = 1 << 14
    ref = oracle.dijkstra(src, dst, w, V, 5)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_kernel", 2)
        for cap, order in ((1 << 17, 0), (256, 2), (512, 0), (256, 2)):
            g.set_param("blk_tile_cap", cap)
            print(f"tile order: cap {cap}, {g.get_param('blk_tiles')} tiles", flush=True)
            assert (g.get_param("blk_tiles") > 512) == (order == 2)
            assert g.get_param("blk_tile_order") == order
            for below in (2.0 ** 26, 0.0):
                g.set_param("plain_below_edges", below)
                for sched in ("heuristic", "plain"):
                    assert np.array_equal(bits(g.solve(5, sched)[0]), bits(ref)), (cap, sched)
        g.set_param("blk_tile_order", 1)
        g.set_param("blk_tile_cap", 1024)
        assert g.get_param("blk_tile_order") == 1


@pytest.mark.gpu
@pytest.mark.parametrize("E,cap", [(1, 1 << 13), (1 << 22, 1 << 13), ((1 << 22) + 1, 1 << 14),
                                   (1 << 23, 1 << 14), ((1 << 23) + 1, 1 << 15)])
def test_default_tile_cap(gpu, oracle, E, cap):
    """The tile cap a graph gets by its edge count, on both sides of a step of
    the rule and of the size up to which light passes wait for a full pass
    that changed much: every schedule ends on the oracle's fixpoint (bits)."""
    rng = np.random.default_rng(5)
    V = 70001
    src = (rng.random(E) ** 3 * V).astype(np.int32)
    dst = (rng.random(E) ** 2 * V).astype(np.int32)
    w = rng.random(E, dtype=np.float32)
    source = int(src[0])
    ref = oracle.dijkstra(src, dst, w, V, source)
    with S.DeviceGraph(src, dst, w, V) as g:
        assert g.get_param("blk_tile_cap") == cap
        for sched in ("heuristic", "learned", "plain"):
            print(f"default tile cap: E {E}, {sched}", flush=True)
            d, _ = g.solve(source, sched)
            assert np.array_equal(bits(d), bits(ref)), sched


@pytest.mark.gpu
def test_batch_u32(gpu, oracle):
    src, dst, w = S.er(1 << 12, 8, seed=4, weight_mode=1)
    V = 1 << 12
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        D, _ = g.solve_batch(np.array([0, 5, 9], np.int32), policy=1)
        for i, s in enumerate((0, 5, 9)):
            assert np.array_equal(D[i], oracle.dijkstra(src, dst, w, V, s))


@pytest.mark.gpu
def test_batch_vertex_major_chunks_and_u32(gpu, oracle):
    """Policy 3 (vertex-major all-edge passes) in chunks of 256 sources: 300
    sources on an R-MAT graph with split blocks (a hub block with more than
    4096 in-edges), repeated sources, and integer weights."""
    src, dst, w = S.rmat(12, 16, seed=23, threads=8)
    V = 1 << 12
    assert np.bincount(dst >> 4).max() > 4096  # at least one split (16-vertex) block
    sources = np.concatenate([S.pick_sources(src, V, 23, 290), np.zeros(10, np.int32)])
    with S.DeviceGraph(src, dst, w, V) as g:
        D, st = g.solve_batch(sources, policy=3)
        assert D.shape == (300, V) and st["t_solve_ms"] > 0
        D1, _ = g.solve_batch(sources, policy=1)
        assert np.array_equal(bits(D), bits(D1))
        for i in (0, 255, 256, 299):
            assert np.array_equal(bits(D[i]), bits(oracle.dijkstra(src, dst, w, V, int(sources[i])))), i
    su, tu, wu = S.er(1 << 12, 8, seed=4, weight_mode=1)
    with S.DeviceGraph(su, tu, wu, 1 << 12) as g:
        D, _ = g.solve_batch(np.array([0, 5, 9], np.int32), policy=3)
        for i, s in enumerate((0, 5, 9)):
            assert np.array_equal(D[i], oracle.dijkstra(su, tu, wu, 1 << 12, s))


def _pack_case(n, seed):
    rng = np.random.default_rng(seed)
    scales = rng.integers(4, 11, n).astype(np.int32)
    s, d, w, offs = S.rmat_many(scales, 8, seed0=seed)
    vcounts = (1 << scales).astype(np.int32)
    srcs = np.array([int(s[offs[k]]) for k in range(n)], np.int32)  # a vertex with out-edges
    return scales, s, d, w, offs, vcounts, srcs


@pytest.mark.gpu
@pytest.mark.parametrize("policy", [1, 2])
def test_pack_matches_per_graph_oracle(gpu, oracle, policy):
    scales, s, d, w, offs, vc, srcs = _pack_case(40, 3)
    p = S.GraphPack(s, d, w, offs, vc)
    try:
        D, st = p.solve(srcs, policy=policy)
    finally:
        p.close()
    voff = np.concatenate([[0], np.cumsum(vc)])
    for k in range(40):
        e0, e1 = offs[k], offs[k + 1]
        ref, _ = oracle.bf(s[e0:e1], d[e0:e1], w[e0:e1], int(vc[k]), int(srcs[k]))
        assert np.array_equal(bits(D[voff[k]:voff[k + 1]]), bits(ref)), k


@pytest.mark.gpu
def test_autotune_batch_and_pack(gpu, tmp_path):
    src, dst, w = S.rmat(12, 8, seed=2, threads=8)
    V = 1 << 12
    sources = S.pick_sources(src, V, 2, 16)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        ref, _ = g.solve_batch(sources, policy=2)
        best = g.autotune_batch(sources, tmp_path / "tune.txt")
        assert best > 0
        text = (tmp_path / "tune.txt").read_text()
        assert text.count("best") == 1 and "workgroup_per_task" in text and "merged_frontier" in text
        assert "vertex_major_all_edge" in text
        D, _ = g.solve_batch(sources, policy=0)
        assert np.array_equal(bits(D), bits(ref))
    # untuned: 32 or more sources on one graph run policy 3, fewer policy 2
    many = S.pick_sources(src, V, 3, 40)
    with S.DeviceGraph(src, dst, w, V) as g:
        D, st = g.solve_batch(many, policy=0)
        assert st["iterations"] == 3
        D2, _ = g.solve_batch(many, policy=1)
        assert np.array_equal(bits(D), bits(D2))
        _, st = g.solve_batch(many[:8], policy=0)
        assert st["iterations"] == 2
    scales, s, d, w2, offs, vc, srcs = _pack_case(24, 5)
    p = S.GraphPack(s, d, w2, offs, vc)
    try:
        a, _ = p.solve(srcs, policy=2)
        assert p.autotune(srcs, tmp_path / "pack.txt") > 0
        b, _ = p.solve(srcs, policy=0)
        assert np.array_equal(bits(a), bits(b))
    finally:
        p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("delta,hub", [(0.01, 0), (0.1, 0), (0.5, 0), (3.0, 0), (0.005, 64),
                                       (0.02, 16)])
def test_far_pile_keeps_the_fixpoint(gpu, oracle, delta, hub):
    """Push rounds defer vertices (d >= min + delta, out-degree >= hub) to the
    far pile; mixed schedules flush it before all-edge and pull rounds."""
    src, dst, w = S.rmat(14, 16, seed=31, threads=16)
    V = 1 << 14
    with S.DeviceGraph(src, dst, w, V, relabel=True) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        g.set_param("delta", delta)
        g.set_param("hub_degree", hub)
        for s in (0, int(src[123])):
            ref = oracle.dijkstra(src, dst, w, V, s)
            for sched in ("push", "heuristic", "learned", "all", "pull"):
                d, st = g.solve(s, sched)
                assert np.array_equal(bits(d), bits(ref)), (delta, hub, s, sched)
                assert st["reached"] == int((d != S.F32_INF).sum())
        ok, counts, _ = g.certify(s)
        assert ok, counts
    su, tu, wu = S.er(1 << 13, 8, seed=9, weight_mode=1)
    with S.DeviceGraph(su, tu, wu, 1 << 13) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        g.set_param("delta", delta * 100)
        g.set_param("hub_degree", hub)
        d, _ = g.solve(0, "push")
        assert np.array_equal(d, oracle.dijkstra(su, tu, wu, 1 << 13, 0))


@pytest.mark.gpu
def test_far_pile_after_failed_solve_and_collection(gpu, oracle):
    """A solve stopped by max_rounds leaves vertices piled and stamps set; the
    next solve and a timing collection must start clean."""
    src, dst, w = S.rmat(13, 16, seed=5, threads=8)
    V = 1 << 13
    ref = oracle.dijkstra(src, dst, w, V, 3)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        g.set_param("delta", 0.01)
        g.set_param("hub_degree", 32)
        g.set_param("max_rounds", 4)
        with pytest.raises(S.SSSPError):
            g.solve(3, "push")
        g.set_param("max_rounds", 100000)
        d, _ = g.solve(3, "push")
        assert np.array_equal(bits(d), bits(ref))
        feats, times = g.collect_timings(3)
        assert len(feats) > 0 and np.all(np.isfinite(times[:, :8]))
        print(f"collection: {len(feats)} rows, {int(g.get_param('collect_rounds'))} rounds run",
              flush=True)
        d, _ = g.solve(3, "heuristic")
        assert np.array_equal(bits(d), bits(ref))
        # a collection past its round budget gives up from the host between
        # rounds (every kernel has ended); the graph stays usable
        g.set_param("collect_budget", 40)
        with pytest.raises(S.SSSPError) as e:
            g.collect_timings(3)
        assert e.value.code == S.ERR_NOT_CONVERGED and "budget" in str(e.value)
        assert g.get_param("collect_rounds") == 41
        d, _ = g.solve(3, "push")
        assert np.array_equal(bits(d), bits(ref))
        g.set_param("collect_budget", 1 << 22)


@pytest.mark.gpu
def test_round_limits_are_bounded(gpu):
    src, dst, w = S.rmat(8, 4, seed=1, threads=1)
    with S.DeviceGraph(src, dst, w, 256) as g:
        for name, bad in (("max_rounds", 0), ("max_rounds", 2.0 ** 28 + 1), ("max_rounds", 2.0 ** 31),
                          ("collect_budget", 0)):
            with pytest.raises(S.SSSPError) as e:
                g.set_param(name, bad)
            assert e.value.code == S.ERR_ARG
        g.set_param("max_rounds", 2 ** 28)
        d, _ = g.solve(0, "push")
        assert g.get_param("max_rounds") == 2 ** 28


# ---- BFS on the same engine (BFS::gpu_bfs, algorithm/bfs/bfs.hpp:213-253) -----

@pytest.mark.gpu
@pytest.mark.parametrize("name,V,src,dst,w", small_graphs(), ids=[g[0] for g in small_graphs()])
def test_bfs_small_graphs_every_schedule(gpu, oracle, name, V, src, dst, w):
    vis_ref, lev_ref, n = oracle.bfs(src, dst, V, 0)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        for sched in SCHEDS:
            vis, lev, st = g.bfs(0, sched)
            assert np.array_equal(vis.view(np.uint8), vis_ref), sched
            assert np.array_equal(lev, lev_ref), sched
            assert st["reached"] == n
        ok, counts, _ = g.certify(0)
        assert ok, counts


@pytest.mark.gpu
def test_bfs_rmat_and_er_every_schedule(gpu, oracle):
    src, dst, w = S.rmat(14, 16, seed=17, threads=16)
    V = 1 << 14
    with S.DeviceGraph(src, dst, w, V, relabel=True) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        for s in [0] + list(S.pick_sources(src, V, 5, 3)):
            vis_ref, lev_ref, _ = oracle.bfs(src, dst, V, int(s))
            for sched in SCHEDS:
                vis, lev, _ = g.bfs(int(s), sched)
                assert np.array_equal(lev, lev_ref), (int(s), sched)
                assert np.array_equal(vis.view(np.uint8), vis_ref)
            ok, counts, par = g.certify(int(s))
            assert ok, counts
            # the tight tree of a BFS: every visited non-source vertex's parent
            # is one level up
            m = (par >= 0)
            assert np.all(lev[m] == lev[par[m]] + 1)
            # BFS levels are not distances: the SSSP result is gone
            with pytest.raises(S.SSSPError):
                g.distances()
        d, _ = g.solve(3, "heuristic")
        assert np.array_equal(bits(d), bits(oracle.dijkstra(src, dst, w, V, 3)))
        ok, counts, _ = g.certify(3)
        assert ok, counts
    su, tu, wu = S.er(1 << 13, 8, seed=11, weight_mode=1)
    with S.DeviceGraph(su, tu, wu, 1 << 13) as g:
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        vis_ref, lev_ref, _ = oracle.bfs(su, tu, 1 << 13, 0)
        for sched in ("plain", "heuristic", "push", "pull"):
            vis, lev, _ = g.bfs(0, sched)
            assert np.array_equal(lev, lev_ref), sched


@pytest.mark.gpu
def test_small_graphs_hand_the_rule_and_network_to_plain_passes(gpu, oracle):
    """Below plain_below_edges a heuristic or learned solve (and BFS) runs the
    plain pass loop -- same fixpoint, no rounds; 0 switches this off."""
    src, dst, w = S.rmat(13, 16, seed=8, threads=8)
    V = 1 << 13
    ref = oracle.dijkstra(src, dst, w, V, 0)
    with S.DeviceGraph(src, dst, w, V) as g:
        assert g.get_param("plain_below_edges") == 2 ** 26
        for sched in ("heuristic", "learned"):
            d, st = g.solve(0, sched)
            assert np.array_equal(bits(d), bits(ref)), sched
            assert st["n_push"] == 0 and st["n_pull"] == 0 and st["mlp_rounds"] == 0
            assert st["n_all"] == st["iterations"] > 0
        vis, lev, st = g.bfs(0, "heuristic")
        assert np.array_equal(lev, oracle.bfs(src, dst, V, 0)[1]) and st["n_push"] == 0
        g.set_param("plain_below_edges", 0)
        d, st = g.solve(0, "heuristic")
        assert np.array_equal(bits(d), bits(ref)) and st["n_push"] > 0


@pytest.mark.gpu
def test_dense_threshold_default_follows_the_graph(gpu, oracle):
    """A graph without hub blocks (uniform random: every block of 2^14
    destinations near the mean in-edge count) runs dense rounds from 0.4 E of
    frontier edges, a skewed one (R-MAT) from 0.15 E; a set value stays."""
    V = 1 << 16
    src, dst, w = S.er(V, 16, seed=3, weight_mode=1)
    ref = oracle.dijkstra(src, dst, w, V, 0)
    with S.DeviceGraph(src, dst, w, V) as g:
        assert g.get_param("dense_all_frac") == 0.4
        g.set_param("plain_below_edges", 0)  # exercise the round engine
        d, _ = g.solve(0, "heuristic")
        assert np.array_equal(bits(d), bits(ref))
        g.set_param("dense_all_frac", 0.2)
        assert g.get_param("dense_all_frac") == 0.2
    src, dst, w = S.rmat(18, 8, seed=3, threads=8)
    with S.DeviceGraph(src, dst, w, 1 << 18) as g:
        assert g.get_param("dense_all_frac") == 0.15


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("frac,unreached", [(0.0, 2.0), (1e9, 0.0), (1e9, 2.0), (0.15, 0.5)])
def test_dense_all_edge_rounds_keep_the_fixpoint(gpu, oracle, frac, unreached, kernel):
    """All-edge rounds run dense when the frontier is large or most of the
    graph is unreached: over the destination-blocked edge list (kernel 0: LDS
    minima, the frontier written by the same kernel) or as the plain pass
    followed by a compaction against a snapshot (kernel 1). Forced on for
    every all-edge round, on only by the unreached rule, and off (the
    fixpoint check stays dense), the distances, levels and frontiers stay
    exact."""
    src, dst, w = S.rmat(14, 16, seed=41, threads=16)
    V = 1 << 14
    su, tu, wu = S.er(1 << 13, 8, seed=13, weight_mode=1)
    with S.DeviceGraph(src, dst, w, V) as g, S.DeviceGraph(su, tu, wu, 1 << 13) as gu:
        for h in (g, gu):
            h.set_param("plain_below_edges", 0)  # exercise the round engine
            h.set_param("dense_all_frac", frac)
            h.set_param("dense_unreached", unreached)
            h.set_param("dense_kernel", kernel)
            assert h.get_param("dense_all_frac") == frac
        for s in (0, int(src[77])):
            ref = oracle.dijkstra(src, dst, w, V, s)
            for sched in ("all", "heuristic", "learned", "push"):
                d, st = g.solve(s, sched)
                assert np.array_equal(bits(d), bits(ref)), (frac, unreached, s, sched)
                assert st["reached"] == int((d != S.F32_INF).sum())
            ok, counts, _ = g.certify(s)
            assert ok, counts
            _, lev, _ = g.bfs(s, "all")
            assert np.array_equal(lev, oracle.bfs(src, dst, V, s)[1])
        for sched in ("all", "heuristic"):
            d, _ = gu.solve(0, sched)
            assert np.array_equal(d, oracle.dijkstra(su, tu, wu, 1 << 13, 0)), sched
        with pytest.raises(S.SSSPError):
            g.set_param("dense_unreached", -1)
        with pytest.raises(S.SSSPError):
            g.set_param("dense_kernel", 2)


@pytest.mark.gpu
def test_dense_rounds_with_split_blocks(gpu, oracle):
    """A destination block with more in-edges than one tile holds is split
    over several tiles, which write back with atomicMin and stamp with an
    exchange; the R-MAT hub block here is split (checked on the host) and
    every dense round stays exact, for f32, u32 and BFS levels."""
    scale = 17
    src, dst, w = S.rmat(scale, 16, seed=44, threads=16)
    V = 1 << scale
    per_block = np.bincount(dst >> 14)
    assert per_block.max() > (1 << 19), per_block.max()  # at least one split block
    wu = (np.arange(len(src)) % 255 + 1).astype(np.uint32)
    with S.DeviceGraph(src, dst, w, V, relabel=True) as g, S.DeviceGraph(src, dst, wu, V) as gu:
        for h in (g, gu):
            h.set_param("plain_below_edges", 0)
            h.set_param("dense_all_frac", 0.0)  # every all-edge round dense
        for s in (0, int(src[999])):
            ref = oracle.dijkstra(src, dst, w, V, s)
            for sched in ("all", "heuristic", "learned"):
                d, st = g.solve(s, sched)
                assert np.array_equal(bits(d), bits(ref)), (s, sched)
            ok, counts, _ = g.certify(s)
            assert ok, counts
            du, _ = gu.solve(s, "all")
            assert np.array_equal(du, oracle.dijkstra(src, dst, wu, V, s)), s
            _, lev, _ = g.bfs(s, "all")
            assert np.array_equal(lev, oracle.bfs(src, dst, V, s)[1]), s


@pytest.mark.gpu
def test_python_mirror_cache_follows_in_place_edits(gpu, oracle):
    """SingleSourceShortestPaths.gpu_bellman_ford caches the device graph; an
    edit of the graph's arrays in place is seen by the next call."""
    g = S.GraphGenerationAPI.R_MAT_parallel(1 << 11, 8, 57, 19, 19, 5, 8, True, 4)
    op = S.SingleSourceShortestPaths()
    d = np.empty(g.vertices_count, np.float32)
    op.gpu_bellman_ford(g, d, 0)
    assert np.array_equal(bits(d), bits(oracle.dijkstra(g.src_ids, g.dst_ids, g.weights,
                                                          g.vertices_count, 0)))
    g.weights[g.src_ids == 0] = 0.0  # in place
    op.gpu_bellman_ford(g, d, 0)
    assert np.array_equal(bits(d), bits(oracle.dijkstra(g.src_ids, g.dst_ids, g.weights,
                                                          g.vertices_count, 0)))


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["one_block", "block_edge", "split", "ties", "equal", "u32",
                                  "ranges", "path"])
def test_light_passes_bit_exact(gpu, oracle, case):
    """Light passes (the lightest edges alone, before a dense round and between
    the full passes of small graphs) end on the oracle's fixpoint: a graph
    of one destination block, one vertex past a block, tiles down to 256 slots
    (split blocks), a few distinct weights, equal weights (no light class), u32,
    tiles by source range, and a long path whose passes outlast the light
    ones. Bit equality: no tolerance."""
    rng = np.random.default_rng(17)
    V = {"one_block": 1 << 14, "block_edge": (1 << 14) + 1, "path": 40000}.get(case, 50021)
    n = 8 * V
    src = (rng.random(n) ** 3 * V).astype(np.int32)
    dst = (rng.random(n) ** 2 * V).astype(np.int32)
    if case in ("u32", "ranges"):
        src, dst = (rng.integers(0, V, n).astype(np.int32) for _ in range(2))
    w = rng.random(n, dtype=np.float32)
    if case == "ties":
        w = (rng.integers(0, 8, n) / 8).astype(np.float32)
    elif case == "equal":
        w = np.full(n, 0.25, np.float32)
    elif case == "u32":
        w = rng.integers(1, 256, n).astype(np.uint32)
    elif case == "path":
        hop = np.arange(V, dtype=np.int32)[::-1].copy()  # against the ids: one hop a pass
        hub = np.full(64, hop[0])  # sparse graphs have a light class only with hubs
        src = np.concatenate([hop[:400], hub, src[:200]])
        dst = np.concatenate([hop[1:401], hop[1000:1064], dst[:200]])
        w = np.concatenate([rng.random(400, dtype=np.float32), np.full(264, 9, np.float32)])
    source = int(src[0])
    ref = oracle.dijkstra(src, dst, w, V, source)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("dense_unreached", 0.0)  # every all-edge round dense
        if case == "split":
            g.set_param("blk_tile_cap", 256)
        if case == "ranges":
            g.set_param("blk_range_bits", 18)
        g.set_param("trace_events", 1)
        light = 0
        for below, kernel in ((2 ** 26, 2), (0, 2)):  # pass loop, round engine
            g.set_param("plain_below_edges", below)
            g.set_param("plain_kernel", kernel)
            for frac in (0.05, 0.0):  # push rounds first, or none
                g.set_param("push_edge_frac", frac)
                for traced in (1, 0):
                    g.set_param("trace_events", traced)
                    print(f"light passes: {case} below {below} push {frac} traced {traced}",
                          flush=True)
                    d, st = g.solve(source, "heuristic")
                    assert np.array_equal(bits(d), bits(ref)), (below, frac, traced)
                    if traced:
                        tr = g.trace()
                        assert len(tr["mode"]) == st["iterations"]
                        light += int((tr["mode"] == S.MODE_LIGHT).sum())
        assert (light == 0) == (case == "equal"), light
        d, st = g.solve(source, "plain")  # the plain schedule stays all-edge passes
        assert np.array_equal(bits(d), bits(ref))
        assert st["edges_relaxed"] == st["iterations"] * len(src)


@pytest.mark.gpu
@pytest.mark.parametrize("V", [1 << 20, (1 << 20) + 1, 4 * (1 << 20) + 3, 5000011])
def test_large_results_reach_the_host_whole(gpu, V):
    """Results above 4 MB are staged through pinned buffers, 4 MB at a time,
    into pages faulted in ahead: at the threshold, one word past it, and sizes
    that end inside a buffer, into memory that starts off a page, every word
    arrives and none beyond it is written. The same copies from two threads
    at once (one of them finds the buffers taken) agree too."""
    import threading

    rng = np.random.default_rng(3)
    src = rng.integers(0, V, 4 * V).astype(np.int32)
    dst = rng.integers(0, V, 4 * V).astype(np.int32)
    w = rng.random(4 * V, dtype=np.float32)
    with S.DeviceGraph(src, dst, w, V, csc=False) as g, \
            S.DeviceGraph(src[:V], dst[:V], w[:V], V, csc=False) as h:
        ref, _ = g.solve(int(src[0]), "plain")
        href, _ = h.solve(int(src[0]), "plain")
        # the fixpoint itself, in numpy: no edge can lower a distance
        ok = ref[src] < S.F32_INF
        assert ref[src[0]] == 0 and not np.any(ref[src[ok]] + w[ok] < ref[dst[ok]])
        room = np.full(V + 64, 7, np.float32)
        out = room[1:1 + V]
        S._check(S.lib().sssp_get_distances(g.handle, S._ptr(out)))
        assert np.array_equal(bits(out), bits(ref))
        assert (room[0] == 7) and (room[1 + V:] == 7).all()
        got = {}

        def fetch(graph, key):
            for k in range(4):
                got[key, k] = graph.distances()

        ts = [threading.Thread(target=fetch, args=a) for a in ((g, "g"), (h, "h"))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for k in range(4):
            assert np.array_equal(bits(got["g", k]), bits(ref))
            assert np.array_equal(bits(got["h", k]), bits(href))


@pytest.mark.gpu
@pytest.mark.parametrize("V,n,kind", [(1, 3, "f32"), (17, 1, "f32"), (4099, 65, "f32"),
                                      (4099, 300, "u32"), (4099, 64, "equal"), (20011, 33, "hub")])
def test_batch_light_and_live_records(gpu, oracle, V, n, kind):
    """Policy 3 relaxes the records whose source row was lowered since, light
    records first: one vertex, a part of one destination block, one source, a
    chunk and a part, u32, equal weights (no light records), a hub block split
    over many tiles, captured and queued. Bit equality: no tolerance."""
    rng = np.random.default_rng(29)
    m = 11 * V
    src = (rng.random(m) ** 2 * V).astype(np.int32)
    dst = rng.integers(0, V, m).astype(np.int32)
    if kind == "hub":
        dst[: m // 2] = 5
    w = rng.random(m, dtype=np.float32)
    if kind == "equal":
        w[:] = 0.5
    elif kind == "u32":
        w = rng.integers(1, 256, m).astype(np.uint32)
    sources = rng.integers(0, V, n).astype(np.int32)
    with S.DeviceGraph(src, dst, w, V) as g:
        for capture in (1, 0):
            g.set_param("batch_capture", capture)
            for rep in range(2):
                print(f"batch records: {kind} V {V} n {n} capture {capture} {rep}", flush=True)
                D, _ = g.solve_batch(sources, policy=3)
                for i in range(0, n, max(1, n // 7)):
                    ref = oracle.dijkstra(src, dst, w, V, int(sources[i]))
                    assert np.array_equal(bits(D[i]), bits(ref)), (capture, i)
                D1, _ = g.solve_batch(sources, policy=1)
                assert np.array_equal(bits(D), bits(D1))


@pytest.mark.gpu
def test_pack_graphs_at_the_edges_of_the_lds_classes(gpu, oracle):
    """Graphs of a pack are solved in LDS up to 2^15 vertices, in classes of
    2^11, 2^14 and 2^15, larger ones together: sizes at and one past each edge,
    a single vertex, a graph without edges, edge ranges that start and end
    inside a 256-edge chunk and span one chunk or less. Bit equality: no
    tolerance."""
    rng = np.random.default_rng(41)
    sizes = [(1, 0), (1, 3), (33, 5), (2047, 9001), (2048, 4096), (2049, 10007), (300, 256),
             (16384, 70001), (16385, 50021), (32768, 100003), (32769, 90001), (40000, 80001),
             (5, 0)]
    for reorder in (False, True):
        if reorder:
            sizes = [sizes[i] for i in rng.permutation(len(sizes))]
        src = [np.minimum((rng.random(m) ** 2 * v).astype(np.int32), v - 1) for v, m in sizes]
        dst = [rng.integers(0, v, m).astype(np.int32) for v, m in sizes]
        w = [rng.random(m, dtype=np.float32) for _, m in sizes]
        offs = np.concatenate([[0], np.cumsum([m for _, m in sizes])]).astype(np.int64)
        vc = np.array([v for v, _ in sizes], np.int32)
        srcs = np.array([int(s[0]) if len(s) else v - 1 for s, (v, _) in zip(src, sizes)], np.int32)
        voff = np.concatenate([[0], np.cumsum(vc)])
        p = S.GraphPack(np.concatenate(src), np.concatenate(dst), np.concatenate(w), offs, vc)
        try:
            for rep in range(2):
                print(f"pack at class edges: reorder {reorder} {rep}", flush=True)
                D, _ = p.solve(srcs, policy=1)
                for k, (v, m) in enumerate(sizes):
                    ref = oracle.dijkstra(src[k], dst[k], w[k], v, int(srcs[k])) if m else \
                        np.where(np.arange(v) == srcs[k], np.float32(0), S.F32_INF)
                    assert np.array_equal(bits(D[voff[k]:voff[k + 1]]), bits(ref)), (rep, v, m)
        finally:
            p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("V", [700, 2048, 9001, 20000, 33000])
def test_batch_policy_1_in_lds_u32(gpu, oracle, V):
    """Policy 1 over the sources of one graph, in each LDS class and past the
    largest, u32 weights with values that saturate."""
    rng = np.random.default_rng(43)
    src, dst = (rng.integers(0, V, 7 * V + 13).astype(np.int32) for _ in range(2))
    w = rng.integers(1, 256, len(src)).astype(np.uint32)
    w[::5] = 0xFFFFFF00
    sources = rng.integers(0, V, 11).astype(np.int32)
    with S.DeviceGraph(src, dst, w, V) as g:
        D, _ = g.solve_batch(sources, policy=1)
        for i, s in enumerate(sources):
            assert np.array_equal(D[i], oracle.dijkstra(src, dst, w, V, int(s))), i


@pytest.mark.gpu
@pytest.mark.parametrize("near", [True, False], ids=["near", "scattered"])
def test_pack_of_large_grids_runs_passes(gpu, oracle, near):
    """The graphs of a pack that are too large for LDS are solved together in
    passes, as one of them alone would be (local passes where ids are near), not
    in rounds that cost a host check per hop: four grids and a small graph
    between them take a few times one grid's time (rounds took 5 and 30 times).
    Bit equality with the oracle."""
    rng = np.random.default_rng(53)
    r, c = 200, 200
    v = np.arange(r * c, dtype=np.int32).reshape(r, c)
    a = np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()])
    b = np.concatenate([v[:, 1:].ravel(), v[1:].ravel()])
    gs = []
    for k in range(4):
        q = v.ravel() if near else rng.permutation(r * c).astype(np.int32)
        s, d = q[np.concatenate([a, b])], q[np.concatenate([b, a])]
        gs.append((s, d, rng.random(len(s), dtype=np.float32), r * c, int(q[k])))
    s, d = (rng.integers(0, 900, 5000).astype(np.int32) for _ in range(2))
    gs.insert(2, (s, d, rng.random(5000, dtype=np.float32), 900, int(s[0])))
    refs = [oracle.dijkstra(s, d, w, n, x) for s, d, w, n, x in gs]
    with S.DeviceGraph(*gs[0][:4]) as g:
        one = min(g.solve(gs[0][4], "heuristic")[1]["t_solve_ms"] for _ in range(4))
    offs = np.concatenate([[0], np.cumsum([len(x[0]) for x in gs])]).astype(np.int64)
    vc = np.array([x[3] for x in gs], np.int32)
    srcs = np.array([x[4] for x in gs], np.int32)
    voff = np.concatenate([[0], np.cumsum(vc)])
    p = S.GraphPack(*(np.concatenate([x[i] for x in gs]) for i in range(3)), offs, vc)
    try:
        for policy in (1, 2):
            times = []
            for rep in range(4):
                print(f"pack of grids: near {near} policy {policy} {rep}", flush=True)
                D, st = p.solve(srcs, policy=policy)
                times.append(st["t_solve_ms"])
                for k, ref in enumerate(refs):
                    assert np.array_equal(bits(D[voff[k]:voff[k + 1]]), bits(ref)), (policy, k)
            assert min(times) < 3 * one, (policy, times, one)
    finally:
        p.close()


@pytest.mark.gpu
def test_pack_merged_in_rounds(gpu, oracle):
    """From 2^25 edges on the graphs of a pack that are too large for LDS share
    the rounds of the engine: bit equality with the oracle."""
    scales = np.full(65, 16, np.int32)
    s, d, w, offs = S.rmat_many(scales, 8, seed0=3)
    assert len(s) > 1 << 25
    vc = (1 << scales).astype(np.int32)
    srcs = np.minimum.reduceat(s, offs[:-1]).astype(np.int32)
    voff = np.concatenate([[0], np.cumsum(vc)])
    p = S.GraphPack(s, d, w, offs, vc)
    try:
        for policy in (1, 2):
            print(f"merged pack in rounds: policy {policy}", flush=True)
            D, _ = p.solve(srcs, policy=policy)
            for k in range(0, 65, 4):
                e0, e1 = offs[k], offs[k + 1]
                ref = oracle.dijkstra(s[e0:e1], d[e0:e1], w[e0:e1], int(vc[k]), int(srcs[k]))
                assert np.array_equal(bits(D[voff[k]:voff[k + 1]]), bits(ref)), (policy, k)
    finally:
        p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("V,E,n,kind", [(16384, 400003, 257, "even"), (16368, 150001, 40, "below_u32"),
                                        (16385, 600007, 65, "one_block"), (20000, 20000, 33, "even")])
def test_batch_tiles_of_even_blocks(gpu, oracle, V, E, n, kind):
    """Policy 3 on graphs without hubs, whose tiles hold whole destination blocks
    from 1024 blocks on, and with one large block, whose tiles stay short: below, at
    and past the line, part of a wave, a chunk and a part, u32, groups of records
    that are and are not whole eights. Captured and queued; bit equality."""
    rng = np.random.default_rng(E + n)
    src, dst = (rng.integers(0, V, E).astype(np.int32) for _ in range(2))
    if kind == "one_block":
        dst[::3] = rng.integers(48, 64, len(dst[::3]))
    w = rng.random(E, dtype=np.float32)
    if kind.endswith("u32"):
        w = rng.integers(1, 256, E).astype(np.uint32)
    sources = src[rng.integers(0, E, n)].astype(np.int32)
    refs = {i: oracle.dijkstra(src, dst, w, V, int(sources[i])) for i in (0, n // 2, n - 1)}
    nblk = (V + 15) // 16
    per = np.bincount(dst // 16, minlength=nblk)
    cap = 512 if nblk >= 1024 and per.max() * nblk <= 4 * E else 128
    assert (cap == 512) == (kind == "even")
    with S.DeviceGraph(src, dst, w, V) as g:
        for capture in (1, 0):
            g.set_param("batch_capture", capture)
            print(f"batch tiles: {kind} V {V} E {E} n {n} capture {capture}", flush=True)
            D, _ = g.solve_batch(sources, policy=3)
            assert g.get_param("multi_tiles") == ((per + cap - 1) // cap).sum()
            for i, ref in refs.items():
                assert np.array_equal(bits(D[i]), bits(ref)), (capture, i)


@pytest.mark.gpu
@pytest.mark.parametrize("V,E,kind", [(4099, 45089, "f32"), (4099, 45089, "u32"),
                                      (1 << 14, 1 << 17, "f32"), (900, 30000, "f32"),
                                      (20011, 220121, "f32"), (4099, 45089, "equal")])
def test_light_list_of_graphs_solved_in_one_workgroup(gpu, oracle, V, E, kind):
    """Graphs whose solves run in one workgroup, or whose passes are too short for
    light ones, are built without the light list; a solve that uses it (plain_kernel
    2, rounds) builds it then, and the light passes are in its trace. Without
    memory for it the solve runs without. Bit equality with the oracle."""
    rng = np.random.default_rng(E)
    src = (rng.random(E) ** 2 * V).astype(np.int32)
    dst = rng.integers(0, V, E).astype(np.int32)
    w = rng.random(E, dtype=np.float32)
    if kind == "u32":
        w = rng.integers(1, 256, E).astype(np.uint32)
    elif kind == "equal":
        w[:] = 0.5
    source = int(src[0])

    def resident(graph):
        b = C.c_int64(0)
        assert S.lib().sssp_graph_info(graph.handle, None, None, None, C.byref(b)) == S.OK
        return b.value

    ref = oracle.dijkstra(src, dst, w, V, source)
    with S.DeviceGraph(src, dst, w, V) as g:
        for traced in (0, 1):
            g.set_param("trace_events", traced)
            d, _ = g.solve(source, "heuristic")
            assert np.array_equal(bits(d), bits(ref)) and g.get_param("light_edges") == 0
        g.set_param("trace_events", 1)
        g.set_param("plain_kernel", 2)
        if E > 1 << 15 and kind != "equal":
            print(f"light list on demand: {kind} V {V} E {E}, no memory", flush=True)
            S.lib().sssp_debug_fail_next_alloc()  # of the light list's build
            d, _ = g.solve(source, "heuristic")
            assert np.array_equal(bits(d), bits(ref))
            assert not (g.trace()["mode"] == S.MODE_LIGHT).any()
        size = resident(g)
        for below in (2 ** 26, 0):  # pass loop, rounds
            print(f"light list on demand: {kind} V {V} E {E}, below {below}", flush=True)
            g.set_param("plain_below_edges", below)
            g.set_param("dense_unreached", 0.0)
            d, _ = g.solve(source, "heuristic")
            assert np.array_equal(bits(d), bits(ref)), below
            assert (g.trace()["mode"] == S.MODE_LIGHT).any() == (kind != "equal"), below
        assert (g.get_param("light_edges") > 0) == (kind != "equal")
        assert (resident(g) > size) == (kind != "equal")


@pytest.mark.gpu
def test_local_tiles_of_graphs_solved_in_one_workgroup(gpu, oracle):
    """The same for the tiles of the local passes: built by the first solve of
    a small grid that runs passes, which are then the local ones."""
    rng = np.random.default_rng(59)
    v = np.arange(3000, dtype=np.int32).reshape(60, 50)
    a = np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()])
    b = np.concatenate([v[:, 1:].ravel(), v[1:].ravel()])
    src, dst = np.concatenate([a, b]), np.concatenate([b, a])
    w = rng.random(len(src), dtype=np.float32)
    ref = oracle.dijkstra(src, dst, w, 3000, 0)
    with S.DeviceGraph(src, dst, w, 3000) as g:
        for rep in range(2):  # in one workgroup, before and after
            d, st = g.solve(0, "heuristic")
            assert np.array_equal(bits(d), bits(ref))
            g.set_param("trace_events", 1)
            for fail in (1, 0) if rep == 0 else (0,):
                print(f"local tiles on demand: {rep} no memory {fail}", flush=True)
                if fail:
                    S.lib().sssp_debug_fail_next_alloc()
                d, st = g.solve(0, "heuristic")
                assert np.array_equal(bits(d), bits(ref))
                plain = g.solve(0, "plain")[1]
                assert (st["iterations"] * 2 < plain["iterations"]) == (fail == 0)
            g.set_param("trace_events", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("V,E,n,kind,light", [
    (4099, 60000, 65, "hubs", False), (30011, (1 << 19) - 1, 33, "hubs", False),
    (30011, 1 << 19, 65, "hubs", True), (30011, 1 << 19, 300, "hubs_u32", True),
    (30011, 1 << 19, 64, "equal", False), (60000, 1 << 19, 33, "hubs", False),
    (100003, (1 << 21) - 1, 33, "even", False), (100003, 1 << 21, 40, "even_u32", True),
    (190000, 1 << 21, 33, "even", False), (16384, 400003, 257, "even", False)])
def test_batch_light_records_where_they_pay(gpu, oracle, V, E, n, kind, light):
    """Policy 3 has light records from the edge counts and mean degrees on where
    they pay, on graphs with hubs and without, and none with equal weights: part of a
    wave, a chunk and a part, u32, tiles that hold whole blocks, captured and
    queued. Bit equality with the oracle."""
    rng = np.random.default_rng(E + n)
    src = (rng.random(E) ** (1 if kind.startswith("even") else 2) * V).astype(np.int32)
    dst = rng.integers(0, V, E).astype(np.int32)
    w = rng.random(E, dtype=np.float32)
    if kind.endswith("u32"):
        w = rng.integers(1, 256, E).astype(np.uint32)
    elif kind == "equal":
        w[:] = 0.5
    sources = rng.integers(0, V, n).astype(np.int32)
    refs = {i: oracle.dijkstra(src, dst, w, V, int(sources[i])) for i in (0, n // 2, n - 1)}
    with S.DeviceGraph(src, dst, w, V) as g:
        for capture in (1, 0):
            g.set_param("batch_capture", capture)
            print(f"light records: {kind} V {V} E {E} n {n} capture {capture}", flush=True)
            D, _ = g.solve_batch(sources, policy=3)
            assert (g.get_param("multi_light_tiles") > 0) == light
            for i, ref in refs.items():
                assert np.array_equal(bits(D[i]), bits(ref)), (capture, i)


def _fresh(n, dtype):
    """An array in memory just mapped, none of it touched."""
    return np.frombuffer(mmap.mmap(-1, n * np.dtype(dtype).itemsize,
                                   flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS), dtype)


def _resident(a):
    """Pages of an array that are in memory, by mincore(2)."""
    libc = C.CDLL(None, use_errno=True)
    page = 4096
    lo = (a.ctypes.data + page - 1) // page * page
    n = (a.ctypes.data + a.nbytes - lo) // page
    vec = (C.c_ubyte * n)()
    assert libc.mincore(C.c_void_p(lo), C.c_size_t(n * page), vec) == 0
    return sum(v & 1 for v in vec), n


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["batch1", "batch2", "batch3", "bfs", "pack"])
def test_result_pages_wait_for_the_allocations(gpu, oracle, call):
    """The pages of a large result are faulted in only once the call's device
    buffers are there (each allocation would wait for the page faults): when
    the first one fails, the call returns SSSP_ERR_OOM with the result's pages untouched. The
    next call succeeds, with every word written."""
    src, dst, w = S.rmat(17, 4, seed=5, threads=8)
    V, n = 1 << 17, 40
    L, sources = S.lib(), S.pick_sources(src, 1 << 17, 2, 40)
    if call == "pack":
        k = 40
        offs = np.arange(k + 1, dtype=np.int64) * len(src)
        many = [np.tile(x, k) for x in (src, dst, w)]
        p = S.GraphPack(*many, offs, np.full(k, V, np.int32))
        same = np.full(k, int(sources[0]), np.int32)
        out, rows, want = _fresh(k * V, np.float32), k, [int(sources[0])] * k
        run = lambda: L.sssp_pack_solve(p._h, S._ptr(same), 0, S._ptr(out), None)  # noqa: E731
        close = p.close
    else:
        if call == "bfs":
            V = 1 << 21
        g = S.DeviceGraph(src, dst, w, V)
        close = g.close
        if call == "bfs":
            out, vis = _fresh(V, np.uint32), np.empty(V, np.uint8)
            run = lambda: L.sssp_bfs(g.handle, int(sources[0]), S.SCHED_HEURISTIC,  # noqa: E731
                                     S._ptr(vis), S._ptr(out), None)
        else:
            out, rows, want = _fresh(n * V, np.float32), n, [int(x) for x in sources]
            run = lambda: L.sssp_solve_batch(g.handle, S._ptr(sources), n, int(call[5:]),  # noqa: E731
                                             S._ptr(out), None)
    try:
        print(f"result pages: {call}", flush=True)
        before, pages = _resident(out)
        assert pages > 1024 and before * 20 < pages
        L.sssp_debug_fail_next_alloc()
        assert run() == S.ERR_OOM
        assert _resident(out)[0] * 20 < pages
        assert run() == S.OK, S.last_error()
        if call == "bfs":
            ref = oracle.bfs(src, dst, V, int(sources[0]))
            assert np.array_equal(out, ref[1]) and np.array_equal(vis, ref[0])
        else:
            for i in range(0, rows, 13):
                ref = oracle.dijkstra(src, dst, w, V, want[i])
                assert np.array_equal(bits(out.reshape(rows, V)[i]), bits(ref)), i
    finally:
        close()


@pytest.mark.gpu
def test_autotuners_try_each_setting_once(gpu, tmp_path):
    """The tuning files list no two candidates that run the same launches: block size
    and workgroups per CU only where a task is too large for LDS, thresholds of the rounds
    only where a solve runs in rounds; the tuned setting solves as the others."""
    def lines(path):
        text = [x for x in path.read_text().splitlines() if not x.startswith("#")]
        assert len({x.split(" ms=")[0] for x in text}) == len(text)
        return [sum(x.startswith("policy=" + k) for x in text)
                for k in ("workgroup_per_task", "merged_frontier", "vertex_major_all_edge")]

    for scale, below, want in ((12, 2 ** 26, [1, 1, 1]), (12, 0, [1, 6, 1]), (16, 2 ** 26, [9, 1, 1])):
        src, dst, w = S.rmat(scale, 8, seed=2, threads=8)
        sources = S.pick_sources(src, 1 << scale, 2, 6)
        print(f"autotune batch: scale {scale} below {below}", flush=True)
        with S.DeviceGraph(src, dst, w, 1 << scale) as g:
            g.set_param("plain_below_edges", below)
            g.autotune_batch(sources, tmp_path / "b.txt")
            assert lines(tmp_path / "b.txt") == want
            a, b = (g.solve_batch(sources, policy=p)[0] for p in (0, 2))
            assert np.array_equal(bits(a), bits(b))
    for scales, want in ((np.full(9, 9), [1, 1, 0]), (np.array([9, 16, 17]), [1, 1, 0]),
                         (np.append(np.full(65, 16), 10), [6, 6, 0])):
        scales = scales.astype(np.int32)
        s, d, w, offs = S.rmat_many(scales, 8, seed0=3)
        srcs = np.minimum.reduceat(s, offs[:-1]).astype(np.int32)
        print(f"autotune pack: {len(scales)} graphs, {len(s)} edges", flush=True)
        p = S.GraphPack(s, d, w, offs, (1 << scales).astype(np.int32))
        try:
            p.autotune(srcs, tmp_path / "p.txt")
            assert lines(tmp_path / "p.txt") == want
            a, b = (p.solve(srcs, policy=q)[0] for q in (0, 2))
            assert np.array_equal(bits(a), bits(b))
        finally:
            p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "light", "local", "rounds"])
def test_decide_spin_off_never_polls(gpu, oracle, kind):
    """decide_spin 0: the host synchronizes the stream, in passes over blocked tiles
    (plain schedule, light and local passes) as in rounds, and polls nothing; 1:
    it polls. Distances are the same, traced or not, and a limit below the solve's
    passes still gives up and leaves the graph usable."""
    if kind == "local":
        V, src, dst = _local_graph("grid", np.random.default_rng(1))
        src, dst = src.astype(np.int32), dst.astype(np.int32)
        w = np.random.default_rng(2).random(len(src), dtype=np.float32)
    else:
        src, dst, w = S.rmat(16, 16, seed=5, threads=8)
        V = 1 << 16
    source, sched = int(src[0]), "plain" if kind == "plain" else "heuristic"
    ref = oracle.dijkstra(src, dst, w, V, source)
    with S.DeviceGraph(src, dst, w, V) as g:
        g.set_param("plain_kernel", 2 if kind == "plain" else 0)
        if kind == "rounds":
            g.set_param("plain_below_edges", 0)
        for spin in (0, 1, 0):
            g.set_param("decide_spin", spin)
            for traced in (0, 1):
                g.set_param("trace_events", traced)
                print(f"decide_spin {spin}: {kind} traced {traced}", flush=True)
                d, st = g.solve(source, sched)
                assert np.array_equal(bits(d), bits(ref)), (spin, traced)
                assert (g.get_param("host_polls") > 0) == (spin == 1), (spin, traced)
            g.set_param("trace_events", 0)
            if kind == "plain":
                g.set_param("max_rounds", 1)
                with pytest.raises(S.SSSPError) as e:
                    g.solve(source, sched)
                assert e.value.code == S.ERR_NOT_CONVERGED
                g.set_param("max_rounds", 100000)


@pytest.mark.gpu
def test_plain_kernel_forces_every_kind_of_graph(gpu, oracle):
    """plain_kernel 2 runs the blocked pass and 1 the edge-list pass also on
    graphs that have local passes: each of their passes relaxes every edge, local ones
    leave tiles out."""
    V, src, dst = _local_graph("grid", np.random.default_rng(1))
    src, dst = src.astype(np.int32), dst.astype(np.int32)
    w = np.random.default_rng(2).random(len(src), dtype=np.float32)
    ref = oracle.dijkstra(src, dst, w, V, 7)
    with S.DeviceGraph(src, dst, w, V) as g:
        for kernel in (0, 1, 2):
            g.set_param("plain_kernel", kernel)
            print(f"plain kernel {kernel} on a grid", flush=True)
            d, st = g.solve(7, "heuristic")
            assert np.array_equal(bits(d), bits(ref)), kernel
            every = st["edges_relaxed"] == st["iterations"] * len(src)
            assert every == (kernel != 0), kernel


@pytest.mark.gpu
@pytest.mark.parametrize("V,E,ends,light", [
    (100003, (1 << 21) - 1, "hubs", False), (100003, 1 << 21, "hubs", True),
    (900001, (3 << 22) - 1, "even", False), (900001, 3 << 22, "even", True),
    (1400003, 3 << 22, "even", False)])
def test_light_passes_where_they_pay(gpu, oracle, V, E, ends, light):
    """The pass loop runs light passes from 2^21 edges on, without hubs from 3 * 2^22
    and a mean of 11 edges; plain_kernel 2 runs them below too. f32, u32 and hops;
    bit equality with the oracle."""
    rng = np.random.default_rng(E)
    src, dst = ((rng.random(E) ** (2 if ends == "hubs" else 1) * V).astype(np.int32)
                for _ in range(2))
    w = rng.random(E, dtype=np.float32) if V % 2 else rng.integers(1, 256, E).astype(np.uint32)
    source = int(src[0])
    ref = oracle.dijkstra(src, dst, w, V, source)
    with S.DeviceGraph(src, dst, w, V, csc=False) as g:
        assert (g.get_param("light_edges") > 0) == light
        for traced in (0, 1):
            g.set_param("trace_events", traced)
            print(f"light line: {ends} V {V} E {E} traced {traced}", flush=True)
            d, st = g.solve(source, "heuristic")
            assert np.array_equal(bits(d), bits(ref)), traced
        assert (g.trace()["mode"] == S.MODE_LIGHT).any() == light
        assert (g.get_param("light_edges") > 0) == light
        g.set_param("plain_kernel", 2)
        d, st = g.solve(source, "heuristic")
        assert np.array_equal(bits(d), bits(ref))
        assert (g.trace()["mode"] == S.MODE_LIGHT).any() and st["n_all"] == st["iterations"]
