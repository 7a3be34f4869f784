// batch.hip -- many SSSP solves in one launch.
//
// Policy 1 (workgroup per task): a workgroup runs a complete frontier
// Bellman-Ford for its task, (graph range, source), with workgroup barriers
// only (no grid barrier, so any occupancy is deadlock-free). Graphs of up to
// 2^15 vertices are solved in LDS (k_lds_solve, one workgroup per task);
// larger ones by a persistent kernel whose workgroups take tasks from an atomic
// counter -- largest tasks first:
//   frontier chunk of BS vertices -> degree scan in LDS -> the chunk's edges
//   dealt over the BS lanes (binary search in LDS) -> check-then-atomicMin ->
//   appends to the next frontier through an LDS counter, deduplicated by a
//   per-workgroup stamp array. The launches are captured once in a hipGraph
//   and replayed.
// Policy 2 (full chip): many disjoint graphs are one union graph, whose solve
//   starts from all their sources: in passes over its blocked list (the pass
//   loop) below 2^25 edges, in frontier rounds from there on. Many sources on one
//   graph are solved one after another, each as sssp_solve does it.
// Policy 3 (many sources on one graph, vertex-major): the distances of up to
//   256 sources are one array D[v * n + s], so a vertex's distances are one
//   contiguous row. All-edge passes over the edges sorted by 16-vertex
//   destination block: a 256-thread workgroup (thread s = source s) holds its
//   block's 16 x 256 minima in LDS (they start unreached, not at the distances).
//   Each of its waves reads the records 64 at a time, one per lane, and takes
//   them in turn (readlane): gather the source vertex's row (coalesced, eight
//   rows in flight) unless no source lowered it since the record was last
//   relaxed, and lower the own LDS column -- no atomics inside a block. The
//   minima below the block's distances are written at the end (atomicMin for
//   blocks split over several tiles).
//   Where light records pay (kMLightEdges), passes over the light edges alone
//   alternate with full ones; they end with a full pass that changes nothing,
//   the Bellman-Ford fixpoint of every source, and the rows are then transposed
//   into the per-source output.
// The autotuner times block size x workgroups per CU for policy 1, frontier
// threshold x push chunk width for policy 2, and policy 3, and keeps the
// fastest; a setting that none of a solve's kernels reads is timed once.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <functional>
#include <numeric>
#include <optional>
#include <string>

#include "sssp_graph.hpp"

namespace sssp {

struct BatchTask {
    int64_t vlo;     // first vertex of the task's graph (global id)
    int64_t doff;    // offset of the task's distance array in the batch output
    int32_t nv;      // vertices of the task's graph
    int32_t source;  // global id
};

namespace {

// Block-wide exclusive scan, BS threads.
template <int BS>
__device__ int64_t bscan(int64_t x, int64_t *total, int64_t *s_warp)
{
    const int lane = __lane_id(), w = threadIdx.x >> 6;
    int64_t inc = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t y = __shfl_up(inc, o);
        if (lane >= o) inc += y;
    }
    if (lane == 63) s_warp[w] = inc;
    __syncthreads();
    int64_t pre = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < BS / 64; i++) {
        if (i < w) pre += s_warp[i];
        tot += s_warp[i];
    }
    __syncthreads();
    *total = tot;
    return pre + inc - x;
}

__global__ void k_batch_reset(int32_t *counter)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        counter[0] = 0;  // next task
        counter[1] = 0;  // error flag
    }
}

template <class WT, int BS>
__global__ __launch_bounds__(BS) void k_wg_solve(const BatchTask *__restrict__ tasks, int32_t ntasks,
                                                 int32_t *counter, const int64_t *__restrict__ row_ptr,
                                                 const int32_t *__restrict__ adj,
                                                 const uint32_t *__restrict__ wts, uint32_t *bdist,
                                                 int32_t *scratch, int64_t maxv, int32_t *round_ctr)
{
    constexpr uint32_t INF = WT::INF;
    __shared__ int s_task, s_n;
    __shared__ int32_t s_v[BS];
    __shared__ int64_t s_start[BS];
    __shared__ int64_t s_off[BS + 1];
    __shared__ uint32_t s_du[BS];
    __shared__ int64_t s_warp[BS / 64];
    const int tid = threadIdx.x;
    int32_t *qa = scratch + (int64_t)blockIdx.x * 3 * maxv;
    int32_t *qb = qa + maxv;
    int32_t *stamp = qb + maxv;  // local index; rounds only ever increase
    int32_t rt = round_ctr[blockIdx.x];
    for (;;) {
        if (tid == 0) s_task = atomicAdd(&counter[0], 1);
        __syncthreads();
        const int t = s_task;
        __syncthreads();
        if (t >= ntasks) break;
        const BatchTask T = tasks[t];
        uint32_t *dist = bdist + T.doff - T.vlo;  // indexed by global vertex id
        for (int64_t v = tid; v < T.nv; v += BS) dist[T.vlo + v] = INF;
        __syncthreads();
        if (tid == 0) {
            dist[T.source] = 0u;
            qa[0] = T.source;
        }
        int32_t n = 1;
        int32_t rounds = 0;
        int32_t *cur = qa, *nxt = qb;
        __syncthreads();
        while (n > 0) {
            if (++rounds > T.nv + 2) {  // cannot happen for w >= 0; bounded anyway
                if (tid == 0) counter[1] = 1;
                break;
            }
            rt++;
            if (tid == 0) s_n = 0;
            __syncthreads();
            for (int32_t base = 0; base < n; base += BS) {
                const int32_t i = base + tid;
                int32_t u = 0;
                int64_t a = 0, deg = 0;
                uint32_t du = INF;
                if (i < n) {
                    u = cur[i];
                    a = row_ptr[u];
                    deg = row_ptr[u + 1] - a;
                    du = dist[u];
                }
                s_v[tid] = u;
                s_start[tid] = a;
                s_du[tid] = du;
                int64_t tot;
                const int64_t off = bscan<BS>(deg, &tot, s_warp);
                s_off[tid] = off;
                if (tid == BS - 1) s_off[BS] = tot;
                __syncthreads();
                for (int64_t e = tid; e < tot; e += BS) {
                    int lo = 0, hi = BS - 1;  // largest j with s_off[j] <= e
                    while (lo < hi) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (s_off[mid] <= e) lo = mid;
                        else hi = mid - 1;
                    }
                    const int64_t edge = s_start[lo] + (e - s_off[lo]);
                    const int32_t v = adj[edge];
                    const uint32_t cand = WT::add(s_du[lo], wts[edge]);
                    // rounds share one launch, so a plain read may be from an
                    // earlier round: the returned old value decides "lowered";
                    // a stale stamp is an older round and falls through to the
                    // exchange
                    if (cand < dist[v]) {
                        const uint32_t old = atomicMin(&dist[v], cand);
                        int32_t *sp = &stamp[v - T.vlo];
                        if (cand < old && *sp != rt && atomicExch(sp, rt) != rt)
                            nxt[atomicAdd(&s_n, 1)] = v;
                    }
                }
                __syncthreads();
            }
            n = s_n;
            int32_t *tmp = cur;
            cur = nxt;
            nxt = tmp;
            __syncthreads();
        }
    }
    if (tid == 0) round_ctr[blockIdx.x] = rt;
}

// Tasks by size: the vertices a workgroup's LDS holds (distances and two
// bitmaps), largest class first; class 0 is solved in global memory.
constexpr int kLdsClasses = 4;
constexpr int32_t kLdsVerts[kLdsClasses] = {0, 1 << 15, 1 << 14, 1 << 11};
static_assert(kLdsVerts[1] == kSoloVerts, "one task may be a whole graph");

inline int lds_class(int64_t nv)
{
    int c = 0;
    while (c + 1 < kLdsClasses && nv <= kLdsVerts[c + 1]) c++;
    return c;
}

// first[c] = source of edge 256 c of the src-sorted list; last entry: V
__global__ __launch_bounds__(kBlock) void k_chunk_sources(const int32_t *src, int64_t nch,
                                                          int32_t V, int32_t *first)
{
    for (int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x; c <= nch;
         c += (int64_t)gridDim.x * kBlock)
        first[c] = c < nch ? src[c * kBlkChunk] : V;
}

// A whole solve in LDS, one workgroup per task: distances and the bitmaps of
// the vertices lowered in the last and in this round. A round deals the
// graph's edges (contiguous in the src-sorted list) to the waves in chunks of
// 256: a lane looks up one chunk's range of sources and tests it against the
// last round's bitmap, and the wave then relaxes every edge of the chunks that
// hold a lowered vertex (16-byte loads, the next chunk's under this one's
// relaxations), so a chunk without one is never read. The graph is solved when
// a round lowers nothing. Bound by latency: LDS and the chunk loads.
// 1024 R-MAT graphs of 2^8-2^14 vertices x 8: 0.39 ms, against 3.86 with
// distances, queues and stamps in global memory (k_wg_solve); 1500 of 2^8-2^10 x 6
// 0.068 against 0.31. One R-MAT graph of 2^11 vertices x 16: 56 us on the device,
// 141 in the pass loop. The class sizes let two workgroups of 1024 threads (2^14
// vertices) or eight of 256 (2^11) share a CU's 160 KB.
// SOLO: one solve of a whole graph (launch_solo), its task in `solo`; the
// workgroup also writes the caller-order copy and reports to the host mirror.
constexpr int kSoloThreads = 1024;
struct SoloArgs {
    BatchTask task;
    const int32_t *vperm;  // slot of the caller's vertex, when relabelled
    uint32_t *dout;        // distances by the caller's ids, when relabelled
    Ctrl *mirror;
    int32_t limit;         // rounds at most
};

// The end of a solo solve: the caller-order copy, and rounds, relaxed edges and
// reached vertices to the host. relaxed: this wave's; buf: room for two values per
// wave that nothing reads any more.
template <uint32_t INF, int BS>
__device__ __forceinline__ void solo_report(const SoloArgs &solo, const uint32_t *s_d,
                                            int64_t relaxed, int32_t rounds, int64_t *buf)
{
    const int tid = threadIdx.x, nv = solo.task.nv;
    if (solo.vperm)
        for (int v = tid; v < nv; v += BS) solo.dout[v] = s_d[solo.vperm[v]];
    int reached = 0;
    for (int v = tid; v < nv; v += BS) reached += s_d[v] != INF ? 1 : 0;
    reached = wave_sum32(reached);
    __syncthreads();
    if (__lane_id() == 0) {
        buf[2 * (tid >> 6)] = reached;
        buf[2 * (tid >> 6) + 1] = relaxed;
    }
    __syncthreads();
    if (tid == 0) {
        int64_t r = 0, c = 0;
        for (int i = 0; i < BS / 64; i++) {
            r += buf[2 * i];
            c += buf[2 * i + 1];
        }
        solo.mirror->n_reached = r;
        solo.mirror->ph_work = c;
        solo.mirror->ph_full = rounds;
        __threadfence_system();
    }
}

template <class WT, int BS, int NV, bool SOLO = false>
__global__ __launch_bounds__(BS) void k_lds_solve(const BatchTask *__restrict__ tasks,
                                                  const SoloArgs solo, int32_t *counter,
                                                  const int64_t *__restrict__ row_ptr,
                                                  const int32_t *__restrict__ src,
                                                  const int32_t *__restrict__ dst,
                                                  const uint32_t *__restrict__ wts, int64_t E,
                                                  const int32_t *__restrict__ first,
                                                  uint32_t *__restrict__ bdist)
{
    typedef int32_t v4i __attribute__((ext_vector_type(4)));
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    constexpr uint32_t INF = WT::INF;
    constexpr int NW = NV / 32;
    constexpr int kWaves = BS / 64;
    __shared__ uint32_t s_d[NV];
    __shared__ uint32_t s_bits[2][NW];
    const int tid = threadIdx.x, lane = __lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const BatchTask T = SOLO ? solo.task : tasks[blockIdx.x];
    const int nv = T.nv;
    int32_t chunks = 0, rounds = 0;  // SOLO: chunks this wave relaxed
    for (int v = tid; v < nv; v += BS) s_d[v] = INF;
    for (int i = tid; i < 2 * NW; i += BS) s_bits[0][i] = 0u;
    __syncthreads();
    if (tid == 0) {
        const int s = (int)(T.source - T.vlo);
        s_d[s] = 0u;
        s_bits[0][s >> 5] = 1u << (s & 31);
    }
    const int64_t e0 = row_ptr[T.vlo], e1 = row_ptr[T.vlo + nv];
    const int64_t c0 = e0 / kBlkChunk, nc = e1 > e0 ? (e1 - 1) / kBlkChunk + 1 - c0 : 0;
    __syncthreads();
    struct Edges {
        v4i s, t;
        v4u w;
    };
    auto load = [&](int64_t c) {  // 4 edges of chunk c per lane (past the list: none)
        const int64_t e = c * kBlkChunk + 4 * lane;
        Edges x{};
        if (e + 4 <= E) {
            x.s = *reinterpret_cast<const v4i *>(src + e);
            x.t = *reinterpret_cast<const v4i *>(dst + e);
            x.w = *reinterpret_cast<const v4u *>(wts + e);
        } else {
            for (int k = 0; k < 4; k++)
                if (e + k < E) {
                    x.s[k] = src[e + k];
                    x.t[k] = dst[e + k];
                    x.w[k] = wts[e + k];
                }
        }
        return x;
    };
    int cur = 0;
    for (int32_t round = 0;; round++) {
        if (SOLO) {
            if (round >= solo.limit) {
                rounds = -1;
                break;
            }
            rounds = round + 1;
        } else if (round > nv + 2) {  // cannot happen for w >= 0; bounded anyway
            if (tid == 0) counter[1] = 1;
            break;
        }
        uint32_t *const now = s_bits[cur], *const nxt = s_bits[cur ^ 1];
        bool low = false;
        // each wave: chunks wave, wave + kWaves, ... of the graph, 64 looked up at a time
        for (int64_t j0 = wave; j0 < nc; j0 += 64 * kWaves) {
            const int64_t j = j0 + (int64_t)lane * kWaves;
            bool live = false;
            if (j < nc) {
                const int a = (int)max((int64_t)first[c0 + j] - T.vlo, (int64_t)0);
                const int b = (int)min((int64_t)first[c0 + j + 1] - T.vlo, (int64_t)nv - 1);
                const int wa = a >> 5, wb = b >> 5;
                for (int i = wa; i <= wb && !live; i++) {
                    uint32_t m = now[i];
                    if (i == wa) m &= ~0u << (a & 31);
                    if (i == wb) m &= ~0u >> (31 - (b & 31));
                    live = m != 0u;
                }
            }
            uint64_t todo = __ballot(live);
            if (SOLO) chunks += __popcll(todo);
            auto next = [&](Edges &x, int64_t &c) {
                const int i = __builtin_ctzll(todo);
                todo &= todo - 1;
                c = c0 + j0 + (int64_t)i * kWaves;
                x = load(c);
            };
            Edges x{};
            int64_t c = 0;
            bool more = todo != 0;
            if (more) next(x, c);
            while (more) {
                const Edges y = x;
                const int64_t e = c * kBlkChunk + 4 * lane;
                more = todo != 0;
                if (more) next(x, c);
                uint32_t cand[4], dv[4];
                int v[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const bool mine = e + k >= e0 && e + k < e1;
                    v[k] = mine ? (int)(y.t[k] - T.vlo) : 0;
                    const uint32_t du = mine ? s_d[(int)(y.s[k] - T.vlo)] : INF;
                    cand[k] = du != INF ? WT::add(du, y.w[k]) : INF;
                }
#pragma unroll
                for (int k = 0; k < 4; k++) dv[k] = s_d[v[k]];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (cand[k] < dv[k] && atomicMin(&s_d[v[k]], cand[k]) > cand[k]) {
                        atomicOr(&nxt[v[k] >> 5], 1u << (v[k] & 31));
                        low = true;
                    }
            }
        }
        if (!__syncthreads_or(low)) break;
        for (int i = tid; i < NW; i += BS) now[i] = 0u;
        cur ^= 1;
        __syncthreads();
    }
    uint32_t *const out = bdist + T.doff;
    for (int v = tid; v < nv; v += BS) out[v] = s_d[v];
    if constexpr (SOLO) {
        // the bitmaps are no longer needed: the waves' counts in their place
        solo_report<INF, BS>(solo, s_d, chunks * kBlkChunk, rounds,
                             reinterpret_cast<int64_t *>(s_bits[0]));
    }
}

// A small graph solved whole with its edges in registers, EPT per thread: a
// round only reads LDS, a source's distance per edge, and relaxes the edges
// whose source fell. Bound by LDS reads and the vector units, 2-3 us a round at
// 32 edges per thread. R-MAT of 2^11 vertices x 16: 35 us on the device against 51
// in k_lds_solve, which reads the live chunks again every round; uniform 7000 x
// 4.6 35 against 75, grid 40 x 50 57 against 141, R-MAT 8 x 8 12 against 17.
template <class WT, int EPT>
__global__ __launch_bounds__(kSoloThreads) void k_reg_solve(const SoloArgs solo,
                                                            const int32_t *__restrict__ src,
                                                            const int32_t *__restrict__ dst,
                                                            const uint32_t *__restrict__ wts, int E,
                                                            uint32_t *__restrict__ dist)
{
    constexpr uint32_t INF = WT::INF;
    constexpr int kStep = EPT > 16 ? 4 : 8;  // distances in flight
    static_assert(EPT % kStep == 0, "whole steps");
    __shared__ uint32_t s_d[kLdsVerts[1]];
    __shared__ int64_t s_rep[2 * kSoloThreads / 64];
    __shared__ int s_more[3];
    const int tid = threadIdx.x, lane = __lane_id(), nv = solo.task.nv;
    uint32_t st[EPT], w[EPT], du[EPT];  // source | destination << 16 (ids below 2^15)
#pragma unroll
    for (int k = 0; k < EPT; k++) {
        const int e = k * kSoloThreads + tid;
        st[k] = w[k] = 0u;
        du[k] = 0u;  // no edge: never lowered
        if (e < E) {
            st[k] = (uint32_t)src[e] | (uint32_t)dst[e] << 16;
            if constexpr (WT::kWeighted) w[k] = wts[e];
            du[k] = INF;
        }
    }
    for (int v = tid; v < nv; v += kSoloThreads) s_d[v] = INF;
    if (tid < 3) s_more[tid] = 0;
    __syncthreads();
    if (tid == 0) s_d[solo.task.source] = 0u;
    __syncthreads();
    int32_t rounds = 0, relaxed = 0;
    for (;; rounds++) {
        if (rounds >= solo.limit) {
            rounds = -1;
            break;
        }
        bool ch = false;
#pragma unroll
        for (int k0 = 0; k0 < EPT; k0 += kStep) {
            uint32_t nu[kStep];
#pragma unroll
            for (int k = 0; k < kStep; k++) {
                // unpacked here every round: kept unpacked, 32 more registers spill
                if constexpr (EPT > 16) asm volatile("" : "+v"(st[k0 + k]));
                nu[k] = *(volatile uint32_t *)&s_d[st[k0 + k] & 0xFFFFu];
            }
            bool lower = false;
#pragma unroll
            for (int k = 0; k < kStep; k++) lower |= nu[k] < du[k0 + k];
            if (__ballot(lower) == 0) continue;
            ch = true;  // a source fell: another round, which may lower nothing
#pragma unroll
            for (int k = 0; k < kStep; k++) {
                if (nu[k] >= du[k0 + k]) continue;
                du[k0 + k] = nu[k];
                relaxed++;
                atomicMin(&s_d[st[k0 + k] >> 16], WT::add(nu[k], w[k0 + k]));
            }
        }
        // flags of three rounds: the one cleared here was read two rounds ago
        if (tid == 0) s_more[(rounds + 1) % 3] = 0;
        if (ch && lane == 0) s_more[rounds % 3] = 1;
        __syncthreads();
        if (s_more[rounds % 3] == 0) {
            rounds++;
            break;
        }
    }
    for (int v = tid; v < nv; v += kSoloThreads) dist[v] = s_d[v];
    solo_report<INF, kSoloThreads>(solo, s_d, wave_sum32(relaxed), rounds, s_rep);
}

template <class WT>
void launch_lds_t(int c, unsigned n, hipStream_t s, const BatchTask *tasks, sssp_graph *g)
{
    switch (c) {
    case 1:
        k_lds_solve<WT, 1024, kLdsVerts[1]><<<n, 1024, 0, s>>>(
            tasks, SoloArgs{}, g->bcounter, g->row_ptr, g->el_src, g->el_dst, g->el_w, g->E, g->el_first,
            g->bdist);
        break;
    case 2:
        k_lds_solve<WT, 1024, kLdsVerts[2]><<<n, 1024, 0, s>>>(
            tasks, SoloArgs{}, g->bcounter, g->row_ptr, g->el_src, g->el_dst, g->el_w, g->E, g->el_first,
            g->bdist);
        break;
    default:
        k_lds_solve<WT, 256, kLdsVerts[3]><<<n, 256, 0, s>>>(
            tasks, SoloArgs{}, g->bcounter, g->row_ptr, g->el_src, g->el_dst, g->el_w, g->E, g->el_first,
            g->bdist);
        break;
    }
    SSSP_LAUNCH_CHECK("k_lds_solve");
}

template <class WT>
void launch_solo_t(sssp_graph *g, int32_t source, int32_t limit)
{
    SoloArgs a{};
    a.task = BatchTask{0, 0, g->V, source};
    a.vperm = g->vperm;
    a.dout = g->dout;
    a.mirror = g->ctrl_host_dev;
    a.limit = limit;
    const int E = (int)g->E;
    auto reg = [&](auto kernel) {
        kernel<<<1, kSoloThreads, 0, g->stream>>>(a, g->el_src, g->el_dst, g->el_w, E, g->dist);
    };
    static_assert(kRegEdges == 32 * kSoloThreads, "more edges need el_first");
    if (E <= 8 * kSoloThreads) reg(k_reg_solve<WT, 8>);
    else if (E <= 16 * kSoloThreads) reg(k_reg_solve<WT, 16>);
    else if (E <= 32 * kSoloThreads) reg(k_reg_solve<WT, 32>);
    else
        k_lds_solve<WT, kSoloThreads, kLdsVerts[1], true><<<1, kSoloThreads, 0, g->stream>>>(
            nullptr, a, nullptr, g->row_ptr, g->el_src, g->el_dst, g->el_w, g->E, g->el_first,
            g->dist);
    SSSP_LAUNCH_CHECK("solve of one small graph");
}

template <int BS>
void launch_wg(int wtype, unsigned grid, hipStream_t s, const BatchTask *tasks, int32_t ntasks,
               int32_t *counter, sssp_graph *g, uint32_t *bdist, int32_t *scratch, int64_t maxv)
{
    if (wtype == SSSP_W_F32)
        k_wg_solve<WF32, BS><<<grid, BS, 0, s>>>(tasks, ntasks, counter, g->row_ptr, g->el_dst,
                                                 g->el_w, bdist, scratch, maxv, g->bround);
    else
        k_wg_solve<WU32, BS><<<grid, BS, 0, s>>>(tasks, ntasks, counter, g->row_ptr, g->el_dst,
                                                 g->el_w, bdist, scratch, maxv, g->bround);
    SSSP_LAUNCH_CHECK("k_wg_solve");
}

struct Config {
    int policy;      // 1 workgroup per task, 2 merged frontier / sequential
    int bs;          // policy 1 block size
    int wgpcu;       // policy 1 workgroups per CU
    double frac;     // policy 2 push/all frontier threshold
    int push_chunk;  // policy 2 sparse push chunk bucket
};

void ensure_batch_buffers(sssp_graph *g, int64_t dist_elems, int32_t ntasks, int32_t nwg,
                          int64_t maxv)
{
    if (dist_elems > g->bdist_elems) {
        dfree(g->bdist);
        g->bdist = nullptr;
        g->bdist = dmalloc<uint32_t>((size_t)dist_elems);
        g->bdist_elems = dist_elems;
    }
    if (ntasks > g->btask_cap) {
        dfree(g->btasks);
        g->btasks = nullptr;
        g->btasks = dmalloc<BatchTask>((size_t)ntasks);
        g->btask_cap = ntasks;
    }
    if (!g->bcounter) g->bcounter = dmalloc<int32_t>(2);
    // per-workgroup scratch = [queue a | queue b | stamps], each `stride`
    // entries; the stride only grows, so stamp regions never move onto old
    // queue contents
    if (nwg > 0 && (maxv > g->bscratch_stride || nwg > g->bround_cap)) {
        const int64_t stride = std::max<int64_t>(maxv, g->bscratch_stride);
        const int32_t cap = std::max<int32_t>(nwg, g->bround_cap);
        const int64_t need = (int64_t)cap * 3 * stride;
        dfree(g->bscratch);
        dfree(g->bround);
        g->bscratch = nullptr;
        g->bround = nullptr;
        g->bscratch = dmalloc<int32_t>((size_t)need);
        g->bscratch_elems = need;
        g->bscratch_stride = stride;
        g->bround = dmalloc<int32_t>((size_t)cap);
        g->bround_cap = cap;
        // stamps start below every round number the kernel will use
        SSSP_HIP(hipMemsetAsync(g->bscratch, 0, 4 * (size_t)need, g->stream));
        SSSP_HIP(hipMemsetAsync(g->bround, 0, 4 * (size_t)cap, g->stream));
    }
}

// Tasks of each class (see kLdsVerts), in the order they are uploaded.
struct TaskCounts {
    int32_t n[kLdsClasses] = {};
};

// Policy 1: tasks already uploaded, class by class; captures the launches (counter
// reset, the kernel of each class) in a hipGraph keyed on their shape and
// replays it.
double run_wg(sssp_graph *g, const TaskCounts &tc, int64_t maxv, int bs, int wgpcu)
{
    hipStream_t s = g->stream;
    const int32_t ntasks = tc.n[0];  // solved in global memory
    if (ntasks > 0 && maxv > g->bscratch_stride)
        throw Error{SSSP_ERR_INTERNAL, "batch scratch too small"};
    maxv = g->bscratch_stride;
    const int32_t nwg = std::min(g->cu_count * wgpcu, ntasks);
    if (ntasks == 0) bs = 0;  // no launch reads it: one capture serves every setting
    ensure_chunk_sources(g);
    const int64_t key[10] = {ntasks, maxv, bs, nwg, (int64_t)(uintptr_t)g->bdist,
                             (int64_t)(uintptr_t)g->bscratch, (int64_t)(uintptr_t)g->btasks,
                             (int64_t)(uintptr_t)g->bround, tc.n[1] + ((int64_t)tc.n[2] << 32),
                             tc.n[3]};
    if (!g->batch_exec || std::memcmp(key, g->batch_key, sizeof(key)) != 0) {
        if (g->batch_exec) {
            (void)hipGraphExecDestroy((hipGraphExec_t)g->batch_exec);
            g->batch_exec = nullptr;
        }
        SSSP_HIP(hipStreamSynchronize(s));
        hipGraph_t graph;
        SSSP_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        k_batch_reset<<<1, 64, 0, s>>>(g->bcounter);
        const BatchTask *tasks = static_cast<const BatchTask *>(g->btasks);
        if (ntasks > 0) {
            switch (bs) {
            case 256: launch_wg<256>(g->wtype, nwg, s, tasks, ntasks, g->bcounter, g, g->bdist, g->bscratch, maxv); break;
            case 512: launch_wg<512>(g->wtype, nwg, s, tasks, ntasks, g->bcounter, g, g->bdist, g->bscratch, maxv); break;
            default: launch_wg<1024>(g->wtype, nwg, s, tasks, ntasks, g->bcounter, g, g->bdist, g->bscratch, maxv); break;
            }
            tasks += ntasks;
        }
        for (int c = 1; c < kLdsClasses; c++) {
            if (tc.n[c] == 0) continue;
            if (g->wtype == SSSP_W_F32) launch_lds_t<WF32>(c, (unsigned)tc.n[c], s, tasks, g);
            else launch_lds_t<WU32>(c, (unsigned)tc.n[c], s, tasks, g);
            tasks += tc.n[c];
        }
        SSSP_HIP(hipStreamEndCapture(s, &graph));
        hipGraphExec_t exec;
        const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        SSSP_HIP(e);
        g->batch_exec = exec;
        std::memcpy(g->batch_key, key, sizeof(key));
    }
    SSSP_HIP(hipEventRecord(g->ev_a, s));
    SSSP_HIP(hipGraphLaunch((hipGraphExec_t)g->batch_exec, s));
    SSSP_HIP(hipEventRecord(g->ev_b, s));
    SSSP_HIP(hipEventSynchronize(g->ev_b));
    float ms = 0.f;
    SSSP_HIP(hipEventElapsedTime(&ms, g->ev_a, g->ev_b));
    int32_t flags[2] = {0, 0};
    SSSP_HIP(hipMemcpy(flags, g->bcounter, sizeof(flags), hipMemcpyDeviceToHost));
    if (flags[1]) throw Error{SSSP_ERR_INTERNAL, "batched solve exceeded its round bound"};
    return ms;
}

TaskCounts upload_tasks(sssp_graph *g, const std::vector<BatchTask> &tasks,
                        const std::vector<int64_t> &work)
{
    // by class, largest tasks first (longest-processing-time order)
    TaskCounts tc;
    std::vector<size_t> order(tasks.size());
    std::iota(order.begin(), order.end(), 0);
    std::vector<int> cls(tasks.size());
    for (size_t i = 0; i < tasks.size(); i++) tc.n[cls[i] = lds_class(tasks[i].nv)]++;
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) {
        return cls[a] != cls[b] ? cls[a] < cls[b] : work[a] > work[b];
    });
    std::vector<BatchTask> sorted(tasks.size());
    for (size_t i = 0; i < order.size(); i++) sorted[i] = tasks[order[i]];
    SSSP_HIP(hipMemcpyAsync(g->btasks, sorted.data(), sizeof(BatchTask) * sorted.size(),
                            hipMemcpyHostToDevice, g->stream));
    return tc;
}

void prepare_multi(sssp_graph *g, int32_t n);
double run_multi(sssp_graph *g, const int32_t *sources, int32_t n);

// ---- many sources on one graph ----------------------------------------------
// ready: called when every allocation is made, before the solves.
using Ready = std::function<void()>;
double batch_sources(sssp_graph *g, const int32_t *sources, int32_t n, const Config &c,
                     const Ready &ready = {})
{
    const int64_t V = g->V;
    if (c.policy == 3) {
        ensure_batch_buffers(g, (int64_t)n * V, 0, 0, 0);
        prepare_multi(g, n);
        if (ready) ready();
        return run_multi(g, sources, n);
    }
    if (c.policy == 1) {
        // (scratch only for tasks solved in global memory)
        const int32_t nwg =
            lds_class(V) == 0 ? std::min<int32_t>(n, g->cu_count * c.wgpcu) : 0;
        ensure_batch_buffers(g, (int64_t)n * V, n, nwg, V);
        ensure_chunk_sources(g);
        if (ready) ready();
        std::vector<BatchTask> tasks((size_t)n);
        std::vector<int64_t> work((size_t)n, 1);
        for (int32_t i = 0; i < n; i++) tasks[(size_t)i] = BatchTask{0, (int64_t)i * V, (int32_t)V, sources[i]};
        // (their work is equal: order is preserved)
        double ms = run_wg(g, upload_tasks(g, tasks, work), V, c.bs, c.wgpcu);
        if (g->vperm) {
            // rows to the caller's vertex order, one row at a time through
            // dout (timed with the solve)
            hipStream_t s = g->stream;
            SSSP_HIP(hipEventRecord(g->ev_a, s));
            for (int32_t i = 0; i < n; i++) {
                uint32_t *row = g->bdist + (int64_t)i * V;
                unpermute_rows(row, g->vperm, V, 1, g->dout, s);
                SSSP_HIP(hipMemcpyAsync(row, g->dout, 4 * (size_t)V, hipMemcpyDeviceToDevice, s));
            }
            SSSP_HIP(hipEventRecord(g->ev_b, s));
            SSSP_HIP(hipEventSynchronize(g->ev_b));
            float extra = 0.f;
            SSSP_HIP(hipEventElapsedTime(&extra, g->ev_a, g->ev_b));
            ms += extra;
        }
        return ms;
    }
    ensure_batch_buffers(g, (int64_t)n * V, 0, 0, 0);
    if (ready) ready();
    const double saved = g->push_edge_frac;
    const int saved_chunk = g->push_chunk;
    g->push_edge_frac = c.frac;
    g->push_chunk = c.push_chunk;
    double total = 0;
    for (int32_t i = 0; i < n; i++) {
        sssp_stats st{};
        solve(g, &sources[i], 1, SSSP_SCHED_HEURISTIC, &st);
        SSSP_HIP(hipMemcpyAsync(g->bdist + (int64_t)i * V, g->dout, 4 * (size_t)V,
                                hipMemcpyDeviceToDevice, g->stream));
        total += st.t_solve_ms;
    }
    SSSP_HIP(hipStreamSynchronize(g->stream));
    g->push_edge_frac = saved;
    g->push_chunk = saved_chunk;
    return total;
}

// ---- policy 3: vertex-major all-edge passes ---------------------------------
constexpr int kMThreads = 256;  // sources per chunk: one thread per source
constexpr int kMBlock = 1 << kMBits;

// Pass state on the device: what each pass ran, whether it lowered anything,
// an estimate of how many rows it lowered (one wave in MultiArgs::every counts:
// one addition per wave to one counter, from 200 thousand waves, took 1.8 ms of
// every light pass at R-MAT scale 20), the last full pass before each, and
// the number of the first pass of the captured run.
struct MultiCtl {
    int32_t kind[64];
    int32_t changed[64];
    int32_t low[64];
    int32_t full[64];
    int32_t base;
};
enum { kMultiLight = 1, kMultiFull = 2, kMultiIdle = 3 };

// One tile of a vertex-major pass: thread s holds source s's minima for the
// tile's 16-vertex destination block in its LDS column, lowers them with the
// tile's records (a record's source row gathered for all sources at once), and
// writes back what is below the distances in global memory. A record is
// relaxed only when its source's row was lowered in pass `since` or later
// (stamp): before that, its list was last relaxed against the row as it still
// is. Rows the tile lowers are stamped with this pass. Returns the rows this
// wave lowered.
// A wave takes 64 records at a time, one per lane: their stamps are one gather,
// the live ones a ballot, and each live record is broadcast from its lane. The
// next 64 records' stamps and the records after those load under this group's
// row gathers. (With a record per step in scalar registers each step waited
// for its records and then for their stamps: a pass took as long as relaxing
// every record.)
template <class WT>
__device__ __forceinline__ int multi_tile(const BlkTile &t, const MRec *__restrict__ rec,
                                          uint32_t *D, int32_t n, int32_t *stamp, int32_t since,
                                          int32_t pass, uint32_t (&ld)[kMBlock][kMThreads])
{
    constexpr uint32_t INF = WT::INF;
    const int s = threadIdx.x, lane = __lane_id();
    const bool act = s < n;
    const int64_t base = (int64_t)t.blk << kMBits;
    // each thread touches only its own column: no barrier is needed
#pragma unroll
    for (int v = 0; v < kMBlock; v++) ld[v][s] = INF;
    struct Rec {
        int32_t src, loc;
        uint32_t w;
    };
    auto fetch = [&](int64_t e) {
        Rec r{0, 0, 0u};
        if (e < t.e1) {
            const MRec m = rec[e];
            r = Rec{m.src, m.loc, m.w};
        }
        return r;
    };
    auto mark = [&](int64_t e, const Rec &r) { return e < t.e1 ? stamp[r.src] : since - 1; };
    const uint32_t *const Ds = D + s;
    auto row = [&](const Rec &r, int i) {  // of lane i's record, this thread's source
        const int32_t u = __builtin_amdgcn_readlane(r.src, i);
        return act ? Ds[(int64_t)u * n] : INF;
    };
    auto relax = [&](const Rec &r, int i, uint32_t du) {
        const uint32_t w = __builtin_amdgcn_readlane(r.w, i);
        const int32_t loc = __builtin_amdgcn_readlane(r.loc, i);
        if (du == INF) return;
        const uint32_t cand = WT::add(du, w);
        if (cand < ld[loc][s]) ld[loc][s] = cand;
    };
    bool any = false;
    Rec r0 = fetch(t.e0 + lane), r1 = fetch(t.e0 + 64 + lane);
    int32_t st = mark(t.e0 + lane, r0);
    for (int64_t e = t.e0; e < t.e1; e += 64) {
        uint64_t m = __ballot(st >= since);
        const Rec r2 = fetch(e + 128 + lane);
        const int32_t st1 = mark(e + 64 + lane, r1);
        any |= m != 0;
        // eight row gathers in flight. Measured at R-MAT scale 20 x 256
        // sources (GTEPS, all records live): 64-vertex blocks (64
        // KB of LDS, 2 waves per SIMD) 23.0 with 8 in flight, 25.8-27.4 with 16;
        // 32-vertex blocks 44.0 (16); 16-vertex blocks (16 KB, 8 workgroups per
        // CU) 51.4 (16), 54.7 (8); 8-vertex blocks 51.1 (16)
        constexpr int R = 8;
        // (whole eights without a test per record: 5-15 % of a pass; sixteen in
        // flight 2-4 % more, not worth the registers)
        for (int left = __popcll(m); left >= R; left -= R) {
            int at[R];
            uint32_t du[R];
#pragma unroll
            for (int q = 0; q < R; q++) {
                at[q] = __builtin_ctzll(m);
                m &= m - 1;
            }
#pragma unroll
            for (int q = 0; q < R; q++) du[q] = row(r0, at[q]);
#pragma unroll
            for (int q = 0; q < R; q++) relax(r0, at[q], du[q]);
        }
        while (m != 0) {
            int at[R];
            uint32_t du[R];
            int k = 0;
#pragma unroll
            for (int q = 0; q < R; q++) {
                at[q] = m != 0 ? __builtin_ctzll(m) : at[q > 0 ? q - 1 : 0];
                if (m != 0) k = q + 1;
                m &= m - 1;
            }
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < k) du[q] = row(r0, at[q]);
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < k) relax(r0, at[q], du[q]);
        }
        r0 = r1;
        r1 = r2;
        st = st1;
    }
    if (!any) return 0;  // wave-uniform
    // the touched rows' distances, all in flight together (a minimum is INF past
    // the end, and where nothing was relaxed into it)
    int rows = 0;
    uint32_t cur[kMBlock];
#pragma unroll
    for (int v = 0; v < kMBlock; v++) {
        cur[v] = 0u;
        if (ld[v][s] != INF) cur[v] = D[(base + v) * n + s];
    }
#pragma unroll
    for (int v = 0; v < kMBlock; v++) {
        const uint32_t nv = ld[v][s];
        const bool low = nv < cur[v];
        if (low) {
            uint32_t *const p = &D[(base + v) * n + s];
            if (t.split)
                __hip_atomic_fetch_min(p, nv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
                *p = nv;  // only this workgroup writes the block
        }
        if (__ballot(low) != 0) {
            rows++;
            if (lane == 0) stamp[base + v] = pass;
        }
    }
    return rows;
}

struct MultiArgs {
    const BlkTile *tile, *ltile;  // of all records, of the light ones
    const MRec *rec, *lrec;
    int32_t n_tile, n_ltile;  // n_ltile 0: full passes only
    uint32_t *D;
    int32_t n;
    int32_t *stamp;
    MultiCtl *ctl;
    int32_t every;       // a power of two: blocks whose hash is 0 modulo it count their rows
    int32_t light_stop;  // light passes go on while their count is this much, or more than
                         // the light pass before
};

// What pass p (from 1) runs; every workgroup reads the same values.
__device__ __forceinline__ int multi_kind(const MultiArgs &a, int32_t p)
{
    if (p == 1) return a.n_ltile > 0 ? kMultiLight : kMultiFull;
    const MultiCtl *c = a.ctl;
    const int i1 = (p - 1) & 63, i2 = (p - 2) & 63;
    const int prev = c->kind[i1];
    const int32_t low = c->low[i1];
    if (prev == kMultiIdle) return kMultiIdle;
    if (prev == kMultiFull) {
        if (c->changed[i1] == 0) return kMultiIdle;
        // few rows lowered: the stamps make another full pass cheap
        return a.n_ltile > 0 && low >= a.light_stop && p < kLightMaxPasses ? kMultiLight
                                                                           : kMultiFull;
    }
    const int32_t before = p > 2 && c->kind[i2] == kMultiLight ? c->low[i2] : 0;
    return (low >= a.light_stop || low > before) && low > 0 && p < kLightMaxPasses ? kMultiLight
                                                                                   : kMultiFull;
}

// One pass per launch, one workgroup per tile. The pass number is the run's
// base + k (base in device memory, so a captured run of passes is replayed as
// the next run). As the blocked passes of a single solve, a pass finds out
// what it runs from the pass before it: light passes (the light records alone)
// until they lower few rows, a full pass, light passes again, until a full pass
// lowers nothing; passes after that return at once. R-MAT 20 x 16, 256 sources:
// 21 passes over every record took 72.6 ms; now two full passes of 2.9 ms (17 GB
// of row gathers at 6 TB/s), 24 light ones of 0.3 ms and a few full ones over the
// few rows still changing, 15.4 ms in all.
template <class WT>
__global__ __launch_bounds__(kMThreads) void k_multi_pass(const MultiArgs a, int32_t k)
{
    MultiCtl *c = a.ctl;
    const int32_t pass = c->base + k;
    const int kind = multi_kind(a, pass);
    const int32_t last_full = pass == 1 ? 0 : c->full[(pass - 1) & 63];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->kind[pass & 63] = kind;
        c->full[pass & 63] = kind == kMultiFull ? pass : last_full;
        c->low[(pass + 1) & 63] = 0;
        c->changed[(pass + 1) & 63] = 0;
    }
    if (kind == kMultiIdle) return;
    const bool light = kind == kMultiLight;
    if ((int)blockIdx.x >= (light ? a.n_ltile : a.n_tile)) return;
    __shared__ uint32_t ld[kMBlock][kMThreads];
    const BlkTile t = (light ? a.ltile : a.tile)[blockIdx.x];
    const int rows = multi_tile<WT>(t, light ? a.lrec : a.rec, a.D, a.n, a.stamp,
                                    light ? pass - 1 : last_full, pass, ld);
    if (rows != 0 && __lane_id() == 0) {
        c->changed[pass & 63] = 1;
        if ((((uint32_t)t.blk * 0x9E3779B1u) >> 16 & (uint32_t)(a.every - 1)) == 0)
            atomicAdd(&c->low[pass & 63], rows);
    }
}

// D[v * n + s] = INF, D[sources[s] * n + s] = 0; stamps: -1 (never lowered),
// k_multi_sources sets the sources'
template <class WT>
__global__ __launch_bounds__(kBlock) void k_multi_init(uint32_t *D, int32_t n, int64_t V,
                                                       const int32_t *sources, int32_t *stamp)
{
    const int64_t total = V * n;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * kBlock) {
        const int64_t v = i / n;
        const int32_t s = (int32_t)(i - v * n);
        D[i] = sources[s] == v ? 0u : WT::INF;
        if (s == 0) stamp[v] = -1;
    }
}

// the sources' rows count as lowered before the first pass; first pass: 1
__global__ void k_multi_sources(const int32_t *sources, int32_t n, int32_t *stamp, MultiCtl *c)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) stamp[sources[i]] = 0;
    if (threadIdx.x == 0) {
        c->base = 1;
        c->low[1] = 0;
        c->changed[1] = 0;
    }
}

// out[s * V + v] = D[slot(v) * n + s] through 64 x 64 LDS tiles (slot(v) =
// vperm[v] on a relabelled graph, else v): per source, caller vertex order
__global__ __launch_bounds__(kBlock) void k_multi_out(const uint32_t *D, int32_t n, int64_t V,
                                                      const int32_t *vperm, uint32_t *out)
{
    __shared__ uint32_t tl[64][65];
    const int64_t v0 = (int64_t)blockIdx.x * 64;
    const int s0 = blockIdx.y * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 64 x 4
    for (int r = ty; r < 64; r += 4) {
        const int64_t v = v0 + r;
        const int s = s0 + tx;
        if (v < V && s < n) tl[r][tx] = D[(vperm ? (int64_t)vperm[v] : v) * n + s];
    }
    __syncthreads();
    for (int r = ty; r < 64; r += 4) {
        const int s = s0 + r;
        const int64_t v = v0 + tx;
        if (v < V && s < n) out[(int64_t)s * V + v] = tl[tx][r];
    }
}

// base[0] += k (the next run of captured passes)
__global__ void k_advance_base(int32_t *base, int32_t k)
{
    if (threadIdx.x == 0) base[0] += k;
}

// Light passes stop once they lower fewer rows than this share of the vertices
// with out-edges: 0.02 / 0.05 / 0.1 / 0.2 took 17.2 / 17.1 / 15.4 / 17.1 ms at
// R-MAT 20 x 16 with 256 sources (the stamps keep the next full pass cheap).
constexpr double kMultiStopFrac = 0.1;
constexpr int32_t kMultiRun = 32;  // passes per captured run (the flag ring has 64)

MultiArgs multi_args(sssp_graph *g, int32_t m)
{
    MultiArgs a{};
    a.tile = g->m_tile;
    a.ltile = g->m_ltile;
    a.rec = g->m_rec;
    a.lrec = g->m_lrec;
    a.n_tile = g->n_mtile;
    a.n_ltile = g->n_mltile;
    a.D = g->mdist;
    a.n = m;
    a.stamp = g->mstamp;
    a.ctl = static_cast<MultiCtl *>(g->mctl);
    a.every = 1;
    // about 2048 blocks count; rows once per wave that lowers them
    while (a.every < 1 << 15 && (g->V >> kMBits) / (2 * a.every) >= 2048) a.every *= 2;
    a.light_stop = (int32_t)std::min<double>(
        kMultiStopFrac * g->n_nzo * ((m + 63) / 64) / a.every, 1 << 30);
    return a;
}

void launch_multi_pass(sssp_graph *g, const MultiArgs &a, int32_t k, hipStream_t s)
{
    const unsigned grid = (unsigned)std::max(a.n_tile, a.n_ltile);
    if (g->wtype == SSSP_W_U32) k_multi_pass<WU32><<<grid, kMThreads, 0, s>>>(a, k);
    else k_multi_pass<WF32><<<grid, kMThreads, 0, s>>>(a, k);
}

void launch_multi_init(sssp_graph *g, const MultiArgs &a, const int32_t *sources, hipStream_t s)
{
    const int64_t V = g->V;
    const unsigned gi = (unsigned)std::min<int64_t>((V * a.n + kBlock - 1) / kBlock, 65536);
    if (g->wtype == SSSP_W_U32)
        k_multi_init<WU32><<<gi, kBlock, 0, s>>>(a.D, a.n, V, sources, a.stamp);
    else k_multi_init<WF32><<<gi, kBlock, 0, s>>>(a.D, a.n, V, sources, a.stamp);
    k_multi_sources<<<1, kBlock, 0, s>>>(sources, a.n, a.stamp, a.ctl);
}

// The captured launches of one chunk of at most 256 sources, keyed on chunk
// shape and buffers: `first` initialises the vertex-major distances, the stamps
// and the pass state, runs kMultiRun passes and transposes the result into the per-source output; `more` (captured when a
// chunk first needs it) advances the pass
// base by kMultiRun and runs the next kMultiRun passes and the transpose.
// Passes after the fixpoint return at once.
hipGraphExec_t capture_multi(sssp_graph *g, int32_t c0, int32_t m, bool first)
{
    hipStream_t s = g->stream;
    const int64_t V = g->V;
    SSSP_HIP(hipStreamSynchronize(s));
    const MultiArgs a = multi_args(g, m);
    hipGraph_t graph;
    SSSP_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    if (first) {
        launch_multi_init(g, a, g->msrc + c0, s);
    } else {
        k_advance_base<<<1, 64, 0, s>>>(&a.ctl->base, kMultiRun);
    }
    if (g->n_mtile > 0)
        for (int32_t k = 0; k < kMultiRun; k++) launch_multi_pass(g, a, k, s);
    k_multi_out<<<dim3((unsigned)((V + 63) / 64), (unsigned)((m + 63) / 64)), kBlock, 0, s>>>(
        g->mdist, m, V, g->vperm, g->bdist + (int64_t)c0 * V);
    const hipError_t le = hipGetLastError();
    const hipError_t ce = hipStreamEndCapture(s, &graph);
    if (le != hipSuccess || ce != hipSuccess) {
        if (ce == hipSuccess) (void)hipGraphDestroy(graph);
        throw Error{SSSP_ERR_HIP, std::string("capturing the batch launch failed: ") +
                                      hipGetErrorString(le != hipSuccess ? le : ce)};
    }
    hipGraphExec_t exec;
    const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    SSSP_HIP(ie);
    return exec;
}

// The slot of a chunk's captured launches, `first` captured.
int multi_graphs(sssp_graph *g, int32_t c0, int32_t m)
{
    const int64_t V = g->V;
    const int64_t key[kMultiKey] = {m,
                                    c0,
                                    V,
                                    g->n_mtile,
                                    (int64_t)(uintptr_t)g->mctl,
                                    (int64_t)(uintptr_t)g->mdist,
                                    (int64_t)(uintptr_t)g->bdist,
                                    (int64_t)(uintptr_t)g->msrc,
                                    g->wtype,
                                    (int64_t)(uintptr_t)g->m_tile};
    for (int i = 0; i < kMultiSlots; i++)
        if (g->mexec[i][0] && std::memcmp(key, g->mkey[i], sizeof(key)) == 0) return i;
    const int slot = g->mnext;
    g->mnext = (g->mnext + 1) % kMultiSlots;
    for (int j = 0; j < 2; j++)
        if (g->mexec[slot][j]) {
            (void)hipGraphExecDestroy((hipGraphExec_t)g->mexec[slot][j]);
            g->mexec[slot][j] = nullptr;
        }
    g->mexec[slot][0] = capture_multi(g, c0, m, true);
    std::memcpy(g->mkey[slot], key, sizeof(key));
    return slot;
}

// Passes among [first, first + count) that did work, from the host's copy of
// what they ran; *done: one of them was idle (the fixpoint was reached).
int32_t multi_ran(const int32_t *kind, int32_t first, int32_t count, bool *done)
{
    for (int32_t i = 0; i < count; i++)
        if (kind[(first + i) & 63] == kMultiIdle) {
            *done = true;
            return i;
        }
    return count;
}

// Passes of one chunk as queued launches (batch_capture = 0): four at a time,
// the host reading what they ran after each four. Returns the passes run.
int32_t multi_passes_launched(sssp_graph *g, const MultiArgs &a)
{
    hipStream_t s = g->stream;
    int32_t ran = 0;
    bool done = g->n_mtile == 0;
    while (!done) {
        for (int i = 0; i < 4; i++) {
            launch_multi_pass(g, a, ran + i, s);
            SSSP_LAUNCH_CHECK("k_multi_pass");
        }
        SSSP_HIP(hipMemcpyAsync(g->ctrl_host->changed, a.ctl->kind, 4 * 64, hipMemcpyDeviceToHost,
                                s));
        SSSP_HIP(hipStreamSynchronize(s));
        ran += multi_ran(g->ctrl_host->changed, ran + 1, 4, &done);
        if (!done && ran > (int64_t)g->V + 4 + kLightMaxPasses)
            throw Error{SSSP_ERR_NOT_CONVERGED, "multi-source passes exceeded V passes"};
    }
    return ran;
}

// Layout, buffers and the first chunk's captured launches of a policy-3 batch.
void prepare_multi(sssp_graph *g, int32_t n)
{
    build_multi_layout(g);
    const int64_t V = g->V;
    const int32_t chunk = std::min<int32_t>(n, kMThreads);
    if ((int64_t)chunk * V > g->mdist_elems) {
        dfree(g->mdist);
        g->mdist = nullptr;
        g->mdist = dmalloc<uint32_t>((size_t)chunk * (size_t)V);
        g->mdist_elems = (int64_t)chunk * V;
    }
    if (n > g->msrc_cap) {
        dfree(g->msrc);
        g->msrc = nullptr;
        g->msrc = dmalloc<int32_t>((size_t)n);
        g->msrc_cap = n;
    }
    if (!g->mctl) g->mctl = dmalloc<MultiCtl>(1);
    if (!g->mstamp) g->mstamp = dmalloc<int32_t>((size_t)V);
    if (g->batch_capture) (void)multi_graphs(g, 0, chunk);
}

double run_multi(sssp_graph *g, const int32_t *sources, int32_t n)
{
    hipStream_t s = g->stream;
    const int64_t V = g->V;
    SSSP_HIP(hipMemcpyAsync(g->msrc, sources, 4 * (size_t)n, hipMemcpyHostToDevice, s));
    float total = 0.f;
    g->multi_passes = 0;
    for (int32_t c0 = 0; c0 < n; c0 += kMThreads) {
        const int32_t m = std::min<int32_t>(kMThreads, n - c0);
        if (g->batch_capture) {
            void **const mg = g->mexec[multi_graphs(g, c0, m)];
            SSSP_HIP(hipEventRecord(g->ev_a, s));
            bool done = g->n_mtile == 0;
            if (done) SSSP_HIP(hipGraphLaunch((hipGraphExec_t)mg[0], s));
            // replay until a run holds an idle pass (at most V + 1 passes and the
            // light ones, as the pass loop)
            for (int32_t run = 0; !done; run++) {
                if ((int64_t)run * kMultiRun > V + 1 + kLightMaxPasses)
                    throw Error{SSSP_ERR_NOT_CONVERGED, "multi-source passes exceeded V passes"};
                if (run == 1 && !mg[1]) mg[1] = capture_multi(g, c0, m, false);
                SSSP_HIP(hipGraphLaunch((hipGraphExec_t)mg[run > 0], s));
                SSSP_HIP(hipMemcpyAsync(g->ctrl_host->changed,
                                        static_cast<MultiCtl *>(g->mctl)->kind, 4 * 64,
                                        hipMemcpyDeviceToHost, s));
                SSSP_HIP(hipStreamSynchronize(s));
                g->multi_passes +=
                    multi_ran(g->ctrl_host->changed, 1 + run * kMultiRun, kMultiRun, &done);
            }
            SSSP_HIP(hipEventRecord(g->ev_b, s));
            SSSP_HIP(hipEventSynchronize(g->ev_b));
        } else {
            SSSP_HIP(hipEventRecord(g->ev_a, s));
            const MultiArgs a = multi_args(g, m);
            launch_multi_init(g, a, g->msrc + c0, s);
            SSSP_LAUNCH_CHECK("k_multi_init");
            g->multi_passes += multi_passes_launched(g, a);
            k_multi_out<<<dim3((unsigned)((V + 63) / 64), (unsigned)((m + 63) / 64)), kBlock, 0,
                          s>>>(g->mdist, m, V, g->vperm, g->bdist + (int64_t)c0 * V);
            SSSP_LAUNCH_CHECK("k_multi_out");
            SSSP_HIP(hipEventRecord(g->ev_b, s));
            SSSP_HIP(hipEventSynchronize(g->ev_b));
        }
        float ms = 0.f;
        SSSP_HIP(hipEventElapsedTime(&ms, g->ev_a, g->ev_b));
        total += ms;
    }
    return total;
}

// What a tuning call may choose from. one_graph: many sources on one graph
// (policy 3 applies); else a pack. workgroups: policy 1 has tasks for the
// persistent kernel, whose block size and workgroups per CU matter; rounds1,
// rounds2: policy 1 / 2 solves in rounds, whose threshold and chunk matter.
// What nothing reads has one candidate.
struct Choices {
    bool one_graph, workgroups, rounds1, rounds2;
};

std::vector<Config> candidates(const Choices &k)
{
    std::vector<Config> c;
    if (k.one_graph) c.push_back(Config{3, kMThreads, 1, 0.0, 0});
    auto thresholds = [&](int policy, int bs, int w, bool rounds) {
        if (!rounds) c.push_back(Config{policy, bs, w, 0.05, 1});
        for (double f : {0.02, 0.05, 0.15})
            for (int pc : {1, 2})
                if (rounds) c.push_back(Config{policy, bs, w, f, pc});
    };
    if (!k.workgroups) thresholds(1, 1024, 1, k.rounds1);
    for (int bs : {256, 512, 1024})
        for (int w : {1, 2, 4})
            if (k.workgroups) c.push_back(Config{1, bs, w, 0.05, 1});
    thresholds(2, 256, 2, k.rounds2);
    return c;
}

std::string describe(const Config &c, const Choices &k)
{
    char buf[160];
    if (c.policy == 1 && !k.workgroups)
        std::snprintf(buf, sizeof(buf), k.rounds1 ? "policy=workgroup_per_task push_edge_frac=%.3f push_chunk=%d"
                                                  : "policy=workgroup_per_task", c.frac, c.push_chunk);
    else if (c.policy == 1)
        std::snprintf(buf, sizeof(buf), "policy=workgroup_per_task block=%d wg_per_cu=%d", c.bs, c.wgpcu);
    else if (c.policy == 3)
        std::snprintf(buf, sizeof(buf), "policy=vertex_major_all_edge sources_per_chunk=%d", c.bs);
    else
        std::snprintf(buf, sizeof(buf), "policy=merged_frontier push_edge_frac=%.3f push_chunk=%d", c.frac,
                      c.push_chunk);
    return buf;
}

template <class Run>
Config autotune(Run &&run, const char *file, double *best_ms, const char *what, const Choices &k)
{
    std::vector<Config> cs = candidates(k);
    std::vector<double> t(cs.size(), 1e300);
    for (size_t i = 0; i < cs.size(); i++) {
        (void)run(cs[i]);  // warm-up (and graph capture)
        t[i] = std::min(run(cs[i]), run(cs[i]));
    }
    const size_t b = std::min_element(t.begin(), t.end()) - t.begin();
    if (file) {
        FILE *f = std::fopen(file, "w");
        if (!f) throw Error{SSSP_ERR_IO, std::string("cannot open tuning file ") + file};
        std::fprintf(f, "# autotune %s: min of 2 timed runs after 1 warm-up, device ms\n", what);
        for (size_t i = 0; i < cs.size(); i++)
            std::fprintf(f, "%s ms=%.4f%s\n", describe(cs[i], k).c_str(), t[i], i == b ? " best" : "");
        std::fclose(f);
    }
    if (best_ms) *best_ms = t[b];
    return cs[b];
}

Config default_config(sssp_graph *g, int32_t n)
{
    if (g->batch_policy)
        return Config{g->batch_policy, g->batch_bs, g->batch_wgpcu, g->push_edge_frac, g->push_chunk};
    // untuned: policy 3 for 32 or more sources on one graph (R-MAT scale 20
    // x 256 sources: 171-180 GTEPS against 11-12 for policy 1, 22-24 for policy 2), policy 2 below
    if (n >= 32) return Config{3, kMThreads, 1, 0.0, 0};
    return Config{2, 256, 2, g->push_edge_frac, g->push_chunk};
}

void fill_stats(sssp_stats *st, double ms, double edges)
{
    if (!st) return;
    std::memset(st, 0, sizeof(*st));
    st->t_solve_ms = ms;
    st->gteps = ms > 0 ? edges / (ms * 1e-3) / 1e9 : 0.0;
}

}  // namespace
}  // namespace sssp

using namespace sssp;

struct sssp_pack {
    sssp_graph *g = nullptr;  // the disjoint union of all graphs
    int32_t n = 0;
    std::vector<int64_t> voff;  // n+1 vertex offsets
    std::vector<int64_t> eoff;  // n+1 edge offsets
    int policy = 0, bs = 256, wgpcu = 2;
    double frac = 0.05;
    int push_chunk = 1;
};

namespace sssp {
namespace {

double pack_run(sssp_pack *p, const int32_t *local_sources, const Config &c)
{
    sssp_graph *g = p->g;
    const int32_t n = p->n;
    // the graphs at `at` as one frontier solve over the union (their distances
    // are in g->dout then; the other graphs' vertices stay unreached)
    auto merged = [&](const std::vector<int32_t> &at) {
        std::vector<int32_t> gs;
        for (int32_t k : at) gs.push_back((int32_t)(p->voff[k] + local_sources[k]));
        const double saved = g->push_edge_frac;
        const int saved_chunk = g->push_chunk;
        g->push_edge_frac = c.frac;
        g->push_chunk = c.push_chunk;
        sssp_stats st{};
        solve(g, gs.data(), (int32_t)gs.size(), SSSP_SCHED_HEURISTIC, &st);
        g->push_edge_frac = saved;
        g->push_chunk = saved_chunk;
        ensure_batch_buffers(g, g->V, 0, 0, 0);
        SSSP_HIP(hipMemcpyAsync(g->bdist, g->dout, 4 * (size_t)g->V, hipMemcpyDeviceToDevice,
                                g->stream));
        return st.t_solve_ms;
    };
    std::vector<int32_t> big;
    if (c.policy == 1) {
        // graphs that fit a workgroup's LDS, one workgroup each; the larger
        // ones share one full-chip solve (one workgroup each, in global
        // memory, 300 graphs of 2^14-2^16 vertices took 16.3 ms; the merged
        // solve of the larger 200 and the rest in LDS take 2.15)
        std::vector<BatchTask> tasks;
        std::vector<int64_t> work;
        for (int32_t k = 0; k < n; k++) {
            const int64_t nv = p->voff[k + 1] - p->voff[k];
            if (lds_class(nv) == 0) {
                big.push_back(k);
                continue;
            }
            tasks.push_back(BatchTask{p->voff[k], p->voff[k], (int32_t)nv,
                                      (int32_t)(p->voff[k] + local_sources[k])});
            work.push_back(p->eoff[k + 1] - p->eoff[k]);
        }
        double ms = big.empty() ? 0.0 : merged(big);
        if (!tasks.empty()) {
            ensure_batch_buffers(g, g->V, (int32_t)tasks.size(), 0, 0);
            ms += run_wg(g, upload_tasks(g, tasks, work), 0, c.bs, c.wgpcu);
        }
        SSSP_HIP(hipStreamSynchronize(g->stream));
        return ms;
    }
    for (int32_t k = 0; k < n; k++) big.push_back(k);
    const double ms = merged(big);
    SSSP_HIP(hipStreamSynchronize(g->stream));
    return ms;
}

std::vector<int32_t> source_slots(const sssp_graph *g, const int32_t *sources, int32_t n)
{
    std::vector<int32_t> out((size_t)n);
    for (int32_t i = 0; i < n; i++) out[(size_t)i] = slot_of(g, sources[i]);
    return out;
}

void check_pack_sources(const sssp_pack *p, const int32_t *sources)
{
    SSSP_REQUIRE(sources, "null sources");
    for (int32_t k = 0; k < p->n; k++)
        SSSP_REQUIRE(sources[k] >= 0 && sources[k] < p->voff[k + 1] - p->voff[k],
                     "pack source out of range for graph " + std::to_string(k));
}

}  // namespace

bool solo_fits(const sssp_graph *g)
{
    return g->V <= kSoloVerts && g->E <= (g->n_ttile > 0 ? kSoloLocalEdges : kSoloEdges);
}

void ensure_chunk_sources(sssp_graph *g)
{
    if (g->el_first) return;
    const int64_t nch = (g->E + kBlkChunk - 1) / kBlkChunk;
    g->el_first = dmalloc<int32_t>((size_t)nch + 1);
    k_chunk_sources<<<(unsigned)std::min<int64_t>(nch / kBlock + 1, 4096), kBlock, 0, g->stream>>>(
        g->el_src, nch, g->V, g->el_first);
    SSSP_LAUNCH_CHECK("k_chunk_sources");
}

void launch_solo(sssp_graph *g, int32_t source, bool hops, int32_t limit)
{
    if (hops) launch_solo_t<WUnit>(g, source, limit);
    else if (g->wtype == SSSP_W_F32) launch_solo_t<WF32>(g, source, limit);
    else launch_solo_t<WU32>(g, source, limit);
}
}  // namespace sssp

extern "C" {

int sssp_solve_batch(sssp_graph *g, const int32_t *sources, int32_t n, int32_t policy,
                     void *dist_out, sssp_stats *stats)
{
    return guard([&] {
        SSSP_REQUIRE(g && sources && n >= 1, "bad arguments");
        SSSP_REQUIRE(policy >= 0 && policy <= 3, "policy must be 0, 1, 2 or 3");
        for (int32_t i = 0; i < n; i++)
            SSSP_REQUIRE(sources[i] >= 0 && sources[i] < g->V, "source vertex out of range");
        SSSP_HIP(hipSetDevice(g->device));
        // the merged/sequential policy solves through g->dist: no single-solve
        // result (distances or BFS levels) survives a batch
        g->have_result = false;
        g->bfs_result = false;
        Config c = default_config(g, n);
        if (policy != 0 && policy != c.policy)
            c = (policy == 1)   ? Config{1, 1024, 1, 0.05, 1}
                : (policy == 3) ? Config{3, kMThreads, 1, 0.0, 0}
                                : Config{2, 256, 2, g->push_edge_frac, g->push_chunk};
        const std::vector<int32_t> slots = source_slots(g, sources, n);
        const size_t bytes = 4 * (size_t)n * (size_t)g->V;
        // the pages are faulted in under the solves alone: an allocation beside
        // it waits for the address space's lock (the first batch of R-MAT 20 x 16
        // with 256 sources, which makes some twenty, 84 ms against 42)
        std::optional<Prefault> pages;
        const double ms = batch_sources(g, slots.data(), n, c,
                                        [&] { pages.emplace(dist_out, bytes); });
        if (dist_out) {
            pages->join();
            download(g, dist_out, g->bdist, bytes);
        }
        fill_stats(stats, ms, (double)g->E * n);
        if (stats) stats->iterations = c.policy;
    });
}

int sssp_autotune_batch(sssp_graph *g, const int32_t *sources, int32_t n, const char *tuning_file,
                        double *best_ms)
{
    return guard([&] {
        SSSP_REQUIRE(g && sources && n >= 1, "bad arguments");
        for (int32_t i = 0; i < n; i++)
            SSSP_REQUIRE(sources[i] >= 0 && sources[i] < g->V, "source vertex out of range");
        SSSP_HIP(hipSetDevice(g->device));
        const std::vector<int32_t> slots = source_slots(g, sources, n);
        const Config b = autotune([&](const Config &c) { return batch_sources(g, slots.data(), n, c); },
                                  tuning_file, best_ms, "batch of sources",
                                  Choices{true, lds_class(g->V) == 0, false, !runs_passes(g, 1)});
        g->batch_policy = b.policy;
        g->batch_bs = b.bs;
        g->batch_wgpcu = b.wgpcu;
        if (b.policy == 2) {
            g->push_edge_frac = b.frac;
            g->push_chunk = b.push_chunk;
        }
    });
}

int sssp_pack_create(const int32_t *src, const int32_t *dst, const float *weights,
                     const int64_t *edge_offsets, const int32_t *vertex_counts, int32_t n_graphs,
                     int32_t device, sssp_pack **out)
{
    sssp_pack *p = nullptr;
    int rc = guard([&] {
        SSSP_REQUIRE(out && edge_offsets && vertex_counts && n_graphs >= 1, "bad arguments");
        *out = nullptr;
        p = new sssp_pack();
        p->n = n_graphs;
        p->voff.assign((size_t)n_graphs + 1, 0);
        p->eoff.assign(edge_offsets, edge_offsets + n_graphs + 1);
        SSSP_REQUIRE(p->eoff[0] == 0, "edge_offsets must start at 0");
        for (int32_t k = 0; k < n_graphs; k++) {
            SSSP_REQUIRE(vertex_counts[k] >= 1, "every graph needs a vertex");
            SSSP_REQUIRE(p->eoff[k + 1] >= p->eoff[k], "edge_offsets must not decrease");
            p->voff[k + 1] = p->voff[k] + vertex_counts[k];
        }
        const int64_t V = p->voff[n_graphs], E = p->eoff[n_graphs];
        SSSP_REQUIRE(V < ((int64_t)1 << 31) - 1, "packed vertex count must fit int32");
        SSSP_REQUIRE(E == 0 || (src && dst && weights), "null edge array");
        std::vector<int32_t> us((size_t)E), ud((size_t)E);
        int64_t bad = 0;
#pragma omp parallel for schedule(dynamic, 16) reduction(+ : bad)
        for (int32_t k = 0; k < n_graphs; k++) {
            const int32_t nv = vertex_counts[k];
            const int32_t o = (int32_t)p->voff[k];
            for (int64_t e = p->eoff[k]; e < p->eoff[k + 1]; e++) {
                if (src[e] < 0 || src[e] >= nv || dst[e] < 0 || dst[e] >= nv) bad++;
                us[(size_t)e] = src[e] + o;
                ud[(size_t)e] = dst[e] + o;
            }
        }
        SSSP_REQUIRE(bad == 0, "pack: edge endpoint outside its graph");
        // the union keeps its ids: a graph's vertices stay one contiguous
        // range, which the workgroup-per-graph policy relies on
        const int rc2 = sssp_graph_create(SSSP_W_F32, us.data(), ud.data(), weights, (int32_t)V, E,
                                          device, SSSP_NO_RELABEL, &p->g);
        if (rc2 != SSSP_OK) throw Error{rc2, sssp_last_error()};
        *out = p;
    });
    if (rc != SSSP_OK && p) {
        if (p->g) sssp_graph_destroy(p->g);
        delete p;
    }
    return rc;
}

int sssp_pack_destroy(sssp_pack *p)
{
    return guard([&] {
        SSSP_REQUIRE(p, "null pack");
        if (p->g) sssp_graph_destroy(p->g);
        delete p;
    });
}

int sssp_pack_solve(sssp_pack *p, const int32_t *sources, int32_t policy, float *dist_out,
                    sssp_stats *stats)
{
    return guard([&] {
        SSSP_REQUIRE(p && p->g, "null pack");
        SSSP_REQUIRE(policy >= 0 && policy <= 2, "policy must be 0, 1 or 2");
        check_pack_sources(p, sources);
        SSSP_HIP(hipSetDevice(p->g->device));
        Config c{p->policy ? p->policy : 1, p->bs, p->wgpcu, p->frac, p->push_chunk};  // as tuned
        if (policy != 0 && policy != p->policy)
            c = policy == 1 ? Config{1, 1024, 1, 0.05, 1} : Config{2, 256, 2, 0.05, 1};
        ensure_batch_buffers(p->g, p->g->V, 0, 0, 0);
        Prefault pages(dist_out, 4 * (size_t)p->g->V);
        const double ms = pack_run(p, sources, c);
        if (dist_out) {
            pages.join();
            download(p->g, dist_out, p->g->bdist, 4 * (size_t)p->g->V);
        }
        fill_stats(stats, ms, (double)p->g->E);
        if (stats) stats->iterations = c.policy;
    });
}

int sssp_autotune_pack(sssp_pack *p, const int32_t *sources, const char *tuning_file,
                       double *best_ms)
{
    return guard([&] {
        SSSP_REQUIRE(p && p->g, "null pack");
        check_pack_sources(p, sources);
        SSSP_HIP(hipSetDevice(p->g->device));
        int32_t large = 0;  // graphs that policy 1 solves together
        for (int32_t k = 0; k < p->n; k++) large += lds_class(p->voff[k + 1] - p->voff[k]) == 0;
        const bool together = !runs_passes(p->g, p->n);
        const Config b = autotune([&](const Config &c) { return pack_run(p, sources, c); },
                                  tuning_file, best_ms, "pack of graphs",
                                  Choices{false, false, large > 0 && !runs_passes(p->g, large), together});
        p->policy = b.policy;
        p->bs = b.bs;
        p->wgpcu = b.wgpcu;
        p->frac = b.frac;
        p->push_chunk = b.push_chunk;
    });
}

}  // extern "C"
