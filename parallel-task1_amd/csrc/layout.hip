// layout.hip -- builds the device layouts of a graph in HBM:
//   * the edge list sorted by src, stable (el_src/el_dst/el_w) with row
//     offsets row_ptr[V+1] (int64, as compressed_adjacency_list.h:13 keeps
//     `long long *edge_ptrs`) -- this is the CSR of the reference
//     (graph.hpp:316-361: per-source order = edge-list order);
//   * the CSC (in-edges grouped by dst, stable) for pull rounds;
//   * static lists of vertices with out-/in-degree > 0 and their tile tables.
// Sorting is a stable LSD radix sort that moves the edges themselves: per tile
// of 8192 an LDS digit histogram, one device-wide scan of the (digit, tile)
// counts, then a pass that ranks the keys inside the tile with ballots (stable
// by construction) and writes keys and payloads out from LDS in runs.
#include "sssp_graph.hpp"

#include <algorithm>

namespace sssp {

namespace {

constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;  // 2048 elements per block
constexpr int kRsThreads = 512;
constexpr int kRsItems = 16;
constexpr int kRsTile = kRsThreads * kRsItems;  // 8192 keys per tile
constexpr int kRsWaves = kRsThreads / 64;

// --------------------------------------------------------------------------
// Generic exclusive scan of int64, three phases.
// --------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_scan_reduce(const int64_t *in, int64_t n, int64_t *blk)
{
    __shared__ int64_t s_warp[kBlock / 64];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++)
        if (base + i < n) s += in[base + i];
    int64_t tot;
    (void)block_excl_scan_i64(s, &tot, s_warp);
    if (threadIdx.x == 0) blk[blockIdx.x] = tot;
}

// single block: exclusive scan of blk[0..nb) in place, blk[nb] = total
__device__ __forceinline__ void scan_blocks_body(int64_t *blk, int64_t nb)
{
    __shared__ int64_t s_warp[kBlock / 64];
    int64_t carry = 0;
    for (int64_t base = 0; base < nb; base += kBlock) {
        int64_t i = base + threadIdx.x;
        int64_t x = i < nb ? blk[i] : 0;
        int64_t tot;
        int64_t ex = block_excl_scan_i64(x, &tot, s_warp);
        if (i < nb) blk[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) blk[nb] = carry;
}

__global__ __launch_bounds__(kBlock) void k_scan_blocks(int64_t *blk, int64_t nb)
{
    scan_blocks_body(blk, nb);
}

// two arrays of nb + 1 values in one launch: workgroup 0 scans a, 1 scans b
__global__ __launch_bounds__(kBlock) void k_scan_blocks_pair(int64_t *a, int64_t *b, int64_t nb)
{
    scan_blocks_body(blockIdx.x == 0 ? a : b, nb);
}

__global__ __launch_bounds__(kBlock) void k_scan_down(const int64_t *in, int64_t *out, int64_t n,
                                                      const int64_t *blk)
{
    __shared__ int64_t s_warp[kBlock / 64];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int64_t v[kScanItems];
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        v[i] = base + i < n ? in[base + i] : 0;
        s += v[i];
    }
    int64_t tot;
    int64_t run = block_excl_scan_i64(s, &tot, s_warp) + blk[blockIdx.x];
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
}

// --------------------------------------------------------------------------
// Input validation: ids in [0, V), weights >= 0 and not NaN.
// --------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Vertex order (slots by descending in- plus out-degree).
// ---------------------------------------------------------------------------
// tot[v] = in- plus out-degree, out[v] = out-degree
__global__ __launch_bounds__(kBlock) void k_degrees(const int32_t *src, const int32_t *dst,
                                                    int64_t E, uint32_t *tot, uint32_t *out)
{
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < E;
         e += (int64_t)gridDim.x * kBlock) {
        const int32_t s = src[e];
        atomicAdd(&tot[s], 1u);
        atomicAdd(&out[s], 1u);
        atomicAdd(&tot[dst[e]], 1u);
    }
}

__global__ __launch_bounds__(kBlock) void k_max_u32(const uint32_t *x, int64_t n, uint32_t *mx)
{
    uint32_t m = 0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock)
        m = max(m, x[i]);
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor(m, o));
    if (__lane_id() == 0 && m) atomicMax(mx, m);
}

// ascending sort key = descending count (counts above kOrderCap tie), of
// vertex at[i] (or of vertex i when `at` is null)
constexpr uint32_t kOrderCap = 1u << 30;
__global__ __launch_bounds__(kBlock) void k_order_keys(const uint32_t *cnt, const uint32_t *at,
                                                       int64_t V, uint32_t *key)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < V;
         i += (int64_t)gridDim.x * kBlock)
        key[i] = kOrderCap - min(cnt[at ? at[i] : i], kOrderCap);
}

// slot i holds vertex by_out[pos[i]] -> vinv, and its inverse vperm
__global__ __launch_bounds__(kBlock) void k_invert_order(const uint32_t *by_out,
                                                         const uint32_t *pos, int64_t V,
                                                         int32_t *vperm, int32_t *vinv)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < V;
         i += (int64_t)gridDim.x * kBlock) {
        const int32_t v = (int32_t)by_out[pos[i]];
        vinv[i] = v;
        vperm[v] = (int32_t)i;
    }
}

__global__ __launch_bounds__(kBlock) void k_relabel_edges(const int32_t *src, const int32_t *dst,
                                                          int64_t E, const int32_t *vperm,
                                                          int32_t *osrc, int32_t *odst)
{
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < E;
         e += (int64_t)gridDim.x * kBlock) {
        osrc[e] = vperm[src[e]];
        odst[e] = vperm[dst[e]];
    }
}

__global__ void k_zero_i64(int64_t *p, int n)
{
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

template <class W>
__global__ __launch_bounds__(kBlock) void k_validate(const int32_t *src, const int32_t *dst,
                                                     const W *w, int64_t E, int32_t V,
                                                     int64_t *bad)
{
    int64_t nb_id = 0, nb_w = 0;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < E;
         e += (int64_t)gridDim.x * kBlock) {
        int32_t s = src[e], d = dst[e];
        if (s < 0 || s >= V || d < 0 || d >= V) nb_id++;
        if (w) {
            const W x = w[e];
            if (!(x >= (W)0)) nb_w++;  // negative or NaN
        }
    }
    nb_id = wave_sum64(nb_id);
    nb_w = wave_sum64(nb_w);
    if (__lane_id() == 0) {
        if (nb_id) atomicAdd((unsigned long long *)&bad[0], (unsigned long long)nb_id);
        if (nb_w) atomicAdd((unsigned long long *)&bad[1], (unsigned long long)nb_w);
    }
}

// --------------------------------------------------------------------------
// Stable LSD radix sort by digits of at most 8 bits.
// counts layout: counts[digit * ntiles + tile] (digit-major) so that one
// exclusive scan yields every tile's output base per digit, in tile order.
// --------------------------------------------------------------------------
// XCD group of an edge: a multiplicative hash of its destination's 64-vertex
// block, so each XCD's L2 serves a disjoint, work-balanced eighth of the
// distance array (R-MAT's per-bit skew makes any bit-sliced split uneven).
__device__ __forceinline__ uint32_t xcd_group(int32_t dst)
{
    return (((uint32_t)dst >> 6) * 0x9E3779B1u) >> 29;
}

// GROUP: the digit is the key's XCD group, else the bits at `shift`.
template <bool GROUP>
__device__ __forceinline__ uint32_t rs_digit(uint32_t key, int shift, uint32_t mask)
{
    return GROUP ? xcd_group((int32_t)key) : (key >> shift) & mask;
}

template <bool GROUP>
__global__ __launch_bounds__(kRsThreads) void k_rs_hist(const uint32_t *keys, int64_t n, int shift,
                                                        int bins, int64_t *counts, int64_t ntiles)
{
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    if (tid < 256) h[tid] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kRsTile;
#pragma unroll 4
    for (int i = 0; i < kRsItems; i++) {
        const int64_t idx = base + i * kRsThreads + tid;
        if (idx < n) {
            const uint32_t d = rs_digit<GROUP>(keys[idx], shift, (uint32_t)bins - 1);
            // 32 copies of the eight group counters: lanes rarely meet
            atomicAdd(&h[GROUP ? d << 5 | (tid & 31) : d], 1u);
        }
    }
    __syncthreads();
    if (tid < bins) {
        uint32_t c = 0;
        if (GROUP)
            for (int k = 0; k < 32; k++) c += h[tid << 5 | k];
        else
            c = h[tid];
        counts[(int64_t)tid * ntiles + blockIdx.x] = c;
    }
}

// One pass: NA arrays (the first holds the keys) from in to out, by digit.
// A wave ranks a run of 1024 keys of the tile on its own (its counters in LDS,
// no barrier between rounds); the counters of the waves before it and the
// digits below complete the rank. Every array then goes through LDS in rank
// order, so a digit's keys are written in one run (128 bytes on average at 64
// of them). Bound by the bandwidth of reading and writing the arrays; moving
// the payloads along (12 bytes an edge each way, 0.13 ms a pass at 2^24 edges)
// replaced a pass over keys and positions (0.31 ms, three barriers per round of
// keys and scattered writes) and a gather of the payloads by position after the
// last one (0.62 ms). in.a[1] null: the positions 0, 1, ... pad: added to every
// position of a digit (or null).
template <int NA>
struct RsArrays {
    uint32_t *a[NA];
};

template <int NA, bool GROUP>
__global__ __launch_bounds__(kRsThreads) void k_rs_split(const RsArrays<NA> in,
                                                         const RsArrays<NA> out, int64_t n,
                                                         int shift, int bins,
                                                         const int64_t *offsets, int64_t ntiles,
                                                         const int64_t *pad)
{
    __shared__ uint32_t s_stage[kRsTile];
    __shared__ uint32_t s_cnt[kRsWaves][256];
    __shared__ uint32_t s_start[256], s_goff[256];
    __shared__ uint32_t s_wave[4];
    const int tid = threadIdx.x, lane = __lane_id(), wv = tid >> 6;
    const uint32_t mask = (uint32_t)bins - 1;
    const int64_t tile = blockIdx.x, base = tile * kRsTile;
    const int cnt = (int)min(n - base, (int64_t)kRsTile);
    for (int i = tid; i < kRsWaves * 256; i += kRsThreads) s_cnt[i >> 8][i & 255] = 0;
    uint32_t key[kRsItems], lp[kRsItems];
    const int first = wv * (kRsTile / kRsWaves) + lane;
#pragma unroll
    for (int r = 0; r < kRsItems; r++) {
        const int i = first + r * 64;
        key[r] = i < cnt ? in.a[0][base + i] : 0u;
    }
    __syncthreads();
    volatile uint32_t *const mine = s_cnt[wv];
#pragma unroll
    for (int r = 0; r < kRsItems; r++) {
        const bool valid = first + r * 64 < cnt;
        const uint32_t dg = rs_digit<GROUP>(key[r], shift, mask);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (dg >> b) & 1u;
            const uint64_t bm = __ballot(bit);
            peers &= bit ? bm : ~bm;
        }
        // every lane reads its digit's counter before the last peer adds to it
        const uint32_t before = mine[dg];
        __builtin_amdgcn_wave_barrier();
        if (valid && (peers >> lane) == 1ull) mine[dg] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        lp[r] = before + (uint32_t)__popcll(peers & lanemask_lt());
    }
    __syncthreads();
    // counters -> keys of the digit in the waves before; exclusive scan of the
    // digits' totals over the tile
    uint32_t total = 0, inc = 0;
    if (tid < 256) {
#pragma unroll
        for (int w = 0; w < kRsWaves; w++) {
            const uint32_t c = s_cnt[w][tid];
            s_cnt[w][tid] = total;
            total += c;
        }
        inc = total;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(inc, o);
            if (lane >= o) inc += y;
        }
        if (lane == 63) s_wave[wv] = inc;
    }
    __syncthreads();
    if (tid < 256) {
        uint32_t start = inc - total;
        for (int w = 0; w < wv; w++) start += s_wave[w];
        s_start[tid] = start;
        if (tid < bins)
            s_goff[tid] = (uint32_t)(offsets[(int64_t)tid * ntiles + tile] + (pad ? pad[tid] : 0)) -
                          start;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRsItems; r++) {
        if (first + r * 64 >= cnt) continue;
        const uint32_t dg = rs_digit<GROUP>(key[r], shift, mask);
        lp[r] += s_start[dg] + s_cnt[wv][dg];
        s_stage[lp[r]] = key[r];
    }
    __syncthreads();
    uint32_t gp[kRsItems];  // where slot r * kRsThreads + tid of the tile goes (n < 2^32)
#pragma unroll
    for (int r = 0; r < kRsItems; r++) {
        const int i = r * kRsThreads + tid;
        if (i >= cnt) continue;
        const uint32_t k = s_stage[i];
        gp[r] = s_goff[rs_digit<GROUP>(k, shift, mask)] + (uint32_t)i;
        out.a[0][gp[r]] = k;
    }
#pragma unroll
    for (int x = 1; x < NA; x++) {
        uint32_t v[kRsItems];
#pragma unroll
        for (int r = 0; r < kRsItems; r++) {
            const int i = first + r * 64;
            v[r] = 0;
            if (i < cnt) v[r] = x > 1 || in.a[x] ? in.a[x][base + i] : (uint32_t)(base + i);
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRsItems; r++)
            if (first + r * 64 < cnt) s_stage[lp[r]] = v[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRsItems; r++) {
            const int i = r * kRsThreads + tid;
            if (i < cnt) out.a[x][gp[r]] = s_stage[i];
        }
    }
}

// --------------------------------------------------------------------------
// Layout assembly kernels.
// --------------------------------------------------------------------------
// Of the counts scanned for the split into XCD groups: goff[x] = where group
// x begins in the padded list (every group a whole number of 16-byte vectors),
// pad[x] = how far that is past its place in the unpadded one.
__global__ void k_group_offsets(const int64_t *offsets, int64_t ntiles, int64_t E, int64_t *goff,
                                int64_t *pad)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int64_t o = 0;
    for (int x = 0; x < 8; x++) {
        const int64_t b = ntiles > 0 ? offsets[x * ntiles] : 0;
        const int64_t e = x < 7 && ntiles > 0 ? offsets[(x + 1) * ntiles] : E;
        goff[x] = o;
        pad[x] = o - b;
        o += (e - b + 3) / 4 * 4;
    }
    goff[8] = o;
    pad[8] = o - E;
}

// The padding of each group's region (up to 3 slots) is a weight-0 self loop
// on vertex 0, which never changes a distance. 32 threads, four per group.
__global__ void k_group_pad(const int64_t *goff, const int64_t *pad, int64_t E, int32_t *xs,
                            int32_t *xd, uint32_t *xw)
{
    const int x = threadIdx.x >> 2;
    // group x ends, unpadded, where group x + 1 begins without its padding
    const int64_t end = (x < 7 ? goff[x + 1] - pad[x + 1] : E) + pad[x];
    const int64_t i = end + (threadIdx.x & 3);
    if (i < goff[x + 1]) {
        xs[i] = 0;
        xd[i] = 0;
        xw[i] = 0u;
    }
}

// Position j of the edges sorted by block, b = dst[j]'s block, goes to
// boff[b] + (j - bptr[b]).
__global__ __launch_bounds__(kBlock) void k_blk_place(const int32_t *src, const uint32_t *dst,
                                                      const uint32_t *w, int64_t E,
                                                      const int64_t *bptr, const int64_t *boff,
                                                      int32_t *bs, uint16_t *bd, uint32_t *bw)
{
    for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < E;
         j += (int64_t)gridDim.x * kBlock) {
        const uint32_t d = dst[j], b = d >> kBlkBits;
        const int64_t o = boff[b] + (j - bptr[b]);
        bs[o] = src[j];
        bd[o] = (uint16_t)(d & ((1u << kBlkBits) - 1));
        bw[o] = w[j];
    }
}

// The padding slots of each block (up to kBlkChunk - 1) copy the block's last
// edge: relaxing it again changes nothing, and its source delta is 0.
__global__ __launch_bounds__(kBlock) void k_blk_pad(const int64_t *bptr, const int64_t *boff,
                                                    int32_t nblk, int32_t *bs, uint16_t *bd,
                                                    uint32_t *bw)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < (int64_t)nblk * kBlkChunk;
         i += (int64_t)gridDim.x * kBlock) {
        const int32_t b = (int32_t)(i / kBlkChunk);
        const int64_t last = boff[b] + (bptr[b + 1] - bptr[b]) - 1;
        const int64_t o = last + 1 + i % kBlkChunk;
        if (o < boff[b + 1]) {  // only blocks with edges have slots
            bs[o] = bs[last];
            bd[o] = bd[last];
            bw[o] = bw[last];
        }
    }
}

// A fixed-stride sample of the edges:
// out[0 .. n) = sampled weights, out[n + 1] += sampled edges between near ids
__global__ __launch_bounds__(kBlock) void k_edge_sample(const int32_t *src, const int32_t *dst,
                                                        const uint32_t *w, int64_t E, int32_t n,
                                                        int32_t near_ids, uint32_t *out)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    bool near = false;
    if (i < n) {
        const int64_t e = i * E / n;
        out[i] = w[e];
        near = abs(src[e] - dst[e]) < near_ids;
    }
    const unsigned long long m = __ballot(near);
    if (m != 0 && __lane_id() == 0) atomicAdd(&out[n + 1], (uint32_t)__popcll(m));
}

// largest out-degree
__global__ __launch_bounds__(kBlock) void k_max_degree(const int64_t *ptr, int64_t V, uint32_t *mx)
{
    uint32_t m = 0;
    for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < V;
         v += (int64_t)gridDim.x * kBlock)
        m = max(m, (uint32_t)(ptr[v + 1] - ptr[v]));
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor(m, o));
    __shared__ uint32_t s_m[kBlock / 64];
    if (__lane_id() == 0) s_m[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {  // one update per workgroup (see k_count_reached)
        for (int w = 1; w < kBlock / 64; w++) m = max(m, s_m[w]);
        if (m) atomicMax(mx, m);
    }
}

// Source deltas of one chunk (one wave, 4 slots per lane, in slot order):
// d[k] = source of slot k - source of the slot before it, 0 for the first.
__device__ __forceinline__ void chunk_deltas(const int32_t *bs, int64_t c, int32_t (&s)[4],
                                             uint32_t (&d)[4])
{
    typedef int32_t v4i __attribute__((ext_vector_type(4)));
    const v4i v = reinterpret_cast<const v4i *>(bs)[c * (kBlkChunk / 4) + __lane_id()];
    s[0] = v.x;
    s[1] = v.y;
    s[2] = v.z;
    s[3] = v.w;
    const int32_t prev = __shfl_up(s[3], 1);
    d[0] = __lane_id() == 0 ? 0u : (uint32_t)(s[0] - prev);
    d[1] = (uint32_t)(s[1] - s[0]);
    d[2] = (uint32_t)(s[2] - s[1]);
    d[3] = (uint32_t)(s[3] - s[2]);
}

// wide[c] = 1 when chunk c has a source gap that does not fit the packed
// delta (sources ascend within a block, so every delta is >= 0)
__global__ __launch_bounds__(kBlock) void k_blk_chunk_wide(const int32_t *bs, int64_t nch,
                                                           uint8_t *wide)
{
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (c >= nch) return;  // wave-uniform
    int32_t s[4];
    uint32_t d[4];
    chunk_deltas(bs, c, s, d);
    bool big = false;
    for (int k = 0; k < 4; k++) big |= d[k] >= (1u << kBlkDeltaBits);
    const uint64_t m = __ballot(big);
    if (__lane_id() == 0) wide[c] = m != 0;
}

// Packs chunk c: widx[c] < 0 -> deltas in the words and the first source in
// cbase; else the destinations alone in the words, the sources whole in
// wide[widx[c] * kBlkChunk ...] and cbase = -(1 + widx[c]).
__global__ __launch_bounds__(kBlock) void k_blk_pack(const int32_t *bs, const uint16_t *bd,
                                                     const int32_t *widx, int64_t nch,
                                                     uint32_t *pk, int32_t *cbase, int32_t *wide)
{
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (c >= nch) return;  // wave-uniform
    int32_t s[4];
    uint32_t d[4];
    chunk_deltas(bs, c, s, d);
    const int32_t wi = widx[c];
    const int64_t o = c * kBlkChunk + 4 * __lane_id();
    for (int k = 0; k < 4; k++)
        pk[o + k] = (wi < 0 ? d[k] << kBlkBits : 0u) | (uint32_t)bd[o + k];
    if (wi >= 0)
        for (int k = 0; k < 4; k++) wide[(int64_t)wi * kBlkChunk + 4 * __lane_id() + k] = s[k];
    if (__lane_id() == 0) cbase[c] = wi < 0 ? s[0] : -(1 + wi);
}

// Light edges of chunk c of a list of n weights (one wave, 4 slots per lane):
// bit k of the result is set when the lane's slot k holds a light edge.
__device__ __forceinline__ int chunk_light(const uint32_t *w, int64_t n, int64_t c, uint32_t thr)
{
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    const int64_t e = c * kBlkChunk + 4 * __lane_id();
    if (e + 4 <= n) {
        const v4u v = *reinterpret_cast<const v4u *>(w + e);
        return (v.x <= thr ? 1 : 0) | (v.y <= thr ? 2 : 0) | (v.z <= thr ? 4 : 0) |
               (v.w <= thr ? 8 : 0);
    }
    int m = 0;
    for (int k = 0; k < 4; k++)
        if (e + k < n && w[e + k] <= thr) m |= 1 << k;
    return m;
}

// light edges of each lane before this one, over the wave
__device__ __forceinline__ int light_before(int m)
{
    int inc = __popc(m);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o);
        if (__lane_id() >= o) inc += y;
    }
    return inc - __popc(m);
}

__global__ __launch_bounds__(kBlock) void k_light_count(const uint32_t *w, int64_t n, int64_t nch,
                                                        uint32_t thr, int64_t *cnt)
{
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (c >= nch) return;  // wave-uniform
    const int k = wave_sum32(__popc(chunk_light(w, n, c, thr)));
    if (__lane_id() == 0) cnt[c] = k;
}

// The light edges of an edge list of n edges, in order (pos: light edges before
// each chunk).
__global__ __launch_bounds__(kBlock) void k_light_select(const int32_t *src, const int32_t *dst,
                                                         const uint32_t *w, int64_t n, int64_t nch,
                                                         uint32_t thr, const int64_t *pos,
                                                         int32_t *ls, int32_t *ld, uint32_t *lw)
{
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (c >= nch) return;  // wave-uniform
    const int m = chunk_light(w, n, c, thr);
    int64_t o = pos[c] + light_before(m);
    for (int k = 0; k < 4; k++) {
        if (!((m >> k) & 1)) continue;
        const int64_t e = c * kBlkChunk + 4 * __lane_id() + k;
        ls[o] = src[e];
        ld[o] = dst[e];
        lw[o] = w[e];
        o++;
    }
}

// out[b] = pos[boff[b] / kBlkChunk]: light edges before block b (nblk + 1 values)
__global__ __launch_bounds__(kBlock) void k_light_starts(const int64_t *pos, const int64_t *boff,
                                                         int32_t nblk, int64_t *out)
{
    for (int64_t b = (int64_t)blockIdx.x * kBlock + threadIdx.x; b <= nblk;
         b += (int64_t)gridDim.x * kBlock)
        out[b] = pos[boff[b] / kBlkChunk];
}

// The light edges of chunk c, in order, to their block's run of the light list:
// pos = light edges before each chunk, lptr / loff = light edges before and
// first slot of each block.
__global__ __launch_bounds__(kBlock) void k_light_gather(const int32_t *bs, const uint16_t *bd,
                                                         const uint32_t *bw, int64_t nch,
                                                         uint32_t thr, const int64_t *pos,
                                                         const int64_t *boff, int32_t nblk,
                                                         const int64_t *lptr, const int64_t *loff,
                                                         int32_t *ls, uint16_t *ld, uint32_t *lw)
{
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (c >= nch) return;  // wave-uniform
    const int m = chunk_light(bw, nch * kBlkChunk, c, thr);
    int32_t lo = 0, hi = nblk - 1;  // the chunk's block: the last with boff <= its first slot
    while (lo < hi) {
        const int32_t mid = (lo + hi + 1) >> 1;
        if (boff[mid] <= c * kBlkChunk) lo = mid;
        else hi = mid - 1;
    }
    int64_t o = loff[lo] + (pos[c] - lptr[lo]) + light_before(m);
    for (int k = 0; k < 4; k++) {
        if (!((m >> k) & 1)) continue;
        const int64_t e = c * kBlkChunk + 4 * __lane_id() + k;
        ls[o] = bs[e];
        ld[o] = bd[e];
        lw[o] = bw[e];
        o++;
    }
}

// off[b * (nfine + 1) + k] = the first slot of block b whose source is at
// least k << fine_bits (sources ascend within a block's padded run), aligned
// down to its chunk; k = nfine gives the end of the run.
__global__ __launch_bounds__(kBlock) void k_blk_range_offsets(const int32_t *bs, const int64_t *boff,
                                                              int32_t nblk, int fine_bits,
                                                              int32_t nfine, int64_t *off)
{
    const int64_t n = (int64_t)nblk * (nfine + 1);
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) {
        const int32_t b = (int32_t)(i / (nfine + 1));
        const int32_t k = (int32_t)(i % (nfine + 1));
        const int64_t b0 = boff[b], b1 = boff[b + 1];
        int64_t pos = b1;
        if (k < nfine) {
            const int64_t key = (int64_t)k << fine_bits;
            int64_t lo = b0, hi = b1;  // first position with bs >= key
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                if ((int64_t)bs[mid] < key) lo = mid + 1;
                else hi = mid;
            }
            pos = b0 + (lo - b0) / kBlkChunk * kBlkChunk;
        }
        off[i] = pos;
    }
}

// record j = edge j of the list sorted by block: destinations, sources,
// weights, n of each
__global__ __launch_bounds__(kBlock) void k_m_place(const uint32_t *sorted, int64_t n, MRec *out)
{
    for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < n;
         j += (int64_t)gridDim.x * kBlock)
        out[j] = MRec{(int32_t)sorted[n + j], sorted[2 * n + j],
                      (int32_t)(sorted[j] & ((1u << kMBits) - 1)), 0};
}

// row_ptr[v] = first position whose sorted key is >= v; row_ptr[V] = E.
// Position i starts the vertices (keys[i-1], keys[i]]; it writes them when
// they are few. A long run of keyless vertices (on a degree-ordered graph
// every isolated vertex sits at the end) is left at -1 for
// k_rowptr_search, so no thread loops over millions of vertices.
constexpr int64_t kRowptrRun = 64;
__global__ __launch_bounds__(kBlock) void k_rowptr_from_sorted(const uint32_t *keys, int64_t E,
                                                               int32_t V, int shift,
                                                               int64_t *row_ptr)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i <= E;
         i += (int64_t)gridDim.x * kBlock) {
        int64_t lo = (i == 0) ? 0 : (int64_t)(keys[i - 1] >> shift) + 1;  // first vertex not yet placed
        int64_t hi = (i == E) ? (int64_t)V : (int64_t)(keys[i] >> shift);  // last vertex starting at i
        if (hi - lo < kRowptrRun)
            for (int64_t v = lo; v <= hi; v++) row_ptr[v] = i;
    }
}

// the entries k_rowptr_from_sorted left at -1: lower bound of v in the keys
__global__ __launch_bounds__(kBlock) void k_rowptr_search(const uint32_t *keys, int64_t E,
                                                          int32_t V, int shift,
                                                          int64_t *row_ptr)
{
    for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v <= V;
         v += (int64_t)gridDim.x * kBlock) {
        if (row_ptr[v] >= 0) continue;
        int64_t lo = 0, hi = E;  // first position with key >= v
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if ((int64_t)(keys[mid] >> shift) < v) lo = mid + 1;
            else hi = mid;
        }
        row_ptr[v] = lo;
    }
}

__global__ __launch_bounds__(kBlock) void k_fill_i64(int64_t *p, int64_t n, int64_t val)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock)
        p[i] = val;
}


__global__ __launch_bounds__(kBlock) void k_nz_flags(const int64_t *ptr, int32_t V, int64_t *flags)
{
    for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < V;
         v += (int64_t)gridDim.x * kBlock)
        flags[v] = ptr[v + 1] > ptr[v] ? 1 : 0;
}

__global__ __launch_bounds__(kBlock) void k_nz_compact(const int64_t *ptr, int32_t V,
                                                       const int64_t *pos, int32_t *nz_v,
                                                       int64_t *nz_scan, int64_t n_nz, int64_t E)
{
    for (int64_t v = (int64_t)blockIdx.x * kBlock + threadIdx.x; v < V;
         v += (int64_t)gridDim.x * kBlock) {
        if (ptr[v + 1] > ptr[v]) {
            int64_t j = pos[v];
            nz_v[j] = (int32_t)v;
            nz_scan[j] = ptr[v];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) nz_scan[n_nz] = E;
}

// tile_out[t] = the entry whose edge range contains edge t * TE; tile_out[ntiles] = n.
__global__ __launch_bounds__(kBlock) void k_tile_table(const int64_t *scan, int32_t n, int64_t TE,
                                                       int64_t ntiles, int32_t *tile_out)
{
    for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < n;
         j += (int64_t)gridDim.x * kBlock) {
        int64_t a = scan[j], b = scan[j + 1];
        for (int64_t t = (a + TE - 1) / TE; t * TE < b; t++) tile_out[t] = (int32_t)j;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) tile_out[ntiles] = n;
}

inline int grid_for(int64_t n, int64_t cap = 8192)
{
    int64_t b = (n + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    return (int)(b < cap ? b : cap);
}

// row_ptr over the keys' bits from `shift` on
void rowptr_from_sorted(const uint32_t *keys, int64_t E, int32_t V, int64_t *row_ptr,
                        hipStream_t s, int shift = 0)
{
    k_fill_i64<<<grid_for((int64_t)V + 1), kBlock, 0, s>>>(row_ptr, (int64_t)V + 1, -1);
    k_rowptr_from_sorted<<<grid_for(E + 1), kBlock, 0, s>>>(keys, E, V, shift, row_ptr);
    k_rowptr_search<<<grid_for((int64_t)V + 1), kBlock, 0, s>>>(keys, E, V, shift, row_ptr);
    SSSP_LAUNCH_CHECK("rowptr_from_sorted");
}

// Scratch of a sort: counts for 256 digits of every tile, the scan's blocks.
struct RsScratch {
    int64_t *counts, *blk_a, *blk_b, n_blk;
};

int key_bits(int64_t max_key)
{
    int bits = 0;
    while (bits < 31 && ((int64_t)1 << bits) <= max_key) bits++;
    return bits;
}

// Counts of one digit, scanned.
template <bool GROUP>
void rs_count(const uint32_t *keys, int64_t n, int shift, int bins, const RsScratch &t,
              hipStream_t s)
{
    const int64_t ntiles = (n + kRsTile - 1) / kRsTile;
    k_rs_hist<GROUP><<<(unsigned)ntiles, kRsThreads, 0, s>>>(keys, n, shift, bins, t.counts, ntiles);
    SSSP_LAUNCH_CHECK("k_rs_hist");
    device_exclusive_scan_i64(t.counts, t.counts, bins * ntiles, t.blk_a, t.blk_b, t.n_blk, s);
}

// Sorts the arrays by bits [lo, lo + bits) of the first, from in to fin, by way
// of tmp (at least one pass: a copy when bits is 0).
template <int NA>
void radix_sort(const RsArrays<NA> &in, const RsArrays<NA> &fin, const RsArrays<NA> &tmp, int64_t n,
                int lo, int bits, const RsScratch &t, hipStream_t s)
{
    if (n <= 0) return;
    const int64_t ntiles = (n + kRsTile - 1) / kRsTile;
    const int passes = std::max(1, (bits + 7) / 8);
    const int width = std::max(1, (bits + passes - 1) / passes);
    RsArrays<NA> from = in;
    for (int p = 0; p < passes; p++) {
        const RsArrays<NA> to = (passes - 1 - p) % 2 == 0 ? fin : tmp;
        const int shift = lo + width * p;
        const int bins = 1 << std::min(width, std::max(1, bits - width * p));
        rs_count<false>(from.a[0], n, shift, bins, t, s);
        k_rs_split<NA, false><<<(unsigned)ntiles, kRsThreads, 0, s>>>(from, to, n, shift, bins,
                                                                      t.counts, ntiles, nullptr);
        SSSP_LAUNCH_CHECK("k_rs_split");
        from = to;
    }
}

inline uint32_t *u32p(const void *p) { return static_cast<uint32_t *>(const_cast<void *>(p)); }

// Short-lived arrays of the build, cut from memory the sorts no longer need
// (an allocation and its release cost 20 us and more, each); allocated where it
// is used up. Used in stream order only.
class Carve {
  public:
    Carve(void *base, size_t bytes) : p_(static_cast<char *>(base)), left_(bytes / 256 * 256) {}
    Carve(const Carve &) = delete;
    Carve &operator=(const Carve &) = delete;
    ~Carve()
    {
        for (void *x : own_) dfree(x);
    }
    template <class T>
    T *get(size_t n)
    {
        const size_t b = (std::max<size_t>(n, 1) * sizeof(T) + 255) / 256 * 256;
        if (b > left_) {
            own_.push_back(dmalloc<char>(b));
            return static_cast<T *>(own_.back());
        }
        T *at = reinterpret_cast<T *>(p_);
        p_ += b;
        left_ -= b;
        return at;
    }

  private:
    char *p_;
    size_t left_;
    std::vector<void *> own_;
};

void build_static_list(const int64_t *ptr, int32_t V, int64_t E, int64_t *tmp_flags,
                       int64_t *tmp_pos, int64_t *blk_a, int64_t *blk_b, int64_t n_blk,
                       hipStream_t s, int32_t **nz_v, int64_t **nz_scan, int32_t *n_nz,
                       int32_t **tiles)
{
    k_nz_flags<<<grid_for(V), kBlock, 0, s>>>(ptr, V, tmp_flags);
    SSSP_LAUNCH_CHECK("k_nz_flags");
    device_exclusive_scan_i64(tmp_flags, tmp_pos, V, blk_a, blk_b, n_blk, s);
    int64_t last_pos = 0, last_flag = 0;
    if (V > 0) {
        SSSP_HIP(hipMemcpyAsync(&last_pos, tmp_pos + V - 1, 8, hipMemcpyDeviceToHost, s));
        SSSP_HIP(hipMemcpyAsync(&last_flag, tmp_flags + V - 1, 8, hipMemcpyDeviceToHost, s));
        SSSP_HIP(hipStreamSynchronize(s));
    }
    const int64_t n = last_pos + last_flag;
    *n_nz = (int32_t)n;
    *nz_v = dmalloc<int32_t>((size_t)n + 1);
    *nz_scan = dmalloc<int64_t>((size_t)n + 1);
    k_nz_compact<<<grid_for(V), kBlock, 0, s>>>(ptr, V, tmp_pos, *nz_v, *nz_scan, n, E);
    SSSP_LAUNCH_CHECK("k_nz_compact");
    // the tables in one allocation, tiles[0]'s
    size_t at[kChunkCount + 1] = {};
    auto count = [&](int c) { return (E + kBlock * kChunkK[c] - 1) / (kBlock * kChunkK[c]); };
    for (int c = 0; c < kChunkCount; c++) at[c + 1] = at[c] + ((size_t)count(c) + 1 + 63) / 64 * 64;
    tiles[0] = dmalloc<int32_t>(at[kChunkCount]);
    for (int c = 0; c < kChunkCount; c++) {
        tiles[c] = tiles[0] + at[c];
        build_tile_table(*nz_scan, (int32_t)n, E, kBlock * kChunkK[c], tiles[c], s);
    }
}

}  // namespace

void scan_blocks_pair_inplace(int64_t *a, int64_t *b, int64_t nb, hipStream_t s)
{
    k_scan_blocks_pair<<<2, kBlock, 0, s>>>(a, b, nb);
    SSSP_LAUNCH_CHECK("k_scan_blocks_pair");
}

int64_t scan_blocks_needed(int64_t n) { return (n + kScanTile - 1) / kScanTile + 2; }

void device_exclusive_scan_i64(const int64_t *in, int64_t *out, int64_t n, int64_t *blk_a,
                               int64_t *blk_b, int64_t n_blk_cap, hipStream_t s)
{
    (void)blk_b;
    if (n <= 0) return;
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    if (nb + 1 > n_blk_cap) throw Error{SSSP_ERR_INTERNAL, "scan scratch too small"};
    k_scan_reduce<<<(unsigned)nb, kBlock, 0, s>>>(in, n, blk_a);
    SSSP_LAUNCH_CHECK("k_scan_reduce");
    k_scan_blocks<<<1, kBlock, 0, s>>>(blk_a, nb);
    SSSP_LAUNCH_CHECK("k_scan_blocks");
    k_scan_down<<<(unsigned)nb, kBlock, 0, s>>>(in, out, n, blk_a);
    SSSP_LAUNCH_CHECK("k_scan_down");
}

void build_tile_table(const int64_t *scan, int32_t n, int64_t total, int32_t tile_edges,
                      int32_t *tile_out, hipStream_t s)
{
    const int64_t ntiles = (total + tile_edges - 1) / tile_edges;
    k_tile_table<<<grid_for(n > 0 ? n : 1), kBlock, 0, s>>>(scan, n, tile_edges, ntiles, tile_out);
    SSSP_LAUNCH_CHECK("k_tile_table");
}

// Packed 12-byte edge records (src, dst, 4-byte weight) of the binary
// edge-list file -> the three edge arrays.
__global__ __launch_bounds__(kBlock) void k_split_records(const uint32_t *__restrict__ rec, int64_t n,
                                                         int32_t *src, int32_t *dst, uint32_t *w)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) {
        src[i] = (int32_t)rec[3 * i];
        dst[i] = (int32_t)rec[3 * i + 1];
        w[i] = rec[3 * i + 2];
    }
}

void split_records(const uint32_t *rec, int64_t n, int32_t *src, int32_t *dst, uint32_t *w,
                   hipStream_t s)
{
    if (n <= 0) return;
    k_split_records<<<grid_for(n), kBlock, 0, s>>>(rec, n, src, dst, w);
    SSSP_LAUNCH_CHECK("k_split_records");
}

// Multi-source records of an edge list of n edges sorted by source (device
// arrays): sorted by destination block, sources ascending within one, and the
// tiles over them.
static void build_records(sssp_graph *g, const int32_t *src, const int32_t *dst, const uint32_t *w,
                          int64_t n, MRec **rec_out, BlkTile **tile_out, int32_t *n_tile)
{
    hipStream_t s = g->stream;
    const int32_t nblk = (int32_t)(((int64_t)g->V + (1 << kMBits) - 1) >> kMBits);
    const int64_t rs_tiles = (n + kRsTile - 1) / kRsTile;
    uint32_t *sorted = dmalloc<uint32_t>(3 * (size_t)n);
    int64_t *counts = dmalloc<int64_t>((size_t)std::max<int64_t>(256 * rs_tiles, (int64_t)nblk + 1));
    int64_t *bptr = dmalloc<int64_t>((size_t)nblk + 1);
    struct Scratch {
        void *p[3];
        ~Scratch()
        {
            for (void *x : p) dfree(x);
        }
    } scratch{{sorted, counts, bptr}};
    MRec *rec = dmalloc<MRec>((size_t)n);
    *rec_out = rec;
    // sorted by way of the records' own memory, which is written afterwards
    uint32_t *via = reinterpret_cast<uint32_t *>(rec);
    radix_sort<3>({{u32p(dst), u32p(src), u32p(w)}}, {{sorted, sorted + n, sorted + 2 * n}},
                  {{via, via + n, via + 2 * n}}, n, kMBits, key_bits(nblk - 1),
                  RsScratch{counts, g->blk_a, g->blk_b, g->n_blk}, s);
    k_m_place<<<grid_for(n), kBlock, 0, s>>>(sorted, n, rec);
    SSSP_LAUNCH_CHECK("k_m_place");
    rowptr_from_sorted(sorted, n, nblk, bptr, s, kMBits);
    std::vector<int64_t> bp((size_t)nblk + 1);
    SSSP_HIP(hipMemcpyAsync(bp.data(), bptr, 8 * bp.size(), hipMemcpyDeviceToHost, s));
    SSSP_HIP(hipStreamSynchronize(s));
    int64_t most = 0;
    for (int32_t b = 0; b < nblk; b++) most = std::max(most, bp[(size_t)b + 1] - bp[(size_t)b]);
    const int64_t cap =
        nblk >= kMEvenBlocks && most * nblk <= 4 * n ? kMTileEven : kMTileEdges;
    std::vector<BlkTile> tiles;
    for (int32_t b = 0; b < nblk; b++) {
        const int64_t c = bp[(size_t)b + 1] - bp[(size_t)b];
        const int64_t nt = (c + cap - 1) / cap;
        for (int64_t k = 0; k < nt; k++) {
            const int64_t e0 = bp[(size_t)b] + k * cap;
            tiles.push_back(BlkTile{b, nt > 1 ? 1 : 0, e0, std::min(e0 + cap, bp[(size_t)b + 1])});
        }
    }
    BlkTile *td = dmalloc<BlkTile>(std::max<size_t>(tiles.size(), 1));
    *tile_out = td;
    SSSP_HIP(hipMemcpyAsync(td, tiles.data(), sizeof(BlkTile) * tiles.size(), hipMemcpyHostToDevice, s));
    SSSP_HIP(hipStreamSynchronize(s));
    *n_tile = (int32_t)tiles.size();
}

// out[0..3) += sampled edges whose source (destination) is near that of the
// edge 256 further on, and edges between near ids. Ids may still be invalid.
constexpr int kOrderSamples = 512;
__global__ __launch_bounds__(kOrderSamples) void k_list_order(const int32_t *src, const int32_t *dst,
                                                              int64_t E, int64_t V, int64_t *out)
{
    const int64_t e = threadIdx.x * E / kOrderSamples, f = min(e + 256, E - 1);
    const int64_t s = src[e], t = dst[e], step = max((int64_t)1, V / 64);
    const bool b[3] = {llabs(src[f] - s) <= step, llabs(dst[f] - t) <= step,
                       llabs(t - s) <= min((int64_t)kListNear, V / 32)};
    for (int i = 0; i < 3; i++) {
        const unsigned long long m = __ballot(b[i]);
        if (m != 0 && __lane_id() == 0)
            atomicAdd((unsigned long long *)&out[i], (unsigned long long)__popcll(m));
    }
}

// Edge-list check on the device: every id in [0, V) and (wtype >= 0) every
// weight >= 0 and not NaN (unsigned weights always are); throws SSSP_ERR_ARG.
// The relaxations rely on it: distances are compared as unsigned bit patterns,
// which orders non-negative IEEE values only. The two counters live in
// `bad_buf` when the caller brings one (device memory, 16 bytes), else in a
// buffer allocated for the call; a kernel clears them either way.
// With `order` (and no bad_buf), the order of the list is sampled on the way.
void validate_edges(const int32_t *src, const int32_t *dst, const void *w, int wtype, int64_t E,
                    int32_t V, hipStream_t s, int64_t *bad_buf, ListOrder *order)
{
    if (E <= 0) return;
    const int n = order ? 5 : 2;
    int64_t *bad = bad_buf ? bad_buf : dmalloc<int64_t>((size_t)n);
    struct Free {
        void *p;
        ~Free() { dfree(p); }
    } fr{bad_buf ? nullptr : bad};
    k_zero_i64<<<1, 64, 0, s>>>(bad, n);
    SSSP_LAUNCH_CHECK("k_zero_i64");
    if (order) {
        k_list_order<<<1, kOrderSamples, 0, s>>>(src, dst, E, V, bad + 2);
        SSSP_LAUNCH_CHECK("k_list_order");
    }
    if (wtype == SSSP_W_F32)
        k_validate<float><<<grid_for(E), kBlock, 0, s>>>(src, dst, static_cast<const float *>(w), E,
                                                         V, bad);
    else if (wtype == SSSP_W_F64)
        k_validate<double><<<grid_for(E), kBlock, 0, s>>>(src, dst, static_cast<const double *>(w),
                                                          E, V, bad);
    else if (wtype == SSSP_W_U32)
        k_validate<uint32_t><<<grid_for(E), kBlock, 0, s>>>(src, dst,
                                                            static_cast<const uint32_t *>(w), E, V,
                                                            bad);
    else
        k_validate<uint32_t><<<grid_for(E), kBlock, 0, s>>>(src, dst, nullptr, E, V, bad);
    SSSP_LAUNCH_CHECK("k_validate");
    int64_t hb[5] = {0, 0, 0, 0, 0};
    SSSP_HIP(hipMemcpyAsync(hb, bad, 8 * n, hipMemcpyDeviceToHost, s));
    SSSP_HIP(hipStreamSynchronize(s));
    if (hb[0]) throw Error{SSSP_ERR_ARG, std::to_string(hb[0]) + " edges have a vertex id outside [0, V)"};
    if (hb[1]) throw Error{SSSP_ERR_ARG, std::to_string(hb[1]) + " edges have a negative or NaN weight"};
    if (order) {
        order->ordered = std::max(hb[2], hb[3]) * 2 >= kOrderSamples;
        order->near = order->ordered && hb[4] * 2 >= kOrderSamples;
    }
}

// The tiles of the destination-blocked list: runs of at most `cap` edge slots
// (a multiple of kBlkChunk) of one block, `split` when a block has several.
// Without source ranges (R.stride == 0) a tile is a run of its block's slots;
// order 0 = smallest tiles first (stable by block), 1 = by block, 2 = largest
// first, 3 = by descending block. With source ranges each block's run is cut
// at the (chunk-aligned) slots where its sources reach multiples of the range
// size, and the tiles are dispatched range by range (by block within one):
// the workgroups running at one time then gather d[src] from one range of
// the distance array, which an XCD's L2 holds. bo: padded block offsets,
// nblk + 1 values (of the blocked list or the light list); off: its cuts.
std::vector<BlkTile> make_blk_tiles(const std::vector<int64_t> &bo, int64_t cap, int order,
                                    const BlkRanges &R, const std::vector<int64_t> &off)
{
    struct T {
        BlkTile t;
        int32_t range;
    };
    std::vector<T> tiles;
    const int32_t nblk = (int32_t)bo.size() - 1;
    const bool ranged = R.stride > 0 && !off.empty();
    const int32_t nr = ranged ? (R.n_fine + R.stride - 1) / R.stride : 1;
    for (int32_t b = 0; b < nblk; b++) {
        const size_t first = tiles.size();
        for (int32_t r = 0; r < nr; r++) {
            int64_t lo = bo[(size_t)b], hi = bo[(size_t)b + 1];
            if (ranged) {
                const size_t row = (size_t)b * (size_t)(R.n_fine + 1);
                lo = off[row + (size_t)std::min(r * R.stride, R.n_fine)];
                hi = off[row + (size_t)std::min((r + 1) * R.stride, R.n_fine)];
            }
            for (int64_t e0 = lo; e0 < hi; e0 += cap)
                tiles.push_back(T{BlkTile{b, 0, e0, std::min(e0 + cap, hi)}, r});
        }
        if (tiles.size() - first > 1)
            for (size_t i = first; i < tiles.size(); i++) tiles[i].t.split = 1;
    }
    if (ranged)
        std::stable_sort(tiles.begin(), tiles.end(),
                         [](const T &a, const T &b) { return a.range < b.range; });
    else if (order == 0 || order == 2)
        std::stable_sort(tiles.begin(), tiles.end(), [order](const T &a, const T &b) {
            const int64_t la = a.t.e1 - a.t.e0, lb = b.t.e1 - b.t.e0;
            return order == 0 ? la < lb : la > lb;
        });
    else if (order == 3)
        std::stable_sort(tiles.begin(), tiles.end(),
                         [](const T &a, const T &b) { return a.t.blk > b.t.blk; });
    std::vector<BlkTile> out;
    out.reserve(tiles.size());
    for (const T &x : tiles) out.push_back(x.t);
    return out;
}

// Slots of a light tile at most: about kLightTiles tiles over the light
// edges, a power of two (whole chunks), never above the full tiles' cap.
static int64_t light_cap(const sssp_graph *g, int64_t cap)
{
    int64_t c = kLightTileMin;
    while (c < cap && c * kLightTiles < g->light_edges) c <<= 1;
    return std::min(c, cap);
}

void retile_blocked(sssp_graph *g, int64_t cap, int order, int range_bits)
{
    if (g->b_off_host.empty()) return;
    BlkRanges R = g->b_ranges;
    R.stride = 0;
    if (range_bits > 0) {
        if (R.off.empty() || range_bits < R.fine_bits || range_bits > 31)
            throw Error{SSSP_ERR_ARG, "blk_range_bits: source ranges unavailable for this size"};
        R.stride = 1 << (range_bits - R.fine_bits);
    }
    // Without an order from the caller: largest first when the tiles are more
    // than run at once, so that the last ones to start are short; smallest
    // first when all start together. Heuristic solve / BFS, smallest against
    // largest first: R-MAT 19 x 32 (529 tiles) 1.08x / 1.10x, 22 x 15 (633)
    // 1.10x / 1.10x, 24 x 10 (1452) 1.07x / 1.17x, 25 x 16 (4391) 1.06x / 1.11x, 21
    // x 40 (683) 0.96x / 0.97x; skewed 4 M x 14 (489) 0.95x / 0.91x, uniform 3.9 M x
    // 6 (477) 0.96x / 0.98x. The plain schedule keeps smallest first: it lowers
    // more within a pass that way (skewed 16 M x 8 0.88x, R-MAT 21 x 40 0.94x, 22
    // x 15 1.09x, 19 x 32 1.15x with the largest first).
    const bool by_count = order < 0 && R.stride == 0;
    auto cut = [&](const std::vector<int64_t> &bo, int64_t c, const std::vector<int64_t> &off) {
        std::vector<BlkTile> t = make_blk_tiles(bo, c, std::max(order, 0), R, off);
        if (by_count && (int64_t)t.size() > kBlkTileWave) t = make_blk_tiles(bo, c, 2, R, off);
        return t;
    };
    const std::vector<BlkTile> tiles = cut(g->b_off_host, cap, R.off);
    const bool largest = by_count && (int64_t)tiles.size() > kBlkTileWave;
    std::vector<BlkTile> ltiles, ptiles;
    if (g->light_edges > 0) ltiles = cut(g->l_off_host, light_cap(g, cap), R.loff);
    if (largest) ptiles = make_blk_tiles(g->b_off_host, cap, 0, R, R.off);
    if (order < 0) order = largest ? 2 : 0;
    auto upload = [&](const std::vector<BlkTile> &t) {
        BlkTile *d = dmalloc<BlkTile>(std::max<size_t>(t.size(), 1));
        SSSP_HIP(hipMemcpyAsync(d, t.data(), sizeof(BlkTile) * t.size(), hipMemcpyHostToDevice,
                                g->stream));
        return d;
    };
    struct Own {
        void *p[4] = {};
        ~Own()
        {
            for (void *x : p) dfree(x);
        }
    } own;
    BlkTile *td = upload(tiles);
    own.p[0] = td;
    BlkTile *ltd = ltiles.empty() ? nullptr : upload(ltiles);
    own.p[1] = ltd;
    uint16_t *ad = dmalloc<uint16_t>(std::max<size_t>(tiles.size(), 1) * kBlkThreads);
    own.p[2] = ad;
    BlkTile *ptd = ptiles.empty() ? nullptr : upload(ptiles);
    own.p[3] = ptd;
    SSSP_HIP(hipStreamSynchronize(g->stream));
    own.p[0] = g->b_tile;
    own.p[1] = g->b_ltile;
    own.p[2] = g->b_app;
    own.p[3] = g->b_ptile;
    g->b_ptile = ptd;
    g->b_tile = td;
    g->b_ltile = ltd;
    g->b_app = ad;
    g->frontier_bits = false;
    g->n_btile = (int32_t)tiles.size();
    g->n_ltile = (int32_t)ltiles.size();
    g->blk_tile_cap = cap;
    g->blk_tile_order = order;
    g->blk_range_bits = range_bits;
}

// The tiles of the local passes (k_blk_local), on graphs they are for.
static void build_local_tiles(sssp_graph *g)
{
    if (!g->local_graph || g->n_ttile > 0) return;
    const std::vector<BlkTile> tiles =
        make_blk_tiles(g->b_off_host, kLocalTileMax, 0, BlkRanges{}, {});
    const size_t n_seg = (g->b_off_host.size() - 1) << (kBlkBits - kSegBits);
    if (!g->t_tile) g->t_tile = dmalloc<BlkTile>(tiles.size());
    if (!g->t_state) g->t_state = dmalloc<TileState>(tiles.size());
    if (!g->t_seg) g->t_seg = dmalloc<int32_t>(n_seg);
    SSSP_HIP(hipMemcpyAsync(g->t_tile, tiles.data(), sizeof(BlkTile) * tiles.size(),
                            hipMemcpyHostToDevice, g->stream));
    tile_spans(g, g->t_tile, (int32_t)tiles.size(), g->t_state);
    SSSP_HIP(hipStreamSynchronize(g->stream));
    g->n_ttile = (int32_t)tiles.size();
    g->n_seg = (int32_t)n_seg;
}

// The weight threshold of the light class: the quantile `frac` of a sample
// of the weights (patterns order like the weights). frac leaves every vertex
// with out-edges about one light edge on a graph with hubs, six on one without
// (the light edges alone have to reach most vertices; hubs shorten the paths),
// between 1/16 and 1/2 of the edges. Measured (ms of a solve, frac 1/16 / 1/8 /
// 1/4 / 3/8 / 1/2; mean degrees are over vertices with out-edges): R-MAT 25 x 16
// 5.6 / 6.7 / 8.2 / 9.2 / - (mean 60), 22 x 32 2.1 / 2.05 / 2.9 / 2.9 / -,
// power-law 4 M x 8 3.2 / 2.5 / 3.0 / 2.9 / 2.8 (mean 8), uniform 6 M x 16
// 9.1 / 9.5 / 5.1 / 4.8 / 5.1, 16 M x 8 - / - / 14.5 / 12.5 / 11.6. The line
// between hubs and none is a largest out-degree of 16 times the mean.
// With many equal weights the class can come out far from that share; below
// half or above three times the target there are no classes (0xFFFFFFFF: every
// edge is light and light passes do not run).
static uint32_t light_threshold(sssp_graph *g, Carve &tmp)
{
    if (g->E == 0) return 0xFFFFFFFFu;
    const int64_t n = std::min<int64_t>(g->E, kLightSample);
    uint32_t *d = tmp.get<uint32_t>((size_t)n + 2);
    SSSP_HIP(hipMemsetAsync(d + n, 0, 8, g->stream));
    k_edge_sample<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, g->stream>>>(
        g->el_src, g->el_dst, g->el_w, g->E, (int32_t)n,
        std::min(kLocalNear, std::max(16, g->V / 32)), d);
    SSSP_LAUNCH_CHECK("k_edge_sample");
    k_max_degree<<<grid_for(g->V, 512), kBlock, 0, g->stream>>>(g->row_ptr, g->V, d + n);
    SSSP_LAUNCH_CHECK("k_max_degree");
    std::vector<uint32_t> s((size_t)n + 2);
    SSSP_HIP(hipMemcpyAsync(s.data(), d, 4 * s.size(), hipMemcpyDeviceToHost, g->stream));
    SSSP_HIP(hipStreamSynchronize(g->stream));
    const double mean = (double)g->E / std::max(g->n_nzo, 1);
    const bool hubs = (double)s[(size_t)n] >= 16.0 * mean;
    g->out_hubs = hubs;
    if (!hubs && mean < kLightMinDegree) {
        // local passes: half the sampled edges join near ids (on random graphs
        // of 2000-7000 vertices, whose edges all lie in one block, they took
        // 1.4 times as long as the edge-list passes)
        g->local_graph = (int64_t)s.back() * 2 >= n;
        return 0xFFFFFFFFu;
    }
    const double per_vertex = hubs ? 1.0 : 6.0;
    const double frac = std::min(0.5, std::max(1.0 / 16, per_vertex / mean));
    s.resize((size_t)n);
    const double target = frac * (double)n;
    const auto nth = s.begin() + std::min<int64_t>(n - 1, (int64_t)target);
    std::nth_element(s.begin(), nth, s.end());
    const uint32_t at = *nth;
    // the class is w <= thr: `at` itself, or the value before it
    const int64_t up = std::count_if(s.begin(), s.end(), [at](uint32_t x) { return x <= at; });
    const int64_t lo = std::count_if(s.begin(), s.end(), [at](uint32_t x) { return x < at; });
    const bool use_lo = at > 0 && std::abs((double)lo - target) < std::abs((double)up - target);
    const double got = use_lo ? (double)lo : (double)up;
    if (got < 0.5 * target || got > 3.0 * target || got > 0.75 * (double)n) return 0xFFFFFFFFu;
    return use_lo ? at - 1 : at;
}

static void sample_weights(sssp_graph *g, Carve &tmp)
{
    if (g->weights_known) return;
    g->light_thr = light_threshold(g, tmp);
    g->weights_known = true;
}

// Packs nch chunks of whole sources and destination offsets (k_blk_pack).
static void pack_chunks(const int32_t *bs, const uint16_t *bd, int64_t nch, hipStream_t s, Carve &tmp,
                        uint32_t **pk, int32_t **cbase, int32_t **wide, int64_t *nwide)
{
    uint8_t *wflag = tmp.get<uint8_t>((size_t)nch);
    int32_t *widx = tmp.get<int32_t>((size_t)nch);
    const unsigned chunk_grid = (unsigned)((nch * 64 + kBlock - 1) / kBlock);
    k_blk_chunk_wide<<<chunk_grid, kBlock, 0, s>>>(bs, nch, wflag);
    SSSP_LAUNCH_CHECK("k_blk_chunk_wide");
    std::vector<uint8_t> wf((size_t)nch);
    SSSP_HIP(hipMemcpyAsync(wf.data(), wflag, (size_t)nch, hipMemcpyDeviceToHost, s));
    SSSP_HIP(hipStreamSynchronize(s));
    std::vector<int32_t> wi((size_t)nch);
    int64_t nw = 0;
    for (int64_t c = 0; c < nch; c++) wi[(size_t)c] = wf[(size_t)c] ? (int32_t)nw++ : -1;
    SSSP_HIP(hipMemcpyAsync(widx, wi.data(), 4 * (size_t)nch, hipMemcpyHostToDevice, s));
    *pk = dmalloc<uint32_t>((size_t)(nch * kBlkChunk));
    *cbase = dmalloc<int32_t>((size_t)nch);
    *wide = nw ? dmalloc<int32_t>((size_t)(nw * kBlkChunk)) : nullptr;
    *nwide = nw;
    k_blk_pack<<<chunk_grid, kBlock, 0, s>>>(bs, bd, widx, nch, *pk, *cbase, *wide);
    SSSP_LAUNCH_CHECK("k_blk_pack");
    SSSP_HIP(hipStreamSynchronize(s));
}

// Source-range cuts of every block's run (k_blk_range_offsets), to the host.
static void range_cuts(const int32_t *bs, const int64_t *boff, int32_t nblk, int32_t nfine,
                       hipStream_t s, Carve &tmp, std::vector<int64_t> *out)
{
    const int64_t n_off = (int64_t)nblk * (nfine + 1);
    int64_t *roff = tmp.get<int64_t>((size_t)n_off);
    k_blk_range_offsets<<<grid_for(n_off), kBlock, 0, s>>>(bs, boff, nblk, kBlkRangeFineBits, nfine,
                                                          roff);
    SSSP_LAUNCH_CHECK("k_blk_range_offsets");
    out->resize((size_t)n_off);
    SSSP_HIP(hipMemcpyAsync(out->data(), roff, 8 * (size_t)n_off, hipMemcpyDeviceToHost, s));
    SSSP_HIP(hipStreamSynchronize(s));
}

// The light list, from the blocked list's edges (bs, bd and b_w, nch chunks,
// boff: first slot of each block on the device): light edges counted per
// chunk, scanned, and gathered in order, each block's run padded to whole
// chunks as the blocked list's. (The padding of the blocked list may be light:
// its copies of an edge are copied too.)
static void build_light_list(sssp_graph *g, const int32_t *bs, const uint16_t *bd,
                             const int64_t *boff, int32_t nblk, int64_t nch, Carve &tmp)
{
    hipStream_t s = g->stream;
    const uint32_t thr = g->light_thr;
    if (thr == 0xFFFFFFFFu) return;
    int64_t *pos = tmp.get<int64_t>((size_t)nch + 1);
    int64_t *lptr = tmp.get<int64_t>(2 * ((size_t)nblk + 1));
    int64_t *loff = lptr + nblk + 1;
    const unsigned chunk_grid = (unsigned)((nch * 64 + kBlock - 1) / kBlock);
    k_light_count<<<chunk_grid, kBlock, 0, s>>>(g->b_w, nch * kBlkChunk, nch, thr, pos);
    SSSP_LAUNCH_CHECK("k_light_count");
    k_fill_i64<<<1, 64, 0, s>>>(pos + nch, 1, 0);  // the last position: the total
    device_exclusive_scan_i64(pos, pos, nch + 1, g->blk_a, g->blk_b, g->n_blk, s);
    k_light_starts<<<grid_for((int64_t)nblk + 1), kBlock, 0, s>>>(pos, boff, nblk, lptr);
    SSSP_LAUNCH_CHECK("k_light_starts");
    std::vector<int64_t> lp((size_t)nblk + 1), lo((size_t)nblk + 1, 0);
    SSSP_HIP(hipMemcpyAsync(lp.data(), lptr, 8 * lp.size(), hipMemcpyDeviceToHost, s));
    SSSP_HIP(hipStreamSynchronize(s));
    for (size_t b = 0; b < (size_t)nblk; b++)
        lo[b + 1] = lo[b] + (lp[b + 1] - lp[b] + kBlkChunk - 1) / kBlkChunk * kBlkChunk;
    const int64_t Lp = lo[(size_t)nblk];
    if (Lp == 0) return;
    SSSP_HIP(hipMemcpyAsync(loff, lo.data(), 8 * lo.size(), hipMemcpyHostToDevice, s));
    int32_t *ls = tmp.get<int32_t>((size_t)Lp);
    uint16_t *ld = tmp.get<uint16_t>((size_t)Lp);
    g->l_w = dmalloc<uint32_t>((size_t)Lp);
    k_light_gather<<<chunk_grid, kBlock, 0, s>>>(bs, bd, g->b_w, nch, thr, pos, boff, nblk, lptr,
                                                 loff, ls, ld, g->l_w);
    SSSP_LAUNCH_CHECK("k_light_gather");
    k_blk_pad<<<grid_for((int64_t)nblk * kBlkChunk), kBlock, 0, s>>>(lptr, loff, nblk, ls, ld,
                                                                     g->l_w);
    SSSP_LAUNCH_CHECK("k_blk_pad light");
    pack_chunks(ls, ld, Lp / kBlkChunk, s, tmp, &g->l_pk, &g->l_cbase, &g->l_wide, &g->l_nwide);
    if (g->b_ranges.n_fine > 0)
        range_cuts(ls, loff, nblk, g->b_ranges.n_fine, s, tmp, &g->b_ranges.loff);
    g->l_off_host = lo;
    g->l_edges = Lp;
    g->light_edges = lp[(size_t)nblk];
}

// f(), which builds what solves can do without: false, with nothing of it
// kept, when there is no memory for it.
template <class F, class Undo>
static bool without_memory_skip(F &&f, Undo &&undo)
{
    try {
        f();
        return true;
    } catch (const Error &e) {
        undo();
        if (e.code != SSSP_ERR_OOM) throw;
        (void)hipGetLastError();
        return false;
    }
}

static void drop_light_list(sssp_graph *g)
{
    (void)hipStreamSynchronize(g->stream);
    for (void *p : {(void *)g->l_w, (void *)g->l_pk, (void *)g->l_cbase, (void *)g->l_wide}) dfree(p);
    g->l_w = g->l_pk = nullptr;
    g->l_cbase = g->l_wide = nullptr;
    g->l_edges = g->l_nwide = g->light_edges = 0;
    g->l_off_host.clear();
    g->b_ranges.loff.clear();
}

// The blocked list's edges again as whole sources and destination offsets
// (one wave per chunk).
__global__ __launch_bounds__(kBlock) void k_blk_unpack(const uint32_t *pk, const int32_t *cbase,
                                                       const int32_t *wide, int64_t nch,
                                                       int32_t *bs, uint16_t *bd)
{
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    if (c >= nch) return;  // wave-uniform
    const int64_t e = c * kBlkChunk + 4 * __lane_id();
    const int32_t cb = cbase[c];
    uint32_t p[4];
    int32_t sum = 0;
    for (int k = 0; k < 4; k++) {
        p[k] = pk[e + k];
        sum += (int32_t)(p[k] >> kBlkBits);
    }
    int32_t at = cb + wave_scan32(sum) - sum;
    for (int k = 0; k < 4; k++) {
        at += (int32_t)(p[k] >> kBlkBits);
        bs[e + k] = cb >= 0 ? at : wide[(int64_t)(-1 - cb) * kBlkChunk + 4 * __lane_id() + k];
        bd[e + k] = (uint16_t)(p[k] & ((1u << kBlkBits) - 1));
    }
}

void ensure_light_list(sssp_graph *g)
{
    if (g->light_built || g->E == 0) return;
    hipStream_t s = g->stream;
    const size_t Ep = (size_t)g->b_edges, nblk = g->b_off_host.size() - 1;
    g->light_built = without_memory_skip(
        [&] {
            Carve tmp(nullptr, 0);
            sample_weights(g, tmp);
            if (g->light_thr == 0xFFFFFFFFu) return;
            int32_t *bs = tmp.get<int32_t>(Ep);
            uint16_t *bd = tmp.get<uint16_t>(Ep);
            int64_t *boff = tmp.get<int64_t>(nblk + 1);
            SSSP_HIP(hipMemcpyAsync(boff, g->b_off_host.data(), 8 * (nblk + 1),
                                    hipMemcpyHostToDevice, s));
            const int64_t nch = (int64_t)Ep / kBlkChunk;
            k_blk_unpack<<<(unsigned)((nch * 64 + kBlock - 1) / kBlock), kBlock, 0, s>>>(
                g->b_pk, g->b_cbase, g->b_wide, nch, bs, bd);
            SSSP_LAUNCH_CHECK("k_blk_unpack");
            build_light_list(g, bs, bd, boff, (int32_t)nblk, nch, tmp);
            if (g->light_edges > 0)
                retile_blocked(g, g->blk_tile_cap, g->blk_order_set ? g->blk_tile_order : -1,
                               g->blk_range_bits);
            SSSP_HIP(hipStreamSynchronize(s));
        },
        [&] { drop_light_list(g); });
}

void ensure_local_tiles(sssp_graph *g)
{
    if (g->local_built || g->E == 0) return;
    g->local_built = without_memory_skip(
        [&] {
            Carve tmp(nullptr, 0);
            sample_weights(g, tmp);
            build_local_tiles(g);
        },
        [] {});
}

// The light edges of the src-sorted list as records of their own, where they
// pay (kMLightEdges).
static void build_light_records(sssp_graph *g, MRec **rec, BlkTile **tile, int32_t *n_tile)
{
    hipStream_t s = g->stream;
    Carve tmp(nullptr, 0);
    sample_weights(g, tmp);
    if (g->light_thr == 0xFFFFFFFFu ||
        g->E < (g->out_hubs ? kMLightEdges : kMLightEvenEdges) || g->E < kMLightMean * g->n_nzo)
        return;
    const int64_t E = g->E, nch = (E + kBlkChunk - 1) / kBlkChunk;
    int64_t *pos = tmp.get<int64_t>((size_t)nch + 1);
    const unsigned grid = (unsigned)((nch * 64 + kBlock - 1) / kBlock);
    k_light_count<<<grid, kBlock, 0, s>>>(g->el_w, E, nch, g->light_thr, pos);
    SSSP_LAUNCH_CHECK("k_light_count");
    k_fill_i64<<<1, 64, 0, s>>>(pos + nch, 1, 0);
    device_exclusive_scan_i64(pos, pos, nch + 1, g->blk_a, g->blk_b, g->n_blk, s);
    int64_t nl = 0;
    SSSP_HIP(hipMemcpyAsync(&nl, pos + nch, 8, hipMemcpyDeviceToHost, s));
    SSSP_HIP(hipStreamSynchronize(s));
    if (nl == 0) return;
    int32_t *ls = tmp.get<int32_t>((size_t)nl), *ld = tmp.get<int32_t>((size_t)nl);
    uint32_t *lw = tmp.get<uint32_t>((size_t)nl);
    k_light_select<<<grid, kBlock, 0, s>>>(g->el_src, g->el_dst, g->el_w, E, nch, g->light_thr, pos,
                                           ls, ld, lw);
    SSSP_LAUNCH_CHECK("k_light_select");
    build_records(g, ls, ld, lw, nl, rec, tile, n_tile);
}

void build_multi_layout(sssp_graph *g)
{
    if (g->m_rec || g->E == 0) return;
    MRec *rec[2] = {};
    BlkTile *tile[2] = {};
    int32_t n[2] = {};
    auto drop = [&](int i) {
        (void)hipStreamSynchronize(g->stream);
        dfree(rec[i]);
        dfree(tile[i]);
        rec[i] = nullptr;
        tile[i] = nullptr;
        n[i] = 0;
    };
    try {
        build_records(g, g->el_src, g->el_dst, g->el_w, g->E, &rec[0], &tile[0], &n[0]);
        (void)without_memory_skip([&] { build_light_records(g, &rec[1], &tile[1], &n[1]); },
                                  [&] { drop(1); });
    } catch (...) {
        drop(0);
        throw;
    }
    g->m_rec = rec[0];
    g->m_tile = tile[0];
    g->n_mtile = n[0];
    g->m_lrec = rec[1];
    g->m_ltile = tile[1];
    g->n_mltile = n[1];
}

void build_layouts(sssp_graph *g, const int32_t *d_src, const int32_t *d_dst, const uint32_t *d_w,
                   bool build_csc)
{
    hipStream_t s = g->stream;
    const int64_t E = g->E;
    const int32_t V = g->V;

    validate_edges(d_src, d_dst, d_w, g->wtype, E, V, s);

    // scratch for the sorts (of E edges, and of V vertices for the order)
    const int64_t n_sort = std::max<int64_t>(E, (int64_t)V);
    const int64_t rs_tiles = (n_sort + kRsTile - 1) / kRsTile;
    const int64_t scan_n = std::max<int64_t>((int64_t)V + 1, 256 * rs_tiles);
    g->n_blk = scan_blocks_needed(scan_n);
    g->blk_a = dmalloc<int64_t>((size_t)g->n_blk);
    g->blk_b = dmalloc<int64_t>((size_t)g->n_blk);
    uint32_t *kA = dmalloc<uint32_t>(4 * (size_t)n_sort);  // four arrays in one allocation
    uint32_t *kB = kA + n_sort, *vA = kB + n_sort, *vB = vA + n_sort;
    int64_t *counts = dmalloc<int64_t>((size_t)std::max<int64_t>(256 * rs_tiles, (int64_t)V + 1));
    int64_t *tmp_pos = dmalloc<int64_t>((size_t)V + 1);
    struct Scratch {
        void *p[8];
        ~Scratch()
        {
            for (void *x : p) dfree(x);
        }
    } scratch{{kA, counts, tmp_pos, nullptr, nullptr, nullptr, nullptr, nullptr}};
    const RsScratch rs{counts, g->blk_a, g->blk_b, g->n_blk};

    // ---- vertex order: slot = rank by descending in- plus out-degree, ties
    // by descending out-degree, then by vertex id (two stable sorts: by
    // out-degree, then by total degree); the edges are renamed into slots
    // before any layout is built. On R-MAT graphs the hubs are vertex ids
    // with few one bits, scattered over the whole id range, so the distance
    // gathers of a dense round touch a cache line per hub; in slot order the
    // hubs' distances are one dense prefix, and among the many vertices of
    // equal small degree the more often gathered come first. Orders measured
    // at R-MAT scale 25 (dense round per launch, learned solve): ids 2.04 /
    // 21.3 ms; total degree, ties by id 1.70 / 20.0; out-degree 1.79 / 20.5;
    // in-degree 1.68 / 20.1; total degree, ties by out-degree 1.61 / 19.0.
    // It pays from 2^23 vertices on skewed graphs (learned R-MAT GTEPS with /
    // without: scale 23 21.4 / 19.0, 24 24.5 / 22.0, 25 +12 %), not below or
    // without hubs (scale 22 x 16 14.6 / 14.6, 22 x 32 20.3 / 22.7, uniform
    // 2^24 x 16 7.9 / 8.2): by default the layouts use it when V >= 2^23 and
    // the largest total degree is at least 16 times the mean.
    uint32_t *tot = nullptr, *outd = nullptr;
    if (g->relabel_mode > 0 || (g->relabel_mode == 0 && V >= (1 << 23))) {
        if (E > 0 && V > 1) {
            tot = dmalloc<uint32_t>((size_t)V);
            scratch.p[6] = tot;
            outd = dmalloc<uint32_t>((size_t)V);
            scratch.p[7] = outd;
            SSSP_HIP(hipMemsetAsync(tot, 0, 4 * (size_t)V, s));
            SSSP_HIP(hipMemsetAsync(outd, 0, 4 * (size_t)V, s));
            k_degrees<<<grid_for(E), kBlock, 0, s>>>(d_src, d_dst, E, tot, outd);
            SSSP_LAUNCH_CHECK("k_degrees");
        }
        g->relabel = tot != nullptr;
        if (g->relabel && g->relabel_mode == 0) {
            uint32_t *mx = dmalloc<uint32_t>(1);
            struct F1 {
                void *p;
                ~F1() { dfree(p); }
            } f1{mx};
            SSSP_HIP(hipMemsetAsync(mx, 0, 4, s));
            k_max_u32<<<grid_for(V, 256), kBlock, 0, s>>>(tot, V, mx);
            SSSP_LAUNCH_CHECK("k_max_u32");
            uint32_t hmax = 0;
            SSSP_HIP(hipMemcpyAsync(&hmax, mx, 4, hipMemcpyDeviceToHost, s));
            SSSP_HIP(hipStreamSynchronize(s));
            // mean total degree = 2E / V
            g->relabel = (double)hmax * (double)V >= 16.0 * 2.0 * (double)E;
        }
    }
    if (g->relabel) {
        uint32_t *okeys = dmalloc<uint32_t>((size_t)V);
        uint32_t *by_out = dmalloc<uint32_t>((size_t)V);
        struct F0 {
            void *p[2];
            ~F0()
            {
                for (void *x : p) dfree(x);
            }
        } f0{{okeys, by_out}};
        // sorted keys with their positions: kB, and by_out, then vB
        uint32_t *const ord = vB;
        k_order_keys<<<grid_for(V), kBlock, 0, s>>>(outd, nullptr, V, okeys);
        SSSP_LAUNCH_CHECK("k_order_keys out");
        radix_sort<2>({{okeys, nullptr}}, {{kB, by_out}}, {{kA, vA}}, V, 0, key_bits(kOrderCap), rs,
                      s);
        k_order_keys<<<grid_for(V), kBlock, 0, s>>>(tot, by_out, V, okeys);
        SSSP_LAUNCH_CHECK("k_order_keys total");
        radix_sort<2>({{okeys, nullptr}}, {{kB, ord}}, {{kA, vA}}, V, 0, key_bits(kOrderCap), rs, s);
        g->vperm = dmalloc<int32_t>((size_t)V);
        g->vinv = dmalloc<int32_t>((size_t)V);
        k_invert_order<<<grid_for(V), kBlock, 0, s>>>(by_out, ord, V, g->vperm, g->vinv);
        SSSP_LAUNCH_CHECK("k_invert_order");
        // the renamed edges take the degree arrays' places in the scratch
        // list: both are dead once the order exists
        SSSP_HIP(hipStreamSynchronize(s));
        dfree(tot);
        dfree(outd);
        scratch.p[6] = scratch.p[7] = nullptr;
        int32_t *rs = dmalloc<int32_t>((size_t)E);
        scratch.p[6] = rs;
        int32_t *rd = dmalloc<int32_t>((size_t)E);
        scratch.p[7] = rd;
        k_relabel_edges<<<grid_for(E), kBlock, 0, s>>>(d_src, d_dst, E, g->vperm, rs, rd);
        SSSP_LAUNCH_CHECK("k_relabel_edges");
        g->vperm_host.resize((size_t)V);
        SSSP_HIP(hipMemcpyAsync(g->vperm_host.data(), g->vperm, 4 * (size_t)V,
                                hipMemcpyDeviceToHost, s));
        SSSP_HIP(hipStreamSynchronize(s));
        d_src = rs;
        d_dst = rd;
    } else {
        dfree(tot);
        dfree(outd);
        scratch.p[6] = scratch.p[7] = nullptr;
    }

    // ---- CSR / src-sorted edge list ----
    g->el_src = dmalloc<int32_t>((size_t)E);
    g->el_dst = dmalloc<int32_t>((size_t)E);
    g->el_w = dmalloc<uint32_t>((size_t)E);
    g->row_ptr = dmalloc<int64_t>((size_t)V + 1);
    const int vbits = key_bits((int64_t)V - 1);
    radix_sort<3>({{u32p(d_src), u32p(d_dst), u32p(d_w)}},
                  {{u32p(g->el_src), u32p(g->el_dst), g->el_w}}, {{kA, kB, vA}}, E, 0, vbits, rs, s);
    rowptr_from_sorted(u32p(g->el_src), E, V, g->row_ptr, s);
    build_static_list(g->row_ptr, V, E, counts, tmp_pos, g->blk_a, g->blk_b, g->n_blk, s,
                      &g->nzo_v, &g->nzo_scan, &g->n_nzo, g->nzo_tile);

    // ---- XCD-partitioned edge list: stable split of the src-sorted list into
    // 8 destination groups (src order kept inside each group) ----
    {
        const size_t Et = (size_t)E + 32;  // at most 3 slots of padding per group
        g->x_src = dmalloc<int32_t>(Et);
        g->x_dst = dmalloc<int32_t>(Et);
        g->x_w = dmalloc<uint32_t>(Et);
        g->xgoff = dmalloc<int64_t>(18);  // the groups' offsets, then the padding before them
        int64_t *const pad = g->xgoff + 9;
        const int64_t ntiles = (E + kRsTile - 1) / kRsTile;
        if (E > 0) rs_count<true>(u32p(g->el_dst), E, 0, 8, rs, s);
        k_group_offsets<<<1, 64, 0, s>>>(counts, ntiles, E, g->xgoff, pad);
        SSSP_LAUNCH_CHECK("k_group_offsets");
        if (E > 0) {
            k_rs_split<3, true><<<(unsigned)ntiles, kRsThreads, 0, s>>>(
                {{u32p(g->el_dst), u32p(g->el_src), g->el_w}},
                {{u32p(g->x_dst), u32p(g->x_src), g->x_w}}, E, 0, 8, counts, ntiles, pad);
            SSSP_LAUNCH_CHECK("k_rs_split (XCD groups)");
            k_group_pad<<<1, 32, 0, s>>>(g->xgoff, pad, E, g->x_src, g->x_dst, g->x_w);
            SSSP_LAUNCH_CHECK("k_group_pad");
        }
        g->xgoff_host.resize(9);
        SSSP_HIP(hipMemcpyAsync(g->xgoff_host.data(), g->xgoff, 72, hipMemcpyDeviceToHost, s));
        SSSP_HIP(hipStreamSynchronize(s));
    }

    // ---- destination-blocked edge list ----
    if (E > 0) {
        const int32_t nblk = (int32_t)(((int64_t)V + (1 << kBlkBits) - 1) >> kBlkBits);
        int64_t *bptr = dmalloc<int64_t>((size_t)nblk + 1);
        int64_t *boff = dmalloc<int64_t>((size_t)nblk + 1);
        // room for every block's padding to whole chunks
        const size_t Em = (size_t)E + (size_t)nblk * (kBlkChunk - 1);
        int32_t *bs = dmalloc<int32_t>(Em);
        uint16_t *bd = dmalloc<uint16_t>(Em);
        struct F3 {
            void *p[4];
            ~F3()
            {
                for (void *x : p) dfree(x);
            }
        } f3{{bptr, boff, bs, bd}};
        g->b_w = dmalloc<uint32_t>(Em);
        // into kA, kB, vA, by way of vB and the list's own arrays
        radix_sort<3>({{u32p(g->el_dst), u32p(g->el_src), g->el_w}}, {{kA, kB, vA}},
                      {{vB, u32p(bs), g->b_w}}, E, kBlkBits, key_bits(nblk - 1), rs, s);
        rowptr_from_sorted(kA, E, nblk, bptr, s, kBlkBits);
        std::vector<int64_t> bp((size_t)nblk + 1), bo((size_t)nblk + 1);
        SSSP_HIP(hipMemcpyAsync(bp.data(), bptr, 8 * bp.size(), hipMemcpyDeviceToHost, s));
        SSSP_HIP(hipStreamSynchronize(s));
        bo[0] = 0;
        // Without hubs (the largest block's in-edges under twice the mean:
        // uniform random graphs) appending all-edge rounds lose to dense ones
        // from a smaller share of the graph on; skewed graphs (R-MAT) keep
        // the appends longer. Measured: ER 2^24 x 16 34.8 ms at 0.4 against
        // 37.5 at 0.15, R-MAT 22 x 32 6.1 ms at 0.15 against 6.5 at 0.4.
        int64_t max_blk = 0;
        for (int32_t b = 0; b < nblk; b++)
            max_blk = std::max(max_blk, bp[(size_t)b + 1] - bp[(size_t)b]);
        const bool no_hubs = (double)max_blk * nblk < 2.0 * (double)E;
        if (no_hubs) g->dense_all_frac = 0.4;
        for (int32_t b = 0; b < nblk; b++)
            bo[(size_t)b + 1] = bo[(size_t)b] +
                                (bp[(size_t)b + 1] - bp[(size_t)b] + kBlkChunk - 1) / kBlkChunk * kBlkChunk;
        // Tile cap. A pass over a small list lasts as long as its longest
        // tile, so the list is cut into about as many parts as run at once
        // (kBlkTileWave); shorter tiles than that only add block write-backs
        // and a second, part-filled wave. Plain solves, ms, at 2^17-edge tiles
        // / at this cap: uniform 400 K x 16 2.2 / 0.74 (2^14), R-MAT 18 x 16
        // 0.95 / 0.34 (2^13), R-MAT 20 x 16 1.32 / 1.25 (2^15), uniform 2 M x 6
        // 3.16 / 2.3 (2^15), skewed 1.2 M x 9 2.33 / 1.45 (2^15); skewed 4 M x
        // 14 2.70 at 2^17 (489 tiles), 3.14 at 2^16. Learned solves: skewed
        // 1.2 M x 9 1.27 / 1.0, R-MAT 22 x 32 and larger graphs the same at
        // 2^16 and 2^17. The cap stays 2^17 up to 2^29 edges and is doubled
        // while more than kBlkTileCount tiles of it fit in the graph -- the
        // 2.08 G-edge
        // R-MAT graph ran 50.9 GTEPS with 2^19-edge tiles, 46.7 with 2^17;
        // R-MAT 25 x 16 (2^29 edges), learned / plain ms, with the dense
        // round's stream loaded a step ahead: 14.9 / 22.3 at 2^17, 15.6 /
        // 23.3 at 2^18, 17.0 / 26.3 at 2^19 (before that change 2^18 was the
        // faster: 19.2 against 19.6 ms). A power of two, so every tile holds
        // whole chunks.
        int64_t tcap = kBlkTileFloor;
        while (tcap * kBlkTileWave < E && tcap < kBlkTileEdges) tcap <<= 1;
        while (tcap * kBlkTileCount < E) tcap <<= 1;
        g->b_off_host = bo;
        const int64_t Ep = bo[(size_t)nblk];
        const int64_t nch = Ep / kBlkChunk;
        SSSP_HIP(hipMemcpyAsync(boff, bo.data(), 8 * bo.size(), hipMemcpyHostToDevice, s));
        // whole sources and destination offsets first, packed below
        g->b_edges = Ep;
        k_blk_place<<<grid_for(E), kBlock, 0, s>>>(reinterpret_cast<const int32_t *>(kB), kA, vA, E, bptr, boff, bs, bd, g->b_w);
        SSSP_LAUNCH_CHECK("k_blk_place");
        k_blk_pad<<<grid_for((int64_t)nblk * kBlkChunk), kBlock, 0, s>>>(bptr, boff, nblk, bs, bd,
                                                                         g->b_w);
        SSSP_LAUNCH_CHECK("k_blk_pad");
        Carve tmp(kA, 16 * (size_t)n_sort);  // the sorted arrays are placed
        pack_chunks(bs, bd, nch, s, tmp, &g->b_pk, &g->b_cbase, &g->b_wide, &g->b_nwide);
        // source-range cuts of every block at 2^kBlkRangeFineBits granularity
        // (for tiles dispatched range by range), when the table is small
        const int64_t nfine = ((int64_t)V + (1 << kBlkRangeFineBits) - 1) >> kBlkRangeFineBits;
        if ((int64_t)nblk * (nfine + 1) <= kBlkRangeMaxEntries) {
            range_cuts(bs, boff, nblk, (int32_t)nfine, s, tmp, &g->b_ranges.off);
            g->b_ranges.fine_bits = kBlkRangeFineBits;
            g->b_ranges.n_fine = (int32_t)nfine;
        }
        // What the graph's solves run passes over, unless they run in one
        // workgroup: the light list where light passes pay (the sample of the
        // weights and the list are 0.1 and 0.15 ms of a small build of 0.7 ms)
        if (V > kSoloVerts || E > std::min(kSoloLocalEdges, kRegEdges)) sample_weights(g, tmp);
        const bool solo = V <= kSoloVerts && E <= (g->local_graph ? kSoloLocalEdges : kSoloEdges);
        if (!solo && (light_pays(g) || E >= g->plain_below_edges))
            g->light_built =
                without_memory_skip([&] { build_light_list(g, bs, bd, boff, nblk, nch, tmp); },
                                    [&] { drop_light_list(g); });
        SSSP_HIP(hipStreamSynchronize(s));
        // Without hubs the d[src] gathers of a tile spread over the whole
        // distance array (degree order cannot gather them), so a graph whose
        // distances outgrow the L2 several times over runs its tiles by source
        // range, 8 ranges (uniform random graphs, ms learned / plain / dense
        // round: 2^24 x 16 31.7 / 71.7 / 2.96 by block, 23.6 / 36.5 / 1.57 in
        // 8 ranges, 26.4 / 37.1 / 1.83 in 16, 23.9 / 41.6 / 1.75 in 4; 2^22 x 16
        // 7.75 / 11.1 / 0.38 by block, 7.09 / 7.93 / 0.38 in 8 ranges). Graphs
        // with hubs lose by it (R-MAT 25 x 16: 17.2 / 24.7 ms by block, 18.5 /
        // 26.4 in 8 ranges).
        int range_bits = 0;
        if (no_hubs && V >= (1 << kBlkRangeMinVertexBits) && !g->b_ranges.off.empty()) {
            int lg = 0;
            while (((int64_t)1 << lg) < (int64_t)V) lg++;
            range_bits = std::max(kBlkRangeFineBits, lg - 3);
        }
        retile_blocked(g, tcap, -1, range_bits);
        if (!solo)
            g->local_built = without_memory_skip([&] { build_local_tiles(g); }, [] {});
    }
    if (solo_fits(g) && E > kRegEdges) ensure_chunk_sources(g);

    // ---- CSC ----
    if (build_csc) {
        g->csc_src = dmalloc<int32_t>((size_t)E);
        g->csc_w = dmalloc<uint32_t>((size_t)E);
        g->col_ptr = dmalloc<int64_t>((size_t)V + 1);
        radix_sort<3>({{u32p(d_dst), u32p(d_src), u32p(d_w)}}, {{vB, u32p(g->csc_src), g->csc_w}},
                      {{kA, kB, vA}}, E, 0, vbits, rs, s);
        rowptr_from_sorted(vB, E, V, g->col_ptr, s);
        build_static_list(g->col_ptr, V, E, counts, tmp_pos, g->blk_a, g->blk_b, g->n_blk, s,
                          &g->nzi_v, &g->nzi_scan, &g->n_nzi, g->nzi_tile);
        g->has_csc = true;
    }
    SSSP_HIP(hipStreamSynchronize(s));
}

}  // namespace sssp
