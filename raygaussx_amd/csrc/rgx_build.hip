// LBVH construction on the GPU: k-sigma AABBs + scene bbox, 63-bit Morton
// codes, LDS-staged LSD radix sort, Karras radix tree, bottom-up refit, skip
// links.  Replaces the OptiX GAS build (optix_raycasting/optix_utils.py:139-142)
// and the AABB pass feeding it (optix_utils.py:36-109).  Also hosts the 30-bit
// Morton ordering of the point cloud (utils/reordering_utils.py:55-104).
#include "rgx_device.h"
#include <float.h>

#include <algorithm>
#include <type_traits>

// ---------------------------------------------------------------------------
// order-preserving float <-> int encoding for atomicMin/atomicMax
__device__ __forceinline__ int32_t enc_f(float f)
{
    int32_t i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float dec_f(int32_t i) { return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff); }

__global__ void k_init_header(WsHeader *h, int64_t n)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        for (int a = 0; a < 3; ++a) {
            h->bb_min_enc[a] = enc_f(INFINITY);
            h->bb_max_enc[a] = enc_f(-INFINITY);
            h->bb_min[a] = INFINITY;
            h->bb_max[a] = -INFINITY;
        }
        h->n = n;
        h->root = 0;
        h->built = 0;
        h->refit_ok = 0;
    }
}

// First kernel of a refit.  A refit walks the parent / child / order arrays the last build left in the
// workspace, so it may only run over a finished tree of exactly n boxes: anything else (a workspace never
// built, built for another n, or left unfinished) would send the refit kernels to indices that mean nothing.
// The check runs on the device, in stream order after whatever build precedes it; when it fails the header is
// left not built, `refit_ok` stays 0 and every later kernel of the refit returns at once (`gate`).
__global__ void k_refit_begin(WsHeader *h, int64_t n)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        const bool ok = h->built == 1 && h->n == n && h->root == 0;
        for (int a = 0; a < 3; ++a) {
            h->bb_min_enc[a] = enc_f(INFINITY);
            h->bb_max_enc[a] = enc_f(-INFINITY);
            if (ok) {
                h->bb_min[a] = INFINITY;
                h->bb_max[a] = -INFINITY;
            }
        }
        h->built = 0;
        h->refit_ok = ok ? 1 : 0;
    }
}
__device__ __forceinline__ bool gate_closed(const int32_t *gate) { return gate != nullptr && *gate == 0; }

// The reductions to a bounding box: every block ends with six atomics, on the same six words of all blocks, so blocks are large and
// few (512 blocks of 256 threads -> these: bounds of 1 M points 16 -> 8 us; tree over 1 M boxes 449 -> 442, 3 M 1 023 -> 1 010).
#define RGX_REDUCE_THREADS 1024
__device__ __forceinline__ void fold_bounds(const float (*red)[6], int a, float &mn, float &mx)
{
    mn = red[0][a];
    mx = red[0][a + 3];
    for (int w = 1; w < RGX_REDUCE_THREADS / 64; ++w) {
        mn = fminf(mn, red[w][a]);
        mx = fmaxf(mx, red[w][a + 3]);
    }
}

// k-sigma AABB of a rotated ellipsoid (optix_utils.py:49-77), canonical arithmetic.
__global__ __launch_bounds__(RGX_REDUCE_THREADS) void k_aabb(const float *__restrict__ pos, const float *__restrict__ scale,
                                              const float *__restrict__ quat, const float *__restrict__ dens,
                                              int64_t n, float thr, float *__restrict__ boxes, int32_t *mn_enc, int32_t *mx_enc)
{
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float t = dens[i] / thr;
        float d = canon_logf(t * t);
        if (!(d > 0.0f)) d = 0.0f;
        d = sqrtf(d);
        float W = quat[4 * i], X = quat[4 * i + 1], Y = quat[4 * i + 2], Z = quat[4 * i + 3];
        const float nn = ((W * W + X * X) + Y * Y) + Z * Z;
        const float invn = 1.0f / sqrtf(nn + 1e-20f);
        W *= invn; X *= invn; Y *= invn; Z *= invn;
        const float L1x = 1.f - 2.f * (Y * Y + Z * Z), L1y = 2.f * (X * Y - W * Z), L1z = 2.f * (X * Z + W * Y);
        const float L2x = 2.f * (X * Y + W * Z), L2y = 1.f - 2.f * (X * X + Z * Z), L2z = 2.f * (Y * Z - W * X);
        const float L3x = 2.f * (X * Z - W * Y), L3y = 2.f * (Y * Z + W * X), L3z = 1.f - 2.f * (X * X + Y * Y);
        const float s0 = scale[3 * i], s1 = scale[3 * i + 1], s2 = scale[3 * i + 2];
        const float hx = d * sqrtf(((s0 * L1x) * (s0 * L1x) + (s1 * L1y) * (s1 * L1y)) + (s2 * L1z) * (s2 * L1z));
        const float hy = d * sqrtf(((s0 * L2x) * (s0 * L2x) + (s1 * L2y) * (s1 * L2y)) + (s2 * L2z) * (s2 * L2z));
        const float hz = d * sqrtf(((s0 * L3x) * (s0 * L3x) + (s1 * L3y) * (s1 * L3y)) + (s2 * L3z) * (s2 * L3z));
        const float c0 = pos[3 * i], c1 = pos[3 * i + 1], c2 = pos[3 * i + 2];
        const float e[6] = {c0 - hx, c1 - hy, c2 - hz, c0 + hx, c1 + hy, c2 + hz};
        if (boxes)
            for (int a = 0; a < 6; ++a) boxes[6 * i + a] = e[a];
        for (int a = 0; a < 3; ++a) {
            b[a] = fminf(b[a], e[a]);
            b[a + 3] = fmaxf(b[a + 3], e[a + 3]);
        }
    }
    __shared__ float red[RGX_REDUCE_THREADS / 64][6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int a = 0; a < 3; ++a) {
        const float mn = wave_min_all(b[a]), mx = wave_max_all(b[a + 3]);
        if (lane == 0) { red[wave][a] = mn; red[wave][a + 3] = mx; }
    }
    __syncthreads();
    if (threadIdx.x < 3 && mn_enc) {
        const int a = threadIdx.x;
        float mn, mx;
        fold_bounds(red, a, mn, mx);
        atomicMin(&mn_enc[a], enc_f(mn));
        atomicMax(&mx_enc[a], enc_f(mx));
    }
}

// stand-alone reductions keep their encoded running min/max in the output buffers themselves
__global__ void k_init_enc(int32_t *mn, int32_t *mx)
{
    if (threadIdx.x < 3) {
        mn[threadIdx.x] = enc_f(INFINITY);
        mx[threadIdx.x] = enc_f(-INFINITY);
    }
}
__global__ void k_decode_enc(int32_t *mn, int32_t *mx)
{
    if (threadIdx.x < 3) {
        ((float *)mn)[threadIdx.x] = dec_f(mn[threadIdx.x]);
        ((float *)mx)[threadIdx.x] = dec_f(mx[threadIdx.x]);
    }
}

__global__ void k_finish_bbox(WsHeader *h, float *bb_min, float *bb_max, const int32_t *gate = nullptr)
{
    const int a = threadIdx.x;
    if (gate_closed(gate)) return;
    if (a < 3) {
        const float mn = dec_f(h->bb_min_enc[a]), mx = dec_f(h->bb_max_enc[a]);
        h->bb_min[a] = mn;
        h->bb_max[a] = mx;
        if (bb_min) bb_min[a] = mn;
        if (bb_max) bb_max[a] = mx;
    }
}

// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t expand21(uint64_t x)
{
    x &= 0x1fffffull;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

// 21 bits per axis of the box centre, relative to the scene bbox (whose final form the first thread leaves in the header)
__global__ __launch_bounds__(256) void k_morton63(const float *__restrict__ boxes, int64_t n, WsHeader *hdr,
                                                  uint64_t *__restrict__ keys, uint32_t *__restrict__ vals)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t q[3];
    for (int a = 0; a < 3; ++a) {
        const float lo = dec_f(hdr->bb_min_enc[a]), hi = dec_f(hdr->bb_max_enc[a]), ext = hi - lo;
        if (i == 0) {
            hdr->bb_min[a] = lo;
            hdr->bb_max[a] = hi;
        }
        const float c = 0.5f * boxes[6 * i + a] + 0.5f * boxes[6 * i + 3 + a];
        float u = ext > 0.f ? (c - lo) / ext : 0.f;
        u = fminf(fmaxf(u, 0.f), 1.f);
        const float s = u * 2097152.0f;
        q[a] = s >= 2097151.0f ? 2097151ull : (uint64_t)s;
    }
    keys[i] = (expand21(q[0]) << 2) | (expand21(q[1]) << 1) | expand21(q[2]);
    vals[i] = (uint32_t)i;
}

// ---------------------------------------------------------------------------
// LSD radix sort, 8 bits per pass, keys u64 + values u32, stable.  Per pass:
// per-tile digit histogram -> exclusive scan over (digit, tile) -> scatter.
// The scatter keeps its per-wave digit cursors in LDS and ranks the 64 keys a
// wave handles at a time with ballot matching, so equal digits leave in input
// order.
template <typename K>
__global__ __launch_bounds__(RGX_RS_THREADS) void k_rs_hist(const K *__restrict__ keys, int64_t n, int shift,
                                                            uint32_t *__restrict__ hist, int nblocks)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * RGX_RS_TILE;
    for (int r = 0; r < RGX_RS_ITEMS; ++r) {
        const int64_t i = base + r * RGX_RS_THREADS + threadIdx.x;
        if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Exclusive scan of the (digit, tile) counts in two levels: block d scans its digit's row of tile
// counts in place and leaves the row total; every block of the scatter scans the 256 totals into
// digit bases for itself (a launch of one block for that cost more than 500 blocks doing it again).
__global__ __launch_bounds__(256) void k_rs_scan_rows(uint32_t *__restrict__ hist, int nblocks, uint32_t *__restrict__ totals)
{
    __shared__ uint32_t part[256];
    uint32_t *row = hist + (size_t)blockIdx.x * nblocks;
    uint32_t carry = 0;
    for (int base = 0; base < nblocks; base += 256) {
        const int i = base + threadIdx.x;
        const uint32_t v = i < nblocks ? row[i] : 0u;
        part[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 256; o <<= 1) { // Hillis-Steele inclusive scan
            const uint32_t t = threadIdx.x >= o ? part[threadIdx.x - o] : 0u;
            __syncthreads();
            part[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < nblocks) row[i] = carry + part[threadIdx.x] - v;
        carry += part[255];
        __syncthreads();
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// One tile's keys to their places.  digit_base: where the keys of digit threadIdx.x begin in the output; before: how many of
// them other tiles put in front of this one's.  put(place, key, value) writes.
template <typename K, int ITEMS, typename Put>
__device__ __forceinline__ void rs_scatter_tile(const K *__restrict__ kin, const uint32_t *__restrict__ vin, int64_t n, int shift,
                                                uint32_t digit_base, uint32_t before, uint32_t (&cnt)[4][256], uint32_t (&wave_total)[4], Put put)
{
    constexpr int TILE = RGX_RS_THREADS * ITEMS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // wave w owns the contiguous 64 ITEMS keys from base, 64 per round
    const int64_t base = (int64_t)blockIdx.x * TILE + (int64_t)wave * (64 * ITEMS);
    K key[ITEMS];
    uint32_t val[ITEMS], place[ITEMS]; // place: in the wave's run of the key's digit
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t i = base + r * 64 + lane;
        key[r] = i < n ? kin[i] : (K)0;
        val[r] = i < n ? vin[i] : 0u;
    }
    // Ranked as they are counted: the lanes of a digit find each other by ballots, and the first of them adds for all.  (An add per key to
    // the counters, and the ranking in a second pass over the keys: order of 1 M points 99 -> 90 us; a build of 150 k boxes 212 -> 205, 3 M 920 -> 885.)
    auto *cur = (__attribute__((address_space(3))) uint32_t *)cnt[wave];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = base + r * 64 + lane < n;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
        uint64_t same = __ballot(valid);
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            same &= bit ? bal : ~bal;
        }
        const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull));
        const uint32_t earlier = __hip_atomic_load(cur + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        place[r] = earlier + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) __hip_atomic_store(cur + d, earlier + (uint32_t)__popcll(same), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // The tile's keys are put in digit order in LDS first and leave from there: keys of one digit are neighbours
    // in the tile's order as they are in the output, so thread after thread writes consecutive words instead of
    // 64 lanes writing to as many streams.  local: where a (wave, digit) run starts in the tile's order;
    // delta[d]: output position minus position in the tile's order, for digit d.
    __shared__ uint32_t delta[256];
    __shared__ K lkey[TILE];
    __shared__ uint32_t lval[TILE];
    {
        const int d = threadIdx.x;
        uint32_t c[4], tile_count = 0;
        for (int w = 0; w < 4; ++w) tile_count += c[w] = cnt[w][d];
        uint32_t upto = tile_count; // inclusive scan of the tile's digit counts
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(upto, o);
            if (lane >= o) upto += t;
        }
        __syncthreads(); // (wave_total's first use is over)
        if (lane == 63) wave_total[wave] = upto;
        __syncthreads();
        uint32_t local = upto - tile_count;
        for (int w = 0; w < wave; ++w) local += wave_total[w];
        delta[d] = digit_base + before - local;
        for (int w = 0; w < 4; ++w) {
            cnt[w][d] = local;
            local += c[w];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        if (base + r * 64 + lane < n) {
            const uint32_t at = cnt[wave][(uint32_t)(key[r] >> shift) & 255u] + place[r];
            lkey[at] = key[r];
            lval[at] = val[r];
        }
    __syncthreads();
    const int64_t tile_base = (int64_t)blockIdx.x * TILE;
    const int tile_n = (int)(n - tile_base < TILE ? n - tile_base : TILE);
    for (int p = threadIdx.x; p < tile_n; p += RGX_RS_THREADS) {
        const K k = lkey[p];
        put((uint32_t)p + delta[(uint32_t)(k >> shift) & 255u], k, lval[p]);
    }
}

// exclusive scan over the 256 threads' values
__device__ __forceinline__ uint32_t rs_sum_before(uint32_t v, uint32_t (&wave_total)[4])
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t incl = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    if (lane == 63) wave_total[wave] = incl;
    __syncthreads();
    uint32_t sum = incl - v;
    for (int w = 0; w < wave; ++w) sum += wave_total[w];
    return sum;
}

// order: where the last pass leaves the values, or null (then vout as every pass)
template <typename K>
__global__ __launch_bounds__(RGX_RS_THREADS) void k_rs_scatter(const K *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                               K *__restrict__ kout, uint32_t *__restrict__ vout, int64_t n,
                                                               int shift, const uint32_t *__restrict__ hist, int nblocks,
                                                               const uint32_t *__restrict__ totals, int64_t *__restrict__ order)
{
    static_assert(RGX_RS_THREADS == 256, "one thread per digit");
    __shared__ uint32_t cnt[4][256];
    __shared__ uint32_t wave_total[4];
    for (int w = 0; w < 4; ++w) cnt[w][threadIdx.x] = 0;
    const uint32_t digit_base = rs_sum_before(totals[threadIdx.x], wave_total);
    rs_scatter_tile<K, RGX_RS_ITEMS>(kin, vin, n, shift, digit_base, hist[(size_t)threadIdx.x * nblocks + blockIdx.x], cnt, wave_total,
                                     [&](uint32_t at, K k, uint32_t v) {
                                         if (order) {
                                             order[at] = (int64_t)v;
                                         } else {
                                             kout[at] = k;
                                             vout[at] = v;
                                         }
                                     });
}

// Fewer keys (rs_short): two launches per pass.  What a pass of three launches takes for them is mostly their latency, some four
// microseconds each; here the tiles' counts lie row by row, and every block of the scatter sums up the rows before its own
// and all of them.  Tree over 9 000, 54 k, 100 k, 150 k, 200 k boxes, three launches a pass / two, us: 211/152 228/198 246/213
// 262/241 271/262 (262 k: 276/274, 500 k: 332/361, the rows are too many then); with 512 keys a tile up to 65 536 and
// 1 024 beyond (54 k with 1 024 or 2 048 a tile 204 and 225, 150 k with 512 or 2 048 260 and 266).  One launch a pass, the next
// pass's digits counted by atomic adds as the keys are written: 152, 206, 248, 349, 355, its adds wait for memory one by one.
template <typename K, int ITEMS>
__global__ __launch_bounds__(RGX_RS_THREADS) void k_rs_count(const K *__restrict__ keys, int64_t n, int shift, uint32_t *__restrict__ counts)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t i = ((int64_t)blockIdx.x * ITEMS + r) * RGX_RS_THREADS + threadIdx.x;
        if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    counts[(size_t)blockIdx.x * 256 + threadIdx.x] = h[threadIdx.x];
}
template <typename K, int ITEMS>
__global__ __launch_bounds__(RGX_RS_THREADS) void k_rs_pass(const K *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                            K *__restrict__ kout, uint32_t *__restrict__ vout, int64_t n, int shift,
                                                            const uint32_t *__restrict__ counts, int tiles, int64_t *__restrict__ order)
{
    __shared__ uint32_t cnt[4][256];
    __shared__ uint32_t wave_total[4];
    for (int w = 0; w < 4; ++w) cnt[w][threadIdx.x] = 0;
    uint32_t before = 0, total = 0;
#pragma unroll 16
    for (int t = 0; t < tiles; ++t) {
        const uint32_t c = counts[(size_t)t * 256 + threadIdx.x];
        total += c;
        before += t < (int)blockIdx.x ? c : 0u;
    }
    const uint32_t digit_base = rs_sum_before(total, wave_total);
    rs_scatter_tile<K, ITEMS>(kin, vin, n, shift, digit_base, before, cnt, wave_total, [&](uint32_t at, K k, uint32_t v) {
        if (order) {
            order[at] = (int64_t)v;
        } else {
            kout[at] = k;
            vout[at] = v;
        }
    });
}

// A sort of few keys: all passes in one workgroup, the keys in registers and their new order in LDS.  What the passes
// above take for them is the latency of their launches, 24 for 64-bit keys (building the tree over 4 096 boxes
// 181 us, with this 98; over 8 192 185 and 125; with a bitonic network, which moves every key through LDS 78 and 91 times
// instead of 8, 117 and 177).  Each wavefront has a run
// of the keys, and ranks 64 at a time as k_rs_scatter does; it ranks as it counts, one lane of each digit adding for all of them (an add per key
// to the counters first: a build of 4 096 boxes 110 -> 107 us, of 8 192 140 -> 135).  The limit is what fits LDS (12 bytes a key, and 16 KB of counters).
template <typename K>
__global__ __launch_bounds__(1024) void k_sort_small(K *__restrict__ keys, uint32_t *__restrict__ vals, int n, int bits)
{
    constexpr int WAVES = 16, ITEMS = RGX_SORT_SMALL / 1024;
    __shared__ K lkey[RGX_SORT_SMALL];
    __shared__ uint32_t lval[RGX_SORT_SMALL];
    __shared__ uint32_t cnt[WAVES][256];
    __shared__ uint32_t wave_total[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rounds = (n + 1023) / 1024, base = wave * rounds * 64; // wave w has the keys [base, base + 64 rounds)
    K key[ITEMS];
    uint32_t val[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int i = base + r * 64 + lane;
        const bool valid = r < rounds && i < n;
        key[r] = valid ? keys[i] : (K)0;
        val[r] = valid ? vals[i] : 0u;
    }
    for (int shift = 0; shift < bits; shift += 8) {
        for (int d = lane; d < 256; d += 64) cnt[wave][d] = 0;
        __builtin_amdgcn_wave_barrier();
        // a key's place in its wavefront's run of its digit: keys of the digit in earlier rounds, then in lower lanes
        uint32_t place[ITEMS];
        auto *cur = (__attribute__((address_space(3))) uint32_t *)cnt[wave];
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            if (r >= rounds) break;
            const bool valid = base + r * 64 + lane < n;
            const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
            uint64_t same = __ballot(valid);
            for (int b = 0; b < 8; ++b) {
                const bool bit = (d >> b) & 1u;
                const uint64_t bal = __ballot(bit);
                same &= bit ? bal : ~bal;
            }
            const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull));
            const uint32_t before = __hip_atomic_load(cur + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            place[r] = before + rank;
            __builtin_amdgcn_wave_barrier();
            if (valid && rank == 0) __hip_atomic_store(cur + d, before + (uint32_t)__popcll(same), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // where each (digit, wave) run starts: digits before waves
        uint32_t total = 0, upto = 0;
        if (threadIdx.x < 256) {
            for (int w = 0; w < WAVES; ++w) total += cnt[w][threadIdx.x];
            upto = total;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t t = __shfl_up(upto, o);
                if (lane >= o) upto += t;
            }
            if (lane == 63) wave_total[wave] = upto;
        }
        __syncthreads();
        if (threadIdx.x < 256) {
            uint32_t at = upto - total;
            for (int w = 0; w < wave; ++w) at += wave_total[w];
            for (int w = 0; w < WAVES; ++w) {
                const uint32_t c = cnt[w][threadIdx.x];
                cnt[w][threadIdx.x] = at;
                at += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r)
            if (r < rounds && base + r * 64 + lane < n) {
                const uint32_t at = cnt[wave][(uint32_t)(key[r] >> shift) & 255u] + place[r];
                lkey[at] = key[r];
                lval[at] = val[r];
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const int i = base + r * 64 + lane;
            if (r < rounds && i < n) {
                key[r] = lkey[i];
                val[r] = lval[i];
            }
        }
        // (the next pass writes lkey and lval after two more barriers)
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int i = base + r * 64 + lane;
        if (r < rounds && i < n) {
            keys[i] = key[r];
            vals[i] = val[r];
        }
    }
}

// the values of a sort in one workgroup, as 64-bit numbers
__global__ __launch_bounds__(256) void k_order64(const uint32_t *__restrict__ v, int64_t n, int64_t *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (int64_t)v[i];
}

// Sorts (k0, v0) by key, stable, with (k1, v1) as the second buffers.  hist: rs_hist_words(n).  order: where the values go in the end, or null.
template <typename K>
static int radix_sort(K *k0, uint32_t *v0, K *k1, uint32_t *v1, int64_t n, int bits, uint32_t *hist, hipStream_t s, int64_t *order = nullptr)
{
    if (n <= RGX_SORT_SMALL) {
        hipLaunchKernelGGL(k_sort_small<K>, dim3(1), dim3(1024), 0, s, k0, v0, (int)n, bits);
        if (order) hipLaunchKernelGGL(k_order64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, v0, n, order);
        RGX_LAUNCH_CHECK();
        return 0;
    }
    const RsShort F = rs_short(n);
    const int nblocks = (int)((n + RGX_RS_TILE - 1) / RGX_RS_TILE);
    K *ki = k0, *ko = k1;
    uint32_t *vi = v0, *vo = v1;
    for (int shift = 0; shift < bits; shift += 8) {
        int64_t *const last = shift + 8 >= bits ? order : nullptr;
        if (F.tiles) {
            const auto pass = [&](auto items) {
                constexpr int ITEMS = decltype(items)::value;
                hipLaunchKernelGGL((k_rs_count<K, ITEMS>), dim3(F.tiles), dim3(RGX_RS_THREADS), 0, s, ki, n, shift, hist);
                hipLaunchKernelGGL((k_rs_pass<K, ITEMS>), dim3(F.tiles), dim3(RGX_RS_THREADS), 0, s, ki, vi, ko, vo, n, shift, hist, F.tiles, last);
            };
            if (F.tile_bits == 9) pass(std::integral_constant<int, 2>{});
            else pass(std::integral_constant<int, 4>{});
        } else {
            hipLaunchKernelGGL(k_rs_hist<K>, dim3(nblocks), dim3(RGX_RS_THREADS), 0, s, ki, n, shift, hist, nblocks);
            uint32_t *totals = hist + (size_t)256 * nblocks;
            hipLaunchKernelGGL(k_rs_scan_rows, dim3(256), dim3(256), 0, s, hist, nblocks, totals);
            hipLaunchKernelGGL(k_rs_scatter<K>, dim3(nblocks), dim3(RGX_RS_THREADS), 0, s, ki, vi, ko, vo, n, shift, hist, nblocks,
                               totals, last);
        }
        K *tk = ki; ki = ko; ko = tk;
        uint32_t *tv = vi; vi = vo; vo = tv;
    }
    RGX_LAUNCH_CHECK();
    return ((bits + 7) / 8) & 1; // 1 when the result ended in (k1, v1)
}

// ---------------------------------------------------------------------------
// Radix tree (Karras 2012), then leaves and boxes in one kernel (leaves of a kernel of their own, read back by this one: a build of 1 M boxes 419 -> 404 us,
// 3 M 935 -> 919, 4 096 113 -> 110).
// Skip links: the node after a subtree is the right child of the one node whose children meet behind the subtree's last leaf;
// after[j] is that child, for j = the last leaf but the tree's (k_karras knows it: every gap between two leaves is
// one node's).  (A kernel of its own that climbed from every node to the first ancestor it was left of took 38 us at 1 M boxes and
// 100 at 3 M.)
__device__ __forceinline__ int32_t skip_link(const int32_t *after, int64_t n, int64_t last_leaf) { return last_leaf < n - 1 ? after[last_leaf] : -1; }

__device__ __forceinline__ int delta(const uint64_t *keys, int64_t n, int64_t i, int64_t j)
{
    if (j < 0 || j >= n) return -1;
    const uint64_t a = keys[i], b = keys[j];
    if (a != b) return __clzll((long long)(a ^ b));
    return 64 + __clz((int)((uint32_t)i ^ (uint32_t)j));
}

// other_end[i]: internal node i covers the sorted leaves between i and other_end[i]
__global__ __launch_bounds__(256) void k_karras(const uint64_t *__restrict__ keys, int64_t n, Node *__restrict__ nodes,
                                                int32_t *__restrict__ parent, int32_t *__restrict__ right,
                                                int32_t *__restrict__ other_end, int32_t *__restrict__ after, int32_t *__restrict__ flags)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1) >= 0 ? 1 : -1;
    const int dmin = delta(keys, n, i, i - d);
    int64_t lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int64_t l = 0;
    for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int64_t j = i + l * d;
    const int dnode = delta(keys, n, i, j);
    int64_t s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
    const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    const int32_t lc = (int32_t)(lo == gamma ? n - 1 + gamma : gamma);
    const int32_t rc = (int32_t)(hi == gamma + 1 ? n - 1 + gamma + 1 : gamma + 1);
    nodes[i].left = lc;
    right[i] = rc;
    after[gamma] = rc;
    parent[lc] = (int32_t)i;
    parent[rc] = (int32_t)i;
    other_end[i] = (int32_t)j;
    flags[i] = 0;
    if (i == 0) parent[0] = -1;
}

// Bottom-up refit: every leaf walks towards the root; the second thread to reach a node
// (counted with an atomic) merges the two child boxes and goes on.  A workgroup owns 512
// consecutive leaves of the sorted order; the nodes whose leaves all lie among them (internal node
// i covers the leaves between i and other_end[i], so its index is one of them) are met in LDS:
// counters, the box of whichever child arrived first, and the links of the 512 nodes, read there at the start: a level
// is then no chain of loads from memory (a build of 4 096 boxes 96.5 -> 92.6 us, 150 k 194 -> 190, 1 M 377 -> 355, 3 M 878 -> 812;
// with 256 leaves 92.4, 190, 359, 820; 1 024: 97.5, 185, 353, 809; 128: 92.5, 193, 376, 869).  Only the few subtree roots a workgroup
// ends up with go on through memory, where box words travel between threads through agent-scope
// atomic stores and loads (write-through to, and read from, the memory all XCDs share).  The thread
// that arrives second at a node may run in another workgroup on another XCD, so the first arriver's
// box stores -- also those it made in the LDS phase -- must have completed before its count becomes
// visible: it waits for them (s_waitcnt vmcnt(0)) before the counter's atomic.  That is the part of
// an agent-scope release these stores need; the full fence also writes the whole L2 back, which
// nothing here depends on (no plain store of this kernel is read by another workgroup) and which made
// the build 2.6 times slower (0.64 -> 1.69 ms at 1 M Gaussians).  The second arriver's loads are
// issued after its atomic has returned (its branch depends on the result).
__device__ __forceinline__ void st_agent(float *p, float v)
{
    __hip_atomic_store((int *)p, __float_as_int(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_agent(const float *p)
{
    return __int_as_float(__hip_atomic_load((const int *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Node `node` for the sweeps by pairs (NodePair): the thread that merges its children's boxes has both.  own: the child it came from.
__device__ __forceinline__ void store_pair(NodePair *pairs, int64_t n, int32_t node, int32_t left, int32_t right, int own,
                                           const float (&lo)[3], const float (&hi)[3], const float (&slo)[3], const float (&shi)[3])
{
    float4 *dst = (float4 *)(pairs + node);
    auto id = [&](int32_t child) { return __int_as_float(child >= n - 1 ? ~(int32_t)(child - (n - 1)) : child); };
    auto extent = [](float a, float b) { return fmaf(fabsf(a) + fabsf(b), 0x1p-22f, (b - a) * (1.0f + 0x1p-19f)); };
    dst[2 * own] = make_float4(lo[0] + hi[0], lo[1] + hi[1], lo[2] + hi[2], own ? 0.f : id(left));
    dst[2 * own + 1] = make_float4(extent(lo[0], hi[0]), extent(lo[1], hi[1]), extent(lo[2], hi[2]), own ? 0.f : id(right));
    dst[2 - 2 * own] = make_float4(slo[0] + shi[0], slo[1] + shi[1], slo[2] + shi[2], own ? id(left) : 0.f);
    dst[3 - 2 * own] = make_float4(extent(slo[0], shi[0]), extent(slo[1], shi[1]), extent(slo[2], shi[2]), own ? id(right) : 0.f);
}

#define RGX_REFIT_LEAVES 512
#define RGX_REFIT_OUTSIDE 0x10000u
#define RGX_REFIT_ARRIVED 0x20000u
__global__ __launch_bounds__(RGX_REFIT_LEAVES) void k_refit(const float *__restrict__ boxes, const uint32_t *__restrict__ order, int64_t n, Node *nodes,
                                               uint32_t *__restrict__ place, const int32_t *__restrict__ parent, const int32_t *__restrict__ right,
                                               const int32_t *__restrict__ other_end, const int32_t *__restrict__ after, int32_t *flags, NodePair *__restrict__ pairs,
                                               WsHeader *h, const int32_t *gate = nullptr)
{
    __shared__ float s_box[2][6][RGX_REFIT_LEAVES]; // [which child][lo xyz, hi xyz][node - first leaf of the workgroup]
    __shared__ int32_t s_up[RGX_REFIT_LEAVES], s_left[RGX_REFIT_LEAVES], s_after[RGX_REFIT_LEAVES]; // parent, nodes[].left, after of the same nodes
    __shared__ uint32_t s_end[RGX_REFIT_LEAVES]; // other_end - first leaf, or RGX_REFIT_OUTSIDE; RGX_REFIT_ARRIVED: a child has arrived
    if (gate_closed(gate)) return; // the whole grid
    const int64_t b0 = (int64_t)blockIdx.x * RGX_REFIT_LEAVES, j = b0 + threadIdx.x;
    if (j < n - 1) {
        s_up[threadIdx.x] = parent[j];
        s_left[threadIdx.x] = nodes[j].left;
        const int64_t end = other_end[j] - b0;
        s_end[threadIdx.x] = end >= 0 && end < RGX_REFIT_LEAVES ? (uint32_t)end : RGX_REFIT_OUTSIDE;
        s_after[threadIdx.x] = after[j];
    } else {
        s_after[threadIdx.x] = -1; // (skip_link)
    }
    __syncthreads();
    if (j >= n) return;
    const int64_t b1 = b0 + RGX_REFIT_LEAVES - 1 < n - 1 ? b0 + RGX_REFIT_LEAVES - 1 : n - 1;
    // node's leaves all among the workgroup's: then it has the index of one of them
    auto met_here = [&](int32_t node) {
        return node >= b0 && node <= b1 && !(s_end[node - b0] & RGX_REFIT_OUTSIDE);
    };
    int32_t child = (int32_t)(n - 1 + j);
    // its leaf
    const int64_t in = order[j];
    place[in] = (uint32_t)j; // the inverse permutation, for the kernels that go through the Gaussians in input order
    float lo[3], hi[3];
    for (int c = 0; c < 3; ++c) {
        lo[c] = boxes[6 * in + c];
        hi[c] = boxes[6 * in + 3 + c];
    }
    int32_t node = n > 1 ? parent[child] : -1;
    {
        const int32_t left = ~(int32_t)j, skip = s_after[threadIdx.x];
        if (node < 0 || met_here(node)) {
            float4 *dst = (float4 *)&nodes[child];
            dst[0] = make_float4(lo[0], lo[1], lo[2], __int_as_float(left));
            dst[1] = make_float4(hi[0], hi[1], hi[2], __int_as_float(skip));
        } else { // its parent is met through memory: see below
            for (int c = 0; c < 3; ++c) {
                st_agent(&nodes[child].lo[c], lo[c]);
                st_agent(&nodes[child].hi[c], hi[c]);
            }
            nodes[child].left = left;
            nodes[child].skip = skip;
        }
    }
    // nodes inside the workgroup's leaves: through LDS
    while (node >= 0) {
        if (!met_here(node)) break;
        const int slot = (int)(node - b0);
        const int32_t left = s_left[slot], side = left == child ? 0 : 1;
        for (int c = 0; c < 3; ++c) {
            s_box[side][c][slot] = lo[c];
            s_box[side][3 + c][slot] = hi[c];
        }
        __threadfence_block();
        const uint32_t end = atomicOr(&s_end[slot], RGX_REFIT_ARRIVED);
        if (!(end & RGX_REFIT_ARRIVED)) return; // the sibling subtree is not done yet
        const int last = max(slot, (int)(end & ~RGX_REFIT_ARRIVED));
        __threadfence_block();
        float slo[3], shi[3];
        for (int c = 0; c < 3; ++c) {
            slo[c] = s_box[1 - side][c][slot];
            shi[c] = s_box[1 - side][3 + c][slot];
        }
        // (the children of a node meet between two neighbours of the sorted order: the right one starts where the left one ends)
        const int32_t split = left >= n - 1 ? left - (int32_t)(n - 1) : left;
        if (pairs) store_pair(pairs, n, node, left, b0 + last == split + 1 ? (int32_t)(n - 1) + split + 1 : split + 1, side, lo, hi, slo, shi);
        for (int c = 0; c < 3; ++c) {
            lo[c] = fminf(lo[c], slo[c]);
            hi[c] = fmaxf(hi[c], shi[c]);
        }
        child = node;
        node = s_up[slot];
        // This box is read again inside this kernel only if the parent is met through memory (then by whichever
        // thread arrives there second, maybe on another XCD): only then does it have to go out as agent-scope
        // stores.  Everything below such a subtree root is next read by other kernels: plain stores.
        const int32_t skip = s_after[last];
        if (node >= 0 && met_here(node)) {
            float4 *dst = (float4 *)&nodes[child];
            dst[0] = make_float4(lo[0], lo[1], lo[2], __int_as_float(left));
            dst[1] = make_float4(hi[0], hi[1], hi[2], __int_as_float(skip));
        } else {
            for (int c = 0; c < 3; ++c) {
                st_agent(&nodes[child].lo[c], lo[c]);
                st_agent(&nodes[child].hi[c], hi[c]);
            }
            nodes[child].skip = skip;
            break;
        }
    }
    // the rest of the way: through memory.  The thread carries its child's box in registers and reads only the
    // sibling's; the indices it will need after the counter (children, next parent) are asked for before the wait,
    // so that each level is three trips to memory one after the other (stores acknowledged, counter, sibling's box)
    // and not five.
    while (node >= 0) {
        const int32_t left = nodes[node].left, rgt = right[node], up = parent[node], end = other_end[node];
        const int32_t skip = skip_link(after, n, node < end ? end : node);
#if defined(__gfx942__) || defined(__gfx950__)
        // (the immediate below is the gfx9 encoding of vmcnt(0) with the other counters left alone, and the
        // argument that the wait suffices rests on how these chips complete agent-scope atomic stores)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup"); // compiler ordering
        __builtin_amdgcn_s_waitcnt(0x0F70);                    // vmcnt(0): this thread's box stores have completed
        if (atomicAdd(&flags[node], 1) == 0) return; // the sibling subtree is not done yet
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
#else
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        if (atomicAdd(&flags[node], 1) == 0) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#endif
        const Node *sibling = &nodes[left == child ? rgt : left];
        float slo[3], shi[3];
        for (int c = 0; c < 3; ++c) {
            slo[c] = ld_agent(&sibling->lo[c]);
            shi[c] = ld_agent(&sibling->hi[c]);
        }
        if (pairs) store_pair(pairs, n, node, left, rgt, left == child ? 0 : 1, lo, hi, slo, shi);
        for (int c = 0; c < 3; ++c) {
            lo[c] = fminf(lo[c], slo[c]);
            hi[c] = fmaxf(hi[c], shi[c]);
            st_agent(&nodes[node].lo[c], lo[c]);
            st_agent(&nodes[node].hi[c], hi[c]);
        }
        nodes[node].skip = skip;
        child = node;
        node = up;
    }
    h->built = 1; // (the thread that has merged the root)
}

__global__ void k_mark_built(WsHeader *h, const int32_t *gate = nullptr) // of an empty scene
{
    if (!gate_closed(gate)) h->built = 1;
}

// ---------------------------------------------------------------------------
static inline dim3 grid_for(int64_t n, int block) { return dim3((unsigned)((n + block - 1) / block)); }
// For the kernels that loop over their input and end with atomics on a few shared words.
static inline dim3 grid_reduce(int64_t n, int most) { return dim3((unsigned)std::min<int64_t>((n + RGX_REDUCE_THREADS - 1) / RGX_REDUCE_THREADS, most)); }

extern "C" int rgx_aabb(const float *pos, const float *scale, const float *quat, const float *dens, int64_t n,
                        float sigma_threshold, float *bboxes, float *bb_min, float *bb_max, void *stream)
{
    const DeviceScope on_device(pos);
    if (n < 0 || (n > 0 && (!pos || !scale || !quat || !dens)) || ((bb_min == nullptr) != (bb_max == nullptr)))
        return RGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    int32_t *mn = (int32_t *)bb_min, *mx = (int32_t *)bb_max;
    if (mn) hipLaunchKernelGGL(k_init_enc, dim3(1), dim3(64), 0, s, mn, mx);
    if (n > 0)
        hipLaunchKernelGGL(k_aabb, grid_reduce(n, 256), dim3(RGX_REDUCE_THREADS), 0, s, pos, scale, quat, dens, n, sigma_threshold, bboxes, mn, mx);
    if (mn) hipLaunchKernelGGL(k_decode_enc, dim3(1), dim3(64), 0, s, mn, mx);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

extern "C" int rgx_build_workspace_bytes(int64_t n, size_t *bytes)
{
    if (n < 0 || !bytes || n > 0x3fffffff) return RGX_EINVAL;
    *bytes = rgx_ws_layout(n).total;
    return RGX_OK;
}

// Copies caller-supplied boxes into the workspace and reduces the scene bbox.
__global__ __launch_bounds__(RGX_REDUCE_THREADS) void k_take_boxes(const float *__restrict__ in, int64_t n, float *__restrict__ boxes, int32_t *__restrict__ flags,
                                                    int32_t *mn_enc, int32_t *mx_enc, const int32_t *gate = nullptr)
{
    if (gate_closed(gate)) return; // the whole grid
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        for (int a = 0; a < 6; ++a) {
            const float v = boxes[6 * i + a] = in[6 * i + a];
            b[a] = a < 3 ? fminf(b[a], v) : fmaxf(b[a], v);
        }
        if (flags) flags[i] = 0; // (k_refit)
    }
    __shared__ float red[RGX_REDUCE_THREADS / 64][6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int a = 0; a < 3; ++a) {
        const float mn = wave_min_all(b[a]), mx = wave_max_all(b[a + 3]);
        if (lane == 0) { red[wave][a] = mn; red[wave][a + 3] = mx; }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        float mn, mx;
        fold_bounds(red, a, mn, mx);
        atomicMin(&mn_enc[a], enc_f(mn));
        atomicMax(&mx_enc[a], enc_f(mx));
    }
}

static int build_impl(const float *pos, const float *scale, const float *quat, const float *dens, const float *in_boxes,
                      int64_t n, float sigma_threshold, void *ws, size_t ws_bytes, void *stream);

extern "C" int rgx_build(const float *pos, const float *scale, const float *quat, const float *dens, int64_t n,
                         float sigma_threshold, void *ws, size_t ws_bytes, void *stream)
{
    if (n > 0 && (!pos || !scale || !quat || !dens)) return RGX_EINVAL;
    return build_impl(pos, scale, quat, dens, nullptr, n, sigma_threshold, ws, ws_bytes, stream);
}

extern "C" int rgx_build_aabbs(const float *bboxes, int64_t n, void *ws, size_t ws_bytes, void *stream)
{
    if (n > 0 && !bboxes) return RGX_EINVAL;
    return build_impl(nullptr, nullptr, nullptr, nullptr, bboxes, n, 0.f, ws, ws_bytes, stream);
}

static int build_impl(const float *pos, const float *scale, const float *quat, const float *dens, const float *in_boxes,
                      int64_t n, float sigma_threshold, void *ws, size_t ws_bytes, void *stream)
{
    const DeviceScope on_device(ws);
    if (n < 0 || n > 0x3fffffff || !ws) return RGX_EINVAL;
    const WsLayout L = rgx_ws_layout(n);
    if (ws_bytes < L.total || ((uintptr_t)ws & 255u)) return RGX_EWORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    char *w = (char *)ws;
    WsHeader *hdr = (WsHeader *)(w + L.header);
    float *boxes = (float *)(w + L.aabb);
    uint64_t *k0 = (uint64_t *)(w + L.keys0), *k1 = (uint64_t *)(w + L.keys1);
    uint32_t *v0 = (uint32_t *)(w + L.vals0), *v1 = (uint32_t *)(w + L.vals1);
    Node *nodes = (Node *)(w + L.nodes);
    int32_t *parent = (int32_t *)(w + L.parent), *right = (int32_t *)(w + L.right), *flags = (int32_t *)(w + L.flags);
    uint32_t *hist = (uint32_t *)(w + L.hist);

    void *span = rgx_span_begin(RGX_T_BUILD, s);
    hipLaunchKernelGGL(k_init_header, dim3(1), dim3(64), 0, s, hdr, n);
    if (n > 0) {
        if (in_boxes)
            hipLaunchKernelGGL(k_take_boxes, grid_reduce(n, 256), dim3(RGX_REDUCE_THREADS), 0, s, in_boxes, n, boxes, (int32_t *)nullptr, hdr->bb_min_enc,
                               hdr->bb_max_enc);
        else
            hipLaunchKernelGGL(k_aabb, grid_reduce(n, 256), dim3(RGX_REDUCE_THREADS), 0, s, pos, scale, quat, dens, n, sigma_threshold, boxes,
                               hdr->bb_min_enc, hdr->bb_max_enc);
        hipLaunchKernelGGL(k_morton63, grid_for(n, 256), dim3(256), 0, s, boxes, n, hdr, k0, v0);
        RGX_LAUNCH_CHECK();
        const int r = radix_sort<uint64_t>(k0, v0, k1, v1, n, 64, hist, s);
        if (r < 0) return r;
        // 8 passes: the sorted keys / permutation are back in (k0, v0)
        int32_t *other_end = (int32_t *)k1, *after = other_end + n; // the sort's second key buffer is free again
        if (n > 1) hipLaunchKernelGGL(k_karras, grid_for(n - 1, 256), dim3(256), 0, s, k0, n, nodes, parent, right, other_end, after, flags);
        hipLaunchKernelGGL(k_refit, grid_for(n, RGX_REFIT_LEAVES), dim3(RGX_REFIT_LEAVES), 0, s, boxes, v0, n, nodes, v1, parent, right, other_end, after, flags,
                           n <= RGX_PAIR_BOXES ? (NodePair *)(w + L.pairs) : nullptr, hdr); // (v1: the sort's second value buffer is free again)
    } else {
        hipLaunchKernelGGL(k_mark_built, dim3(1), dim3(1), 0, s, hdr);
    }
    rgx_span_end(span, s);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

// Refit: the tree's shape (children, parents, sorted order) stays as the last build into `ws` left it;
// leaf boxes are taken from `bboxes`, internal boxes and the scene box recomputed bottom-up.
// Precondition, checked on the device by the refit's first kernel: `ws` holds a finished tree over exactly
// `n` boxes.  If it does not, no kernel of the refit touches the tree, the workspace is left marked not
// built (rgx_scene_bbox then reports RGX_EWORKSPACE) and the call still returns RGX_OK: the check runs in
// stream order and the host does not wait for it.
extern "C" int rgx_refit_aabbs(const float *bboxes, int64_t n, void *ws, size_t ws_bytes, void *stream)
{
    if (n < 0 || n > 0x3fffffff || !ws || (n > 0 && !bboxes)) return RGX_EINVAL;
    const DeviceScope on_device(ws);
    const WsLayout L = rgx_ws_layout(n);
    if (ws_bytes < L.total || ((uintptr_t)ws & 255u)) return RGX_EWORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    char *w = (char *)ws;
    WsHeader *hdr = (WsHeader *)(w + L.header);
    float *boxes = (float *)(w + L.aabb);
    const uint32_t *order = (const uint32_t *)(w + L.vals0);
    Node *nodes = (Node *)(w + L.nodes);
    int32_t *parent = (int32_t *)(w + L.parent), *right = (int32_t *)(w + L.right), *flags = (int32_t *)(w + L.flags);
    const int32_t *other_end = (const int32_t *)(w + L.keys1); // left there by the build
    void *span = rgx_span_begin(RGX_T_BUILD, s);
    const int32_t *gate = &hdr->refit_ok;
    hipLaunchKernelGGL(k_refit_begin, dim3(1), dim3(64), 0, s, hdr, n);
    if (n > 0) {
        hipLaunchKernelGGL(k_take_boxes, grid_reduce(n, 256), dim3(RGX_REDUCE_THREADS), 0, s, bboxes, n, boxes, flags, hdr->bb_min_enc, hdr->bb_max_enc, gate);
        hipLaunchKernelGGL(k_finish_bbox, dim3(1), dim3(64), 0, s, hdr, (float *)nullptr, (float *)nullptr, gate);
        const int32_t *after = other_end + n;
        hipLaunchKernelGGL(k_refit, grid_for(n, RGX_REFIT_LEAVES), dim3(RGX_REFIT_LEAVES), 0, s, boxes, order, n, nodes, (uint32_t *)(w + L.vals1), parent, right, other_end,
                           after, flags, n <= RGX_PAIR_BOXES ? (NodePair *)(w + L.pairs) : nullptr, hdr, gate);
    } else {
        hipLaunchKernelGGL(k_mark_built, dim3(1), dim3(1), 0, s, hdr, gate);
    }
    rgx_span_end(span, s);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

extern "C" int rgx_build_layout(int64_t n, size_t *host_out6)
{
    if (n < 0 || n > 0x3fffffff || !host_out6) return RGX_EINVAL;
    const WsLayout L = rgx_ws_layout(n);
    host_out6[0] = L.aabb;
    host_out6[1] = L.vals0;
    host_out6[2] = L.nodes;
    host_out6[3] = L.parent;
    host_out6[4] = L.right;
    host_out6[5] = L.header;
    return RGX_OK;
}

// ---------------------------------------------------------------------------
// Synchronous / small read-backs of a built workspace.
extern "C" int rgx_scene_bbox(const void *ws, float *host_out6, void *stream)
{
    const DeviceScope on_device(ws);
    if (!ws || !host_out6) return RGX_EINVAL;
    WsHeader h;
    RGX_HIP(hipMemcpyAsync(&h, ws, sizeof h, hipMemcpyDeviceToHost, (hipStream_t)stream));
    RGX_HIP(hipStreamSynchronize((hipStream_t)stream));
    if (h.built != 1) return RGX_EWORKSPACE; // never built, or a refit that found no tree of its size to refit
    for (int a = 0; a < 3; ++a) {
        host_out6[a] = h.bb_min[a];
        host_out6[3 + a] = h.bb_max[a];
    }
    return RGX_OK;
}

__global__ __launch_bounds__(256) void k_copy_order(const uint32_t *__restrict__ v, int64_t n, int32_t *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (int32_t)v[i];
}

extern "C" int rgx_build_order(const void *ws, int64_t n, int32_t *order_out, void *stream)
{
    const DeviceScope on_device(ws);
    if (!ws || n < 0 || (n > 0 && !order_out)) return RGX_EINVAL;
    if (n == 0) return RGX_OK;
    const WsLayout L = rgx_ws_layout(n);
    hipLaunchKernelGGL(k_copy_order, grid_for(n, 256), dim3(256), 0, (hipStream_t)stream,
                       (const uint32_t *)((const char *)ws + L.vals0), n, order_out);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

// ---------------------------------------------------------------------------
// 30-bit Morton ordering of the point cloud (utils/reordering_utils.py:55-104,
// classes/point_cloud.py:1017-1024).
__global__ __launch_bounds__(RGX_REDUCE_THREADS) void k_pos_minmax(const float *__restrict__ pos, int64_t n, int32_t *mn_enc, int32_t *mx_enc)
{
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += 4 * step) {
        float v[4][3];
#pragma unroll
        for (int k = 0; k < 4; ++k) { // (four points in flight; past the end: the first again)
            const int64_t j = i + k * step < n ? i + k * step : i;
            for (int a = 0; a < 3; ++a) v[k][a] = pos[3 * j + a];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            for (int a = 0; a < 3; ++a) {
                b[a] = fminf(b[a], v[k][a]);
                b[a + 3] = fmaxf(b[a + 3], v[k][a]);
            }
    }
    __shared__ float red[RGX_REDUCE_THREADS / 64][6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int a = 0; a < 3; ++a) {
        const float mn = wave_min_all(b[a]), mx = wave_max_all(b[a + 3]);
        if (lane == 0) { red[wave][a] = mn; red[wave][a + 3] = mx; }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        float mn, mx;
        fold_bounds(red, a, mn, mx);
        atomicMin(&mn_enc[a], enc_f(mn));
        atomicMax(&mx_enc[a], enc_f(mx));
    }
}

__global__ __launch_bounds__(256) void k_morton30(const float *__restrict__ pos, int64_t n, const int32_t *__restrict__ mn_enc,
                                                  const int32_t *__restrict__ mx_enc, uint32_t *__restrict__ keys,
                                                  uint32_t *__restrict__ vals, int64_t *__restrict__ codes)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t code = 0;
    for (int a = 0; a < 3; ++a) {
        const float mn = dec_f(mn_enc[a]), mx = dec_f(mx_enc[a]);
        const float scale = 1023.0f / ((mx - mn) + 1e-9f); // reordering_utils.py:73
        const int32_t q = (int32_t)((pos[3 * i + a] - mn) * scale); // .to(torch.int32): truncation
        for (int b = 0; b < 10; ++b) code |= (uint32_t)((q >> b) & 1) << (3 * b + a); // reordering_utils.py:98-102
    }
    keys[i] = code;
    vals[i] = (uint32_t)i;
    if (codes) codes[i] = (int64_t)code;
}

struct MortonLayout {
    size_t enc, keys0, keys1, vals0, vals1, hist, total;
};
static inline MortonLayout morton_layout(int64_t n)
{
    MortonLayout L;
    const size_t nn = (size_t)(n > 0 ? n : 1);
    size_t off = 0;
    L.enc = off;   off = rgx_align_up(off + 8 * sizeof(int32_t), 256);
    L.keys0 = off; off = rgx_align_up(off + nn * 4, 256);
    L.keys1 = off; off = rgx_align_up(off + nn * 4, 256);
    L.vals0 = off; off = rgx_align_up(off + nn * 4, 256);
    L.vals1 = off; off = rgx_align_up(off + nn * 4, 256);
    L.hist = off;  off = rgx_align_up(off + rs_hist_words((int64_t)nn) * 4, 256);
    L.total = off;
    return L;
}

extern "C" int rgx_morton_workspace_bytes(int64_t n, size_t *bytes)
{
    if (n < 0 || !bytes || n > 0x3fffffff) return RGX_EINVAL;
    *bytes = morton_layout(n).total;
    return RGX_OK;
}

extern "C" int rgx_morton_order(const float *pos, int64_t n, int64_t *codes, int64_t *order, void *ws, size_t ws_bytes,
                                void *stream)
{
    const DeviceScope on_device(pos);
    if (n < 0 || n > 0x3fffffff || !ws || (n > 0 && !pos)) return RGX_EINVAL;
    const MortonLayout L = morton_layout(n);
    if (ws_bytes < L.total || ((uintptr_t)ws & 255u)) return RGX_EWORKSPACE;
    if (n == 0) return RGX_OK;
    hipStream_t s = (hipStream_t)stream;
    char *w = (char *)ws;
    int32_t *mn = (int32_t *)(w + L.enc), *mx = mn + 4;
    uint32_t *k0 = (uint32_t *)(w + L.keys0), *k1 = (uint32_t *)(w + L.keys1);
    uint32_t *v0 = (uint32_t *)(w + L.vals0), *v1 = (uint32_t *)(w + L.vals1);
    hipLaunchKernelGGL(k_init_enc, dim3(1), dim3(64), 0, s, mn, mx);
    hipLaunchKernelGGL(k_pos_minmax, grid_reduce(n, 128), dim3(RGX_REDUCE_THREADS), 0, s, pos, n, mn, mx);
    hipLaunchKernelGGL(k_morton30, grid_for(n, 256), dim3(256), 0, s, pos, n, mn, mx, k0, v0, codes);
    RGX_LAUNCH_CHECK();
    if (order) {
        const int r = radix_sort<uint32_t>(k0, v0, k1, v1, n, 32, (uint32_t *)(w + L.hist), s, order);
        if (r < 0) return r;
    }
    return RGX_OK;
}

// ---------------------------------------------------------------------------
// Fused multi-tensor gather for the periodic reordering of the point cloud: every
// per-Gaussian tensor (parameters, Adam moments, statistics) is permuted with the same index
// (classes/point_cloud.py:1031-1044, classes/optimizer.py:54-66: one `tensor[index]` launch per
// tensor there).  A workgroup takes RGX_GATHER_ROWS consecutive output rows, fetches their source rows'
// numbers once and moves the rows of one tensor after the other, in the widest pieces that the rows'
// length and the tensors' alignment allow (16, 12, 8 or 4 bytes): writes are coalesced, the reads of a
// row are contiguous, and every thread has up to four reads in flight.  Bound by memory: one 32-bit word per
// thread, its row found by a 64-bit division and its number fetched per word, took 0.743 ms for the 15
// tensors of a 1 M cloud (1.42 GB); this takes 0.438 ms (3.2 TB/s), and short rows have a way of their own below.
#define RGX_GATHER_MAX 24
#define RGX_GATHER_ROWS 128
#define RGX_GATHER_LONG 4096 // a row of at least this many pieces is moved by the workgroup on its own
struct GatherArgs {
    const uint32_t *src[RGX_GATHER_MAX];
    uint32_t *dst[RGX_GATHER_MAX];
    int32_t pieces[RGX_GATHER_MAX];  // per row
    uint32_t magic[RGX_GATHER_MAX];  // floor(2^32 / pieces) + 1: p / pieces = umulhi(p, magic) for p * pieces < 2^32
    uint8_t words[RGX_GATHER_MAX];   // 32-bit words of a piece
    int32_t count;
};
template <int W>
struct Piece {
    uint32_t v[W];
};
template <int W>
__device__ __forceinline__ Piece<W> piece_load(const uint32_t *p)
{
    Piece<W> x;
    if constexpr (W == 4) {
        const uint4 u = *(const uint4 *)p;
        x.v[0] = u.x; x.v[1] = u.y; x.v[2] = u.z; x.v[3] = u.w;
    } else if constexpr (W == 2) {
        const uint2 u = *(const uint2 *)p;
        x.v[0] = u.x; x.v[1] = u.y;
    } else {
#pragma unroll
        for (int k = 0; k < W; ++k) x.v[k] = p[k];
    }
    return x;
}
template <int W>
__device__ __forceinline__ void piece_store(uint32_t *p, const Piece<W> &x)
{
    if constexpr (W == 4) *(uint4 *)p = make_uint4(x.v[0], x.v[1], x.v[2], x.v[3]);
    else if constexpr (W == 2) *(uint2 *)p = make_uint2(x.v[0], x.v[1]);
    else {
#pragma unroll
        for (int k = 0; k < W; ++k) p[k] = x.v[k];
    }
}

template <int W>
__device__ __forceinline__ void gather_tensor(const uint32_t *src, uint32_t *dst, int pieces, uint32_t magic, const int64_t *s_row,
                                              int64_t row0, int rows)
{
    uint32_t *out = dst + row0 * ((int64_t)pieces * W);
    if (pieces >= RGX_GATHER_LONG) {
        for (int r = 0; r < rows; ++r)
            for (int q = threadIdx.x; q < pieces; q += 256)
                piece_store<W>(out + ((int64_t)r * pieces + q) * W, piece_load<W>(src + (s_row[r] * pieces + q) * W));
        return;
    }
    const int total = rows * pieces; // < RGX_GATHER_ROWS * RGX_GATHER_LONG
    auto from = [&](int p) {
        const int r = pieces == 1 ? p : (int)__umulhi((uint32_t)p, magic);
        return src + (s_row[r] * pieces + (p - r * pieces)) * W;
    };
    int p = threadIdx.x;
    for (; p + 3 * 256 < total; p += 4 * 256) {
        Piece<W> x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = piece_load<W>(from(p + k * 256));
#pragma unroll
        for (int k = 0; k < 4; ++k) piece_store<W>(out + (int64_t)(p + k * 256) * W, x[k]);
    }
    for (; p < total; p += 256) piece_store<W>(out + (int64_t)p * W, piece_load<W>(from(p)));
}

__global__ __launch_bounds__(256) void k_gather_rows(const GatherArgs A, const int64_t *__restrict__ order, int64_t n)
{
    __shared__ int64_t s_row[RGX_GATHER_ROWS];
    const int64_t row0 = (int64_t)blockIdx.x * RGX_GATHER_ROWS;
    const int rows = (int)(n - row0 < RGX_GATHER_ROWS ? n - row0 : RGX_GATHER_ROWS);
    if ((int)threadIdx.x < rows) s_row[threadIdx.x] = order[row0 + threadIdx.x];
    __syncthreads();
    for (int t = blockIdx.y; t < A.count; t += gridDim.y) {
        switch (A.words[t]) {
        case 4: gather_tensor<4>(A.src[t], A.dst[t], A.pieces[t], A.magic[t], s_row, row0, rows); break;
        case 3: gather_tensor<3>(A.src[t], A.dst[t], A.pieces[t], A.magic[t], s_row, row0, rows); break;
        case 2: gather_tensor<2>(A.src[t], A.dst[t], A.pieces[t], A.magic[t], s_row, row0, rows); break;
        default: gather_tensor<1>(A.src[t], A.dst[t], A.pieces[t], A.magic[t], s_row, row0, rows); break;
        }
    }
}

// Short rows.  A row of a few words read wherever it lies costs the whole line it lies in: the twelve short tensors of a 1 M
// cloud (positions, scales, quaternions and densities with both Adam moments, 132 bytes a Gaussian) took 230 us of the
// reordering's 439, the three tensors of 192-byte rows 249.  So the short rows of a Gaussian are first put together in a record of up to 128
// bytes, read and written in order, and the records gathered: one line instead of one per tensor.  Both kernels go through a
// tile of 128 rows in LDS, so that every tensor's rows are read and written as one run of words: 1 M 439 -> 398 us for all tensors
// (72 to put them together, 67 to gather them, one tensor too many for the record's 32 words; 3.7 and 4.4 TB/s),
// 3 M 1 454 -> 1 192.
#define RGX_PACK_WORDS 32    // of a record
#define RGX_PACK_ROW 8       // words of the longest row that counts as short
#define RGX_PACK_STRIDE 36   // words from row to row in LDS
#define RGX_PACK_MIN 2       // tensors that make a record worth while
#define RGX_PACK_ROWS 262144 // rows from which on it is (300 k 129 -> 125 us, 400 k 174 -> 161; below, the caches hold the short tensors)
struct PackArgs {
    const uint32_t *src[RGX_PACK_WORDS];
    uint32_t *dst[RGX_PACK_WORDS];
    uint32_t magic[RGX_PACK_WORDS]; // as in GatherArgs, of the row's words
    uint8_t words[RGX_PACK_WORDS], at[RGX_PACK_WORDS]; // of the row; where it begins in the record
    uint8_t owner[RGX_PACK_WORDS]; // the tensor that a word of the record belongs to
    int32_t count, quads, total;   // tensors; 16-byte pieces and words of a record
    int32_t aligned;               // all tensors begin on a 16-byte boundary
};
// Goes through the words that the tensors have in a whole tile, in pieces of 16 bytes: a word of the record stands for
// RGX_GATHER_ROWS / 4 of them.  each(tensor, piece of the tensor's run of words, where its four words are in the tile)
template <typename Each>
__device__ __forceinline__ void pack_pieces(const PackArgs &A, Each each)
{
    constexpr int PER = RGX_GATHER_ROWS / 4;
    for (int p = threadIdx.x; p < A.total * PER; p += 256) {
        const int c = p / PER, t = A.owner[c];
        const uint32_t w = A.words[t], piece = (uint32_t)(c - A.at[t]) * PER + (uint32_t)p % PER;
        uint32_t r = w == 1 ? 4 * piece : __umulhi(4 * piece, A.magic[t]), k = 4 * piece - r * w;
        uint32_t at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            at[i] = r * RGX_PACK_STRIDE + A.at[t] + k;
            if (++k == w) {
                k = 0;
                ++r;
            }
        }
        each(t, piece, at);
    }
}
__global__ __launch_bounds__(256) void k_pack_rows(const PackArgs A, int64_t n, uint4 *__restrict__ rec)
{
    __shared__ __align__(16) uint32_t s_tile[RGX_GATHER_ROWS * RGX_PACK_STRIDE];
    const int64_t row0 = (int64_t)blockIdx.x * RGX_GATHER_ROWS;
    const int rows = (int)(n - row0 < RGX_GATHER_ROWS ? n - row0 : RGX_GATHER_ROWS);
    if (rows == RGX_GATHER_ROWS && A.aligned) {
        pack_pieces(A, [&](int t, uint32_t piece, const uint32_t (&at)[4]) {
            const uint4 v = ((const uint4 *)(A.src[t] + row0 * A.words[t]))[piece];
            s_tile[at[0]] = v.x; s_tile[at[1]] = v.y; s_tile[at[2]] = v.z; s_tile[at[3]] = v.w;
        });
    } else {
        for (int t = 0; t < A.count; ++t) {
            const uint32_t w = A.words[t];
            const uint32_t *src = A.src[t] + row0 * w;
            for (uint32_t p = threadIdx.x; p < rows * w; p += 256) {
                const uint32_t r = w == 1 ? p : __umulhi(p, A.magic[t]);
                s_tile[r * RGX_PACK_STRIDE + A.at[t] + (p - r * w)] = src[p];
            }
        }
    }
    __syncthreads();
    for (int p = threadIdx.x; p < rows * A.quads; p += 256) {
        const int r = p / A.quads, q = p - r * A.quads;
        rec[row0 * A.quads + p] = *(const uint4 *)(s_tile + r * RGX_PACK_STRIDE + 4 * q);
    }
}
__global__ __launch_bounds__(256) void k_unpack_rows(const PackArgs A, const int64_t *__restrict__ order, int64_t n, const uint4 *__restrict__ rec)
{
    __shared__ __align__(16) uint32_t s_tile[RGX_GATHER_ROWS * RGX_PACK_STRIDE];
    const int64_t row0 = (int64_t)blockIdx.x * RGX_GATHER_ROWS;
    const int rows = (int)(n - row0 < RGX_GATHER_ROWS ? n - row0 : RGX_GATHER_ROWS);
    for (int p = threadIdx.x; p < rows * A.quads; p += 256) {
        const int r = p / A.quads, q = p - r * A.quads;
        *(uint4 *)(s_tile + r * RGX_PACK_STRIDE + 4 * q) = rec[order[row0 + r] * A.quads + q];
    }
    __syncthreads();
    if (rows == RGX_GATHER_ROWS && A.aligned) {
        pack_pieces(A, [&](int t, uint32_t piece, const uint32_t (&at)[4]) {
            ((uint4 *)(A.dst[t] + row0 * A.words[t]))[piece] = make_uint4(s_tile[at[0]], s_tile[at[1]], s_tile[at[2]], s_tile[at[3]]);
        });
        return;
    }
    for (int t = 0; t < A.count; ++t) {
        const uint32_t w = A.words[t];
        uint32_t *dst = A.dst[t] + row0 * w;
        for (uint32_t p = threadIdx.x; p < rows * w; p += 256) {
            const uint32_t r = w == 1 ? p : __umulhi(p, A.magic[t]);
            dst[p] = s_tile[r * RGX_PACK_STRIDE + A.at[t] + (p - r * w)];
        }
    }
}

// Tensors are gone through RGX_GATHER_SET at a time, a bit each (no memory of the host's is asked for).
#define RGX_GATHER_SET 64
// The tensors of `todo` that share the next record (first fit, in order).
static uint64_t pack_group(const int64_t *row_bytes, uint64_t todo)
{
    uint64_t members = 0;
    int words = 0;
    for (; todo; todo &= todo - 1) {
        const int i = __builtin_ctzll(todo);
        const int64_t w = row_bytes[i] / 4;
        if (w > RGX_PACK_ROW || words + w > RGX_PACK_WORDS) continue;
        members |= 1ull << i;
        words += (int)w;
    }
    return members;
}

static int gather_check(int32_t count, const int64_t *row_bytes, int64_t n)
{
    if (count < 0 || n < 0 || (count > 0 && !row_bytes)) return RGX_EINVAL;
    for (int i = 0; i < count; ++i)
        if (row_bytes[i] <= 0 || (row_bytes[i] & 3) || row_bytes[i] > 0x7fffffff) return RGX_EINVAL;
    return RGX_OK;
}

extern "C" int rgx_gather_workspace_bytes(int32_t count, const int64_t *row_bytes, int64_t n, size_t *bytes)
{
    const int rc = gather_check(count, row_bytes, n);
    if (rc != RGX_OK || !bytes) return RGX_EINVAL;
    int shorts = 0;
    for (int i = 0; i < count; ++i) shorts += row_bytes[i] / 4 <= RGX_PACK_ROW;
    *bytes = n >= RGX_PACK_ROWS && shorts >= RGX_PACK_MIN ? (size_t)n * RGX_PACK_WORDS * 4 : 0;
    return RGX_OK;
}

static int gather_direct(uint64_t todo, const void *const *src, void *const *dst, const int64_t *row_bytes, const int64_t *order, int64_t n, hipStream_t s)
{
    while (todo) {
        GatherArgs A;
        int m = 0;
        for (; todo && m < RGX_GATHER_MAX; todo &= todo - 1, ++m) {
            const int t = __builtin_ctzll(todo), i = m;
            A.src[i] = (const uint32_t *)src[t];
            A.dst[i] = (uint32_t *)dst[t];
            const int32_t words = (int32_t)(row_bytes[t] / 4);
            const uintptr_t at = (uintptr_t)A.src[i] | (uintptr_t)A.dst[i];
            const int w = words % 4 == 0 && (at & 15) == 0 ? 4 : words % 3 == 0 ? 3 : words % 2 == 0 && (at & 7) == 0 ? 2 : 1;
            A.words[i] = (uint8_t)w;
            A.pieces[i] = words / w;
            A.magic[i] = (uint32_t)((1ull << 32) / (uint32_t)A.pieces[i] + 1);
        }
        A.count = m;
        const int64_t blocks = (n + RGX_GATHER_ROWS - 1) / RGX_GATHER_ROWS;
        // a workgroup goes through all tensors where there are enough of them to fill the chip several times over
        const int split = blocks >= 2048 ? 1 : m;
        hipLaunchKernelGGL(k_gather_rows, dim3((unsigned)blocks, (unsigned)split), dim3(256), 0, s, A, order, n);
        RGX_LAUNCH_CHECK();
    }
    return RGX_OK;
}

// ws, ws_bytes: rgx_gather_workspace_bytes(); with less (or none) every tensor is gathered by itself.
extern "C" int rgx_gather_rows_packed(int32_t count, const void *const *src, void *const *dst, const int64_t *row_bytes,
                                      const int64_t *order, int64_t n, void *ws, size_t ws_bytes, void *stream)
{
    const DeviceScope on_device(order);
    const int rc = gather_check(count, row_bytes, n);
    if (rc != RGX_OK) return rc;
    if ((count > 0 && (!src || !dst)) || (n > 0 && count > 0 && !order) || ((uintptr_t)ws & 255u)) return RGX_EINVAL;
    for (int i = 0; i < count; ++i)
        if (((!src[i] || !dst[i]) && n > 0) || src[i] == dst[i]) return RGX_EINVAL;
    if (n == 0) return RGX_OK;
    size_t need = 0;
    rgx_gather_workspace_bytes(count, row_bytes, n, &need);
    const bool pack = need > 0 && ws && ws_bytes >= need;
    hipStream_t s = (hipStream_t)stream;
    const unsigned blocks = (unsigned)((n + RGX_GATHER_ROWS - 1) / RGX_GATHER_ROWS);
    for (; count > 0; count -= RGX_GATHER_SET, src += RGX_GATHER_SET, dst += RGX_GATHER_SET, row_bytes += RGX_GATHER_SET) {
        uint64_t todo = count < RGX_GATHER_SET ? (1ull << count) - 1 : ~0ull;
        for (uint64_t members; pack && __builtin_popcountll(members = pack_group(row_bytes, todo)) >= RGX_PACK_MIN; todo &= ~members) {
            PackArgs A;
            A.count = (int32_t)__builtin_popcountll(members);
            A.aligned = 1;
            int at = 0, i = 0;
            for (uint64_t left = members; left; left &= left - 1, ++i) {
                const int t = __builtin_ctzll(left);
                const int32_t w = (int32_t)(row_bytes[t] / 4);
                A.src[i] = (const uint32_t *)src[t];
                A.dst[i] = (uint32_t *)dst[t];
                A.words[i] = (uint8_t)w;
                A.at[i] = (uint8_t)at;
                for (int k = 0; k < w; ++k) A.owner[at + k] = (uint8_t)i;
                A.aligned &= (((uintptr_t)A.src[i] | (uintptr_t)A.dst[i]) & 15) == 0;
                A.magic[i] = (uint32_t)((1ull << 32) / (uint32_t)w + 1);
                at += w;
            }
            A.quads = (at + 3) / 4;
            A.total = at;
            hipLaunchKernelGGL(k_pack_rows, dim3(blocks), dim3(256), 0, s, A, n, (uint4 *)ws);
            hipLaunchKernelGGL(k_unpack_rows, dim3(blocks), dim3(256), 0, s, A, order, n, (const uint4 *)ws);
            RGX_LAUNCH_CHECK();
        }
        const int gathered = gather_direct(todo, src, dst, row_bytes, order, n, s);
        if (gathered != RGX_OK) return gathered;
    }
    return RGX_OK;
}

extern "C" int rgx_gather_rows(int32_t count, const void *const *src, void *const *dst, const int64_t *row_bytes,
                               const int64_t *order, int64_t n, void *stream)
{
    return rgx_gather_rows_packed(count, src, dst, row_bytes, order, n, nullptr, 0, stream);
}

// ---------------------------------------------------------------------------
// Mean squared distance of every point to its three nearest neighbours: distCUDA2 of the
// simple-knn extension (submodules/simple-knn/simple_knn.cu:186-222; used to initialise the scales,
// classes/point_cloud.py:252).  As there: points sorted along a Morton curve, boxes of consecutive
// sorted points, boxes that cannot hold one of the three nearest are left out (the pruning is exact,
// so the result is the exact 3-NN mean whatever the order and the box size).
// Here the curve is a Hilbert curve (k_knn_keys), and a wavefront searches for the consecutive points of it that it owns, in two steps.
// Together: three levels of boxes (8 points, 64 leaves, 64 boxes), of which each lane tests one child against the bounds of the
// wavefront's points, as a few runs, and the largest distance any of them still has to beat; the leaves that are left wait in a list.  Then each
// lane by itself: it tests its share of the list for its own point, some twenty instructions a leaf, and meets the few leaves that can hold one of
// its three.  A wavefront owns 32 points, or 16 or 8 whose 4 or 8 lanes share the list (knn_lanes): a large cloud is bound by the issue of the tests
// and distances, a small one by its longest wavefront, which gets shorter with the stretch of the curve whose bounds it has to search.
// The whole call, sort and boxes included, us; before (a Morton curve of the box between the outermost points, leaves of 16 met by all lanes of
// the wavefront for all its points, 30 bits sorted at every size) / now:
//     heavy-tailed cloud of 1 000, 5 000, 20 000, 54 k, 150 k, 300 k, 1 M, 3 M   36/29 57/48 78/66 119/83 177/109 472/150 681/351 1 612/924
//     ball of as many                                                          35/26 53/39 77/56 112/70 159/102 230/142 537/309 1 362/795
// On a Hilbert curve consecutive cells touch: a run of the Morton curve spans jumps, and its bounds meet twice the leaves (counted on the CPU).
// Distances are (dx*dx + dy*dy) + dz*dz without contraction; rounding is monotone, so the distance to a
// box that holds a point, computed the same way, is never larger than the distance to the point.
#define RGX_KNN_LEAF 8
#define RGX_KNN_FAN 64
#define RGX_KNN_BOX (RGX_KNN_LEAF * RGX_KNN_FAN)
#define RGX_KNN_SEGS(C) ((C) == 8 ? 2 : 4) // runs that a wavefront's points are taken as: with two of 32 points 3 M heavy-tailed take 2.96 ms instead of 0.92
#define RGX_KNN_QUEUE 64 // leaves that wait before the points choose among them

// What the order of the points is made from (k_knn_begin).
#define RGX_KNN_SAMPLE 1024
struct KnnGrid {
    float centre[3], inv_spread[3], inv_reach[3]; // 1 / what knn_warp makes of the sample's outermost points, and a little more
    int32_t crowded;                              // so many points share a cell of that grid that it is not taken
    float line[3][RGX_KNN_SAMPLE];                // the sample's coordinates, ascending: the lines of the other grid
};

// How far along a Hilbert curve of 2^(3 bits) cells a cell lies (the transposed form of J. Skilling, "Programming the Hilbert curve", 2004).
__device__ __forceinline__ uint32_t hilbert_place(uint32_t (&q)[3], int bits)
{
    const uint32_t top = 1u << (bits - 1);
    for (uint32_t m = top; m > 1; m >>= 1)
        for (int a = 0; a < 3; ++a) {
            const uint32_t t = (q[0] ^ q[a]) & (m - 1);
            if (q[a] & m) {
                q[0] ^= m - 1;
            } else {
                q[0] ^= t;
                q[a] ^= t;
            }
        }
    q[1] ^= q[0];
    q[2] ^= q[1];
    uint32_t t = 0;
    for (uint32_t m = top; m > 1; m >>= 1) t ^= q[2] & m ? m - 1 : 0u;
    uint32_t code = 0;
    for (int b = bits - 1; b >= 0; --b)
        for (int a = 0; a < 3; ++a) code = code << 1 | ((q[a] ^ t) >> b & 1u);
    return code;
}

// The points of a crowded box, in the order of a curve through the box alone (there the cells of the whole cloud's say too little): thread t has the t-th of them
// then.  p, id: a point and its index, what comes behind the last one with valid = false.
__device__ __forceinline__ void knn_sort_box(float4 &p, uint32_t &id, bool valid)
{
    __shared__ float x[3][RGX_KNN_BOX], bound[RGX_KNN_BOX / 64][6];
    __shared__ uint32_t ids[RGX_KNN_BOX];
    __shared__ __align__(16) uint32_t key[RGX_KNN_BOX];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool fin = fabsf(p.x) < 1e30f && fabsf(p.y) < 1e30f && fabsf(p.z) < 1e30f;
    const float v[3] = {p.x, p.y, p.z};
    for (int a = 0; a < 3; ++a) {
        const float lo = wave_min_all(fin ? v[a] : INFINITY), hi = wave_max_all(fin ? v[a] : -INFINITY);
        if (lane == 0) {
            bound[wave][a] = lo;
            bound[wave][a + 3] = hi;
        }
        x[a][t] = v[a];
    }
    ids[t] = id;
    __syncthreads();
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
        float lo = bound[0][a], hi = bound[0][a + 3];
        for (int w = 1; w < RGX_KNN_BOX / 64; ++w) {
            lo = fminf(lo, bound[w][a]);
            hi = fmaxf(hi, bound[w][a + 3]);
        }
        const float scale = hi - lo > 1e-30f ? 128.f / (hi - lo) : 0.f;
        q[a] = fin ? (uint32_t)fminf((v[a] - lo) * scale, 127.f) : 127u;
    }
    static_assert(RGX_KNN_BOX == 512, "a key is 21 bits of the curve and nine of the place");
    const uint32_t k = (valid ? hilbert_place(q, 7) : 1u << 21) << 9 | (uint32_t)t;
    key[t] = k;
    __syncthreads();
    int rank = 0;
#pragma unroll 8
    for (int o = 0; o < RGX_KNN_BOX; o += 4) {
        const uint4 other = *(const uint4 *)&key[o];
        rank += (other.x < k) + (other.y < k) + (other.z < k) + (other.w < k);
    }
    __syncthreads();
    key[rank] = (uint32_t)t;
    __syncthreads();
    const uint32_t from = key[t];
    p = make_float4(x[0][from], x[1][from], x[2][from], 0.f);
    id = ids[from];
}

// Gathers the sorted points and bounds them: one workgroup per box.  A point with a coordinate that is
// not a number is at no distance from any other: it becomes a point at infinity, and such points, like the
// padding behind the last one, are in no box's bounds.
__global__ __launch_bounds__(RGX_KNN_BOX) void k_knn_gather(const float *__restrict__ pos, uint32_t *__restrict__ order, const KnnGrid *__restrict__ grid,
                                                            int64_t n, float4 *__restrict__ pts, float4 *__restrict__ leaves,
                                                            float4 *__restrict__ boxes, int32_t *supers_enc)
{
    const int64_t i = (int64_t)blockIdx.x * RGX_KNN_BOX + threadIdx.x;
    float4 p = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
    uint32_t id = 0;
    if (i < n) {
        id = order[i];
        const int64_t j = id;
        const float x = pos[3 * j], y = pos[3 * j + 1], z = pos[3 * j + 2];
        if (x == x && y == y && z == z) p = make_float4(x, y, z, 0.f);
    }
    if (grid->crowded) { // (the whole launch)
        knn_sort_box(p, id, i < n);
        if (i < n) order[i] = id;
    }
    pts[i] = p;
    const bool fin = fabsf(p.x) < INFINITY && fabsf(p.y) < INFINITY && fabsf(p.z) < INFINITY;
    float mn[3] = {fin ? p.x : INFINITY, fin ? p.y : INFINITY, fin ? p.z : INFINITY};
    float mx[3] = {fin ? p.x : -INFINITY, fin ? p.y : -INFINITY, fin ? p.z : -INFINITY};
    auto spread = [&](auto ctrl, auto rows) {
        for (int a = 0; a < 3; ++a) {
            mn[a] = fminf(mn[a], dpp_f<decltype(ctrl)::value, decltype(rows)::value>(INFINITY, mn[a]));
            mx[a] = fmaxf(mx[a], dpp_f<decltype(ctrl)::value, decltype(rows)::value>(-INFINITY, mx[a]));
        }
    };
    const std::integral_constant<int, 0xf> all{};
    spread(std::integral_constant<int, 0xB1>{}, all); // over two, four and the eight lanes of a leaf
    spread(std::integral_constant<int, 0x4E>{}, all);
    spread(std::integral_constant<int, 0x141>{}, all);
    if ((threadIdx.x & (RGX_KNN_LEAF - 1)) == 0) {
        const int64_t l = i / RGX_KNN_LEAF;
        leaves[2 * l] = make_float4(mn[0], mn[1], mn[2], 0.f);
        leaves[2 * l + 1] = make_float4(mx[0], mx[1], mx[2], 0.f);
    }
    spread(std::integral_constant<int, 0x140>{}, all); // over the row, and over the rows, in the last lane
    spread(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
    spread(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    __shared__ float red[RGX_KNN_BOX / 64][6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 63)
        for (int a = 0; a < 3; ++a) {
            red[wave][a] = mn[a];
            red[wave][a + 3] = mx[a];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float v = red[0][a];
        for (int w = 1; w < RGX_KNN_BOX / 64; ++w) v = a < 3 ? fminf(v, red[w][a]) : fmaxf(v, red[w][a]);
        ((float *)(boxes + 2 * (int64_t)blockIdx.x))[a < 3 ? a : a + 1] = v;
        int32_t *super = supers_enc + 6 * (int64_t)(blockIdx.x / RGX_KNN_FAN);
        if (a < 3) atomicMin(&super[a], enc_f(v));
        else atomicMax(&super[a], enc_f(v));
    }
}

// What the order of the points is made from, and the bounds of the boxes of boxes before any point is in them.
// The order only decides how many boxes a search has to open, never what it finds, so it may be any curve.  It is a Hilbert
// curve, whose consecutive cells always touch, through a grid that a sample of the cloud shapes: per axis linear where the bulk of the
// points lies, logarithmic beyond (knn_warp).  A grid between the outermost points instead, as a few far points stretch it, leaves
// thousands of the others in one cell, in whose order they say nothing of where they lie.
// Where there is no one bulk -- clumps far apart, points along a line -- a cell of that grid holds hundreds.  So a cloud of which the sample says that knn_crowd
// others or more share a point's cell is sorted along the grid of the sample's quantiles, as many points between any two lines of an axis, and box by box once more along
// a curve through the box (knn_sort_box).  Not the other clouds: the cells of sparse points far out become long and thin (54 k heavy-tailed 81 us, by quantiles 179).
// Clouds like those of the table above come out below 10, up to a million points, clumps above 30.  The whole call, us: by a Morton curve of 30 bits through the
// box between the outermost points and leaves of 16 / by the first grid always / now:
//     points                             54 k              150 k                500 k                   1 M
//     10 clumps of 0.005 in a cube    124/130/91       196/432/133       440/3 183/255        850/1 180/501
//     3 clumps of 0.002               120/242/87       252/1 090/129     635/11 640/267     1 550/3 830/538
//     100 clumps of 0.002             104/83/79        157/236/120       430/1 580/254      1 030/1 380/462
//     20 clumps of 0.001 to 0.3       146/142/102      270/395/166     1 260/3 250/355      1 800/1 900/1 050
//     along a line                     77/142/88       106/310/124       246/1 024/287        620/1 190/548
// (A line is what a Morton curve sorts best.  A ball or a heavy-tailed cloud pays 1 to 2 us for being asked.)
#define RGX_KNN_RANKED 64 // of the sample: a workgroup ranks so many, along one axis
// Up to so many points nothing is asked: what it and the other grid take is more than crowded cells do (5 000 points in 10 clumps 41 us, asked 52; in a ball 40 and 41).
#define RGX_KNN_ASKED 8192
// From so many others in a point's cell on a cloud is crowded: the fewer points, the more (16 384 in 10 clumps, some 90 others: 54 us, by quantiles 73; 32 768, some 180: 87 and 68).
__device__ __forceinline__ float knn_crowd(int64_t n) { return fminf(fmaxf(0x1p21f / (float)n, 16.f), 128.f); }
// Bits of the grid per axis: 24-bit keys are sorted in three passes, 30-bit keys in four.  Beyond half a million points a cell of the coarser grid
// holds too many of them where a cloud is dense (us with 8 / 10 bits: 54 k heavy-tailed 83 / 101, 300 k 178 / 184, 1 M 408 / 352, ball 293 / 309).
static inline int knn_bits(int64_t n) { return n <= 1 << 19 ? 8 : 10; }
__device__ __forceinline__ float knn_warp(float x, float centre, float inv_spread)
{
    const float u = (x - centre) * inv_spread, m = fabsf(u);
    return copysignf(m < 1.f ? m : 1.f + __logf(m), u);
}
// the t-th point of the sample.  A few points: all of them; else places without a period that the points' own order could share
__device__ __forceinline__ int64_t knn_sample(int t, int64_t n)
{
    return n <= RGX_KNN_SAMPLE ? (t < n ? t : n - 1) : (int64_t)(((uint64_t)((uint32_t)t * 2654435761u) * (uint64_t)n) >> 32);
}
// Which cell of the warped grid a point lies in, per axis.
__device__ __forceinline__ void knn_cell(const float (&x)[3], const float (&centre)[3], const float (&inv_spread)[3], const float (&inv_reach)[3], int bits, uint32_t (&q)[3])
{
    const float half = (float)(1u << (bits - 1));
    for (int a = 0; a < 3; ++a) {
        const float u = knn_warp(x[a], centre[a], inv_spread[a]) * inv_reach[a];
        q[a] = (uint32_t)(half + (half - 1.f) * fminf(fmaxf(u, -1.f), 1.f)); // (not a number: the grid's edge)
    }
}
// One workgroup for the warped grid, `ranking` of them for the lines of the other (none: it is not asked for), the others for the bounds.
__global__ __launch_bounds__(RGX_KNN_SAMPLE) void k_knn_begin(const float *__restrict__ pos, int64_t n, int bits, int ranking, KnnGrid *grid, int32_t *supers_enc, int64_t ns)
{
    __shared__ __align__(16) uint32_t s_words[4 * RGX_KNN_SAMPLE];
    if ((int)blockIdx.x > ranking) {
        for (int64_t k = (int64_t)((int)blockIdx.x - 1 - ranking) * blockDim.x + threadIdx.x; k < 6 * ns; k += (int64_t)((int)gridDim.x - 1 - ranking) * blockDim.x)
            supers_enc[k] = enc_f(k % 6 < 3 ? INFINITY : -INFINITY);
        return;
    }
    if (blockIdx.x > 0) {
        const int axis = (blockIdx.x - 1) % 3, first = (blockIdx.x - 1) / 3 * RGX_KNN_RANKED;
        float *const x = (float *)s_words;
        int *const count = (int *)(s_words + RGX_KNN_SAMPLE);
        const float mine = pos[3 * knn_sample(threadIdx.x, n) + axis];
        x[threadIdx.x] = mine == mine ? mine : INFINITY;
        __syncthreads();
        // how many of a sixteenth of the sample come before each (the sixteenth is a wavefront's); of equal ones the earlier of the sample
        const int s = first + (threadIdx.x & 63), from = threadIdx.x & ~63;
        const float v = x[s];
        int before = 0;
#pragma unroll 4
        for (int t = from; t < from + 64; t += 4) {
            const float4 o = *(const float4 *)&x[t];
            if (from < first) before += (o.x <= v) + (o.y <= v) + (o.z <= v) + (o.w <= v);
            else if (from > first) before += (o.x < v) + (o.y < v) + (o.z < v) + (o.w < v);
            else before += (t < s ? o.x <= v : o.x < v) + (t + 1 < s ? o.y <= v : o.y < v) + (t + 2 < s ? o.z <= v : o.z < v) + (t + 3 < s ? o.w <= v : o.w < v);
        }
        count[threadIdx.x] = before;
        __syncthreads();
        if (threadIdx.x < RGX_KNN_RANKED) {
            int rank = 0;
            for (int k = 0; k < RGX_KNN_SAMPLE; k += 64) rank += count[threadIdx.x + k];
            grid->line[axis][rank] = v;
        }
        return;
    }
    constexpr int EACH = RGX_KNN_SAMPLE / 256;
    if (threadIdx.x >= 256) return; // (four wavefronts meet sooner than sixteen)
    for (int k = threadIdx.x; k < 4 * RGX_KNN_SAMPLE; k += 256) s_words[k] = ~0u;
    __shared__ float red[4][4][6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto sum = [&](int use, float *v, int m, bool most) { // over the workgroup, in every thread; or the largest of the last three
        for (int a = 0; a < m; ++a) {
            v[a] = most && a >= m - 3 ? wave_max_all(v[a]) : wave_sum_all(v[a]);
            if (lane == 0) red[use][wave][a] = v[a];
        }
        __syncthreads();
        for (int a = 0; a < m; ++a) {
            const float *r = &red[use][0][a];
            v[a] = most && a >= m - 3 ? fmaxf(fmaxf(r[0], r[6]), fmaxf(r[12], r[18])) : (r[0] + r[6]) + (r[12] + r[18]);
        }
    };
    float x[EACH][3], w[EACH]; // w: 0 for a point that has a coordinate without a finite value
    for (int k = 0; k < EACH; ++k) {
        const int64_t i = knn_sample(k * 256 + threadIdx.x, n);
        for (int a = 0; a < 3; ++a) x[k][a] = pos[3 * i + a];
    }
    float v[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < EACH; ++k) {
        w[k] = fabsf(x[k][0]) < 1e30f && fabsf(x[k][1]) < 1e30f && fabsf(x[k][2]) < 1e30f ? 1.f : 0.f;
        for (int a = 0; a < 3; ++a) {
            x[k][a] = w[k] != 0.f ? x[k][a] : 0.f;
            v[a] += x[k][a];
        }
        v[3] += w[k];
    }
    sum(0, v, 4, false);
    const float count = fmaxf(v[3], 1.f);
    float c[3], off[3]; // the mean, and the mean distance from it
    for (int a = 0; a < 3; ++a) {
        c[a] = v[a] / count;
        v[a] = 0.f;
        for (int k = 0; k < EACH; ++k) v[a] += w[k] * fabsf(x[k][a] - c[a]);
    }
    sum(1, v, 3, false);
    for (int a = 0; a < 3; ++a) {
        off[a] = v[a] / count;
        v[a] = v[a + 3] = 0.f;
        for (int k = 0; k < EACH; ++k) { // from the mean towards the median: weights fall with the distance
            const float g = w[k] / (fabsf(x[k][a] - c[a]) + 0.05f * off[a] + 1e-30f);
            v[a] += g * x[k][a];
            v[a + 3] += g;
        }
    }
    sum(2, v, 6, false);
    for (int a = 0; a < 3; ++a) {
        c[a] = v[a + 3] > 0.f ? v[a] / v[a + 3] : 0.f;
        v[a] = v[a + 3] = 0.f;
        for (int k = 0; k < EACH; ++k) {
            const float d = fabsf(x[k][a] - c[a]);
            v[a] += w[k] * __logf(fmaxf(d, 1e-3f * off[a]) + 1e-30f);
            v[a + 3] = fmaxf(v[a + 3], w[k] * d);
        }
    }
    sum(3, v, 6, true);
    float inv_spread[3], inv_reach[3];
    for (int a = 0; a < 3; ++a) {
        // the spread: the geometric mean distance from the centre; e of it is where an even spread ends
        const float spread = 2.7f * __expf(v[a] / count);
        inv_spread[a] = spread > 1e-25f ? 1.f / spread : 0.f;
        inv_reach[a] = 1.f / fmaxf(1.05f * knn_warp(v[a + 3], 0.f, inv_spread[a]), 1e-3f);
    }
    v[0] = 0.f;
    if (ranking) {
        // How many of the sample lie in a cell that others of it lie in: a place for each cell, maybe others' too, holds who was there last.
        uint32_t before[EACH], cell[EACH];
        for (int k = 0; k < EACH; ++k) {
            uint32_t q[3];
            knn_cell(x[k], c, inv_spread, inv_reach, bits, q);
            cell[k] = w[k] != 0.f ? (q[0] << bits | q[1]) << bits | q[2] : ~0u - 1u;
            before[k] = atomicExch(&s_words[cell[k] * 2654435761u >> 20], cell[k]);
        }
        for (int k = 0; k < EACH; ++k) v[0] += w[k] != 0.f && before[k] == cell[k] ? 1.f : 0.f;
        sum(0, v, 1, false);
    }
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        grid->centre[a] = a == 0 ? c[0] : a == 1 ? c[1] : c[2];
        grid->inv_spread[a] = a == 0 ? inv_spread[0] : a == 1 ? inv_spread[1] : inv_spread[2];
        grid->inv_reach[a] = a == 0 ? inv_reach[0] : a == 1 ? inv_reach[1] : inv_reach[2];
        // as many as of points spread over so few cells that as many share one
        const float cells = (float)n / knn_crowd(n);
        if (a == 0) grid->crowded = ranking && v[0] >= RGX_KNN_SAMPLE - cells * (1.f - __expf(-RGX_KNN_SAMPLE / cells));
    }
}

// The place of every point along the curve.
__global__ __launch_bounds__(256) void k_knn_keys(const float *__restrict__ pos, int64_t n, const KnnGrid *__restrict__ grid, int bits,
                                                  uint32_t *__restrict__ keys, uint32_t *__restrict__ vals)
{
    __shared__ float line[3][RGX_KNN_SAMPLE];
    const bool crowded = grid->crowded; // (the whole launch)
    if (crowded) {
        const int each = RGX_KNN_SAMPLE >> bits; // of the sample's coordinates to a cell
        for (int k = threadIdx.x; k < 3 << bits; k += 256) line[k >> bits][k & ((1 << bits) - 1)] = grid->line[k >> bits][(k & ((1 << bits) - 1)) * each + each - 1];
        __syncthreads();
    }
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float x[3];
    uint32_t q[3] = {0u, 0u, 0u};
    for (int a = 0; a < 3; ++a) x[a] = pos[3 * i + a];
    if (crowded) {
        for (uint32_t m = 1u << (bits - 1); m > 0; m >>= 1) // how many lines are below it (not a number: none)
            for (int a = 0; a < 3; ++a) q[a] += line[a][q[a] + m - 1] < x[a] ? m : 0u;
    } else {
        knn_cell(x, grid->centre, grid->inv_spread, grid->inv_reach, bits, q);
    }
    keys[i] = hilbert_place(q, bits);
    vals[i] = (uint32_t)i;
}

// Squared distance between two boxes (a point is a box of no size): simple_knn.cu:124-135 distBoxPoint.
__device__ __forceinline__ float knn_box_dist(f3 lo, f3 hi, f3 qlo, f3 qhi)
{
    const float dx = fmaxf(fmaxf(lo.x - qhi.x, qlo.x - hi.x), 0.f);
    const float dy = fmaxf(fmaxf(lo.y - qhi.y, qlo.y - hi.y), 0.f);
    const float dz = fmaxf(fmaxf(lo.z - qhi.z, qlo.z - hi.z), 0.f);
    return (dx * dx + dy * dy) + dz * dz;
}

// Lanes per point (us with 8 / 4 / 2 lanes, keys of 30 bits: heavy-tailed 5 000 52 / 59 / 80, 54 k 101 / 101 / 244, 150 k 120 / 126 / 230, 300 k
// 184 / 167 / 215, 1 M 474 / 375 / 352, 3 M 1 133 / 976 / 924; ball 54 k 85 / 85 / 95, 300 k 161 / 160 / 154, 1 M 360 / 345 / 309, 3 M 991 / 920 / 795).
static inline int knn_lanes(int64_t n) { return n <= 1 << 18 ? 8 : n <= 1 << 19 ? 4 : 2; }

// the smallest of the first P lanes' values (all lanes must be active)
template <int P> __device__ __forceinline__ float first_min(float v)
{
    v = fminf(v, dpp_f<0xB1, 0xf>(INFINITY, v));
    v = fminf(v, dpp_f<0x4E, 0xf>(INFINITY, v));
    v = fminf(v, dpp_f<0x141, 0xf>(INFINITY, v));
    if constexpr (P > 8) v = fminf(v, dpp_f<0x140, 0xf>(INFINITY, v));
    if constexpr (P > 16) v = fminf(v, dpp_f<0x142, 0xa>(INFINITY, v));
    if constexpr (P > 32) v = fminf(v, dpp_f<0x143, 0xc>(INFINITY, v));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), P - 1));
}
template <int P> __device__ __forceinline__ float first_max(float v) { return -first_min<P>(-v); }

// simple_knn.cu:137-184 updateKBest<3>, boxMeanDist.  C: lanes per point.
template <int C>
__global__ __launch_bounds__(256) void k_knn3(const float4 *__restrict__ pts, const uint32_t *__restrict__ order, int64_t n,
                                              const float4 *__restrict__ leaves, const float4 *__restrict__ boxes, int64_t nb,
                                              const int32_t *__restrict__ supers_enc, int64_t ns, float *__restrict__ out)
{
    static_assert(RGX_KNN_LEAF == 8, "eight lanes hold a leaf");
    constexpr int P = 64 / C, SHARE = 2 * RGX_KNN_QUEUE / C; // points of a wavefront; waiting leaves that a lane looks at, at most
    constexpr int WORDS = (SHARE + 31) / 32;
    constexpr int SEGS = RGX_KNN_SEGS(C);
    __shared__ int queue[4][2 * RGX_KNN_QUEUE];
    const int lane = threadIdx.x & 63, copy = lane / P;
    int *const list = queue[threadIdx.x >> 6];
    const int64_t first = __builtin_amdgcn_readfirstlane((int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6)) * (int64_t)P;
    if (first >= n) return; // whole wave
    const int64_t i = first + (lane & (P - 1));
    const float4 p4 = pts[i]; // (the array is padded to whole boxes)
    const f3 p = mk3(p4.x, p4.y, p4.z);
    const bool act = fabsf(p.x) < INFINITY && fabsf(p.y) < INFINITY && fabsf(p.z) < INFINITY;
    // The wavefront's points as SEGS runs of the curve, cut where it jumps farthest: the bounds of a run that
    // spans such a jump would meet most of the cloud.
    uint64_t cuts = 0; // over the first P lanes
    {
        const f3 step = p - mk3(__shfl_up(p.x, 1), __shfl_up(p.y, 1), __shfl_up(p.z, 1));
        float gap = lane > 0 && lane < P ? dot3(step, step) : -1.f;
        if (!(gap < INFINITY)) gap = -1.f;
        for (int k = 1; k < SEGS; ++k) {
            const float g = first_max<P>(gap);
            const uint64_t at = __ballot(gap == g && g > 0.f);
            if (at == 0) break;
            cuts |= at & -at;
            if (lane == __builtin_ctzll(at)) gap = -1.f;
        }
    }
    const int seg = __popcll(cuts & (~0ull >> (63 - (lane & (P - 1)))));
    f3 slo[SEGS], shi[SEGS];
    float reach[SEGS]; // the largest distance a point of the run still has to beat
    for (int k = 0; k < SEGS; ++k) {
        const bool in = act && seg == k;
        slo[k] = mk3(first_min<P>(in ? p.x : INFINITY), first_min<P>(in ? p.y : INFINITY), first_min<P>(in ? p.z : INFINITY));
        shi[k] = mk3(first_max<P>(in ? p.x : -INFINITY), first_max<P>(in ? p.y : -INFINITY), first_max<P>(in ? p.z : -INFINITY));
    }
    float b0 = FLT_MAX, b1 = FLT_MAX, b2 = FLT_MAX; // the three smallest that this lane has met, ascending
    auto put = [](float &c0, float &c1, float &c2, float d) {
        c2 = __builtin_amdgcn_fmed3f(c1, c2, d);
        c1 = __builtin_amdgcn_fmed3f(c0, c1, d);
        c0 = fminf(c0, d);
    };
    auto meet = [&](f3 q, bool not_itself = true) {
        const float dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
        const float d = (dx * dx + dy * dy) + dz * dz;
        put(b0, b1, b2, not_itself ? d : FLT_MAX);
    };
    float t0, t1, worst; // the three smallest that the point's lanes have met
    auto measure = [&]() {
        t0 = b0;
        t1 = b1;
        worst = b2;
        for (int o = P; o < 64; o <<= 1) {
            const float o0 = __shfl_xor(t0, o), o1 = __shfl_xor(t1, o), o2 = __shfl_xor(worst, o);
            put(t0, t1, worst, o0);
            put(t0, t1, worst, o1);
            put(t0, t1, worst, o2);
        }
        for (int k = 0; k < SEGS; ++k) reach[k] = first_max<P>(act && seg == k ? worst : -1.f);
    };
    // The points nearby on the curve first, those of the point's own leaf and of the two beside it: they leave little for the boxes.
    // Eight lanes hold a leaf and hand its points around among themselves.
    const int own = (int)(i / RGX_KNN_LEAF), n_leaves = (int)(nb * RGX_KNN_FAN);
    for (int turn = copy; turn < (C > 3 ? C : 3); turn += C) { // (a leaf's eight lanes take the same turns)
        const int l = turn == 0 ? own : turn == 1 ? own - 1 : own + 1;
        const bool there = turn < 3 && l >= 0 && l < n_leaves;
        const float4 q4 = pts[(int64_t)(there ? l : own) * RGX_KNN_LEAF + (lane & (RGX_KNN_LEAF - 1))];
        const f3 q = mk3(there ? q4.x : INFINITY, q4.y, q4.z);
        auto across = [](f3 v, auto ctrl) {
            constexpr int X = decltype(ctrl)::value;
            return mk3(dpp_f<X, 0xf>(v.x, v.x), dpp_f<X, 0xf>(v.y, v.y), dpp_f<X, 0xf>(v.z, v.z));
        };
        const std::integral_constant<int, 0xB1> by1{}; // lanes of a quad exchanged: with the neighbour,
        const std::integral_constant<int, 0x4E> by2{}; // with the one after it,
        const std::integral_constant<int, 0x1B> by3{}; // mirrored
        const f3 r = across(q, std::integral_constant<int, 0x141>{}); // the eight lanes mirrored
        meet(q, l != own);
        meet(across(q, by1));
        meet(across(q, by2));
        meet(across(q, by3));
        meet(r);
        meet(across(r, by1));
        meet(across(r, by2));
        meet(across(r, by3));
    }
    measure();
    auto open = [&](f3 lo, f3 hi) { // is the box within some run's reach?
        bool o = false;
        for (int k = 0; k < SEGS; ++k) o |= knn_box_dist(lo, hi, slo[k], shi[k]) < reach[k];
        return o;
    };
    int waiting = 0; // leaves in the list
    // Of its share of the leaves in the list every lane chooses those that can hold one of its point's three, and meets them by itself.
    auto choose = [&]() {
        __builtin_amdgcn_wave_barrier();
        uint32_t mine[WORDS] = {};
        const int rounds = (waiting + C - 1) / C;
#pragma unroll
        for (int w = 0; w < WORDS; ++w)
            for (int c0 = 32 * w; c0 < rounds && c0 < 32 * w + 32; c0 += 4) {
                int l[4];
                float4 lo[4], hi[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    l[k] = list[std::min((c0 + k) * C + copy, waiting - 1)];
                    lo[k] = leaves[2 * (int64_t)l[k]];
                    hi[k] = leaves[2 * (int64_t)l[k] + 1];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const bool near = knn_box_dist(mk3(lo[k].x, lo[k].y, lo[k].z), mk3(hi[k].x, hi[k].y, hi[k].z), p, p) < worst &&
                                      (uint32_t)(l[k] - own + 1) > 2u && (c0 + k) * C + copy < waiting;
                    mine[w] |= near ? 1u << (c0 + k - 32 * w) : 0u;
                }
            }
#pragma unroll
        for (int w = 0; w < WORDS; ++w) {
            if (!act) mine[w] = 0;
            while (mine[w]) {
                const int l = list[(32 * w + __builtin_ctz(mine[w])) * C + copy];
                mine[w] &= mine[w] - 1;
                const float4 *q = pts + (int64_t)l * RGX_KNN_LEAF;
#pragma unroll
                for (int k = 0; k < RGX_KNN_LEAF; ++k) meet(mk3(q[k].x, q[k].y, q[k].z));
            }
        }
        __builtin_amdgcn_wave_barrier();
        waiting = 0;
        measure();
    };
    // The children that lie within reach, one in each lane, one after the other.  More than MANY of them are open to a run that has not met
    // its neighbours yet (points between a dense part and a sparse one): then the nearest first, and the others only if they
    // are still within reach.
    auto each_open = [&](bool there, f3 lo, f3 hi, int many, auto visit) {
        uint64_t todo = __ballot(there && open(lo, hi));
        while (todo) {
            int t = __builtin_ctzll(todo);
            const bool nearest = __popcll(todo) > many;
            if (nearest) {
                float d = INFINITY;
                for (int k = 0; k < SEGS; ++k) d = fminf(d, knn_box_dist(lo, hi, slo[k], shi[k]));
                if (!(todo >> lane & 1)) d = INFINITY;
                const uint64_t at = __ballot(d == wave_min_all(d)) & todo;
                if (at) t = __builtin_ctzll(at);
            }
            todo &= ~(1ull << t);
            visit(t);
            if (nearest) {
                if (waiting) choose();
                todo &= __ballot(open(lo, hi));
            }
        }
    };
    for (int64_t s0 = 0; s0 < ns; s0 += 64) {
        const int32_t *e = supers_enc + 6 * std::min(s0 + lane, ns - 1);
        each_open(s0 + lane < ns, mk3(dec_f(e[0]), dec_f(e[1]), dec_f(e[2])), mk3(dec_f(e[3]), dec_f(e[4]), dec_f(e[5])), 4, [&](int ts) {
            const int64_t box0 = (s0 + ts) * RGX_KNN_FAN;
            const float4 *b = boxes + 2 * std::min(box0 + lane, nb - 1);
            const float4 blo = b[0], bhi = b[1];
            each_open(box0 + lane < nb, mk3(blo.x, blo.y, blo.z), mk3(bhi.x, bhi.y, bhi.z), 8, [&](int tb) {
                const int l = (int)(box0 + tb) * RGX_KNN_FAN + lane;
                const float4 lo = leaves[2 * (int64_t)l], hi = leaves[2 * (int64_t)l + 1];
                const bool wanted = open(mk3(lo.x, lo.y, lo.z), mk3(hi.x, hi.y, hi.z));
                const uint64_t some = __ballot(wanted);
                if (wanted) list[waiting + __popcll(some & ((1ull << lane) - 1ull))] = l;
                waiting += __popcll(some);
                if (waiting >= RGX_KNN_QUEUE) choose();
            });
        });
    }
    if (waiting) choose();
    if (i < n && copy == 0) out[order[i]] = act ? ((t0 + t1) + worst) / 3.0f : INFINITY;
}

struct KnnLayout {
    MortonLayout m;
    size_t pts, leaves, boxes, supers, grid, total;
    int64_t nb, ns;
};
static inline KnnLayout knn_layout(int64_t n)
{
    KnnLayout K;
    K.m = morton_layout(n);
    const size_t nn = (size_t)(n > 0 ? n : 1);
    K.nb = (int64_t)((nn + RGX_KNN_BOX - 1) / RGX_KNN_BOX);
    K.ns = (K.nb + RGX_KNN_FAN - 1) / RGX_KNN_FAN;
    size_t off = K.m.total;
    K.pts = off;    off = rgx_align_up(off + (size_t)K.nb * RGX_KNN_BOX * 16, 256);
    K.leaves = off; off = rgx_align_up(off + (size_t)K.nb * RGX_KNN_FAN * 32, 256);
    K.boxes = off;  off = rgx_align_up(off + (size_t)K.nb * 32, 256);
    K.supers = off; off = rgx_align_up(off + (size_t)K.ns * 24, 256);
    K.grid = off;   off = rgx_align_up(off + sizeof(KnnGrid), 256);
    K.total = off;
    return K;
}

extern "C" int rgx_knn_workspace_bytes(int64_t n, size_t *bytes)
{
    if (n < 0 || !bytes || n > 0x3fffffff) return RGX_EINVAL;
    *bytes = knn_layout(n).total;
    return RGX_OK;
}

extern "C" int rgx_dist2_knn3(const float *pos, int64_t n, float *mean_dist2, void *ws, size_t ws_bytes, void *stream)
{
    const DeviceScope on_device(pos);
    if (n < 0 || n > 0x3fffffff || !ws || (n > 0 && (!pos || !mean_dist2))) return RGX_EINVAL;
    const KnnLayout K = knn_layout(n);
    if (ws_bytes < K.total || ((uintptr_t)ws & 255u)) return RGX_EWORKSPACE;
    if (n == 0) return RGX_OK;
    hipStream_t s = (hipStream_t)stream;
    char *w = (char *)ws;
    uint32_t *k0 = (uint32_t *)(w + K.m.keys0), *k1 = (uint32_t *)(w + K.m.keys1);
    uint32_t *v0 = (uint32_t *)(w + K.m.vals0), *v1 = (uint32_t *)(w + K.m.vals1);
    float4 *pts = (float4 *)(w + K.pts), *leaves = (float4 *)(w + K.leaves), *boxes = (float4 *)(w + K.boxes);
    int32_t *supers = (int32_t *)(w + K.supers);
    KnnGrid *grid = (KnnGrid *)(w + K.grid);
    const int bits = knn_bits(n);
    const int ranking = n > RGX_KNN_ASKED ? 3 * RGX_KNN_SAMPLE / RGX_KNN_RANKED : 0;
    hipLaunchKernelGGL(k_knn_begin, dim3(1 + ranking + (unsigned)std::min<int64_t>((6 * K.ns + RGX_KNN_SAMPLE - 1) / RGX_KNN_SAMPLE, 256)), dim3(RGX_KNN_SAMPLE), 0, s, pos, n, bits, ranking,
                       grid, supers, K.ns);
    hipLaunchKernelGGL(k_knn_keys, grid_for(n, 256), dim3(256), 0, s, pos, n, grid, bits, k0, v0);
    RGX_LAUNCH_CHECK();
    const int r = radix_sort<uint32_t>(k0, v0, k1, v1, n, 3 * bits, (uint32_t *)(w + K.m.hist), s);
    if (r < 0) return r;
    uint32_t *order = r ? v1 : v0;
    hipLaunchKernelGGL(k_knn_gather, dim3((unsigned)K.nb), dim3(RGX_KNN_BOX), 0, s, pos, order, grid, n, pts, leaves, boxes, supers);
    const auto search = [&](auto lanes) {
        constexpr int C = decltype(lanes)::value;
        hipLaunchKernelGGL(k_knn3<C>, grid_for(n * C, 256), dim3(256), 0, s, pts, order, n, leaves, boxes, K.nb, supers, K.ns, mean_dist2);
    };
    switch (knn_lanes(n)) {
    case 8: search(std::integral_constant<int, 8>{}); break;
    case 4: search(std::integral_constant<int, 4>{}); break;
    default: search(std::integral_constant<int, 2>{});
    }
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}
