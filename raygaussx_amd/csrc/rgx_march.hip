// Ray-march kernels: forward compositing, its viewer variant, and the two backward passes.
// Replace the OptiX programs of optix_raycasting/cuda_train/forward/gaussians_aabb.cu
// (also cuda_test/, byte-identical), cuda_gui/gaussians_aabb.cu and
// cuda_train/backward/gaussians_aabb.cu, and their launchers
// (optix_raycasting/optix_utils.py:222-322, 363-500, 503-601).
//
// Mapping: one lane per ray, one 64-lane wavefront (= one workgroup) per 8x8 pixel
// tile, all rays of a tile sharing the camera origin.  Per slab iteration the wave
//   1. makes its candidate table (LDS) cover the lanes' slab intervals: it reuses the resident
//      window, or sweeps the BVH cooperatively (node stack in LDS, one node per lane per step,
//      starting from the tile's cut through the tree) for the Gaussians whose ellipsoids meet
//      the tile's frustum in the depth range wanted;
//   2. filters: a wave-uniform loop over the table in which every lane tests ITS ray and slab against the
//      entry, without the hit predicate's roots unless a decision is close, and then by the exact
//      predicate (so hit sets are those of a per-ray query); the result is the tile's list of entries hit,
//      per lane its hit bits over that list, and per 4x4 pixel row which entries reach each half of the samples;
//   3. shades: every lane walks its own hits (forward, the backward's density pass), or groups of lanes
//      walk the entries that one of their rays hits, in lock step, and sum each entry's 13 whitened-frame
//      sums over their rays with DPP adds (the backward's gradient pass: half rows of 8 lanes in a replay, rows
//      of 16 in the backward that searches the tree).
// An image of few tiles is marched by parts of tiles (Part, launch_forward).
// The forward can record what 1 and 2 produced, and the per-sample density and colour sums of 3;
// the replaying backward then needs no tree, no table, no predicate and no density pass, sums a window's
// gradients in LDS before adding them to memory, and replays a tile in several pieces side by side.
// The first-hit query (once per ray, and after an empty slab) runs on the same candidate tables.
// The per-lane skip-link queries below serve the segment test hooks (arbitrary rays).
#include "rgx_device.h"
#include <hip/hip_fp16.h>

#include <mutex>
#include <type_traits>

#ifndef RGX_QCAP
#define RGX_QCAP 432       // node stack entries per wave (LDS)
#endif
#ifndef RGX_CCAP
#define RGX_CCAP 112       // candidate table entries per wave (LDS): with 112 (and a 432-entry stack) a tile needs 12 800 bytes, and 12 tiles fit a CU
#endif
#ifndef RGX_KHI
#define RGX_KHI ((RGX_CCAP * 3) / 4) // a window that filled its table beyond this looks half as many slabs ahead next time
#endif
#ifndef RGX_KLO
#define RGX_KLO (RGX_CCAP / 3)       // one that stayed below this, twice as many
#endif
#define RGX_MASK_WORDS ((RGX_CCAP + 31) / 32) // 32-bit words of a hit mask over the list
// Above QCAP - margin the sweep pops one node at a time (depth-first).  A breadth-first step pops
// up to 64 nodes and pushes up to 128, so it leaves at most QCAP - margin + 64 entries; a
// depth-first step adds at most one entry per level it descends, and a Karras tree over 63-bit
// keys with ties broken by a 30-bit index is at most 63 + 30 = 93 deep: with a margin of 160 the
// stack never holds more than QCAP - 96 + 93 < QCAP entries, whatever the scene.
#define RGX_DFS_MARGIN 160
#define RGX_LDS_HITS 32    // per-lane list of the stand-alone collect hook
// The march kernels are sized (registers and LDS) for three wavefronts per SIMD.
#ifndef RGX_WAVES_ATTR
#define RGX_WAVES_ATTR __attribute__((amdgpu_waves_per_eu(3, 3)))
#endif
// The forward that leaves a record by parts of tiles, for two: what it keeps of a part's record does not fit 168 registers beside the rest (112 bytes of
// spills a lane), and a launch by parts seldom fills more (4 k Gaussians 128x128 0.82 -> 0.74 ms a step, 100 k in a ball 256x240 1.22 -> 1.16).
#define RGX_WAVES_ATTR_FWD(two) __attribute__((amdgpu_waves_per_eu((two) ? 2 : 3, (two) ? 2 : 3)))

struct MarchParams {
    RgxCamera cam;
    RgxMarch m;
    const Node *nodes;
    const int32_t *right; // right child of internal node i
    const float4 *pairs;  // the same tree, internal node by internal node (NodePair; up to RGX_PAIR_BOXES boxes)
    const uint32_t *order; // sorted position -> input index
    const uint32_t *place; // input index -> sorted position
    const WsHeader *hdr;
    const Prim *prims;
    int64_t n;
    float *ray_colors;       // fwd: output
    uint8_t *frame;          // viewer: uchar4 colours
    float *depth;            // viewer: expected depth
    const float *fwd_colors; // bwd: forward output (C + T*bg)
    const float *dloss;      // bwd
    float *gbuf;             // bwd: (n,16) gradient block in Morton order
    RgxStats *stats;
    int32_t tiles_x, tiles_y;
    uint32_t *records;      // hit-list record stream, rec_tile_words per tile or part of one, or null
    int32_t rec_tile_words;
    int32_t only_overflow;  // backward: handle only the tiles (parts) whose record overflowed
    int32_t rec_pieces, rec_first, rec_equal, rec_turn; // the pieces of a tile's record (record_pieces)
    uint32_t *tile_order;   // launch order lists (or null: as launched)
    int32_t use_tile_order; // 0: as launched; 1: per XCD, its tiles' list positions from the heaviest to the lightest (k_tile_order);
                            // 2: per XCD, the blocks of tiles it renders, heaviest first (k_block_order)
    int32_t part_bits;      // each tile by 2^part_bits workgroups (launch_forward)
    float4 *sum_pool;       // sample-sum slots of the record (RGX_SUM_SLOT_WORDS each), or null
    uint32_t *sum_next;     // next free slot (bump counter in the record's pool header)
    int32_t sum_slots;      // slots in the pool (a part's: 2^part_bits to one of the bump counter's)
    int32_t sum_slot_words; // words per slot: RGX_SUM_SLOT_WORDS, or RGX_SUM_SLOT_WORDS_HALF with half-precision colour sums, >> part_bits
    uint32_t *faults;       // march workspace: [0] replays that lost their record, [1] sweeps that dropped nodes; or null
    uint32_t *ray_counts;   // counting forward only: per ray, slabs blended and the sum of their hit-list lengths; or null
    // (at the end: where the others lie decides which of them one load fetches)
    int32_t rec_bits;       // each tile has 2^rec_bits regions of the record
    uint32_t sum_first;     // the first slot of the pool that is not a part's own to begin with
};

// The kernel's arguments once more, from the kernel's argument segment: what is read through this is loaded where it is used.
// Only in a kernel whose first argument is its MarchParams, and in functions that are always inlined into one: in a function that is called, the
// segment's pointer is none.
__device__ __forceinline__ const MarchParams &args_again()
{
    auto p = (const __attribute__((address_space(4))) MarchParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const MarchParams *)p;
}

// Section census (diagnostic builds only: -DRGX_SECTION_CLOCKS, `python -m raygaussx_amd.build --sections`;
// the product library has none of it).  Every wave of a kernel launched without a statistics block keeps
// one running time stamp; RGX_SEC(cn, k) adds the cycles since the previous stamp to section k, so the
// sections of a wave add up to its lifetime.  At its end a wave adds its sections to a device table that
// rgx_debug_section_cycles() reads back.
#ifdef RGX_SECTION_CLOCKS
#define RGX_NSEC 12
enum { RGX_SEC_SWEEP = 0, RGX_SEC_FILTER = 1, RGX_SEC_SHADE = 2, RGX_SEC_LISTS = 3, RGX_SEC_BLEND = 4, RGX_SEC_SUMS = 5,
       RGX_SEC_SETUP = 6, RGX_SEC_TOP = 7, RGX_SEC_END = 8, RGX_SEC_EPILOGUE = 9, RGX_SEC_WALK = 10, RGX_SEC_FLUSH = 11 };
enum { RGX_SEC_PARSE = RGX_SEC_SWEEP, RGX_SEC_COUNT = RGX_SEC_FILTER, RGX_SEC_PRETRIP = RGX_SEC_LISTS }; // the replaying backward's names for sections it has no other use for
enum { RGX_SECK_FWD_RECORD = 0, RGX_SECK_FWD_PLAIN = 1, RGX_SECK_BWD_SUMS = 2, RGX_SECK_BWD_LISTS = 3, RGX_SECK_BWD_TREE = 4, RGX_NSECK = 5 };
#define RGX_SEC_ROWS 65536 // rows of the table: a workgroup's own up to that many (a 1920x1080 launch has 33 024), shared beyond
// [forward / backward][workgroup][section]; word RGX_NSEC of a row counts the waves that used it, the next word names their
// kernel, words 14 and 15 are the start and end of the last wave that used it on the 100 MHz wall clock.
// The sums live in memory, not in registers: the march kernels have no registers to spare, and a census that made them
// spill would time another kernel.
__device__ unsigned g_section_cycles[2][RGX_SEC_ROWS][16];
struct SectionClock {
    unsigned last = 0;
    unsigned *row = nullptr;
    __device__ __forceinline__ void start(int pass)
    {
        row = g_section_cycles[pass][blockIdx.x % RGX_SEC_ROWS]; // (a replay in pieces has more workgroups than rows)
        if (threadIdx.x == 0) row[14] = (unsigned)wall_clock64(); // when the wave started, 100 MHz ticks (the last launch's)
        last = (unsigned)__builtin_readcyclecounter();
    }
    __device__ __forceinline__ void to(int k)
    {
        const unsigned now = (unsigned)__builtin_readcyclecounter();
        if (threadIdx.x == 0) atomicAdd(row + k, now - last);
        last = now;
    }
    __device__ __forceinline__ void flush(int kernel)
    {
        if (threadIdx.x != 0) return;
        atomicAdd(row + RGX_NSEC, 1u);
        row[RGX_NSEC + 1] = (unsigned)kernel;
        row[15] = (unsigned)wall_clock64(); // and when it ended
    }
};
struct NoSectionClock {
    __device__ __forceinline__ void start(int) {}
    __device__ __forceinline__ void to(int) {}
    __device__ __forceinline__ void flush(int) {}
};
#define RGX_SEC(cn, k) (cn).clock.to(k)
#define RGX_SEC_START(cn, pass) (cn).clock.start(pass)
#define RGX_SEC_FLUSH(cn, kernel) (cn).clock.flush(kernel)
#else
#define RGX_SEC(cn, k) ((void)0)
#define RGX_SEC_START(cn, pass) ((void)0)
#define RGX_SEC_FLUSH(cn, kernel) ((void)0)
#endif

// Launch statistics (RgxStats).  Kernels launched without a statistics block carry none of it:
// the counters live in registers for the whole march, and the march has none to spare.
struct Counters {
    unsigned hit_pairs = 0, slabs = 0, empty = 0, overflow = 0, rays_hit = 0;
    unsigned long long nodes = 0;
    unsigned cands = 0, cands_hit = 0; // per wave (lane 0 counts)
    unsigned replay_lost = 0;          // per wave: the backward's replay did not consume its record exactly
    unsigned grad_atomics = 0;         // fp32 atomic adds to the gradient block in memory
#ifdef RGX_SECTION_CLOCKS
    NoSectionClock clock;              // the census is taken on the kernels without counters
#endif
};
struct NoCount { // accepts what the kernels do to a counter, keeps nothing
    template <typename T>
    __device__ __forceinline__ NoCount &operator+=(T) { return *this; }
    template <typename T>
    __device__ __forceinline__ NoCount &operator=(T) { return *this; }
    __device__ __forceinline__ NoCount &operator++() { return *this; }
    __device__ __forceinline__ NoCount &operator++(int) { return *this; }
};
struct NoCounters {
    NoCount hit_pairs, slabs, empty, overflow, rays_hit, nodes, cands, cands_hit, replay_lost, grad_atomics;
#ifdef RGX_SECTION_CLOCKS
    SectionClock clock;
#endif
};
template <bool STATS>
using CountersFor = typename std::conditional<STATS, Counters, NoCounters>::type;

// ---------------------------------------------------------------------------
// Per-lane queries through the skip links.
//
// First-hit query: optixTrace with SBT offset 0 (gaussians_aabb.cu:234-247, 300-313),
// __closesthit__ch / __miss__ms_ch (370-380).  Smallest reported t, or -1.
template <typename Cn>
__device__ float first_hit(const MarchParams &P, f3 o, f3 dir, float tlo, float thi, Cn &cn)
{
    const RayBox rb = make_raybox(o, dir, thi);
    float best = -1.0f;
    int32_t node = P.n > 0 ? 0 : -1;
    const float4 *nodes4 = (const float4 *)P.nodes;
    // a sound tree is walked in < 2n steps and never leaves [0, 2n-1); both bounds are enforced
    // so that a corrupted workspace ends the query instead of hanging or faulting the GPU
    const uint32_t n_nodes = (uint32_t)(2 * P.n - 1);
    uint32_t steps = 0;
    while ((uint32_t)node < n_nodes && steps++ < n_nodes) {
        const float4 a = nodes4[2 * node], b = nodes4[2 * node + 1];
        cn.nodes++;
        int32_t next = __float_as_int(b.w);
        if (box_overlaps(rb, a, b, tlo, thi)) {
            const int32_t left = __float_as_int(a.w);
            if (left < 0) {
                const Prim *p = P.prims + (~left);
                float r1, r2, t;
                if (line_roots(p->pos4, p->inv_inter4, p->quat4, dir, r1, r2) && segment_hit(r1, r2, tlo, thi, t)) {
                    thi = t; // OptiX shrinks the interval to the closest accepted hit
                    best = t;
                }
            } else {
                next = left;
            }
        }
        node = next;
    }
    return best;
}

struct HitList {
    int32_t *lds;   // &hits[0][lane]
    int32_t *spill; // entries beyond RGX_LDS_HITS
    __device__ __forceinline__ void put(int j, int32_t v) const
    {
        if (j < RGX_LDS_HITS) lds[j * 64] = v;
        else spill[j - RGX_LDS_HITS] = v;
    }
    __device__ __forceinline__ int32_t get(int j) const { return j < RGX_LDS_HITS ? lds[j * 64] : spill[j - RGX_LDS_HITS]; }
};

// Collect query, one ray at a time: optixTrace with SBT offset 1 + __anyhit__ah
// (gaussians_aabb.cu:282-295, 349-367).  Used by the segment test hook.
template <typename Cn>
__device__ int collect(const MarchParams &P, f3 o, f3 dir, float tlo, float thi, int cap, const HitList &hl, bool &overflow,
                       Cn &cn)
{
    const RayBox rb = make_raybox(o, dir, thi);
    int p0 = 0;
    overflow = false;
    int32_t node = P.n > 0 ? 0 : -1;
    const float4 *nodes4 = (const float4 *)P.nodes;
    const uint32_t n_nodes = (uint32_t)(2 * P.n - 1);
    uint32_t steps = 0;
    while ((uint32_t)node < n_nodes && steps++ < n_nodes) {
        const float4 a = nodes4[2 * node], b = nodes4[2 * node + 1];
        cn.nodes++;
        int32_t next = __float_as_int(b.w);
        if (box_overlaps(rb, a, b, tlo, thi)) {
            const int32_t left = __float_as_int(a.w);
            if (left < 0) {
                const Prim *p = P.prims + (~left);
                float r1, r2, t;
                if (line_roots(p->pos4, p->inv_inter4, p->quat4, dir, r1, r2) && segment_hit(r1, r2, tlo, thi, t)) {
                    if (p0 >= cap) { // optixTerminateRay at max_prim_slice (gaussians_aabb.cu:352-356)
                        overflow = true;
                        next = -1;
                    } else {
                        hl.put(p0++, ~left);
                    }
                }
            } else {
                next = left;
            }
        }
        node = next;
    }
    return p0;
}

// ---------------------------------------------------------------------------
// Tile frustum: the four planes through the eye that hold the tile's first and last pixel columns and rows
// (every pixel ray of the tile lies inside, the image-plane grid being affine) and
// the shell T0 <= |x - eye| <= T1 (ray directions are unit vectors).  pad (world
// units) covers the rounding of the exact predicate and of these tests.
struct Frustum {
    f3 o;
    f3 n[4]; // unit normals pointing out of the frustum
    f3 dc;       // the tile's central direction
    float delta; // no ray of the tile is further than this angle from dc
    float t0, t1, pad;
    float near2, far2; // frustum_misses: bounds on the squares of twice the distance to a box's furthest and of that to its nearest point
    __device__ __forceinline__ void range(float from, float to, float padding)
    {
        t0 = from;
        t1 = to;
        pad = padding;
        const float near_t = t0 - pad, far_t = t1 + pad;
        near2 = near_t > 0.f ? near_t * near_t * (4.0f * 0.9999f) : -1.0f;
        far2 = far_t * far_t * 1.0001f;
    }
    int32_t cut_node; // per lane: one node of the tile's cut through the tree (frustum_cut, frustum_cut_pairs), or -1
    int cut_n;        // nodes in the cut (wave-uniform); 0: sweeps start at the root
    int cut_inner;    // (frustum_cut_pairs) so many of them, the first ones, are internal nodes; the others are leaves
};

__device__ __forceinline__ f3 cross3(f3 a, f3 b) { return mk3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x); }

__device__ __forceinline__ f3 plane_normal(f3 a, f3 b, f3 inside)
{
    f3 n = cross3(a, b);
    n = n * (1.0f / sqrtf(fmaxf(dot3(n, n), 1e-30f)));
    return dot3(n, inside) > 0.f ? n * -1.0f : n;
}

// width, height: in pixels (of a tile, or of the part of one that a wavefront marches).
// The rays of a pixel column lie in the plane of v and w + x u, those of a row in that of u and w + y v: a plane spanned by two such vectors, nearly at right
// angles, has a normal good to a few ulps, however few and narrow the pixels.  (Spanned by two rays its error is theirs over the angle between them: of a 4x2 part's,
// one pixel apart, 1e-4 of the distance with 220 pixels across 5 degrees, where pad is 1.6e-5, and Gaussians that a ray only grazed were lost.)
__device__ __forceinline__ void frustum_planes(const RgxCamera &cam, int px0, int py0, Frustum &F, int width = 8, int height = 8)
{
    const f3 d00 = compute_ray(cam, (unsigned)px0, (unsigned)py0), d10 = compute_ray(cam, (unsigned)(px0 + width - 1), (unsigned)py0);
    const f3 d01 = compute_ray(cam, (unsigned)px0, (unsigned)(py0 + height - 1));
    const f3 d11 = compute_ray(cam, (unsigned)(px0 + width - 1), (unsigned)(py0 + height - 1));
    const f3 in = (d00 + d10) + (d01 + d11);
    const f3 u = mk3(cam.u[0], cam.u[1], cam.u[2]), v = mk3(cam.v[0], cam.v[1], cam.v[2]), w = mk3(cam.w[0], cam.w[1], cam.w[2]);
    const float x0 = column_x(cam, (unsigned)px0), x1 = column_x(cam, (unsigned)(px0 + width - 1));
    const float y0 = row_y(cam, (unsigned)py0), y1 = row_y(cam, (unsigned)(py0 + height - 1));
    const f3 right = u * (x1 - x0), down = v * (y1 - y0); // from one edge to the other
    F.o = mk3(cam.eye[0], cam.eye[1], cam.eye[2]);
    F.n[0] = plane_normal(w + u * x0, v, right);
    F.n[1] = plane_normal(w + u * x1, v, right * -1.0f);
    F.n[2] = plane_normal(w + v * y0, u, down);
    F.n[3] = plane_normal(w + v * y1, u, down * -1.0f);
    F.dc = in * (1.0f / sqrtf(dot3(in, in)));
    // the rays' directions lie, before normalisation, in a plane quadrilateral with these four as
    // corners, so the largest angle to dc is at a corner; |d - dc| = 2 sin(angle / 2)
    const f3 e00 = d00 - F.dc, e10 = d10 - F.dc, e01 = d01 - F.dc, e11 = d11 - F.dc;
    F.delta = 1.02f * sqrtf(fmaxf(fmaxf(dot3(e00, e00), dot3(e10, e10)), fmaxf(dot3(e01, e01), dot3(e11, e11)))) + 1e-6f;
    // the planes are the same in every lane: keep them in scalar registers
    auto uni = [](float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); };
    F.o = mk3(uni(F.o.x), uni(F.o.y), uni(F.o.z));
    F.dc = mk3(uni(F.dc.x), uni(F.dc.y), uni(F.dc.z));
    F.delta = uni(F.delta);
    F.cut_node = -1;
    F.cut_n = F.cut_inner = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) F.n[k] = mk3(uni(F.n[k].x), uni(F.n[k].y), uni(F.n[k].z));
}

// Whether the box [a, b] may meet the frustum: in twice its centre c and extent e from the eye, plane k's distance to the
// corner furthest inside is n.c - |n|.e, six multiply-adds and no select per axis (a step of the descent costs a
// third less than with the corner picked by the normal's signs, and 24 scalar registers of those signs are free).  A large
// box's near corner comes out of large terms: e is widened by more than their rounding (16 ulps).
__device__ __forceinline__ bool frustum_misses(const Frustum &F, float4 a, float4 b)
{
    const f3 lo = mk3(a.x - F.o.x, a.y - F.o.y, a.z - F.o.z), hi = mk3(b.x - F.o.x, b.y - F.o.y, b.z - F.o.z);
    const f3 c = lo + hi, e = (hi - lo) * (1.0f + 0x1p-19f);
    float d[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const f3 n = F.n[k];
        d[k] = fmaf(n.x, c.x, fmaf(-fabsf(n.x), e.x, fmaf(n.y, c.y, fmaf(-fabsf(n.y), e.y, fmaf(n.z, c.z, -fabsf(n.z) * e.z)))));
    }
    // distance shell (dmax: of twice the furthest corner)
    const float nx = fmaxf(fmaxf(lo.x, -hi.x), 0.f), ny = fmaxf(fmaxf(lo.y, -hi.y), 0.f), nz = fmaxf(fmaxf(lo.z, -hi.z), 0.f);
    const float fx = fabsf(c.x) + e.x, fy = fabsf(c.y) + e.y, fz = fabsf(c.z) + e.z;
    const float dmin2 = fmaf(nx, nx, fmaf(ny, ny, nz * nz)), dmax2 = fmaf(fx, fx, fmaf(fy, fy, fz * fz));
    return (fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3])) > 2.0f * F.pad) | (dmax2 < F.near2) | (dmin2 > F.far2);
}

// The same of a box given as twice its centre and twice its half extents (NodePair): nine instructions fewer.
__device__ __forceinline__ bool frustum_misses_pair(const Frustum &F, f3 c, f3 e)
{
    c = mk3(fmaf(-2.0f, F.o.x, c.x), fmaf(-2.0f, F.o.y, c.y), fmaf(-2.0f, F.o.z, c.z));
    float d[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const f3 n = F.n[k];
        d[k] = fmaf(n.x, c.x, fmaf(-fabsf(n.x), e.x, fmaf(n.y, c.y, fmaf(-fabsf(n.y), e.y, fmaf(n.z, c.z, -fabsf(n.z) * e.z)))));
    }
    const float nx = fmaxf(fabsf(c.x) - e.x, 0.f), ny = fmaxf(fabsf(c.y) - e.y, 0.f), nz = fmaxf(fabsf(c.z) - e.z, 0.f);
    const float fx = fabsf(c.x) + e.x, fy = fabsf(c.y) + e.y, fz = fabsf(c.z) + e.z;
    const float dmin2 = fmaf(nx, nx, fmaf(ny, ny, nz * nz)), dmax2 = fmaf(fx, fx, fmaf(fy, fy, fz * fz)); // of twice the distances
    return (fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3])) > 2.0f * F.pad) | (dmax2 < F.near2) | (dmin2 > 4.0f * F.far2);
}

// Candidate table.  A Gaussian that survives the sweep is turned, by the lane that found
// it, into everything the per-ray work needs and parked in LDS, where all lanes later read
// it as a broadcast: rotation columns, the ray-independent half of the hit predicate
// (S^-1 R^T (eye - centre) and its squared norm - 1), and the distance shell [dmin, dmax]
// from the eye that bounds the ellipsoid.  The values are produced by the same operations,
// in the same order, as in line_roots(), so using them changes no rounding.
//   U.xyz V.xyz W.xyz inv_inter.xyz | Oe.xyz, sorted index | dmin, dmax, k, c
// in this order without gaps: the filter reads the first sixteen words, as four LDS reads and without holes in the
// registers they land in (three words of a quadruple take four).
// (80 bytes, sized so that 12 wavefronts' tables fit one CU's LDS; what only the shading of an
// actual hit needs -- eye - centre and the colour -- is read from the primitive record.)
#define RGX_TAB 20
enum { RGX_TAB_PID = 15, RGX_TAB_DMIN = 16, RGX_TAB_DMAX = 17, RGX_TAB_K = 18, RGX_TAB_C = 19 };
__device__ __forceinline__ void table_store(float4 *e, f3 U, f3 V, f3 W, f3 inv, f3 Oe, int32_t pid, float dmin, float dmax, float k, float c)
{
    e[0] = make_float4(U.x, U.y, U.z, V.x);
    e[1] = make_float4(V.y, V.z, W.x, W.y);
    e[2] = make_float4(W.z, inv.x, inv.y, inv.z);
    e[3] = make_float4(Oe.x, Oe.y, Oe.z, __int_as_float(pid));
    e[4] = make_float4(dmin, dmax, k, c);
}
__device__ __forceinline__ void table_frame(const float4 *e, f3 &U, f3 &V, f3 &W, f3 &inv)
{
    const float4 a = e[0], b = e[1], c = e[2];
    U = mk3(a.x, a.y, a.z);
    V = mk3(a.w, b.x, b.y);
    W = mk3(b.z, b.w, c.x);
    inv = mk3(c.y, c.z, c.w);
}

// Cooperative sweep of the BVH: the node stack is shared by the wave, every step pops up to
// 64 nodes (one per lane) and tests their boxes against the frustum.  Internal nodes that pass
// push their children.  A leaf that passes is tested again with its actual ellipsoid -- exact
// support distance against the four frustum planes, bounding sphere against the shell -- and,
// if it still passes, written to the candidate table.  Returns the number of table entries
// when the stack is empty (done) or the table might not take another step's leaves; call again
// to continue with an emptied table.
// Correctly rounded a / b and sqrt(x) for operands of ordinary size: the instruction sequences the
// compiler emits for `/` and sqrtf(), without their range handling (v_div_scale / v_div_fixup,
// the 2^32 pre-scaling of small sqrt arguments, the special-value checks).  Where that handling
// would do nothing -- b and a / b far from the ends of the exponent range, |a| >= 2^-104,
// 2^-96 <= x < infinity -- the results are bit-identical to `/` and sqrtf().  (Kept for rgx_check_plain_arith: no kernel takes roots where
// their cost shows.)
__device__ __forceinline__ float div_rn_plain(float a, float b)
{
    float r = __builtin_amdgcn_rcpf(b);
    r = fmaf(fmaf(-b, r, 1.0f), r, r);
    float q = a * r;
    q = fmaf(fmaf(-b, q, a), r, q);
    return fmaf(fmaf(-b, q, a), r, q);
}
__device__ __forceinline__ float sqrt_rn_plain(float x)
{
    const float y = __builtin_amdgcn_sqrtf(x); // within one ulp: the answer is y or a neighbour
    const float down = __int_as_float(__float_as_int(y) - 1), up = __int_as_float(__float_as_int(y) + 1);
    const float r_down = fmaf(-down, y, x), r_up = fmaf(-up, y, x);
    const float z = r_down <= 0.0f ? down : y;
    return r_up > 0.0f ? up : z;
}

// Whether every ray through a Gaussian has a quadratic of ordinary size, which the filter's margin is derived for, and the plain forms' range: inv = (1 / scale) / k per axis, c = |S^-1 R^T (eye - centre)|^2 - 1.
// For a unit direction a = |De|^2 lies in [min inv^2, max inv^2]; where the line hits
// (disc > 1e-7) disc * a >= 1e-7 min inv^2 and |q| lies in [sqrt(1e-7) min inv, (sqrt(c + 1) + 1) max inv].
__device__ __forceinline__ bool plain_roots(f3 inv, float c)
{
    const float lo = fminf(inv.x, fminf(inv.y, inv.z)), hi = fmaxf(inv.x, fmaxf(inv.y, inv.z));
    return lo >= 0x1p-23f && hi <= 0x1p22f && fabsf(c) >= 0x1p-46f && fabsf(c) <= 0x1p46f;
}

// how many of the mask's lanes come before this one
__device__ __forceinline__ int rank_in(uint64_t mask)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

struct Sweep {
    int qn;  // stack entries (wave-uniform)
    int lqn; // leaves waiting for their ellipsoid test (wave-uniform)
};

// The orders in which a sweep can find a tile's Gaussians.  Where max_prim_slice cuts a ray's list the order decides which hits are
// kept, so a backward that has to search the tree for a tile takes the order of the forward that wrote the tile's record.
//   BY_NODES  up to 64 nodes a step; where nothing speaks for another
//   BY_PAIRS  the children of up to 64 nodes a step
enum { BY_NODES, BY_PAIRS };

template <int ORDER>
__device__ __forceinline__ void sweep_begin(const MarchParams &P, Sweep &S, const Frustum &F, int32_t *s_queue, int32_t *s_leafq)
{
    S.lqn = 0;
    if constexpr (ORDER == BY_PAIRS) {
        S.qn = F.cut_inner;
        S.lqn = F.cut_n - F.cut_inner;
        const int lane = threadIdx.x;
        if (lane < F.cut_n) *(lane < F.cut_inner ? s_queue + lane : s_leafq + (lane - F.cut_inner)) = F.cut_node;
    } else if (F.cut_n > 0) {
        S.qn = F.cut_n;
        if ((int)threadIdx.x < F.cut_n) s_queue[threadIdx.x] = F.cut_node;
    } else {
        S.qn = P.n > 0 ? 1 : 0;
        if (threadIdx.x == 0) s_queue[0] = 0;
    }
    __syncthreads();
}

// A leaf's ellipsoid against the frustum, and the range of distances from the eye that bounds it along the tile's rays.
// (Bounds only: hardware reciprocal and square root and multiply-adds, their last-bit errors are inside the 1.001 factors.)
__device__ __forceinline__ bool leaf_meets(const Frustum &F, const Prim &p, f3 U, f3 V, f3 W, float &dmin, float &dmax)
{
    auto dot = [](f3 a, f3 b) { return fmaf(a.x, b.x, fmaf(a.y, b.y, a.z * b.z)); };
    const f3 O = mk3(p.pos4.x, p.pos4.y, p.pos4.z);
    // semi-axes of the k-sigma ellipsoid: k * scale = 1 / inv_inter
    const f3 ax = mk3(__builtin_amdgcn_rcpf(p.inv_inter4.x), __builtin_amdgcn_rcpf(p.inv_inter4.y), __builtin_amdgcn_rcpf(p.inv_inter4.z));
    // how far the ellipsoid reaches beyond its centre along n
    auto extent = [&](f3 n) {
        const float a = dot(U, n) * ax.x, b = dot(V, n) * ax.y, c = dot(W, n) * ax.z;
        return __builtin_amdgcn_sqrtf(fmaf(a, a, fmaf(b, b, c * c))) * 1.001f;
    };
    const float dist = __builtin_amdgcn_sqrtf(dot(O, O));
    const float amax = fmaxf(ax.x, fmaxf(ax.y, ax.z));
    const float rad = amax * 1.001f + 1e-5f * dist + F.pad;
    // Along a ray of direction d the ellipsoid lies within (centre - eye).d -+ |A R^T d|.  For
    // d = dc that is depth -+ h; a ray at angle <= delta from dc moves the centre term by at
    // most |depth| delta^2 / 2 + |offset of the centre from the central ray| delta and the
    // extent by at most amax delta.  The bounding sphere's shell bounds the same range.
    const float depth = -dot(O, F.dc);
    const f3 off = mk3(fmaf(depth, F.dc.x, O.x), fmaf(depth, F.dc.y, O.y), fmaf(depth, F.dc.z, O.z));
    const float ext = extent(F.dc);
    const float slack = 1.5f * (0.5f * fabsf(depth) * F.delta * F.delta + (__builtin_amdgcn_sqrtf(dot(off, off)) + amax) * F.delta) +
                        1e-5f * dist + F.pad;
    dmin = fmaxf(dist - rad, depth - ext - slack);
    dmax = fminf(dist + rad, depth + ext + slack);
    bool ok = (p.inv_inter4.w == p.inv_inter4.w) & (dmax >= F.t0) & (dmin <= F.t1); // k is NaN below the density threshold: never hit
#pragma unroll
    for (int k = 0; k < 4; ++k) ok = ok & !(-dot(F.n[k], O) - extent(F.n[k]) > F.pad); // centre - eye = -O
    return ok;
}

// The tile's cut through the tree.  Every sweep of a tile tests the same top of the tree against the
// same four planes -- a dozen steps of one to a few dozen nodes, each waiting on memory.  Done once
// instead: descend from the root, level by level, keeping the nodes that meet the frustum at any
// depth, until the next level would not fit one node per lane; the sweeps then start from those
// nodes.  t_far: the largest distance any sweep of this tile will ask for (sets the planes' pad).
__device__ __forceinline__ void frustum_cut(const MarchParams &P, Frustum &F, float t_far, int32_t *s_queue)
{
    const int lane = threadIdx.x;
    const uint64_t lt = (1ull << lane) - 1ull;
    const float4 *nodes4 = (const float4 *)P.nodes;
    const uint32_t n_nodes = (uint32_t)(2 * P.n - 1);
    F.range(0.f, INFINITY, 2.0f * RGX_PAD_REL * fmaxf(t_far, 1.0f)); // no distance shell
    int32_t node = lane == 0 && P.n > 0 ? 0 : -1;
    int count = P.n > 0 ? 1 : 0;
    for (int level = 0; level < 64 && count > 0; ++level) {
        bool keep = false, inner = false;
        int32_t left = 0, right = 0;
        if ((uint32_t)node < n_nodes) {
            const float4 a = nodes4[2 * node], b = nodes4[2 * node + 1];
            right = P.right[max(0, min(node, (int32_t)P.n - 2))]; // with the box, not after the test (n = 1: no internal node, word 0 of the padded array)
            if (!frustum_misses(F, a, b)) {
                left = __float_as_int(a.w);
                inner = left >= 0;
                keep = !inner;
            }
        }
        const uint64_t bk = __ballot(keep), bi = __ballot(inner);
        const int next = __popcll(bk) + 2 * __popcll(bi);
        if (bi == 0 || next > 64) break; // nothing to open, or the next level does not fit: keep this one
        // next level: the leaves kept, then the children of the inner nodes
        if (keep) s_queue[__popcll(bk & lt)] = node;
        if (inner) {
            const int at = __popcll(bk) + 2 * __popcll(bi & lt);
            s_queue[at] = left;
            s_queue[at + 1] = right;
        }
        __syncthreads();
        node = lane < next ? s_queue[lane] : -1;
        count = next;
        __syncthreads();
    }
    // nodes that failed the planes in the last round stay in the cut: the sweeps test them again
    F.cut_n = count;
    const uint64_t have = __ballot((uint32_t)node < n_nodes);
    F.cut_node = node;
    if (have != (count >= 64 ? ~0ull : ((1ull << count) - 1ull))) F.cut_n = 0; // (cannot happen) fall back to the root
}

// The same with a node's two children at a time (NodePair): what is in the cut has passed the test itself.  Entries >= 0 are
// internal nodes, they come first; the others are ~leaf.
__device__ __forceinline__ void frustum_cut_pairs(const MarchParams &P, Frustum &F, float t_far, int32_t *s_queue)
{
    const int lane = threadIdx.x;
    F.range(0.f, INFINITY, 2.0f * RGX_PAD_REL * fmaxf(t_far, 1.0f)); // no distance shell
    int32_t node = P.n == 1 ? ~0 : 0;
    int inner_n = P.n > 1 ? 1 : 0, count = P.n > 0 ? 1 : 0;
    for (int level = 0; level < 96 && inner_n > 0; ++level) {
        const bool open = lane < inner_n;
        const float4 *q = P.pairs + 4 * (int64_t)(open ? min(node, (int32_t)P.n - 2) : 0);
        const float4 a = q[0], b = q[1], c = q[2], d = q[3];
        const int32_t left = __float_as_int(a.w), right = __float_as_int(b.w);
        const uint64_t here = __ballot(open);
        const uint64_t p0 = here & ~__ballot(frustum_misses_pair(F, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z)));
        const uint64_t p1 = here & ~__ballot(frustum_misses_pair(F, mk3(c.x, c.y, c.z), mk3(d.x, d.y, d.z)));
        const uint64_t l0 = __ballot(left < 0), l1 = __ballot(right < 0);
        const int inners = __popcll(p0 & ~l0) + __popcll(p1 & ~l1), leaves = __popcll(p0 & l0) + __popcll(p1 & l1) + count - inner_n;
        if (inners + leaves > 64) break; // the next level does not fit: keep this one
        // next level: inner children, then leaves (those there were already last)
        const int left_inner = __popcll(p0 & ~l0), left_leaf = __popcll(p0 & l0), right_leaf = __popcll(p1 & l1);
        if (__builtin_amdgcn_inverse_ballot_w64(p0)) s_queue[left < 0 ? inners + rank_in(p0 & l0) : rank_in(p0 & ~l0)] = left;
        if (__builtin_amdgcn_inverse_ballot_w64(p1)) s_queue[right < 0 ? inners + left_leaf + rank_in(p1 & l1) : left_inner + rank_in(p1 & ~l1)] = right;
        if (lane >= inner_n && lane < count) s_queue[inners + left_leaf + right_leaf + lane - inner_n] = node;
        __syncthreads();
        count = inners + leaves;
        inner_n = inners;
        node = lane < count ? s_queue[lane] : 0;
        __syncthreads();
    }
    F.cut_n = count;
    F.cut_inner = inner_n;
    F.cut_node = node;
}

template <int ORDER, bool AGAIN, typename Cn>
__device__ __forceinline__ int sweep_next(const MarchParams &P, Sweep &S, const Frustum &F, int32_t *s_queue, int32_t *s_leafq, float *s_tab,
                          bool &done, bool &plain, Cn &cn)
{
    constexpr bool PAIRS = ORDER == BY_PAIRS;
    plain = true;
    const int lane = threadIdx.x;
    const float4 *nodes4 = (const float4 *)P.nodes;
    const uint32_t n_nodes = (uint32_t)(2 * P.n - 1);
    int C = 0;
    const MarchParams *again = &P;
    while (C < RGX_CCAP) {
        if constexpr (AGAIN) again = &args_again();
        while (S.qn > 0 && S.lqn < 64) {
            // A step of the descent: up to 64 nodes, one per lane.  (Lanes beyond them repeat the last one, and their results are
            // masked: straight-line code.  The wavefront's LDS accesses take place in program order.)
            const int m = S.qn > RGX_QCAP - RGX_DFS_MARGIN ? 1 : (S.qn < 64 ? S.qn : 64);
            const int base = S.qn - m;
            if constexpr (PAIRS) {
                const MarchParams &A = AGAIN ? *again : P;
                const int32_t top = (int32_t)A.n - 2; // the last internal node (with fewer than two Gaussians the stack stays empty)
                const uint32_t popped = (uint32_t)s_queue[base + min(lane, m - 1)], node = min(popped, (uint32_t)top);
                __builtin_amdgcn_wave_barrier();
                const float4 *q = (const float4 *)((const char *)A.pairs + ((uint64_t)node << 6));
                const float4 a = q[0], b = q[1], c = q[2], d = q[3];
                const int32_t left = __float_as_int(a.w), right = __float_as_int(b.w);
                const uint64_t here = (~0ull >> (64 - m)) & __ballot(popped <= (uint32_t)top);
                const uint64_t p0 = here & ~__ballot(frustum_misses_pair(F, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z)));
                const uint64_t p1 = here & ~__ballot(frustum_misses_pair(F, mk3(c.x, c.y, c.z), mk3(d.x, d.y, d.z)));
                const uint64_t l0 = __ballot(left < 0), l1 = __ballot(right < 0);
                if (lane == 0) cn.nodes += 2u * (unsigned)m;
                // fewer than 64 leaves waiting + at most 128 new <= 192
                if (__builtin_amdgcn_inverse_ballot_w64(p0 & l0)) s_leafq[S.lqn + rank_in(p0 & l0)] = left;
                S.lqn += __popcll(p0 & l0);
                if (__builtin_amdgcn_inverse_ballot_w64(p1 & l1)) s_leafq[S.lqn + rank_in(p1 & l1)] = right;
                S.lqn += __popcll(p1 & l1);
                const uint64_t i0 = p0 & ~l0, i1 = p1 & ~l1;
                const int rights = __popcll(i1), pushed = rights + __popcll(i0);
                if (__builtin_expect(base + pushed <= RGX_QCAP, 1)) {
                    const int lefts = pushed - rights;
                    if (__builtin_amdgcn_inverse_ballot_w64(i0)) s_queue[base + rank_in(i0)] = left;
                    if (__builtin_amdgcn_inverse_ballot_w64(i1)) s_queue[base + lefts + rank_in(i1)] = right;
                    S.qn = base + pushed;
                } else { // cannot happen (see RGX_DFS_MARGIN); if it did, the drop is counted, not silent
                    S.qn = base;
                    if (lane == 0 && P.faults) atomicAdd(&P.faults[1], (uint32_t)pushed);
                }
                __builtin_amdgcn_wave_barrier();
                continue;
            }
            const uint32_t popped = (uint32_t)s_queue[base + min(lane, m - 1)], node = min(popped, n_nodes - 1u);
            __builtin_amdgcn_wave_barrier();
            const float4 *box = (const float4 *)((const char *)nodes4 + ((uint64_t)node << 5));
            const float4 a = box[0], b = box[1];
            // the right child is fetched along with the box, not after the test: one memory round trip per step, not two
            const int32_t right = P.right[min(node, (uint32_t)max((int32_t)P.n - 2, 0))]; // (a leaf has none)
            const int32_t left = __float_as_int(a.w);
            const uint64_t pass = (~0ull >> (64 - m)) & ~__ballot(frustum_misses(F, a, b)) & __ballot(popped < n_nodes);
            const uint64_t leaves = pass & __ballot(left < 0), inner = pass & ~leaves;
            if (lane == 0) cn.nodes += (unsigned)m;
            if (__builtin_amdgcn_inverse_ballot_w64(leaves)) s_leafq[S.lqn + rank_in(leaves)] = left; // fewer than 64 waiting + at most 64 new <= 128
            S.lqn += __popcll(leaves);
            S.qn = base + 2 * __popcll(inner);
            if (__builtin_expect(S.qn <= RGX_QCAP, 1)) {
                if (__builtin_amdgcn_inverse_ballot_w64(inner)) {
                    const int pos = base + 2 * rank_in(inner);
                    s_queue[pos] = right;
                    s_queue[pos + 1] = left;
                }
            } else { // cannot happen (see RGX_DFS_MARGIN); if it did, the drop is counted, not silent
                S.qn = base;
                if (lane == 0 && P.faults) atomicAdd(&P.faults[1], (uint32_t)__popcll(inner));
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (S.lqn == 0) break;
        // Leaves whose boxes passed wait in a queue until there are 64 of them (or no node is
        // left): the expensive part -- fetch the Gaussian, test its ellipsoid, build its table
        // entry -- then runs with every lane busy, not with the few leaves one step turns up.
        const int m = S.lqn < 64 ? S.lqn : 64;
        S.lqn -= m;
        const int32_t left = s_leafq[S.lqn + min(lane, m - 1)]; // (as in a step of the descent)
        const Prim p = P.prims[(uint32_t)~left];
        f3 U, V, W;
        quat_to_cols(p.quat4, U, V, W);
        float dmin, dmax;
        uint64_t hits = (~0ull >> (64 - m)) & __ballot(leaf_meets(F, p, U, V, W, dmin, dmax));
        const int rank = rank_in(hits), room = RGX_CCAP - C;
        if (__popcll(hits) > room) {
            // the table takes what it has room for; the rest goes back to the queue for the next table
            const uint64_t back = hits & __ballot(rank >= room);
            if (__builtin_amdgcn_inverse_ballot_w64(back)) s_leafq[S.lqn + rank - room] = left;
            S.lqn += __popcll(back);
            hits &= ~back;
        }
        const f3 inv = mk3(p.inv_inter4.x, p.inv_inter4.y, p.inv_inter4.z);
        const f3 Oe = apply_sinv_rt(mk3(p.pos4.x, p.pos4.y, p.pos4.z), U, V, W, inv);
        const float c = fmaf(Oe.x, Oe.x, fmaf(Oe.y, Oe.y, fmaf(Oe.z, Oe.z, -1.0f)));
        if (__builtin_amdgcn_inverse_ballot_w64(hits)) {
            table_store((float4 *)(s_tab + (C + rank) * RGX_TAB), U, V, W, inv, Oe, ~left, dmin, dmax, p.inv_inter4.w, c);
        }
        plain = plain && (hits & ~__ballot(plain_roots(inv, c))) == 0;
        C += __popcll(hits);
        __syncthreads();
    }
    done = S.qn == 0 && S.lqn == 0;
    return C;
}

// Workgroups are dealt round-robin to the 8 XCDs (workgroup i runs on XCD i % 8), each with its
// own L2.  The image is cut into square blocks of tiles and the blocks are dealt to the XCDs in
// turn: an XCD works through adjacent tiles, so its L2 sees one region of the scene at a time, and
// every XCD gets blocks from all over the image, so the expensive middle of a scene is not one
// XCD's alone.  Blocks are 8 x 8 tiles where that still leaves every XCD some 32 blocks, else
// 4 x 4.  The number of blocks per row of blocks is kept odd (by a phantom block column if need
// be): with an even count the same few block columns would go to the same XCD in every row.
struct TileGrid {
    int bw, bh, blocks_x, per_xcd; // block width (clipped to the image) and height in tiles, blocks per row of blocks, blocks per XCD
};
__host__ __device__ __forceinline__ TileGrid tile_grid(int tiles_x, int tiles_y)
{
    TileGrid g;
    g.bh = ((tiles_x + 7) / 8) * ((tiles_y + 7) / 8) >= 256 ? 8 : 4;
    g.bw = tiles_x < g.bh ? tiles_x : g.bh;
    g.blocks_x = ((tiles_x + g.bw - 1) / g.bw) | 1;
    const int blocks_y = (tiles_y + g.bh - 1) / g.bh;
    g.per_xcd = (g.blocks_x * blocks_y + 7) >> 3;
    return g;
}
__device__ __forceinline__ bool tile_origin(const MarchParams &P, unsigned id, int &px0, int &py0, int *tile_out = nullptr, int part_bits = 0, int *part = nullptr)
{
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    const int xcd = id & 7;
    const int per_block = g.bw * g.bh;
    int j = id >> 3;
    if (part) {
        *part = j & ((1 << part_bits) - 1);
        j >>= part_bits;
    }
    int block;
    if (P.use_tile_order == 2) {
        block = (int)P.tile_order[xcd * g.per_xcd + j / per_block];
    } else {
        if (P.use_tile_order) j = (int)P.tile_order[xcd * (g.per_xcd * per_block) + j];
        block = xcd + 8 * (j / per_block);
    }
    const int within = j % per_block;
    const int tx = (block % g.blocks_x) * g.bw + within % g.bw;
    const int ty = (block / g.blocks_x) * g.bh + within / g.bw;
    px0 = tx * 8;
    py0 = ty * 8;
    if (tile_out) *tile_out = ty * P.tiles_x + tx;
    return tx < P.tiles_x && ty < P.tiles_y;
}

__device__ __forceinline__ void flush_stats(RgxStats *, const NoCounters &) {}
__device__ __forceinline__ void flush_stats(RgxStats *st, const Counters &c)
{
    if (!st) return;
    unsigned long long v[10] = {c.hit_pairs, c.slabs, c.empty, c.overflow, c.rays_hit, c.nodes, c.cands, c.cands_hit, c.replay_lost,
                                c.grad_atomics};
    for (int k = 0; k < 10; ++k) {
        unsigned long long x = v[k];
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
        v[k] = x;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&st->hit_pairs, v[0]); atomicAdd(&st->slabs, v[1]); atomicAdd(&st->empty_slabs, v[2]);
        atomicAdd(&st->overflow_rays, v[3]); atomicAdd(&st->rays_hit, v[4]); atomicAdd(&st->nodes_visited, v[5]);
        atomicAdd(&st->candidates, v[6]); atomicAdd(&st->candidates_hit, v[7]);
        if (v[8]) atomicAdd(&st->replay_lost, v[8]);
        if (v[9]) atomicAdd(&st->grad_atomics, v[9]);
    }
}

// State of one ray between slab iterations; the slab loop itself is wave-uniform.
// A ray is either marching (its next slab is [tbuffer, tbuffer + 32 dt]) or searching:
// looking for the first Gaussian at or after tbuffer -- the reference's first-hit query
// (optixTrace SBT offset 0), issued once per ray (gaussians_aabb.cu:234-257) and after
// every empty slab (297-319).  The search runs on the same candidate tables as the slabs,
// one window per iteration: if no Gaussian of the window is hit at or after tbuffer, every
// hit lies beyond the window, so searching on from the window's end returns the same
// closest t as one query over [tbuffer, texit] would.
struct RayState {
    f3 dir;
    float tenter, texit, tbuffer, T, dt, slab_spacing;
    bool active, searching, first;
};

// Ray set-up: computeRay and the scene-bbox slab test (fwd: gaussians_aabb.cu:207-231;
// bwd: backward/gaussians_aabb.cu:211-233, which divides by the direction where the forward
// multiplies by its reciprocal).  The ray starts out searching from the box entry.
__device__ __forceinline__ void ray_begin(const MarchParams &P, int px, int py, bool valid, bool divide, RayState &R)
{
    const f3 o = mk3(P.cam.eye[0], P.cam.eye[1], P.cam.eye[2]);
    R.dir = compute_ray(P.cam, (unsigned)px, (unsigned)py);
    const float *bmn = P.hdr->bb_min, *bmx = P.hdr->bb_max;
    float t0x, t1x, t0y, t1y, t0z, t1z;
    if (divide) {
        t0x = (bmn[0] - o.x) / R.dir.x; t1x = (bmx[0] - o.x) / R.dir.x;
        t0y = (bmn[1] - o.y) / R.dir.y; t1y = (bmx[1] - o.y) / R.dir.y;
        t0z = (bmn[2] - o.z) / R.dir.z; t1z = (bmx[2] - o.z) / R.dir.z;
    } else {
        const f3 inv = mk3(1.0f / R.dir.x, 1.0f / R.dir.y, 1.0f / R.dir.z);
        t0x = (bmn[0] - o.x) * inv.x; t1x = (bmx[0] - o.x) * inv.x;
        t0y = (bmn[1] - o.y) * inv.y; t1y = (bmx[1] - o.y) * inv.y;
        t0z = (bmn[2] - o.z) * inv.z; t1z = (bmx[2] - o.z) * inv.z;
    }
    R.tenter = fmaxf(0.0f, fmaxf(fminf(t0x, t1x), fmaxf(fminf(t0y, t1y), fminf(t0z, t1z))));
    R.texit = fminf(fmaxf(t0x, t1x), fminf(fmaxf(t0y, t1y), fmaxf(t0z, t1z)));
    R.dt = P.m.dt_step;
    R.slab_spacing = R.dt * RGX_BUFFER_SIZE;
    R.T = 1.0f;
    R.tbuffer = R.tenter;
    R.searching = true;
    R.first = true;
    // a first hit can only be reported inside [tenter, texit]; with tenter >= texit the ray keeps
    // the background either way (gaussians_aabb.cu:249-260, 333-339)
    R.active = valid && P.n > 0 && R.tenter < R.texit;
}

// Top of an iteration: loop condition, adaptive step (gaussians_aabb.cu:266-276) and the interval
// this ray asks about: its slab when marching (returns true), or one slab length ahead of tbuffer
// when searching (returns false; the search itself runs to the end of the candidate window).
// clip: the forward clips the slab to [tenter, texit] (275-276), the backward does not (279-280).  t_floor: t_eps.
__device__ __forceinline__ bool slab_begin(const MarchParams &P, bool clip, float t_floor, RayState &R, float &tlo, float &thi)
{
    R.active = R.active && R.tbuffer < R.texit && R.T > t_floor;
    // a step below one ulp of t cannot advance the ray: stop instead of spinning
    R.active = R.active && (R.tbuffer + R.slab_spacing > R.tbuffer);
    if (R.active && !R.searching && P.m.dynamic_sampling) {
        const float dt_dist = fmaxf(R.tbuffer / 1024.0f, P.m.dt_step);
        const float coeff = rcbrtf(R.T);
        R.dt = fminf(dt_dist * coeff, 4.0f * P.m.dt_step);
        R.slab_spacing = R.dt * RGX_BUFFER_SIZE;
    }
    if (R.searching) {
        tlo = R.tbuffer;
        thi = fminf(R.texit, R.tbuffer + R.slab_spacing);
        return false;
    }
    tlo = clip ? fmaxf(R.tenter, R.tbuffer) : R.tbuffer;
    thi = clip ? fminf(R.texit, R.tbuffer + R.slab_spacing) : R.tbuffer + R.slab_spacing;
    return R.active && thi > R.tenter;
}

// End of an iteration.  Marching ray: step to the next slab; after an empty slab start searching
// from there (gaussians_aabb.cu:297-319, 324).  Searching ray: `found` (< 0: nothing in
// [tbuffer, searched_to]) either restarts the march at the hit or moves the search on.
template <typename Cn>
__device__ __forceinline__ void slab_end(RayState &R, bool need, int p0, float found, float searched_to, Cn &cn)
{
    if (!R.active) return;
    if (R.searching) {
        if (found >= 0.0f) {
            if (R.first) {
                R.first = false;
                cn.rays_hit++;
                R.tenter = found;
                R.active = found < R.texit;
            }
            R.tbuffer = found;
            R.searching = false;
        } else {
            R.tbuffer = searched_to;
            R.active = searched_to < R.texit;
        }
        return;
    }
    R.tbuffer += R.slab_spacing;
    if (need && p0 == 0) {
        cn.empty++;
        R.searching = true;
    }
}

// OR over the 16 lanes of each row, left in every lane of the row
__device__ __forceinline__ uint32_t row_or(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false); // row_half_mirror
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false); // row_mirror
    return v;
}

// ---------------------------------------------------------------------------
struct TileLds {
    int32_t *queue;        // [RGX_QCAP]
    int32_t *leafq;        // [128], by pairs [192]: leaves waiting for the sweep's ellipsoid test
    float *tab;            // [RGX_CCAP * RGX_TAB]
    uint8_t *list;         // [RGX_CCAP]: table slots that some ray of the tile hits
    uint32_t (*mask)[64];  // [RGX_MASK_WORDS][64]: per lane, hit bits over the list
    uint32_t (*half)[4][RGX_MASK_WORDS]; // [2][row][word]: list entries with samples in the slab's first / second 16
};

// Ray-interval-independent half of __intersection__gaussian (gaussians_aabb.cu:43-82) on a table
// entry: same arithmetic as line_roots(), with the precomputed ray-independent parts.
__device__ __forceinline__ bool lane_roots(const float4 *e, f3 dir, float &r1, float &r2)
{
    f3 U, V, W, inv;
    table_frame(e, U, V, W, inv);
    const float4 e4 = e[3];
    const f3 De = apply_sinv_rt(dir, U, V, W, inv);
    const f3 Oe = mk3(e4.x, e4.y, e4.z);
    const float a = fmaf(De.x, De.x, fmaf(De.y, De.y, De.z * De.z));
    const float b = -fmaf(Oe.x, De.x, fmaf(Oe.y, De.y, Oe.z * De.z));
    const float c = ((const float *)e)[RGX_TAB_C];
    const float inv_a = 1.0f / a;
    const float b_inv_a = b * inv_a;
    const f3 Pc = mk3(fmaf(b_inv_a, De.x, Oe.x), fmaf(b_inv_a, De.y, Oe.y), fmaf(b_inv_a, De.z, Oe.z));
    const float d2 = fmaf(Pc.x, Pc.x, fmaf(Pc.y, Pc.y, Pc.z * Pc.z));
    const float disc = 1.0f - d2;
    // no branch per lane: where the line misses (disc <= 1e-7) the roots are garbage and the result false
    const float sdisc = sqrtf(disc * a);
    const float q = b + copysignf(sdisc, b);
    r1 = c / q;
    r2 = q * inv_a;
    return disc > 1e-7f;
}

// A Gaussian as the shading code sees it: its record in HBM plus its rotation columns,
// inverse scales / k and k -- read from the LDS table entry when there is one; otherwise the
// rotation columns come from the 9-word frame the replay keeps per window slot (same operations,
// same values) and the scales from the record.
template <bool FROM_TABLE>
struct Entry {
    const float4 *tab; // LDS table entry (FROM_TABLE), or the slot's column of the replay's frame array
    const Prim *prim;
    int32_t pid;       // index in Morton order
    int slot;          // its slot in the candidate table of the current window
    __device__ __forceinline__ float4 position() const { return prim->pos4; }
    __device__ __forceinline__ float4 colour() const { return prim->rgba4; }
    __device__ __forceinline__ void frame(f3 &U, f3 &V, f3 &W, f3 &inv, float &k) const
    {
        if constexpr (FROM_TABLE) {
            table_frame(tab, U, V, W, inv);
            k = ((const float *)tab)[RGX_TAB_K];
        } else {
            const float *f = (const float *)tab; // component-major: word c of this slot at f[c * RGX_CCAP]
            U = mk3(f[0], f[RGX_CCAP], f[2 * RGX_CCAP]);
            V = mk3(f[3 * RGX_CCAP], f[4 * RGX_CCAP], f[5 * RGX_CCAP]);
            W = mk3(f[6 * RGX_CCAP], f[7 * RGX_CCAP], f[8 * RGX_CCAP]);
            const float4 i4 = prim->inv_inter4;
            inv = mk3(i4.x, i4.y, i4.z);
            k = i4.w;
        }
    }
};

// An entry of the replay whose record has been asked for beforehand (replay_lists).
struct EntryAhead {
    const float4 *tab;
    const Prim *prim;
    int32_t pid;
    int slot;
    float4 pos4, inv4, rgba4;
    __device__ __forceinline__ float4 position() const { return pos4; }
    __device__ __forceinline__ float4 colour() const { return rgba4; }
    __device__ __forceinline__ void frame(f3 &U, f3 &V, f3 &W, f3 &inv, float &k) const
    {
        const float *f = (const float *)tab; // as in Entry<false>
        U = mk3(f[0], f[RGX_CCAP], f[2 * RGX_CCAP]);
        V = mk3(f[3 * RGX_CCAP], f[4 * RGX_CCAP], f[5 * RGX_CCAP]);
        W = mk3(f[6 * RGX_CCAP], f[7 * RGX_CCAP], f[8 * RGX_CCAP]);
        inv = mk3(inv4.x, inv4.y, inv4.z);
        k = inv4.w;
    }
};

// exp(-power / 2) as one multiply and the hardware's exp2: -0.5 and log2(e) folded into one constant.
__device__ __forceinline__ float gauss_weight(float power) { return __builtin_amdgcn_exp2f(power * -0.72134752044448170f); }

// Per-hit constants of the sample recurrence (gaussians_aabb.cu:135-164).
struct HitSetup {
    float power, inc, inc_st, cut;
    f3 Mx0, Md; // the first sample point and the ray direction in the Gaussian's whitened frame
};
__device__ __forceinline__ HitSetup hit_setup(f3 U, f3 V, f3 W, f3 inv, float k, float4 pos4, f3 dir, f3 ray_dir_tmid, float dt)
{
    const f3 inv_s = mk3(inv.x * k, inv.y * k, inv.z * k);
    const f3 xhit = mk3(pos4.x, pos4.y, pos4.z) + ray_dir_tmid;
    const f3 Mx0 = apply_sinv_rt(xhit, U, V, W, inv_s);
    const f3 Md = apply_sinv_rt(dir, U, V, W, inv_s);
    const float Md2 = dot3(Md, Md);
    const float Md_dt_2 = (dt * dt) * Md2;
    HitSetup h;
    h.power = dot3(Mx0, Mx0);
    h.inc = Md_dt_2 + 2.0f * dot3(Mx0, Md) * dt;
    h.inc_st = 2.0f * Md_dt_2;
    h.cut = k * k;
    h.Mx0 = Mx0;
    h.Md = Md;
    return h;
}

// How close to zero the filter's u (below) may come before it stops deciding.  With N = |Oe| = sqrt(c + 1), e = 2^-24,
// a ray that meets the ellipsoid or nearly so, and the same computed a, b, De, Oe in both forms: the
// predicate's r2 = (b + s) / a is within 3 e (N + 1) + 6 e of the exact root of those numbers in whitened
// units; its r1 = c / q within 16 e N, since c is rounded (3 e N^2) and a, b need not belong to that c exactly
// (9 e N^2), over q > 0.86 N; u's own point tc is within 3 e N, and its square as far again with half-chord
// and distance at most one: 38 e N + 40 e, plus 470 (e N)^2, which up to N = 2^15 is below 2 e N + 24 e.
// A quotient c / q is that well behaved, and a line with b < 0 that surely missed, only with the eye outside the
// ellipsoid's double (c >= 3): entries nearer than that, or further than N = 2^15, are decided by their roots.
__device__ __forceinline__ float filter_margin(float c)
{
    return c >= 3.0f && c <= 0x1p30f ? fmaf(__builtin_amdgcn_sqrtf(c + 1.0f), 41.0f * 0x1p-24f, 66.0f * 0x1p-24f) : INFINITY;
}

// Adds a hit's samples to the half's sums: those within the cut-off, by the execution mask (a comparison that writes it
// and a scalar move that restores it cost less than a comparison, two wait states and a select).
// What the compiler cannot see inside the assembly is arranged there:
//   a sum is written before the last inputs are read: early-clobber ("+&v"), no input shares its register;
//   gw comes from a transcendental, whose result the next instruction may not read yet: the comparison, which reads
//     only the power, comes first;
//   a vector write of the mask needs five instructions before a data-parallel or cross-lane instruction, and one of vcc
//     four before v_div_fmas or v_readlane take it: the four multiply-adds and the scalar move are those five;
//   a vector write of a register needs two before a data-parallel or permlane read of it: the scalar move is one, and the
//     sums are next read after the hit's branch has ended, whose scalar instructions are more than the other.
__device__ __forceinline__ void accumulate_samples(HitSetup hs, float4 col, float (&sg)[RGX_CHUNK_SIZE], float (&cr)[RGX_CHUNK_SIZE],
                                                   float (&cg)[RGX_CHUNK_SIZE], float (&cb)[RGX_CHUNK_SIZE])
{
    const uint64_t lanes = __builtin_amdgcn_read_exec();
#pragma unroll
    for (int i = 0; i < RGX_CHUNK_SIZE; ++i) {
        const float gw = gauss_weight(hs.power);
        asm("v_cmpx_lt_f32_e32 vcc, %[p], %[cut]\n\tv_fmac_f32_e32 %[a], %[w], %[g]\n\tv_fmac_f32_e32 %[r], %[x], %[g]\n\t"
            "v_fmac_f32_e32 %[gg], %[y], %[g]\n\tv_fmac_f32_e32 %[b], %[z], %[g]\n\ts_mov_b64 exec, %[l]"
            : [a] "+&v"(sg[i]), [r] "+&v"(cr[i]), [gg] "+&v"(cg[i]), [b] "+&v"(cb[i])
            : [p] "v"(hs.power), [cut] "v"(hs.cut), [g] "v"(gw), [x] "v"(col.x), [y] "v"(col.y), [z] "v"(col.z), [w] "v"(col.w), [l] "s"(lanes)
            : "vcc");
        hs.power += hs.inc;
        hs.inc += hs.inc_st;
    }
}

// Four samples of the recurrence: their powers, and for each the rays for which it lies inside the cut-off.  The rays of a
// trip walk lists of one order and so are at similar depths: for many a block of four no ray has a sample, and then its
// exponentials and sums are left out: 23 % of the backward's blocks at 1 M Gaussians 800x800 (5.27 -> 5.07 ms), 58 % at 3 M
// 1237x822 (10.1 -> 8.4 ms).  The others run for the rays that have a sample in them only (`any`): the same instructions, and
// less power, which is what the clock of a card under this load depends on (1 M 800x800 5.03 -> 4.86 ms).
// Where tiles are light and few a wavefront has its SIMD to itself and waits for the branch:
// 4 k Gaussians 128x128 0.142 -> 0.161 ms, 100 k 400x400 0.567 -> 0.590, 300 k 440x440 1.47 -> 1.51 (the replay of lists
// alone the same); up to 3 000 tiles other scenes gain as much as these lose (3 M 256x256 2.32 -> 2.04, 1 M 440x440 2.75 -> 2.55), so
// one form serves all.  In the forward, whose walks have two chunks and more rays per trip, it is 9 and 30 % of the blocks, and
// the branches cost more than that (3 M 1920x1080: 17.4 -> 17.7 ms; masks without the branches 16.9 -> 17.3).
#define RGX_SAMPLE_BLOCK 4
struct SampleBlock {
    float power[RGX_SAMPLE_BLOCK];
    uint64_t in[RGX_SAMPLE_BLOCK];
    uint64_t any; // the rays with a sample in the block
    __device__ __forceinline__ void step(HitSetup &h, float cut)
    {
        any = 0;
#pragma unroll
        for (int k = 0; k < RGX_SAMPLE_BLOCK; ++k) {
            power[k] = h.power;
            in[k] = __ballot(h.power < cut);
            any |= in[k];
            h.power += h.inc;
            h.inc += h.inc_st;
        }
    }
};

// a's upper 32 lanes and b's lower 32 lanes change places; the same with the rows of 16 of each half
__device__ __forceinline__ void swap32(float &a, float &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float &a, float &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
// the value of each of the four copies of a ray, in every copy
__device__ __forceinline__ void copies(float v, float (&out)[4])
{
    float a = v, b = v; // -> a: copies 0 and 1 (in the lower and upper rows of both halves), b: copies 2 and 3
    swap32(a, b);
    float a1 = a, b1 = b;
    swap16(a, a1);
    swap16(b, b1);
    out[0] = a; out[1] = a1; out[2] = b; out[3] = b1;
}
// 16 values per lane -> four: copy `sub` gets the sums over the copies of v[4 sub .. 4 sub + 3]
__device__ __forceinline__ void sum_copies(float (&v)[RGX_CHUNK_SIZE], float (&out)[4])
{
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        swap32(v[i], v[i + 8]);
        v[i] += v[i + 8];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        swap16(v[i], v[i + 4]);
        out[i] = v[i] + v[i + 4];
    }
}

// Parts of tiles.  A wavefront that marches only RAYS of a tile's 64 rays has each of them 64 / RAYS times over (lane = RAYS * copy + ray).  The
// copies test as many table entries at a time, and each shades every 64 / RAYS-th hit.
template <int RAYS>
struct Part {
    static_assert(RAYS == 64 || RAYS == 32 || RAYS == 16 || RAYS == 8, "a tile; its upper or lower half; a 4x4 block; 4x2 pixels");
    static constexpr int COPIES = 64 / RAYS, BITS = RAYS == 64 ? 0 : RAYS == 32 ? 1 : RAYS == 16 ? 2 : 3;
    static constexpr int WIDTH = RAYS < 32 ? 4 : 8, HEIGHT = RAYS / WIDTH; // in pixels
    static constexpr int EACH = RGX_CHUNK_SIZE / COPIES;                   // samples of a chunk that a copy blends
    static constexpr int LISTS_HEAD = RAYS == 64 ? 8 : 2;                  // words of a LISTS item before its slots
    static constexpr int ROWS = RAYS > 16 ? RAYS / 16 : 1;                 // rows of lanes that hold all rays
    // a lane's ray and copy (with one copy: what the compiler need not find out)
    static __device__ __forceinline__ int ray(int lane) { return RAYS == 64 ? lane : lane % RAYS; }
    static __device__ __forceinline__ int copy(int lane) { return RAYS == 64 ? 0 : lane / RAYS; }
    // what the lanes of copy s say, said by all copies
    static __device__ __forceinline__ uint64_t spread(uint64_t lanes, int s)
    {
        const uint32_t own = (uint32_t)(lanes >> (RAYS * s));
        const uint32_t word = RAYS == 32 ? own : RAYS == 16 ? (own & 0xffffu) * 0x10001u : (own & 0xffu) * 0x1010101u;
        return (uint64_t)word << 32 | word;
    }
    // hits without the first n of them, n < COPIES
    static __device__ __forceinline__ uint32_t skip(uint32_t bits, int n)
    {
        for (int k = 0; k < COPIES - 1; ++k) bits = n > k ? bits & (bits - 1u) : bits;
        return bits;
    }
    static __device__ __forceinline__ float other_half_row(float v) // (row_ror:8)
    {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));
    }
    // the value of each copy of a ray, in every copy
    static __device__ __forceinline__ void of_all(float v, float (&out)[COPIES])
    {
        if constexpr (RAYS == 32) {
            float a = v, b = v;
            swap32(a, b);
            out[0] = a;
            out[1] = b;
        } else if constexpr (RAYS == 16) {
            copies(v, out);
        } else {
            const float o = other_half_row(v);
            const bool odd = threadIdx.x & 8;
            float even_ones[4], odd_ones[4];
            copies(odd ? o : v, even_ones);
            copies(odd ? v : o, odd_ones);
#pragma unroll
            for (int k = 0; k < COPIES; ++k) out[k] = k & 1 ? odd_ones[k >> 1] : even_ones[k >> 1];
        }
    }
    static __device__ __forceinline__ float sum_of_all(float v)
    {
        float c[COPIES];
        of_all(v, c);
        float sum = c[0];
        for (int k = 1; k < COPIES; ++k) sum += c[k];
        return sum;
    }
    static __device__ __forceinline__ float least_of_all(float v)
    {
        float c[COPIES];
        of_all(v, c);
        float least = c[0];
        for (int k = 1; k < COPIES; ++k) least = fminf(least, c[k]);
        return least;
    }
    // a chunk's values per lane -> copy c gets the sums over the copies of the c-th run of EACH of them
    static __device__ __forceinline__ void sums(float (&v)[RGX_CHUNK_SIZE], float (&out)[EACH])
    {
        if constexpr (RAYS == 32) {
#pragma unroll
            for (int i = 0; i < EACH; ++i) {
                swap32(v[i], v[i + EACH]);
                out[i] = v[i] + v[i + EACH];
            }
        } else if constexpr (RAYS == 16) {
            sum_copies(v, out);
        } else {
            float four[4];
            sum_copies(v, four); // over the copies of the lane's half of the row: samples 4 row .. 4 row + 3
            const bool odd = threadIdx.x & 8;
#pragma unroll
            for (int i = 0; i < EACH; ++i) { // two of the four, from both halves
                const float mine = odd ? four[i + EACH] : four[i], theirs = odd ? four[i] : four[i + EACH];
                out[i] = mine + other_half_row(theirs);
            }
        }
    }
};

// What one lane asks of the candidate table in this iteration.
struct LaneQuery {
    f3 dir;
    bool need;      // marching: collect the hits of [tlo, thi] (the collect query, gaussians_aabb.cu:282-295, 349-367)
    float tlo, thi;
    bool search;    // searching: smallest hit t in [slo, shi] (the first-hit query, 234-247, 370-380)
    float slo, shi;
    int cap;        // max_prim_slice
    float tmid;     // tbuffer + 16 dt: where the slab's second 16 samples begin
};

// Filter: every lane tests the table entries whose distance shell meets [t0, t1] (the union of
// the lanes' intervals).  An entry hit by any marching lane is appended to the iteration's list, and each lane
// keeps its own hit bits over it.  A wave is four 16-lane rows, each row a 4x4 pixel block: per list entry a row
// also notes whether any of its rays can have
// samples inside the Gaussian in the slab's first 16 samples and in its second 16 (the chord
// [r1, r2] against tmid; a sample lies half a step from tmid, rounding moves a root by far less),
// so that each half is shaded from its own, shorter list.  len (wave-uniform) is the list length; p0 / ov count this lane's
// hits and note the max_prim_slice cut (__anyhit__ah's optixTerminateRay, 352-356); found is
// the running minimum of the searching lanes.
// part (the same for all lanes): 0: all hits of [tlo, thi]; 1: only those reaching the first 16
// samples; 2: only those reaching the second 16, of which the ones that also reach the first are
// not counted again.  plain: every entry of the table passed plain_roots().
//
// The filter is bound by the number of its instructions, of whatever kind, and by how long each waits for the one
// before: three wavefronts per SIMD issue at most one each in some five clocks.  The reference's
// predicate is two divisions and a square root, correctly rounded, one after the other.  What decides is
// whether the ray's segment meets the ellipsoid, and for nearly every ray and entry that does not take the roots:
// with tc the line's closest point to the centre and d2 its squared whitened distance there, the point of
// the segment closest to tc lies at u = (x - tc)^2 a + d2 - 1 from the surface, and u < 0 says hit.  Where
// some ray's |u| is within filter_margin() of zero -- u and the predicate's comparisons may then fall on different
// sides -- the wavefront takes the exact roots for that entry, as it does where a searching ray may have
// found something, whose t it needs.  What the lanes decide stays in scalar registers, one list serves the
// whole wavefront, and the entries' slots are collected in a register.
template <typename Cn>
__device__ __forceinline__ void filter_table(const TileLds &L, int C, float t0, float t1, const LaneQuery &Q, int part, bool plain,
                                             int &p0, bool &ov, float &found, int &len_out, uint32_t (&own)[2], Cn &cn)
{
    const int lane = threadIdx.x;
    int len = 0;
    uint32_t first = 0, second = 0; // this lane's hits with samples in the first / second half
    int slots = 0;                  // lane i: slot of entry i of the list's current 64
    own[0] = own[1] = 0u;
    const bool asks = Q.need && !Q.search;
    const uint64_t searching = __ballot(Q.search);
    // the segment and where its halves meet (rays that ask nothing: far from everything)
    const float none = 1e15f;
    const float lo = Q.search ? Q.slo : asks ? Q.tlo : none, hi = Q.search ? Q.shi : asks ? Q.thi : none;
    const float mid = Q.search ? hi : asks ? fminf(Q.tmid, hi) : none;
    // max_prim_slice cuts a ray's list in the order of the entries: where it could, entry by entry
    const bool slow = !plain || __any(asks && (ov || p0 + C > Q.cap));
    const uint64_t take_first = part != 2 ? ~0ull : 0ull, take_second = part != 1 ? ~0ull : 0ull;
    auto flush = [&](int w) {
        const uint32_t bits = (part != 2 ? first : 0u) | (part != 1 ? second : 0u);
        L.mask[w][lane] = bits;
        if (!slow) p0 += __popc(part == 2 ? second & ~first : bits);
        if (w == 0) { // the ray's own notes on the list's first 32 entries stay with it (see shade_lanes)
            own[0] = first;
            own[1] = second;
        }
        const uint32_t f = row_or(first), g = row_or(second);
        if ((lane & 15) == 0) {
            L.half[0][lane >> 4][w] = f;
            L.half[1][lane >> 4][w] = g;
        }
        first = second = 0;
        if (lane < len - (w & ~1) * 32) L.list[(w & ~1) * 32 + lane] = (uint8_t)slots;
    };
    for (int h = 0; h < RGX_CCAP; h += 64) {
        const int cl = h + lane;
        bool rel = false;
        float margins = INFINITY;
        if (cl < C) {
            const float dmin = L.tab[cl * RGX_TAB + RGX_TAB_DMIN], dmax = L.tab[cl * RGX_TAB + RGX_TAB_DMAX];
            rel = dmax >= t0 && dmin <= t1;
            margins = slow ? INFINITY : filter_margin(L.tab[cl * RGX_TAB + RGX_TAB_C]);
        }
        uint64_t m = __ballot(rel);
        if (lane == 0) cn.cands += (unsigned)__popcll(m);
        while (m) {
            const int i = __builtin_ctzll(m), c = h + i;
            m &= m - 1;
            const float margin = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(margins), i));
            const float4 *e = (const float4 *)((const char *)L.tab + __builtin_amdgcn_readfirstlane(c * (RGX_TAB * 4)));
            f3 U, V, W, inv;
            table_frame(e, U, V, W, inv);
            const float4 e4 = e[3];
            const f3 De = apply_sinv_rt(Q.dir, U, V, W, inv);
            const float a = fmaf(De.x, De.x, fmaf(De.y, De.y, De.z * De.z));
            const float b = -fmaf(e4.x, De.x, fmaf(e4.y, De.y, e4.z * De.z));
            const float tc = b * __builtin_amdgcn_rcpf(a);
            const f3 Pc = mk3(fmaf(tc, De.x, e4.x), fmaf(tc, De.y, e4.y), fmaf(tc, De.z, e4.z));
            const float out = fmaf(Pc.x, Pc.x, fmaf(Pc.y, Pc.y, Pc.z * Pc.z)) - 1.0f;
            const float x1 = __builtin_amdgcn_fmed3f(tc, lo, mid) - tc, x2 = __builtin_amdgcn_fmed3f(tc, mid, hi) - tc;
            const float u1 = fmaf(x1 * x1, a, out), u2 = fmaf(x2 * x2, a, out);
            uint64_t f = __ballot(!(u1 > margin)), g = __ballot(!(u2 > margin));
            const uint64_t sure = __ballot(fminf(fabsf(u1), fabsf(u2)) > margin);
            if ((f | g) == 0) continue;
            if (__builtin_expect((~sure | ((f | g) & searching)) != 0, 0)) {
                float r1, r2;
                const bool ok = lane_roots(e, Q.dir, r1, r2);
                // first-hit query (searching lanes): smallest max(slo, r1) over the entries hit in [slo, shi]
                const float ts = fmaxf(Q.slo, r1);
                const bool sfound = Q.search && ok && ts <= fminf(Q.shi, r2);
                found = sfound ? (found < 0.0f ? ts : fminf(found, ts)) : found;
                // collect query (marching lanes); every hit is noted for a half at least
                bool seg = asks && !ov && ok && fmaxf(Q.tlo, r1) <= fminf(Q.thi, r2);
                const bool to_second = r2 > Q.tmid, to_first = r1 < Q.tmid || !to_second;
                if (slow) {
                    const bool counts = part != 2 || !to_first, over = seg && counts && p0 >= Q.cap;
                    ov = ov || over;
                    seg = seg && !over;
                    p0 += seg && counts && (part != 1 || to_first) ? 1 : 0;
                }
                f = __ballot(seg && to_first);
                g = __ballot(seg && to_second);
            }
            if (((f & take_first) | (g & take_second)) == 0) continue;
            if (lane == 0) cn.cands_hit++;
            const uint32_t bit = 1u << (len & 31);
            first |= __builtin_amdgcn_inverse_ballot_w64(f) ? bit : 0u;
            second |= __builtin_amdgcn_inverse_ballot_w64(g) ? bit : 0u;
            slots = lane == (len & 63) ? c : slots;
            ++len;
            if ((len & 31) == 0) flush((len >> 5) - 1);
        }
    }
    if (len & 31) flush(len >> 5);
    len_out = len;
    __syncthreads();
}

// filter_table for a part of a tile: as many entries at a time as a ray has copies.
template <int RAYS, typename Cn>
__device__ __forceinline__ void filter_part(const TileLds &L, int C, float t0, float t1, const LaneQuery &Q, int part, bool plain,
                                            int &p0, bool &ov, float &found, int &len_out, uint32_t (&own)[2], Cn &cn)
{
    constexpr int COPIES = 64 / RAYS;
    const int lane = threadIdx.x, copy = Part<RAYS>::copy(lane);
    int len = 0;
    uint32_t first = 0, second = 0; // the ray's hits with samples in the first / second half (the same in all copies)
    int slots = 0;                  // lane i: slot of entry i of the list's current 64
    own[0] = own[1] = 0u;
    const bool asks = Q.need && !Q.search;
    const uint64_t searching = __ballot(Q.search);
    const float none = 1e15f;
    const float lo = Q.search ? Q.slo : asks ? Q.tlo : none, hi = Q.search ? Q.shi : asks ? Q.thi : none;
    const float mid = Q.search ? hi : asks ? fminf(Q.tmid, hi) : none;
    const bool slow = !plain || __any(asks && (ov || p0 + C > Q.cap)); // (then one entry at a time, which the first copy decides)
    const uint64_t take_first = part != 2 ? ~0ull : 0ull, take_second = part != 1 ? ~0ull : 0ull;
    auto flush = [&](int w) {
        const uint32_t bits = (part != 2 ? first : 0u) | (part != 1 ? second : 0u);
        L.mask[w][lane] = bits;
        if (!slow) p0 += __popc(part == 2 ? second & ~first : bits);
        if (w == 0) {
            own[0] = first;
            own[1] = second;
        }
        const uint32_t f = row_or(first), g = row_or(second);
        if ((lane & 15) == 0) {
            L.half[0][lane >> 4][w] = f;
            L.half[1][lane >> 4][w] = g;
        }
        first = second = 0;
        if (lane < len - (w & ~1) * 32) L.list[(w & ~1) * 32 + lane] = (uint8_t)slots;
    };
    for (int h = 0; h < RGX_CCAP; h += 64) {
        const int cl = h + lane;
        bool rel = false;
        float margins = INFINITY;
        if (cl < C) {
            const float dmin = L.tab[cl * RGX_TAB + RGX_TAB_DMIN], dmax = L.tab[cl * RGX_TAB + RGX_TAB_DMAX];
            rel = dmax >= t0 && dmin <= t1;
            margins = slow ? INFINITY : filter_margin(L.tab[cl * RGX_TAB + RGX_TAB_C]);
        }
        uint64_t m = __ballot(rel);
        if (lane == 0) cn.cands += (unsigned)__popcll(m);
        while (m) {
            int at[COPIES], c = 0;
            float margin = 0.f;
            int there = 0; // copies with an entry (the others go through the first one's again, to no effect)
#pragma unroll
            for (int s = 0; s < COPIES; ++s) {
                at[s] = s == 0 || (m && !slow) ? __builtin_ctzll(m) : at[0];
                const bool is = s == 0 || (m && !slow);
                const float ms = is ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(margins), at[s])) : -INFINITY;
                if (is) {
                    m &= m - 1;
                    ++there;
                }
                c = copy == s ? at[s] : c;
                margin = copy == s ? ms : margin;
            }
            const float4 *e = (const float4 *)(L.tab + (h + c) * RGX_TAB);
            f3 U, V, W, inv;
            table_frame(e, U, V, W, inv);
            const float4 e4 = e[3];
            const f3 De = apply_sinv_rt(Q.dir, U, V, W, inv);
            const float a = fmaf(De.x, De.x, fmaf(De.y, De.y, De.z * De.z));
            const float b = -fmaf(e4.x, De.x, fmaf(e4.y, De.y, e4.z * De.z));
            const float tc = b * __builtin_amdgcn_rcpf(a);
            const f3 Pc = mk3(fmaf(tc, De.x, e4.x), fmaf(tc, De.y, e4.y), fmaf(tc, De.z, e4.z));
            const float out = fmaf(Pc.x, Pc.x, fmaf(Pc.y, Pc.y, Pc.z * Pc.z)) - 1.0f;
            const float x1 = __builtin_amdgcn_fmed3f(tc, lo, mid) - tc, x2 = __builtin_amdgcn_fmed3f(tc, mid, hi) - tc;
            const float u1 = fmaf(x1 * x1, a, out), u2 = fmaf(x2 * x2, a, out);
            uint64_t f = __ballot(!(u1 > margin)), g = __ballot(!(u2 > margin));
            const uint64_t sure = __ballot(fminf(fabsf(u1), fabsf(u2)) > margin);
            const uint64_t valid = there * RAYS < 64 ? (1ull << (there * RAYS)) - 1ull : ~0ull;
            f &= valid;
            g &= valid;
            if ((f | g) == 0) continue;
            if (__builtin_expect(((~sure & valid) | ((f | g) & searching)) != 0, 0)) {
                float r1, r2;
                const bool ok = lane_roots(e, Q.dir, r1, r2) && copy < there;
                const float ts = fmaxf(Q.slo, r1);
                const bool sfound = Q.search && ok && ts <= fminf(Q.shi, r2);
                found = sfound ? (found < 0.0f ? ts : fminf(found, ts)) : found;
                bool seg = asks && !ov && ok && fmaxf(Q.tlo, r1) <= fminf(Q.thi, r2);
                const bool to_second = r2 > Q.tmid, to_first = r1 < Q.tmid || !to_second;
                if (slow) {
                    const bool counts = part != 2 || !to_first, over = seg && counts && p0 >= Q.cap;
                    seg = seg && !over;
                    ov = ov || __builtin_amdgcn_inverse_ballot_w64(Part<RAYS>::spread(__ballot(over), 0));
                    p0 += __builtin_amdgcn_inverse_ballot_w64(Part<RAYS>::spread(__ballot(seg && counts && (part != 1 || to_first)), 0)) ? 1 : 0;
                }
                f = __ballot(seg && to_first);
                g = __ballot(seg && to_second);
            }
            if (((f & take_first) | (g & take_second)) == 0) continue;
#pragma unroll
            for (int s = 0; s < COPIES; ++s) {
                const uint64_t fs = Part<RAYS>::spread(f, s), gs = Part<RAYS>::spread(g, s);
                if (((fs & take_first) | (gs & take_second)) == 0) continue;
                if (lane == 0) cn.cands_hit++;
                const uint32_t bit = 1u << (len & 31);
                first |= __builtin_amdgcn_inverse_ballot_w64(fs) ? bit : 0u;
                second |= __builtin_amdgcn_inverse_ballot_w64(gs) ? bit : 0u;
                slots = lane == (len & 63) ? h + at[s] : slots;
                ++len;
                if ((len & 31) == 0) flush((len >> 5) - 1);
            }
        }
    }
    if (len & 31) flush(len >> 5);
    len_out = len;
    if (searching) {
        const float best = Part<RAYS>::least_of_all(found < 0.0f ? INFINITY : found);
        found = best < INFINITY ? best : -1.0f;
    }
    __syncthreads();
}

// Tag telling a shading body which 16 of the slab's 32 samples its walk is for.
template <int H>
struct Half {
    static constexpr int value = H;
    static constexpr int group = 16; // lanes that share a trip's entry: a row
};
// Tag of a walk in which the two halves of a row (8 lanes each) walk on their own.  (Groups of 4 make
// still fewer trips, but four times a row's adds to the window's sums in LDS: measured slower.)
struct HalfRows {
    static constexpr int value = 0;
    static constexpr int group = 8;
};

// Shade: the four rows walk the entries that one of their own rays hits in lock step; body(entry, hit, live) runs whenever
// some lane hits (hit: this lane hits this entry; live: this lane's row still has an entry).
template <typename Body>
__device__ __forceinline__ void shade_rows(const MarchParams &P, const TileLds &L, int len, bool run, Body body)
{
    const int lane = threadIdx.x;
    const int nw = (len + 31) >> 5;
    int w = 0;
    uint32_t own = nw > 0 ? L.mask[0][lane] : 0u, bits = row_or(own);
    for (;;) {
        // (all lanes of a row hold the same bits and the same w)
        while (__any(bits == 0u && w + 1 < nw)) {
            const bool next = bits == 0u && w + 1 < nw;
            const uint32_t m = next ? L.mask[w + 1][lane] : 0u;
            const uint32_t o = row_or(m);
            if (next) {
                ++w;
                own = m;
                bits = o;
            }
        }
        const bool live = bits != 0u;
        if (!__any(live)) break;
        const int at = live ? __builtin_ctz(bits) : 0;
        bits &= bits - 1u;
        const bool hit = run && live && ((own >> at) & 1u);
        if (__ballot(hit)) {
            const int c = live ? L.list[w * 32 + at] : 0;
            const float4 *tab = (const float4 *)(L.tab + c * RGX_TAB);
            const int32_t pid = __float_as_int(L.tab[c * RGX_TAB + RGX_TAB_PID]);
            body(Entry<true>{tab, P.prims + pid, pid, c}, hit, live, Half<0>{});
        }
    }
}

// Shade, one ray at a time: every lane walks its own hits (the set bits of its mask over the
// list), so the trip count is the longest hit list of a ray.
// For bodies that need no sum over the rays of a row.  The order of a ray's hits is that of
// shade_rows.  Only the entries that can reach half `half` of the slab's samples are visited; the
// body gets Half<TAG>.  For the list's first 32 entries the ray goes by its own chords (own[half]: its
// hits with samples in that half, as the filter left them), for the rest by its row's notes, which
// also hold for rays whose own chord stays in the other half.
// RAYS < 64: each copy of a ray takes every 64 / RAYS-th of the ray's hits.
template <int TAG, int RAYS = 64, typename Body>
__device__ __forceinline__ void shade_lanes(const MarchParams &P, const TileLds &L, int len, bool run, int half,
                                            const uint32_t (&own)[2], Body body)
{
    const int lane = threadIdx.x, row = lane >> 4;
    const int nw = (len + 31) >> 5;
    int w = 0;
    const int copy = Part<RAYS>::copy(lane);
    uint32_t bits = (run && nw > 0) ? Part<RAYS>::skip(half ? own[1] : own[0], copy) : 0u;
    for (;;) {
        while (bits == 0u && run && w + 1 < nw) {
            ++w;
            bits = Part<RAYS>::skip(L.mask[w][lane] & L.half[half][row][w], copy);
        }
        const bool has = bits != 0u;
        if (!__any(has)) break;
        int c = 0;
        if (has) {
            c = L.list[w * 32 + __builtin_ctz(bits)];
            bits &= bits - 1u;
            for (int k = 1; k < 64 / RAYS; ++k) bits &= bits - 1u;
        }
        const float4 *tab = (const float4 *)(L.tab + c * RGX_TAB);
        const int32_t pid = __float_as_int(L.tab[c * RGX_TAB + RGX_TAB_PID]);
        body(Entry<true>{tab, P.prims + pid, pid, c}, has, has, Half<TAG>{});
    }
}

// ---------------------------------------------------------------------------
// Hit-list records.  What the sweep and the filter produce -- per window the Gaussians of the
// candidate table, per slab iteration and 4x4 row the table slots some ray of the row hits, per ray
// its hit bits over that list, per searching ray the first-hit t -- is a few hundred bytes per
// iteration.  The forward can stream it to memory so that the backward replays the same lists
// instead of sweeping the tree and evaluating the predicate again.  Per tile a region of
// rec_tile_words 32-bit words:
//   word 0: status (RGX_REC_COMPLETE, _OVERFLOWED, _COMPLETE_SUMS);  word 1: words used;
//   words 4 .. 4 + RGX_REC_PIECES_MAX: where a backward can start in the middle of a tile (below);
//   from word RGX_REC_HEAD, per iteration: WINDOW when a table was built, one LISTS per table, then TRAIL
//   WINDOW: {tag | C, -, -, -}, pid[pad4(C)]            the table's Gaussians, by slot
//   LISTS:  {tag | last << 8 | nw, len[4] (four times the same), -, -, -}, slot bytes in pad4(len) / 4 words,
//           mask[nw][64], half[2][4][nw]   (the TileLds arrays of the same names; bytes past the list's length are junk)
//   TRAIL:  {tag | any_search, cover (float), sample-sum slot + 1, -}, found[64] when any_search
// Where a tile is marched by parts (record_part_lines) each of them has that share of the region and of a slot, laid out the same with as many rays as
// the part has in the place of 64, as many rows in the place of 4, and two words before a list's slots.  Their lists together need more than the tile's, so a
// part whose share is used up goes on in a slot of the pool, or, where the pool is empty, in its own, and leaves lists alone.  (The pool's first
// slots, where it has more than those, are one for each part, which holds its first sums.  Kept for the lists alone they left the sums without: 4 k Gaussians in a cube
// 240x240, sums for 5.3 slots a tile in a pool of six and no list that goes on: two parts in three, now one in sixty.)  The
// word RGX_REC_MORE + 1 of a region is that slot + 1 (0: none), word RGX_REC_MORE the offset of the first item there; the slot's words count from the
// end of the share.
//
// Sample sums.  A record with room beyond RGX_REC_LIST_WORDS per tile also has a pool of slots
// shared by all tiles: per slab iteration that blends something, the per-sample density and colour
// sums the forward blended -- sum rho w, then the red, green and blue of sum rgb rho w, each as [8][64 rays][4 consecutive
// samples]: 16 bytes per lane and access, and in registers a multiple of the even-aligned tuples that loads land
// in (three colours of a sample together take four registers while they are on their way).  The
// backward reads them back instead of walking the hit lists a second time to rebuild them.  The
// iteration's TRAIL item names its slot (word 2: slot + 1, 0 = none).  Tiles take slots from a
// bump counter; a tile that found the pool empty is marked lists-only (status 0).
#define RGX_REC_LIST_WORDS 16384   // hit-list words per tile when the record also holds sample sums
#define RGX_SUM_SLOT_WORDS 8192    // 32 samples x 64 rays x 4 words
// With RgxMarch::record_format 1 a slot keeps the colour sums in half precision: the density sums as before
// (floats: the transmittance must replay bit for bit), then per chunk of 16 samples and ray
// the 48 colour sums divided by a power of two that brings the largest to [1/2, 1) and rounded to binary16, two to a
// word ([2 chunks][24 words][64 rays]), then that power of two per chunk and ray ([2][64] floats).  The scale makes
// the format safe for any density (plain binary16 overflows at 65504); the sums keep 11 bits relative to each
// value down to 2^-14 of the chunk's largest.
typedef float quad __attribute__((ext_vector_type(4)));
typedef uint32_t quad_bits __attribute__((ext_vector_type(4)));
#define RGX_SUM_SLOT_WORDS_HALF (2048 + 2 * 24 * 64 + 2 * 64)
#ifndef RGX_SUM_SLOT_BATCH
#define RGX_SUM_SLOT_BATCH 2       // slots a tile takes from the pool at a time (the last batch's unused ones stay empty)
#endif
#define RGX_REC_COMPLETE 0u        // word 0 of a tile: hit lists complete
#define RGX_REC_OVERFLOWED 1u      //   the region overflowed (record unusable)
#define RGX_REC_COMPLETE_SUMS 2u   //   hit lists and sample sums complete
#define RGX_REC_OVERFLOWED_UNCUT 3u //  (parts) as 1, and no list was cut at max_prim_slice: a search in any order finds the same hits
#define RGX_REC_WINDOW 0x57000000u
#define RGX_REC_LISTS 0x4C000000u
#define RGX_REC_TRAIL 0x54000000u
// Pieces of a tile's record.  A tile is a serial march for the forward, but with the rays' state at a few of its
// iterations (transmittance, colour so far, position, step) the backward can replay the stretches between
// them side by side, each with a wavefront of its own: a launch no longer lasts as long as its longest tile.
// A piece ends once it has enough blending iterations, where a new window begins anyway or it has become half as long
// again (the next one then begins with the resident window's WINDOW item once more).  The states, state[piece][8][64],
// go to a slot of the sample-sum pool; word 4 of the tile's region: how many | slot << 8, words 5 ..: where in the
// region the iterations of the pieces after the first begin.
// How many, and how long, by the number of tiles (3072 wavefronts are resident at a time):
//   up to half of that: up to 16 short pieces, to fill the chip (4 k Gaussians, 128x128: 0.61 -> 0.17 ms);
//   beyond: up to 8, the first two 4 iterations long and each later one half as long again, so that short and
//     long tiles alike have several (300 k Gaussians, 800x800: 3.24 -> 2.94 ms; 1 M: 6.46 -> 6.29);
//   beyond four rounds of tiles the end of a launch is a small part of it, and what a piece costs (its state, its window
//     set up and flushed once more) weighs as much: none (3 M, 1237x822: 15.1 ms, 15.5 with pieces from 4 iterations, 14.8
//     with pieces from 8, but 0.2 more in the forward).
#define RGX_REC_PIECES_MAX 16
#define RGX_REC_HEAD (4 + RGX_REC_PIECES_MAX)
#define RGX_REC_MORE (RGX_REC_HEAD - 2)
#define RGX_REC_STATE_WORDS (8 * 64)
static_assert((RGX_REC_PIECES_MAX - 1) * RGX_REC_STATE_WORDS <= RGX_SUM_SLOT_WORDS, "a slot holds the states of a tile");
struct RecordPieces {
    int most;  // pieces
    int first; // blending iterations of the first ones
    int equal; // as many as this have that length; then they grow
    bool turn; // the XCDs replay different pieces at a time
};
static inline RecordPieces record_pieces(int tiles)
{
    if (tiles <= 1536) return {RGX_REC_PIECES_MAX, 2, 8, false};
    // (up to two rounds of tiles, the deepest pieces of all tiles would run at once, and add to the same few far
    // Gaussians: 150 k Gaussians, 619x411: 1.82 ms, turned 1.62.  The pieces that one XCD replays at a time stay at
    // one depth: its L2 holds the Gaussians of one depth, not of all (1 M, 800x800: 6.3 ms, 9.7 with mixed depths).)
    if (tiles <= 2 * 3072) return {RGX_REC_PIECES_MAX / 2, 4, 2, true};
    if (tiles <= 4 * 3072) return {RGX_REC_PIECES_MAX / 2, 4, 2, false};
    return {1, 0, 0, false};
}

// Words 2 and 3 of a tile's region name the launch the record belongs to (number of Gaussians,
// image size, step, fixed or adaptive), so that a backward handed a record of another scene or view recomputes the
// tile instead of following indices that mean nothing in its own tables.  (Size and kind of step also say by which parts of tiles a region
// is laid out: record_part_lines.)
__device__ __forceinline__ uint32_t record_mark(const MarchParams &P, int which)
{
    return which == 0 ? (uint32_t)P.n ^ ((uint32_t)P.m.record_format << 31)
                      : ((uint32_t)P.cam.width << 16 ^ (uint32_t)P.cam.height ^ __float_as_uint(P.m.dt_step) ^ (P.m.dynamic_sampling ? 0x55555555u : 0u));
}
// Status of a tile's record if it is this launch's and complete, else RGX_REC_OVERFLOWED.
__device__ __forceinline__ uint32_t record_status(const MarchParams &P, const uint32_t *reg)
{
    const uint32_t st = (uint32_t)__builtin_amdgcn_readfirstlane((int)reg[0]);
    const bool mine = (uint32_t)__builtin_amdgcn_readfirstlane((int)reg[2]) == record_mark(P, 0) &&
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)reg[3]) == record_mark(P, 1);
    return mine && (st == RGX_REC_COMPLETE || (st == RGX_REC_COMPLETE_SUMS && P.sum_pool)) ? st : RGX_REC_OVERFLOWED;
}
// Of a part: overflowed, without a list that was cut (each lane may ask of another region).
__device__ __forceinline__ bool record_uncut(const MarchParams &P, const uint32_t *reg)
{
    return reg[0] == RGX_REC_OVERFLOWED_UNCUT && reg[2] == record_mark(P, 0) && reg[3] == record_mark(P, 1);
}
__device__ __forceinline__ bool record_usable(const MarchParams &P, const uint32_t *reg)
{
    return record_status(P, reg) != RGX_REC_OVERFLOWED;
}

template <int RAYS>
struct Recorder {
    uint32_t *reg;  // the region of this tile, or part of one, or null
    int off;        // next free word (wave-uniform)
    int cap;        // words in the region
    bool ovf;       // the region is exhausted
    bool sums;      // every blending iteration so far got a sample-sum slot
    int slot;       // the current iteration's sample-sum slot, or -1
    int length;     // blending iterations of the current piece after which the next one is due
    int states = 0;      // states kept: pieces before the current one
    int state_slot = -1; // where
    int since = 0;       // blending iterations of the current piece
    uint32_t batch_next = 0; // the next slot of the batch this tile last took from the pool
    int batch_left = 0;      // slots left in that batch
    uint32_t *more = nullptr; // (parts) where the region goes on, less the share's size
    int more_from = 0, more_slot = -1;
    bool cut = false;         // (parts) max_prim_slice has cut a ray's list
    __device__ __forceinline__ bool on() const { return reg != nullptr && !ovf; }
    __device__ __forceinline__ uint32_t *item() const { return (RAYS < 64 && more ? more : reg) + off; }
    // room for an item and the iteration's trailer?
    __device__ __forceinline__ bool fits(const MarchParams &P, int size)
    {
        if (__builtin_expect(off + size + 72 > cap, 0)) {
            if (RAYS < 64 && !more && P.sum_next) {
                constexpr int COPIES = Part<RAYS>::COPIES;
                const uint32_t units = (uint32_t)P.sum_slots / COPIES;
                uint32_t s = 0;
                if (threadIdx.x == 0) s = atomicAdd(P.sum_next, 1u);
                s = (uint32_t)__builtin_amdgcn_readfirstlane((int)s);
                if (s >= units && P.sum_first) {
                    s = (uint32_t)((reg - P.records) / P.rec_tile_words); // its own
                    sums = false;
                    __threadfence(); // (what lanes stored there before is behind what others store now)
                }
                if (s < units && size + 72 <= P.sum_slot_words * COPIES) {
                    more_slot = (int)s * COPIES;
                    more_from = off;
                    more = (uint32_t *)(P.sum_pool + (int64_t)more_slot * (P.sum_slot_words / 4)) - cap;
                    off = cap;
                    cap += P.sum_slot_words * COPIES;
                    return true;
                }
            }
            ovf = true;
        }
        return !ovf;
    }

    // A slot of the pool, or -1 where it is empty.
    // (RGX_SUM_SLOT_BATCH slots per request: a request is a round trip to one counter that every tile of the
    // launch shares, and where iterations are short the tiles spend a good part of their time waiting on it)
    __device__ __forceinline__ int take_slot(const MarchParams &P)
    {
        if (batch_left == 0) {
            uint32_t s = 0;
            constexpr int COPIES = Part<RAYS>::COPIES; // (a part's slots are that share of a tile's: the counter's unit holds as many)
            if (threadIdx.x == 0) s = atomicAdd(P.sum_next, COPIES > 1 ? 1u : (uint32_t)RGX_SUM_SLOT_BATCH);
            batch_next = (uint32_t)__builtin_amdgcn_readfirstlane((int)s) * (uint32_t)COPIES;
            batch_left = COPIES > 1 ? COPIES : RGX_SUM_SLOT_BATCH;
        }
        const uint32_t s = batch_next++;
        --batch_left;
        return s < (uint32_t)P.sum_slots ? (int)s : -1;
    }

    // Does the next piece begin with this iteration?  reuse: the iteration goes on with the resident window.
    __device__ __forceinline__ bool piece_due(const MarchParams &P, bool reuse) const
    {
        return since >= (reuse ? length + (length >> 1) : length) && states < P.rec_pieces - 1 && on() && sums;
    }
    __device__ __forceinline__ void begin_piece(const MarchParams &P, const RayState &R, float Cr, float Cg, float Cb)
    {
        if (state_slot < 0) {
            state_slot = take_slot(P);
            if (state_slot < 0) {
                sums = false; // the pool is empty
                return;
            }
        }
        if (threadIdx.x == 0) reg[5 + states] = (uint32_t)off;
        float *st = (float *)(P.sum_pool + (int64_t)state_slot * (P.sum_slot_words / 4)) + states * (8 * RAYS) + threadIdx.x;
        if (RAYS == 64 || threadIdx.x < RAYS) {
            st[0] = R.T; st[RAYS] = R.tbuffer; st[2 * RAYS] = R.tenter; st[3 * RAYS] = R.dt;
            st[4 * RAYS] = Cr; st[5 * RAYS] = Cg; st[6 * RAYS] = Cb;
            ((uint32_t *)st)[7 * RAYS] = (R.active ? 1u : 0u) | (R.searching ? 2u : 0u) | (R.first ? 4u : 0u);
        }
        ++states;
        since = 0;
        if (states >= P.rec_equal) length += (length + 1) >> 1;
    }

    __device__ __forceinline__ void write_window(const MarchParams &P, const TileLds &L, int C)
    {
        if (!on() || !fits(P, 4 + ((C + 3) & ~3))) return;
        uint32_t *it = item();
        if (threadIdx.x == 0) it[0] = RGX_REC_WINDOW | (uint32_t)C;
        for (int i = threadIdx.x; i < C; i += 64) it[4 + i] = __float_as_uint(L.tab[i * RGX_TAB + RGX_TAB_PID]);
        off += 4 + ((C + 3) & ~3);
    }

    __device__ __forceinline__ void write_lists(const MarchParams &P, const TileLds &L, int len, bool last)
    {
        if (!on()) return;
        const int lane = threadIdx.x, row = lane >> 4;
        const int nw = (len + 31) >> 5, q = (len + 3) >> 2;
        constexpr int ROWS = Part<RAYS>::ROWS;
        constexpr int HEAD = Part<RAYS>::LISTS_HEAD;
        const int size = HEAD + q + nw * (RAYS + 2 * ROWS);
        if (!fits(P, size)) return;
        uint32_t *it = item();
        if (lane < (RAYS == 64 ? 5 : 2)) it[lane] = lane == 0 ? RGX_REC_LISTS | (last ? 0x100u : 0u) | (uint32_t)nw : (uint32_t)len;
        if (lane < q) it[HEAD + lane] = ((const uint32_t *)L.list)[lane];
        static_assert(RGX_CCAP <= 4 * 64, "a word of the list per lane");
        if (RAYS == 64 || lane < RAYS)
            for (int w = 0; w < nw; ++w) it[HEAD + q + w * RAYS + lane] = L.mask[w][lane];
        if ((lane & 15) < 2 && (ROWS == 4 || row < ROWS)) // two lanes per row: one per half
            for (int w = 0; w < nw; ++w) it[HEAD + q + nw * RAYS + ((lane & 15) * ROWS + row) * nw + w] = L.half[lane & 15][row][w];
        off += size;
    }

    // blends: some ray of the wave has hits to blend in this iteration
    __device__ __forceinline__ void write_trailer(const MarchParams &P, bool any_search, float cover, float found, bool blends)
    {
        slot = -1;
        if (!on()) return;
        since += blends ? 1 : 0;
        if (blends && P.sum_next) {
            // every blending iteration asks, also those of a tile that has gone without once: the counter then
            // ends at the launch's whole demand, which is what the next record of this view's shape is sized from
            const int s = take_slot(P);
            if (sums && s >= 0) slot = s;
            else sums = false;
        }
        uint32_t *it = item();
        if (threadIdx.x == 0) {
            it[0] = RGX_REC_TRAIL | (any_search ? 1u : 0u);
            it[1] = __float_as_uint(cover);
            it[2] = (uint32_t)(slot + 1);
        }
        if (any_search && (RAYS == 64 || threadIdx.x < RAYS)) it[4 + threadIdx.x] = __float_as_uint(found);
        off += 4 + (any_search ? RAYS : 0);
    }

    __device__ __forceinline__ void finish(const MarchParams &P)
    {
        if (reg && threadIdx.x == 0) {
            reg[0] = ovf ? (RAYS < 64 && !cut ? RGX_REC_OVERFLOWED_UNCUT : RGX_REC_OVERFLOWED) : (sums ? RGX_REC_COMPLETE_SUMS : RGX_REC_COMPLETE);
            reg[1] = (uint32_t)off;
            reg[4] = (uint32_t)states | (uint32_t)max(state_slot, 0) << 8;
            if (RAYS < 64) {
                reg[RGX_REC_MORE] = (uint32_t)more_from;
                reg[RGX_REC_MORE + 1] = (uint32_t)(more_slot + 1);
            }
            reg[2] = record_mark(P, 0);
            reg[3] = record_mark(P, 1);
        }
    }
};

// Stand-in where nothing is recorded: an image that no backward follows, or (WholeLists) one whose backward will search the tree.
struct NoRecorder {
    __device__ __forceinline__ void write_window(const MarchParams &, const TileLds &, int) {}
    __device__ __forceinline__ void write_lists(const MarchParams &, const TileLds &, int, bool) {}
    static constexpr int slot = -1;
    __device__ __forceinline__ void write_trailer(const MarchParams &, bool, float, float, bool) {}
    __device__ __forceinline__ void finish(const MarchParams &) {}
};
struct WholeLists : NoRecorder {};

__device__ __forceinline__ uint32_t uni_u32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// What the backward sums per Gaussian over rays and slabs, 13 words: sum y (d density), the colour
// gradient (3), sum y (Mx) (3) and the symmetric sum y (Mx)(Mx)^T (xx, yy, zz, xy, xz, yz), where
// Mx = S^-1 R^T (x - centre) is the sample point in the Gaussian's whitened frame.  Every
// gradient of the Gaussian is linear in these, so the change of variables below runs once per
// Gaussian and window (or row), not once per ray.
#define RGX_NSUM 13

// The 14 gradient words (density, rgb, position, scale, quaternion) from the 13 sums
// (backward/gaussians_aabb.cu:443-481).
__device__ __forceinline__ void sums_to_gradients(const Prim *pr, const float *s, float *out)
{
    const float4 q4 = pr->quat4, i4 = pr->inv_inter4;
    const float rho = pr->rgba4.w;
    f3 U, V, W;
    quat_to_cols(q4, U, V, W);
    const f3 inv_s = mk3(i4.x * i4.w, i4.y * i4.w, i4.z * i4.w);
    const f3 sc = mk3(1.0f / inv_s.x, 1.0f / inv_s.y, 1.0f / inv_s.z);
    const f3 Us = U * inv_s.x, Vs = V * inv_s.y, Ws = W * inv_s.z; // rows of M
    const f3 Vy = mk3(s[4], s[5], s[6]);
    out[0] = s[0];
    out[1] = s[1]; out[2] = s[2]; out[3] = s[3];
    // d position = rho M^T sum y (Mx)
    out[4] = rho * (Us.x * Vy.x + Vs.x * Vy.y + Ws.x * Vy.z);
    out[5] = rho * (Us.y * Vy.x + Vs.y * Vy.y + Ws.y * Vy.z);
    out[6] = rho * (Us.z * Vy.x + Vs.z * Vy.y + Ws.z * Vy.z);
    // d scale_a = rho sum y (Mx)_a^2 / scale_a
    out[7] = rho * s[7] * inv_s.x; out[8] = rho * s[8] * inv_s.y; out[9] = rho * s[9] * inv_s.z;
    // Q_a = sum y x (Mx)_a with x = R S (Mx);  d R column a = -rho Q_a / scale_a
    const f3 Ux = U * sc.x, Vx = V * sc.y, Wx = W * sc.z;
    const f3 Qx = (Ux * s[7] + Vx * s[10]) + Wx * s[11];
    const f3 Qy = (Ux * s[10] + Vx * s[8]) + Wx * s[12];
    const f3 Qz = (Ux * s[11] + Vx * s[12]) + Wx * s[9];
    const f3 d1 = Qx * (-rho * inv_s.x), d2 = Qy * (-rho * inv_s.y), d3 = Qz * (-rho * inv_s.z);
    const float qx = q4.x, qy = q4.y, qz = q4.z, qw = q4.w;
    // backward/gaussians_aabb.cu:469-481
    out[10] = 2 * qw * d1.y - 2 * qz * d1.z - 2 * qw * d2.x + 2 * qy * d2.z + 2 * qz * d3.x - 2 * qy * d3.y;
    out[11] = 2 * qz * d1.y + 2 * qw * d1.z + 2 * qz * d2.x - 4 * qy * d2.y + 2 * qx * d2.z + 2 * qw * d3.x - 2 * qx * d3.y -
              4 * qy * d3.z;
    out[12] = -4 * qz * d1.x + 2 * qy * d1.y - 2 * qx * d1.z + 2 * qy * d2.x + 2 * qw * d2.z + 2 * qx * d3.x + 2 * qw * d3.y -
              4 * qz * d3.z;
    out[13] = -4 * qw * d1.x + 2 * qx * d1.y + 2 * qy * d1.z - 2 * qx * d2.x - 4 * qw * d2.y + 2 * qz * d2.z + 2 * qy * d3.x +
              2 * qz * d3.y;
}

// The replaying backward keeps, per tile, the sums of the current window's Gaussians in LDS (one
// row of RGX_NSUM per table slot): the groups of lanes add their shares there (GroupAdd), and the
// gradients go to memory once per window instead of once per row, slab and Gaussian.
// The record as the replay reads it: the tile's region in memory, of which the words
// [at, at + RGX_STAGE_WORDS) are also held in LDS once stage() has fetched them.  An iteration's items are
// read word by word, each read depending on the last (a head gives a size gives the next head), and from
// memory every link of that chain is a round trip; staged, the chain costs one.  Words outside the staged
// range are read from memory as before.
#define RGX_STAGE_WORDS 448 // (as many as fit beside the rest: twelve tiles per CU)
template <bool STAGED, bool PARTS>
struct RecordView {
    const uint32_t *reg; // the tile's region
    uint32_t *lds;       // [RGX_STAGE_WORDS] (STAGED)
    int at;              // first staged word (wave-uniform)
    int used;            // words the forward wrote
    const uint32_t *more; // (PARTS) where words from `share` on are, less as many
    int share, more_from; // more_from: the item after which the stream goes on at `share`, or -1
    __device__ __forceinline__ uint32_t from_memory(int i) const
    {
        if constexpr (PARTS) return (i < share ? reg : more)[i];
        else return reg[i];
    }
    // where the next item after the one that ends at i begins
    __device__ __forceinline__ int next(int i) const { return PARTS && i == more_from ? share : i; }
    __device__ __forceinline__ uint32_t word(int i) const
    {
        if constexpr (STAGED) {
            const unsigned o = (unsigned)(i - at);
            return o < (unsigned)RGX_STAGE_WORDS ? lds[o] : from_memory(i);
        } else {
            return from_memory(i);
        }
    }
    __device__ __forceinline__ uint32_t uni(int i) const { return (uint32_t)__builtin_amdgcn_readfirstlane((int)word(i)); }
    __device__ __forceinline__ uint32_t byte(int i, int b) const { return (word(i + (b >> 2)) >> ((b & 3) * 8)) & 0xffu; } // byte b after word i
    __device__ __forceinline__ void stage(int from)
    {
        if constexpr (STAGED) {
            uint32_t v[RGX_STAGE_WORDS / 64];
#pragma unroll
            for (int k = 0; k < RGX_STAGE_WORDS / 64; ++k) {
                const int i = from + k * 64 + (int)threadIdx.x;
                v[k] = i < used ? from_memory(i) : 0u;
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < RGX_STAGE_WORDS / 64; ++k) lds[k * 64 + threadIdx.x] = v[k];
            at = from;
            __syncthreads();
        }
    }
};

struct ReplayLds {
    float *acc;        // [RGX_CCAP][RGX_NSUM]: a group's lanes meet a row in different banks
    uint32_t *pid;     // [RGX_CCAP]: the window's Gaussians by slot
    uint8_t *mark;     // [RGX_CCAP]: 0, or (the slot has something in acc) 1 + the group that last claimed it (GroupAdd)
    float *frame;      // [9][RGX_CCAP]: rotation columns U, V, W of the window's Gaussians
    uint8_t *rowlist;  // [4][RGX_CCAP]: the slot lists of the LISTS item whose gradient pass is running
};

// The window's sums go to memory, as gradients.  The lanes that turned a slot's sums into its 14 words leave them in LDS (in the place
// of the window's frames, which nobody needs any more), and 16 lanes add a Gaussian's words together: its 64 bytes are one
// request to memory.  Adding them from the lane that made them, 14 requests of 4 bytes for each Gaussian, was the bound of
// this kernel at 3 M Gaussians 1237x822 (12.2 -> 10.0 ms; 300 k 800x800: 2.8 -> 2.0).
#define RGX_FLUSH_ROW 15 // 14 words and the Gaussian
template <typename Cn>
__device__ __forceinline__ void replay_flush(const MarchParams &P, const ReplayLds &RL, Cn &cn)
{
    RGX_SEC(cn, RGX_SEC_WALK);
    __syncthreads();
    static_assert(64 * RGX_FLUSH_ROW <= 9 * RGX_CCAP, "a row per lane in the place of the frames");
    const int lane = threadIdx.x;
    for (int first = 0; first < RGX_CCAP; first += 64) {
        const int slot = first + lane;
        const bool mine = slot < RGX_CCAP && RL.mark[slot] != 0;
        const uint64_t touched = __ballot(mine);
        if (mine) {
            const uint32_t pid = RL.pid[slot];
            RL.mark[slot] = 0;
            cn.grad_atomics += 14;
            float sums[RGX_NSUM], out[14];
#pragma unroll
            for (int c = 0; c < RGX_NSUM; ++c) {
                sums[c] = RL.acc[slot * RGX_NSUM + c];
                RL.acc[slot * RGX_NSUM + c] = 0.f;
            }
            sums_to_gradients(P.prims + pid, sums, out);
            float *row = RL.frame + rank_in(touched) * RGX_FLUSH_ROW;
#pragma unroll
            for (int c = 0; c < 14; ++c) row[c] = out[c];
            row[14] = __uint_as_float(pid);
        }
        __syncthreads();
        const int n = __popcll(touched), c = lane & 15;
        for (int at = lane >> 4; at < n; at += 4) {
            const float *row = RL.frame + at * RGX_FLUSH_ROW;
            if (c < 14) unsafeAtomicAdd(P.gbuf + (int64_t)__float_as_uint(row[14]) * 16 + c, row[c]);
        }
        __syncthreads();
    }
    RGX_SEC(cn, RGX_SEC_FLUSH);
}

// Makes the WINDOW item at `at` the current window (sums of the previous one go to memory first).
template <typename Cn, typename Rv>
__device__ __forceinline__ void replay_window(const MarchParams &P, const ReplayLds &RL, const Rv &rv, int at, int &win_at, Cn &cn)
{
    if (at == win_at) return;
    replay_flush(P, RL, cn);
    const int C = (int)(rv.uni(at) & 0xffffu);
    for (int i = threadIdx.x; i < C && i < RGX_CCAP; i += 64) {
        const uint32_t pid = min(rv.word(at + 4 + i), (uint32_t)(P.n - 1));
        RL.pid[i] = pid;
        const Prim *pr = P.prims + pid;
        f3 U, V, W;
        quat_to_cols(pr->quat4, U, V, W);
        float *f = RL.frame + i;
        f[0] = U.x; f[RGX_CCAP] = U.y; f[2 * RGX_CCAP] = U.z;
        f[3 * RGX_CCAP] = V.x; f[4 * RGX_CCAP] = V.y; f[5 * RGX_CCAP] = V.z;
        f[6 * RGX_CCAP] = W.x; f[7 * RGX_CCAP] = W.y; f[8 * RGX_CCAP] = W.z;
    }
    win_at = at;
    __syncthreads();
}

// Replays one LISTS item.  WALK_ROWS: as shade_rows (the four rows walk their recorded lists in lock
// step); WALK 0 / 1: as shade_lanes over one half's entries; WALK_LANES_ALL: every ray walks all
// its hits; WALK_NONE: no walk.  COUNT adds the lane's hits to p0.  Returns the item's size.
enum { WALK_LANES_ALL = 2, WALK_ROWS_ALL = 3, WALK_NONE = 4 };
template <bool COUNT, int WALK, int RAYS, typename Body, typename Cn, typename Rv>
__device__ __forceinline__ int replay_lists(const MarchParams &P, const ReplayLds &RL, const Rv &rv, int it, bool run, int &p0, Body body, Cn &cn)
{
    const int lane = threadIdx.x, row = lane >> 4;
    const int nw = (int)(rv.uni(it) & 0xffu), len = (int)rv.uni(it + 1), q = (len + 3) >> 2;
    constexpr int HEAD = Part<RAYS>::LISTS_HEAD;
    const int slots_at = it + HEAD;                      // the slot bytes start at this word
    const int masks_at = slots_at + q + Part<RAYS>::ray(lane);    // word w of this lane: masks_at + w * RAYS
    if constexpr (WALK == WALK_NONE) {
        const int nwr = run ? min((len + 31) >> 5, nw) : 0;
        if (COUNT)
            for (int w = 0; w < nwr; ++w) p0 += __popc(rv.word(masks_at + w * RAYS));
    } else if constexpr (WALK != WALK_ROWS_ALL) {
        const int nwr = run ? min((len + 31) >> 5, nw) : 0;
        const int half_at = slots_at + q + nw * RAYS + ((WALK & 1) * Part<RAYS>::ROWS + (RAYS == 64 ? row : row % Part<RAYS>::ROWS)) * nw;
        auto word = [&](int w) { return WALK == WALK_LANES_ALL ? rv.word(masks_at + w * RAYS) : rv.word(masks_at + w * RAYS) & rv.word(half_at + w); };
        if (COUNT)
            for (int w = 0; w < nwr; ++w) p0 += __popc(rv.word(masks_at + w * RAYS));
        int w = 0;
        uint32_t bits = nwr > 0 ? word(0) : 0u;
        for (;;) {
            while (bits == 0u && w + 1 < nwr) bits = word(++w);
            const bool has = bits != 0u;
            if (!__any(has)) break;
            int slot = 0;
            if (has) {
                slot = min((int)rv.byte(slots_at, w * 32 + __builtin_ctz(bits)), RGX_CCAP - 1);
                bits &= bits - 1u;
            }
            const int32_t pid = (int32_t)RL.pid[slot];
            body(Entry<false>{(const float4 *)(RL.frame + slot), P.prims + pid, pid, slot}, has, has, Half<(WALK & 1)>{});
        }
    } else {
        RGX_SEC(cn, RGX_SEC_WALK);
        // the rows' slot lists go to LDS first: every trip starts by looking its slot up, and from memory that
        // look-up is a round trip at the head of the trip's chain of dependent loads
        const uint8_t *slots = RL.rowlist + row * RGX_CCAP;
        {
            uint32_t *dst = (uint32_t *)(RL.rowlist + row * RGX_CCAP);
            for (int i = lane & 15; i < min((len + 3) >> 2, RGX_CCAP / 4); i += 16) dst[i] = rv.word(slots_at + i);
            __syncthreads();
        }
        static_assert(!COUNT, "the rows' walk counts nothing");
        // Each half of a row (8 lanes, 2 x 4 pixels) walks the entries that one of its own rays hits: the set bits
        // of the OR of its lanes' masks.  Fewer trips than with whole rows in lock step (a trip lasts until the
        // longest list of the wave is done, and half a row's list is shorter than the row's).  Where a ray has copies the groups of the
        // same rays share their entries among themselves.
        using Pt = Part<RAYS>;
        const int copy = Pt::copy(lane);
        const int nwr = min((len + 31) >> 5, nw);
        auto lane_word = [&](int w) {
            const int left = len - w * 32;
            return (run ? rv.word(masks_at + w * RAYS) : 0u) & (left >= 32 ? ~0u : ((1u << left) - 1u));
        };
        auto group_or = [](uint32_t m) {
            m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xf, 0xf, true);  // quad_perm [1,0,3,2]
            m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xf, 0xf, true);  // quad_perm [2,3,0,1]
            m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, true); // row_half_mirror
            return m;
        };
        int w = 0;
        uint32_t mword = nwr > 0 ? lane_word(0) : 0u;
        uint32_t bits = Pt::skip(group_or(mword), copy);
#ifdef RGX_SECTION_CLOCKS
        asm volatile("" :: "v"(bits)); // the first words have arrived: their wait belongs to the set-up, not to the first trip
#endif
        RGX_SEC(cn, RGX_SEC_PRETRIP);
        // A trip's chain -- position in the list, slot, Gaussian, its record in memory -- is walked one trip ahead: the record's
        // words arrive while the trip before goes through its samples.
        struct Ahead {
            bool live, hit;
            int slot;
            int32_t pid;
            float4 pos4, inv4, rgba4;
        };
        auto ahead = [&]() {
            // (all lanes of a group hold the same bits and the same w: the DPP moves below run with the whole group active)
            while (nw > 1 && __any(bits == 0u && w + 1 < nwr)) {
                const bool next = bits == 0u && w + 1 < nwr;
                const uint32_t m = next ? lane_word(w + 1) : 0u;
                const uint32_t o = Pt::skip(group_or(m), copy);
                if (next) {
                    ++w;
                    mword = m;
                    bits = o;
                }
            }
            Ahead a;
            a.live = bits != 0u;
            const int pos = __builtin_ctz(bits | 0x80000000u);
            for (int k = 0; k < Pt::COPIES; ++k) bits &= bits - 1u;
            a.hit = a.live && ((mword >> pos) & 1u);
            a.slot = min((int)slots[min(w * 32 + pos, RGX_CCAP - 1)], RGX_CCAP - 1);
            a.pid = (int32_t)RL.pid[a.slot];
            const Prim *prim = P.prims + (uint32_t)a.pid;
            a.pos4 = prim->pos4;
            a.inv4 = prim->inv_inter4;
            a.rgba4 = prim->rgba4;
            return a;
        };
        Ahead next = ahead();
        while (__any(next.live)) {
            const Ahead a = next;
            next = ahead();
            body(EntryAhead{(const float4 *)(RL.frame + a.slot), P.prims + (uint32_t)a.pid, a.pid, a.slot, a.pos4, a.inv4, a.rgba4}, a.hit, a.live, HalfRows{});
        }
    }
    return HEAD + q + nw * (RAYS + 2 * Part<RAYS>::ROWS);
}

// Resident candidate window: the table holds every Gaussian of the tile frustum between the
// wave's nearest slab start and `hi`, so the next slab iterations reuse it without sweeping.
struct Window {
    float hi;
    int n;
    bool resident;
    int k;        // slabs to look ahead when a window is built
    bool crowded; // the last iteration's Gaussians did not fit one table
    bool plain;   // the resident table's entries all passed plain_roots()
};

__device__ __forceinline__ void frustum_range(Frustum &F, float t0, float t1)
{
    F.range(t0, t1, 2.0f * RGX_PAD_REL * fmaxf(t1, 1.0f));
}

// One slab iteration's work on the candidate tables, in two phases that share a single copy of
// the sweep and filter code:
//   phase 0  make the table cover the wave's intervals (reuse the resident window, or sweep a new
//            one looking Wn.k slabs ahead, or -- when even this iteration's own range overflows
//            the table -- walk it in table-sized batches), filter, body_a over the row lists;
//   mid(split) per lane, between the phases; returns whether the lane takes part in phase 1;
//   phase 1  body_b over the same row lists, or over freshly swept and filtered batches when the
//            candidates did not fit one table.
// WALK_FORWARD: body_a per ray over the entries reaching the first 16 samples, body_b per ray over
// those reaching the second 16.  WALK_BACKWARD: body_a per ray, once for each half; body_b over the
// row lists in lock step (it sums over the rays of a row).  WALK_ROWS: both bodies over the row lists.
// Returns the phase-1 participation flag of this lane.
enum { WALK_FORWARD, WALK_BACKWARD, WALK_ROWS };
template <int WALK, int ORDER, int RAYS = 64, typename Cn, typename Rec, typename BodyA, typename Mid, typename BodyB>
__device__ __forceinline__ bool slab_tables(const MarchParams &P, const TileLds &L, Frustum &F, Window &Wn, const RayState &R,
                                            bool need, float tlo, float thi, int &p0, bool &ov, float &found, float &searched_to,
                                            Cn &cn, Rec &rec, BodyA body_a, Mid mid, BodyB body_b)
{
    const bool srch = R.active && R.searching, want = need || srch;
    const float t0 = wave_min_all(want ? tlo : INFINITY), t1 = wave_max_all(want ? thi : -INFINITY);
    const bool any_search = __any(srch);
    const float tmid = fmaf(R.dt, (float)RGX_CHUNK_SIZE, R.tbuffer);
    // Where slabs hold more Gaussians than a table (the previous iteration found so), a forward
    // that no backward follows sweeps each half of the slab's depth range for its own phase instead
    // of the whole range twice: phase 0 takes the Gaussians that reach the first 16 samples,
    // phase 1 those that reach the second 16, and a Gaussian of both halves is counted once.
    // (A backward sweeps the whole range: where max_prim_slice cuts a ray's list, the halves keep other hits.  What a forward without a
    // record, but with a backward to come (WholeLists), takes for the whole range: 3 M Gaussians 1237x822 7.70 -> 9.0 ms, before a search of 53;
    // 1 M 800x800 4.78 -> 4.74.  A kernel of its own: with the choice at run time, images were 0.3 to 0.7 % slower.)
    const bool split = WALK == WALK_FORWARD && std::is_same<Rec, NoRecorder>::value && Wn.crowded && __any(need);
    int len = 0, q0 = 0, seen = 0;
    uint32_t own[2] = {0u, 0u}; // this ray's hits among the list's first 32 entries, by half of the samples
    bool run = need, qov = false;
    for (int phase = 0; phase < 2; ++phase) {
        const bool reuse = !split && Wn.resident && t1 <= Wn.hi;
        float lo = t0, hi = t1; // depth range of this phase's tables
        if (split) {
            if (phase == 0) hi = wave_max_all(need ? fminf(thi, tmid) : -INFINITY); // searching rays look as far as that
            else lo = wave_min_all(run && tmid < thi ? fmaxf(tlo, tmid) : INFINITY), hi = wave_max_all(run ? thi : -INFINITY);
            if (!(lo <= hi)) break; // no ray reaches into the second half
        }
        RGX_SEC(cn, RGX_SEC_TOP);
        Sweep S = {0, 0};
        if (!reuse) {
            float wend = hi;
            if (!split && phase == 0 && Wn.k > 1)
                wend = fmaxf(t1, wave_max_all(want ? tlo + (float)Wn.k * R.slab_spacing : -INFINITY));
            frustum_range(F, lo, wend);
            sweep_begin<ORDER>(P, S, F, L.queue, L.leafq);
        }
        bool first = true, more = true;
        while (more) {
            int C;
            bool plain;
            if (reuse) {
                C = Wn.n;
                plain = Wn.plain;
                more = false;
            } else {
                bool done;
                C = sweep_next<ORDER, ORDER == BY_PAIRS && std::is_same<Rec, NoRecorder>::value>(P, S, F, L.queue, L.leafq, L.tab, done, plain, cn);
                if (split) {
                    seen += C;
                } else if (phase == 0 && first) {
                    if (done) {
                        Wn.hi = F.t1;
                        Wn.n = C;
                        Wn.resident = true;
                        Wn.plain = plain;
                        Wn.crowded = false;
                        if (C > RGX_KHI) Wn.k = Wn.k > 1 ? Wn.k / 2 : 1;
                        else if (C < RGX_KLO && Wn.k < 32) Wn.k *= 2;
                    } else if (Wn.k > 1) {
                        Wn.k = 1; // too many Gaussians ahead: start over with this iteration's range only
                        frustum_range(F, t0, t1);
                        sweep_begin<ORDER>(P, S, F, L.queue, L.leafq);
                        continue;
                    } else {
                        Wn.resident = false;
                        Wn.crowded = true;
                    }
                }
                first = false;
                more = !done;
            }
            RGX_SEC(cn, RGX_SEC_SWEEP);
            if (phase == 0 && !reuse) rec.write_window(P, L, C);
            RGX_SEC(cn, RGX_SEC_LISTS);
            if (phase == 0 || !Wn.resident || split) {
                // phase 0 asks the lane's real question; a phase-1 re-filter only recounts the slab hits
                const float cover = split ? hi : (Wn.resident ? Wn.hi : t1); // this iteration's tables cover [t0, cover]
                const LaneQuery Q = {R.dir, run, tlo, thi, phase == 0 && srch, R.tbuffer, fminf(R.texit, cover), P.m.max_prim_slice, tmid};
                const bool real = phase == 0 || split; // counts into the lane's own p0 / ov
                int cnt = real ? p0 : q0;
                bool cut = real ? ov : qov;
                float best = phase == 0 ? found : -1.0f;
                const float to = phase == 0 && any_search ? cover : hi;
                if constexpr (RAYS == 64) filter_table(L, C, lo, to, Q, split ? 1 + phase : 0, plain, cnt, cut, best, len, own, cn);
                else filter_part<RAYS>(L, C, lo, to, Q, split ? 1 + phase : 0, plain, cnt, cut, best, len, own, cn);
                if (real) {
                    p0 = cnt;
                    ov = cut;
                } else {
                    q0 = cnt;
                    qov = cut;
                }
                RGX_SEC(cn, RGX_SEC_FILTER);
                if (phase == 0) {
                    found = best;
                    searched_to = fmaxf(Q.slo, Q.shi); // a split phase may end before a searching ray's start
                    rec.write_lists(P, L, len, !more);
                }
                RGX_SEC(cn, RGX_SEC_LISTS);
            }
            if constexpr (WALK == WALK_FORWARD) {
                static_assert(std::is_same<BodyA, BodyB>::value, "the forward shades both halves with one body");
                shade_lanes<0, RAYS>(P, L, len, run, phase, own, body_a);
            } else if constexpr (WALK == WALK_BACKWARD) {
                if (phase == 0) {
                    shade_lanes<0>(P, L, len, run, 0, own, body_a);
                    shade_lanes<1>(P, L, len, run, 1, own, body_a);
                } else {
                    shade_rows(P, L, len, run, body_b);
                }
            } else {
                if (phase == 0) shade_rows(P, L, len, run, body_a);
                else shade_rows(P, L, len, run, body_b);
            }
            RGX_SEC(cn, RGX_SEC_SHADE);
        }
        if (phase == 0) {
            rec.write_trailer(P, any_search, split ? hi : (Wn.resident ? Wn.hi : t1), found, __any(need && p0 > 0));
            RGX_SEC(cn, RGX_SEC_LISTS);
            run = mid(split);
            if (!__any(run)) break;
        }
    }
    if (split && seen < RGX_CCAP / 2) Wn.crowded = false; // sparse again: go back to resident windows
    if constexpr (WALK == WALK_FORWARD && std::is_same<Cn, Counters>::value) {
        // What is counted are whole lists: the hits of the second half for the rays that have ended in the first, which nothing shades.
        const bool ask = split && need && !run && tmid < thi;
        if (__any(ask)) {
            const Cn work = cn; // (nodes and candidates: those of the march)
            const float lo = wave_min_all(ask ? fmaxf(tlo, tmid) : INFINITY), hi = wave_max_all(ask ? thi : -INFINITY);
            frustum_range(F, lo, hi);
            Sweep S = {0, 0};
            sweep_begin<ORDER>(P, S, F, L.queue, L.leafq);
            for (bool done = false; !done;) {
                bool plain;
                const int C = sweep_next<ORDER, ORDER == BY_PAIRS && std::is_same<Rec, NoRecorder>::value>(P, S, F, L.queue, L.leafq, L.tab, done, plain, cn);
                const LaneQuery Q = {R.dir, ask, tlo, thi, false, 0.f, 0.f, P.m.max_prim_slice, tmid};
                float none = -1.0f;
                if constexpr (RAYS == 64) filter_table(L, C, lo, hi, Q, 2, plain, p0, ov, none, len, own, cn);
                else filter_part<RAYS>(L, C, lo, hi, Q, 2, plain, p0, ov, none, len, own, cn);
            }
            cn.nodes = work.nodes;
            cn.cands = work.cands;
            cn.cands_hit = work.cands_hit;
        }
    }
    return run;
}

// Size in words of the LISTS item at `it`.
template <int RAYS, typename Rv>
__device__ __forceinline__ int lists_size(const Rv &rv, int it)
{
    return Part<RAYS>::LISTS_HEAD + (((int)rv.uni(it + 1) + 3) >> 2) + (int)(rv.uni(it) & 0xffu) * (RAYS + 2 * Part<RAYS>::ROWS);
}

// Walks the record stream of one tile, or part of one, for the backward.
template <bool STAGED, int RAYS>
struct Replayer {
    RecordView<STAGED, (RAYS < 64)> rv; // the tile's region
    int at;              // next item
    int win_at;          // the WINDOW item whose Gaussians sit in RL.pid (-1: none yet)
    bool lost;           // the stream did not hold the items an iteration expects (the caller stops)
    ReplayLds RL;

    // The backward's iteration driven by the record instead of the tree: body_a per ray over the
    // recorded lists, once per half of the samples; mid(); body_b over the lists row by row.
    // SUMS: body_a(slot) reads the iteration's sample sums instead of walking the lists for them
    template <bool SUMS, typename Cn, typename BodyA, typename Mid, typename BodyB>
    __device__ __forceinline__ bool slab(const MarchParams &P, const RayState &R, bool need, int &p0, float &found,
                                         float &searched_to, Cn &cn, BodyA body_a, Mid mid, BodyB body_b)
    {
        const int start = rv.next(at), used = rv.used;
        rv.stage(start);
        int end = start; // the iteration's TRAIL item
        for (;;) {
            end = rv.next(end);
            if (end + 4 > used) break;
            const uint32_t head = rv.uni(end);
            int size;
            if ((head & 0xff000000u) == RGX_REC_WINDOW) size = 4 + (((int)(head & 0xffffu) + 3) & ~3);
            else if ((head & 0xff000000u) == RGX_REC_LISTS && end + 2 <= used) size = lists_size<RAYS>(rv, end);
            else break;
            if (end + size > used) break;
            end += size;
        }
        const uint32_t tr = end + 4 <= used ? rv.uni(end) : 0u;
        const bool any_search = tr & 1u;
        if ((tr & 0xff000000u) != RGX_REC_TRAIL || end + 4 + (any_search ? RAYS : 0) > used) {
            lost = true;
            mid(false);
            return false;
        }
        int dummy = 0;
        RGX_SEC(cn, RGX_SEC_PARSE);
        if constexpr (SUMS) {
            auto none = [](const auto &, bool, bool, auto) {};
            for (int a = start; a < end; a = rv.next(a)) {
                const uint32_t head = rv.uni(a);
                if ((head & 0xff000000u) == RGX_REC_WINDOW) {
                    replay_window(P, RL, rv, a, win_at, cn); // later iterations of the window carry no WINDOW item
                    a += 4 + (((int)(head & 0xffffu) + 3) & ~3);
                } else {
                    a += replay_lists<true, WALK_NONE, RAYS>(P, RL, rv, a, need, p0, none, cn);
                }
            }
            RGX_SEC(cn, RGX_SEC_COUNT);
            if (__any(need && p0 > 0)) {
                const uint32_t slot1 = rv.uni(end + 2);
                if (slot1 == 0u || slot1 > (uint32_t)P.sum_slots) {
                    lost = true;
                    mid(false);
                    return false;
                }
                body_a(P.sum_pool + (int64_t)(slot1 - 1u) * (P.sum_slot_words / 4));
            }
        } else {
            for (int a = start; a < end; a = rv.next(a)) {
                const uint32_t head = rv.uni(a);
                if ((head & 0xff000000u) == RGX_REC_WINDOW) {
                    replay_window(P, RL, rv, a, win_at, cn);
                    a += 4 + (((int)(head & 0xffffu) + 3) & ~3);
                } else {
                    replay_lists<true, 0, RAYS>(P, RL, rv, a, need, p0, body_a, cn);
                    a += replay_lists<false, 1, RAYS>(P, RL, rv, a, need, dummy, body_a, cn);
                }
            }
        }
        const float cover = __uint_as_float(rv.uni(end + 1));
        found = any_search ? __uint_as_float(rv.word(end + 4 + Part<RAYS>::ray(threadIdx.x))) : -1.0f;
        searched_to = fminf(R.texit, cover);
        at = end + 4 + (any_search ? RAYS : 0);
        const bool run = mid(false);
        if (__any(run)) {
            for (int b = start; b < end; b = rv.next(b)) {
                const uint32_t head = rv.uni(b);
                if ((head & 0xff000000u) == RGX_REC_WINDOW) {
                    replay_window(P, RL, rv, b, win_at, cn);
                    b += 4 + (((int)(head & 0xffffu) + 3) & ~3);
                } else {
                    b += replay_lists<false, WALK_ROWS_ALL, RAYS>(P, RL, rv, b, run, dummy, body_b, cn);
                }
            }
        }
        return run;
    }
};

#define RGX_TILE_LDS(ORDER)                                           \
    __shared__ int32_t s_queue[RGX_QCAP];                             \
    __shared__ int32_t s_leafq[(ORDER) == BY_PAIRS ? 192 : 128];      \
    __shared__ __align__(16) float s_tab[RGX_CCAP * RGX_TAB];         \
    __shared__ __align__(4) uint8_t s_list[RGX_CCAP];                 \
    __shared__ uint32_t s_mask[RGX_MASK_WORDS][64];                   \
    __shared__ uint32_t s_half[2][4][RGX_MASK_WORDS];                 \
    const TileLds L = {s_queue, s_leafq, s_tab, s_list, s_mask, s_half}

// lane -> pixel: row r = lane / 16 is the 4x4 block (r & 1, r >> 1) of the 8x8 tile
__device__ __forceinline__ void lane_pixel(int px0, int py0, int lane, int &px, int &py)
{
    const int row = lane >> 4, j = lane & 15;
    px = px0 + (row & 1) * 4 + (j & 3);
    py = py0 + (row >> 1) * 4 + (j >> 2);
}

// ---------------------------------------------------------------------------
// cuda_gui/helpers.h:45-50
__device__ __forceinline__ uint8_t quantize8(float x)
{
    x = fminf(fmaxf(x, 0.0f), 1.0f);
    const unsigned v = (unsigned)(x * 256.0f);
    return (uint8_t)(v < 255u ? v : 255u);
}

// Forward: __raygen__rg (gaussians_aabb.cu:205-340), accumulateChunk (112-180),
// colorBlendingT_chunked (182-203).  VIEWER: the interactive viewer's variant of the same march
// (cuda_gui/gaussians_aabb.cu): black background, uchar4 colours, and the expected depth
// sum T (1 - w) t over the samples (its colorBlendingT_chunked, 183-205).
// PAIRS: how the sweeps descend (sweep_next).  WHOLE: no record, and a backward that will search the tree (slab_tables).
// RAYS: of a tile that one wavefront marches (launch_forward).
template <bool PAIRS, bool RECORD, bool VIEWER, bool STATS, bool HALF = false, bool WHOLE = false, int RAYS = 64>
RGX_WAVES_ATTR_FWD(RECORD && RAYS < 64) __global__ __launch_bounds__(64) void k_march_fwd(const MarchParams P)
{
    static_assert(RECORD || !HALF, "the colour sums' format is a property of the record");
    static_assert(RAYS == 64 || !WHOLE, "a backward that searches the tree without a record goes tile by tile");
    // Fifty-two bytes, run once, that put the loops of the filter and of the shading elsewhere in the 64-byte lines they are fetched by.  The same instructions without them, or with 2 to 11 of the
    // thirteen, take 1 % longer for an image (30 k Gaussians in a ball 800x800 735 us, with them 728; 300 k with lobes 2 290, 2 262; 335 k 896x559 3 640, 3 608); every loop
    // at the beginning of a line costs 3 % (the padding before it is run).
    if constexpr (!RECORD && RAYS == 64) asm volatile(".rept 13\n\ts_nop 0\n\t.endr");
    using Pt = Part<RAYS>;
    static_assert(!(RECORD || PAIRS) || !WHOLE, "a search without a record goes by nodes");
    RGX_TILE_LDS(PAIRS);
    int px0, py0, tile, part = 0;
    if (!tile_origin(P, blockIdx.x, px0, py0, &tile, Pt::BITS, &part)) return; // whole wave
    const int copy = Pt::copy(threadIdx.x);
    px0 += Pt::WIDTH == 4 ? 4 * (part & 1) : 0;
    py0 += Pt::HEIGHT * (Pt::WIDTH == 4 ? part >> 1 : part);
    typename std::conditional<RECORD, Recorder<RAYS>, typename std::conditional<WHOLE, WholeLists, NoRecorder>::type>::type rec;
    if constexpr (RECORD) {
        const int64_t region = ((int64_t)tile << Pt::BITS) + part;
        rec = Recorder<RAYS>{P.records + region * P.rec_tile_words, RGX_REC_HEAD, P.rec_tile_words, false, P.sum_pool != nullptr, -1, P.rec_first};
        if (RAYS < 64 && P.sum_first) { // (the slot that it has to begin with)
            rec.batch_next = (uint32_t)region * (uint32_t)Pt::COPIES;
            rec.batch_left = Pt::COPIES;
        }
    }
    int px, py;
    lane_pixel(px0, py0, Pt::ray(threadIdx.x), px, py);
    const bool valid = px < P.cam.width && py < P.cam.height;
    CountersFor<STATS> cn;
    RGX_SEC_START(cn, 0);
    Frustum F;
    frustum_planes(P.cam, px0, py0, F, Pt::WIDTH, Pt::HEIGHT);
    RayState R;
    ray_begin(P, px, py, valid, false, R);
    {
        const float t_far = wave_max_all(R.active && R.texit < 1e30f ? R.texit : 0.f);
        if constexpr (PAIRS) frustum_cut_pairs(P, F, t_far, L.queue);
        else frustum_cut(P, F, t_far, L.queue);
    }
    const f3 dir = R.dir;
    float Cr = 0.f, Cg = 0.f, Cb = 0.f, depth = 0.f;
    Window Wn = {0.f, 0, false, 4, false, false};
    RGX_SEC(cn, RGX_SEC_SETUP);

    while (__any(R.active)) {
        float tlo, thi;
        const bool need = slab_begin(P, true, P.m.t_eps, R, tlo, thi);
        int p0 = 0;
        bool ov = false;
        float found = -1.0f, searched_to = 0.f;
        if (__any(need || (R.active && R.searching))) {
            const float dt = R.dt;
            if constexpr (RECORD) {
                if (rec.piece_due(P, false)) {
                    const bool reuse = Wn.resident && wave_max_all(need || (R.active && R.searching) ? thi : -INFINITY) <= Wn.hi;
                    if (rec.piece_due(P, reuse)) {
                        if constexpr (RAYS == 64) rec.begin_piece(P, R, Cr, Cg, Cb);
                        else rec.begin_piece(P, R, Pt::sum_of_all(Cr), Pt::sum_of_all(Cg), Pt::sum_of_all(Cb));
                        if (reuse) rec.write_window(P, L, Wn.n);
                    }
                }
            }
            float sg[RGX_CHUNK_SIZE], cr[RGX_CHUNK_SIZE], cg[RGX_CHUNK_SIZE], cb[RGX_CHUNK_SIZE];
#pragma unroll
            for (int i = 0; i < RGX_CHUNK_SIZE; ++i) sg[i] = cr[i] = cg[i] = cb[i] = 0.f;
            f3 rdt = dir * fmaf(dt, 0.5f, R.tbuffer); // samples 0..15
            auto accumulate = [&](const auto &e, bool hit, bool, auto) {
                if (hit) {
                    const float4 col = e.prim->rgba4;
                    f3 U, V, W, inv;
                    float k;
                    e.frame(U, V, W, inv, k);
                    HitSetup hs = hit_setup(U, V, W, inv, k, e.prim->pos4, dir, rdt, dt);
                    accumulate_samples(hs, col, sg, cr, cg, cb);
                }
            };
            [[maybe_unused]] float sum[4][Pt::EACH]; // (parts) a copy's run of the chunk's sums
            auto blend = [&](bool second_chunk) { // gaussians_aabb.cu:195-201
                const float first_sample = second_chunk ? 16.5f : 0.5f; // (viewer: cuda_gui/gaussians_aabb.cu:189)
                if constexpr (RAYS < 64) { // each copy has its run of the samples: all lanes, also of rays whose sums are zero
                    constexpr int N = Pt::EACH;
                    Pt::sums(sg, sum[0]);
                    Pt::sums(cr, sum[1]);
                    Pt::sums(cg, sum[2]);
                    Pt::sums(cb, sum[3]);
                    float w[N], s[N], T = R.T;
                    [[maybe_unused]] const float tbuffer = need ? R.tbuffer : 0.0f; // (a ray that is not marching may be at no finite place)
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        const float x = sum[0][i] * dt;
                        w[i] = __expf(-x);
                        s[i] = dt * ((1.0f - w[i]) * __builtin_amdgcn_rcpf(fmaxf(x, 1e-6f)));
                    }
                    if constexpr (RECORD) {
                        // one sample after the other, in every copy: a replay of the record rounds the transmittance the same way
                        float ws[N][Pt::COPIES];
#pragma unroll
                        for (int i = 0; i < N; ++i) Pt::of_all(w[i], ws[i]);
#pragma unroll
                        for (int k = 0; k < Pt::COPIES; ++k) {
                            T = copy == k ? R.T : T;
#pragma unroll
                            for (int i = 0; i < N; ++i) R.T *= ws[i][k];
                        }
                    } else {
                        float through[Pt::COPIES], all = w[0];
#pragma unroll
                        for (int i = 1; i < N; ++i) all *= w[i];
                        Pt::of_all(all, through);
#pragma unroll
                        for (int k = 0; k < Pt::COPIES; ++k) {
                            T = copy == k ? R.T : T;
                            R.T *= through[k];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        const float ts = T * s[i];
                        Cr = fmaf(ts, sum[1][i], Cr);
                        Cg = fmaf(ts, sum[2][i], Cg);
                        Cb = fmaf(ts, sum[3][i], Cb);
                        if constexpr (VIEWER) depth += T * (1.0f - w[i]) * fmaf(dt, first_sample + (float)(N * copy + i), tbuffer);
                        T *= w[i];
                    }
                    return;
                }
#pragma unroll
                for (int i = 0; i < RGX_CHUNK_SIZE; ++i) {
                    const float x = sg[i] * dt;
                    const float w = __expf(-x);
                    const float s = dt * ((1.0f - w) * __builtin_amdgcn_rcpf(fmaxf(x, 1e-6f))); // the reference's __fdividef
                    const float ts = R.T * s;
                    Cr = fmaf(ts, cr[i], Cr);
                    Cg = fmaf(ts, cg[i], Cg);
                    Cb = fmaf(ts, cb[i], Cb);
                    if constexpr (VIEWER) {
                        depth += R.T * (1.0f - w) * fmaf(dt, first_sample + (float)i, R.tbuffer);
                    }
                    R.T *= w;
                }
            };
            // the chunk's sums go to the iteration's sample-sum slot, if it has one
            auto keep_sums = [&](int first_sample, [[maybe_unused]] bool blended) {
                if constexpr (RECORD && RAYS < 64) {
                    if (rec.slot >= 0) {
                        if (!blended) {
#pragma unroll
                            for (int c = 0; c < 4; ++c)
#pragma unroll
                                for (int i = 0; i < Pt::EACH; ++i) sum[c][i] = 0.f;
                        }
                        float *slot = (float *)(P.sum_pool + (int64_t)rec.slot * (P.sum_slot_words / 4));
                        const int sample = first_sample + Pt::EACH * copy, ray = Pt::ray(threadIdx.x);
                        auto keep = [&](int c) { // [component][8][RAYS][4 samples]: 8 or 16 bytes at a time
                            constexpr int RUN = Pt::EACH < 4 ? Pt::EACH : 4;
                            typedef float run __attribute__((ext_vector_type(RUN)));
#pragma unroll
                            for (int i = 0; i < Pt::EACH; i += RUN) {
                                run v;
#pragma unroll
                                for (int k = 0; k < RUN; ++k) v[k] = sum[c][i + k];
                                __builtin_nontemporal_store(v, (run *)(slot + ((c * RGX_BUFFER_SIZE + sample + i) / 4 * RAYS + ray) * 4 + (sample + i) % 4));
                            }
                        };
                        keep(0);
                        if constexpr (!HALF) {
                            keep(1);
                            keep(2);
                            keep(3);
                        } else {
                            float big = 0.f;
#pragma unroll
                            for (int i = 0; i < Pt::EACH; ++i) big = fmaxf(big, fmaxf(fabsf(sum[1][i]), fmaxf(fabsf(sum[2][i]), fabsf(sum[3][i]))));
                            big = -Pt::least_of_all(-big);
                            const int e = big > 0.f ? __builtin_amdgcn_frexp_expf(big) : 0;
                            const float down = __builtin_amdgcn_ldexpf(1.0f, -e);
                            const int chunk = first_sample / RGX_CHUNK_SIZE;
                            uint32_t *col = (uint32_t *)slot + RGX_BUFFER_SIZE * RAYS + chunk * (24 * RAYS) + 3 * Pt::EACH / 2 * copy * RAYS + ray;
                            auto value = [&](int k) { return sum[1 + k % 3][k / 3] * down; };
#pragma unroll
                            for (int j = 0; j < 3 * Pt::EACH / 2; ++j) {
                                const __half2 two = __floats2half2_rn(value(2 * j), value(2 * j + 1));
                                __builtin_nontemporal_store(*(const uint32_t *)&two, col + j * RAYS);
                            }
                            if (copy == 0)
                                __builtin_nontemporal_store(__builtin_amdgcn_ldexpf(1.0f, e), slot + RGX_BUFFER_SIZE * RAYS + 2 * 24 * RAYS + chunk * RAYS + ray);
                        }
                    }
                } else if constexpr (RECORD) {
                    if (rec.slot >= 0) {
                        float *slot = (float *)(P.sum_pool + (int64_t)rec.slot * (P.sum_slot_words / 4));
                        // written once, read once by the backward: keep them out of the caches' way
                        const auto desc = __builtin_amdgcn_make_buffer_rsrc(slot, 0, P.sum_slot_words * 4, 0x00020000);
                        auto keep = [&](const float (&v)[RGX_CHUNK_SIZE], int component) {
#pragma unroll
                            for (int i = 0; i < RGX_CHUNK_SIZE; i += 4) {
                                const quad four = {v[i], v[i + 1], v[i + 2], v[i + 3]};
                                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(quad_bits, four), desc, threadIdx.x * 16,
                                                                       (component * RGX_BUFFER_SIZE + first_sample + i) * 256, 2);
                                // A store of 16 bytes reads its registers until one instruction later.  The compiler knows that of every form but this
                                // one, with an offset in a scalar register: a row's last four lanes have stored what the next instruction wrote there.
                                asm volatile("s_nop 0" ::"v"(four));
                            }
                        };
                        keep(sg, 0);
                        if constexpr (!HALF) {
                            keep(cr, 1);
                            keep(cg, 2);
                            keep(cb, 3);
                        } else {
                            const int chunk = first_sample / RGX_CHUNK_SIZE;
                            float big = 0.f;
#pragma unroll
                            for (int i = 0; i < RGX_CHUNK_SIZE; ++i) big = fmaxf(big, fmaxf(fabsf(cr[i]), fmaxf(fabsf(cg[i]), fabsf(cb[i]))));
                            // big = f * 2^e with f in [1/2, 1): everything times 2^-e lies in (-1, 1)
                            const int e = big > 0.f ? __builtin_amdgcn_frexp_expf(big) : 0;
                            const float down = __builtin_amdgcn_ldexpf(1.0f, -e);
                            uint32_t *col = (uint32_t *)slot + RGX_BUFFER_SIZE * 64 + chunk * (24 * 64) + threadIdx.x;
                            auto value = [&](int k) { return (k % 3 == 0 ? cr[k / 3] : k % 3 == 1 ? cg[k / 3] : cb[k / 3]) * down; };
#pragma unroll
                            for (int j = 0; j < 24; ++j) {
                                const __half2 two = __floats2half2_rn(value(2 * j), value(2 * j + 1));
                                __builtin_nontemporal_store(*(const uint32_t *)&two, col + j * 64);
                            }
                            __builtin_nontemporal_store(__builtin_amdgcn_ldexpf(1.0f, e),
                                                        slot + RGX_BUFFER_SIZE * 64 + 2 * 24 * 64 + chunk * 64 + threadIdx.x);
                        }
                    }
                }
            };
            auto second_half = [&](bool split) { // split: the hits of the second half are not known yet
                const bool has = need && (p0 > 0 || split);
                const bool blends = RAYS < 64 ? __any(has) : has;
                if (blends) blend(false);
                RGX_SEC(cn, RGX_SEC_BLEND);
                keep_sums(0, blends);
                RGX_SEC(cn, RGX_SEC_SUMS);
                // samples 16..31, only for rays still above the transmittance floor (gaussians_aabb.cu:190)
#pragma unroll
                for (int i = 0; i < RGX_CHUNK_SIZE; ++i) sg[i] = cr[i] = cg[i] = cb[i] = 0.f;
                rdt = dir * fmaf(dt, 16.5f, R.tbuffer);
                return has && R.T > P.m.t_eps;
            };
            const bool run2 = slab_tables<WALK_FORWARD, PAIRS, RAYS>(P, L, F, Wn, R, need, tlo, thi, p0, ov, found, searched_to, cn, rec, accumulate,
                                          second_half, accumulate);
            RGX_SEC(cn, RGX_SEC_TOP); // (what slab_tables did after its last section: nothing to speak of)
            const bool blends2 = RAYS < 64 ? __any(run2) : run2;
            if (blends2) blend(true);
            RGX_SEC(cn, RGX_SEC_BLEND);
            keep_sums(RGX_CHUNK_SIZE, blends2);
            RGX_SEC(cn, RGX_SEC_SUMS);
            if (need && p0 > 0 && copy == 0) {
                cn.slabs++;
                cn.hit_pairs += p0;
            }
            if constexpr (RECORD && RAYS < 64) rec.cut = rec.cut || __any(ov);
            if (ov && copy == 0) cn.overflow++;
        }
        if constexpr (STATS && RAYS < 64) {
            Counters mine = {};
            slab_end(R, need, p0, found, searched_to, mine);
            if (copy == 0) {
                cn.rays_hit += mine.rays_hit;
                cn.empty += mine.empty;
            }
        } else {
            slab_end(R, need, p0, found, searched_to, cn);
        }
        RGX_SEC(cn, RGX_SEC_END);
    }
    if constexpr (RAYS < 64) {
        Cr = Pt::sum_of_all(Cr);
        Cg = Pt::sum_of_all(Cg);
        Cb = Pt::sum_of_all(Cb);
        if constexpr (VIEWER) depth = Pt::sum_of_all(depth);
    }
    if (valid && copy == 0) {
        const int64_t ray = (int64_t)py * P.cam.width + px;
        if constexpr (VIEWER) {
            *(uchar4 *)(P.frame + 4 * ray) = make_uchar4(quantize8(Cr), quantize8(Cg), quantize8(Cb), 255);
            P.depth[ray] = depth;
        } else {
            const float bg = P.m.white_background ? 1.0f : 0.0f;
            P.ray_colors[3 * ray] = Cr + R.T * bg;
            P.ray_colors[3 * ray + 1] = Cg + R.T * bg;
            P.ray_colors[3 * ray + 2] = Cb + R.T * bg;
        }
    }
    if constexpr (STATS) {
        if (valid && copy == 0 && P.ray_counts) {
            const int64_t ray = (int64_t)py * P.cam.width + px;
            P.ray_counts[2 * ray] = cn.slabs;
            P.ray_counts[2 * ray + 1] = cn.hit_pairs;
        }
    }
    rec.finish(P);
    flush_stats(P.stats, cn);
    RGX_SEC(cn, RGX_SEC_EPILOGUE);
    RGX_SEC_FLUSH(cn, RECORD ? RGX_SECK_FWD_RECORD : RGX_SECK_FWD_PLAIN);
}

// ---------------------------------------------------------------------------
// sum over the 16 lanes of each row, left in every lane of the row.  (Every lane of these four
// patterns reads a lane of its own row, so bound_ctrl changes nothing but the instruction: without
// it the last stage, whose add the compiler sinks into the one-lane-per-row branch that uses it,
// costs a zeroed register and a move per value.)
template <int CTRL>
__device__ __forceinline__ float row_take(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int GROUP>
__device__ __forceinline__ float group_sum(float v)
{
    v += row_take<0xB1>(v);  // quad_perm [1,0,3,2]
    v += row_take<0x4E>(v);  // quad_perm [2,3,0,1]
    if constexpr (GROUP >= 8) v += row_take<0x141>(v); // row_half_mirror
    if constexpr (GROUP == 16) v += row_take<0x140>(v); // row_mirror
    return v;
}

// The 13 sums of a gradient trip over the 8 lanes of a group, in seven registers: r[c] is the group's sum of out[c]
// in the group's first four lanes and that of out[c + 7] in its last four (r[6] there: undefined).  The step between
// the two quads of a group writes with a bank mask (a bank = four lanes): the even banks add up component c, the odd
// banks component c + 7, so that the two steps inside the quads run on seven registers instead of thirteen.
// (Inline assembly because the compiler has no masked form of the data-parallel add.  The s_nop at either end is the
// two wait states this chip needs between a vector instruction's write and a data-parallel read of the register:
// the compiler counts them for its own instructions only.)
__device__ __forceinline__ void group_sums_split(const float (&out)[RGX_NSUM], float (&r)[7])
{
    static_assert(RGX_NSUM == 13, "seven and six");
    asm volatile("s_nop 1\n\t"
                 "v_add_f32_dpp %0, %7, %7 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %1, %8, %8 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %2, %9, %9 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %3, %10, %10 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %4, %11, %11 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %5, %12, %12 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %6, %13, %13 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %0, %14, %14 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "v_add_f32_dpp %1, %15, %15 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "v_add_f32_dpp %2, %16, %16 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "v_add_f32_dpp %3, %17, %17 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "v_add_f32_dpp %4, %18, %18 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "v_add_f32_dpp %5, %19, %19 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "s_nop 1"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6])
                 : "v"(out[0]), "v"(out[1]), "v"(out[2]), "v"(out[3]), "v"(out[4]), "v"(out[5]), "v"(out[6]), "v"(out[7]),
                   "v"(out[8]), "v"(out[9]), "v"(out[10]), "v"(out[11]), "v"(out[12]));
#pragma unroll
    for (int c = 0; c < 7; ++c) r[c] += row_take<0xB1>(r[c]); // quad_perm [1,0,3,2]
    __builtin_amdgcn_sched_barrier(0); // (a component's two steps one right after the other would wait for each other)
#pragma unroll
    for (int c = 0; c < 7; ++c) {
        r[c] += row_take<0x4E>(r[c]); // quad_perm [2,3,0,1]
        asm volatile("" : "+v"(r[c])); // (here, for all lanes: otherwise the last add moves under the condition of the adds to LDS and leaves a move behind)
    }
}

// LDS words that the lanes of one wavefront hand to each other: a wavefront's LDS accesses take place in program order,
// and these stay in it (plain ones the compiler may forward, or move past each other where lanes differ in address).
template <typename T>
__device__ __forceinline__ T lds_get(const T *p)
{
    return __hip_atomic_load((const __attribute__((address_space(3))) T *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
template <typename T>
__device__ __forceinline__ void lds_put(T *p, T v)
{
    __hip_atomic_store((__attribute__((address_space(3))) T *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Adds the groups' sums of a trip to those of their slots in LDS, every lane one or two of its group's.  An atomic float
// add takes the LDS unit, which all of a CU's wavefronts share, some four clocks a lane: at 3 M Gaussians 1237x822, with
// 5.9 groups adding in a trip, that was a seventh of the kernel's time.  So
//   where a row's two groups are at one slot, as often in dense scenes, the first adds for both (between rows it costs as much
//     as it saves);
//   of the groups that are then left at a slot, one adds by reading and writing it: every group leaves its number in the
//     slot's mark, and the one that finds its own there reads the slot's sums beforehand -- begin(), long enough before
//     end() that no wait is left -- and writes them back with its own added;
//   the others (a third to a quarter of the groups that add) add atomically after those writes.
// Backward with all groups adding atomically -> now: 3 M 1237x822 8.53 -> 7.58 ms, 300 k 800x800 2.00 -> 1.91, 1 M 800x800
// 4.98 -> 4.89.  (Without any adds it would take 7.37, 1.89 and 4.85.)
struct GroupAdd {
    bool todo, both, first; // this lane's group adds; for the row's other group as well; reading and writing the slot
    float old0, old1;       // what the slot's sums were before this trip
    // adds: the lane's group has something for `slot`
    __device__ __forceinline__ void begin(const float *acc, uint8_t *mark, int slot, bool adds)
    {
        const int lane = threadIdx.x, q = lane & 3;
        const int key = adds ? slot : -1 - lane;
        both = key == __builtin_amdgcn_update_dpp(0, key, 0x128, 0xf, 0xf, true); // row_ror:8
        todo = adds && !(both && (lane & 8));
        const uint8_t group = (uint8_t)((lane >> 3) + 1);
        if (todo) lds_put(mark + slot, group);
        first = lds_get(mark + slot) == group;
        const float *src = acc + slot * RGX_NSUM + ((lane & 4 ? 7 : 0) + q);
        old0 = lds_get(src);
        old1 = lds_get(src + (q < (lane & 4 ? 2 : 3) ? 4 : 0));
    }
    // r: as group_sums_split leaves it
    __device__ __forceinline__ void end(float *acc, const float (&r)[7], int slot) const
    {
        const int lane = threadIdx.x, q = lane & 3;
        const bool upper = lane & 4, two = q < (upper ? 2 : 3); // lane q of a quad: its components q and q + 4
        const float r0 = r[0], r1 = r[1], r2 = r[2], r3 = r[3], r4 = r[4], r5 = r[5], r6 = r[6];
        float v0 = q == 0 ? r0 : q == 1 ? r1 : q == 2 ? r2 : r3, v1 = q == 0 ? r4 : q == 1 ? r5 : r6;
        const float other0 = row_take<0x128>(v0), other1 = row_take<0x128>(v1);
        v0 = both ? v0 + other0 : v0;
        v1 = both ? v1 + other1 : v1;
        float *dst = acc + slot * RGX_NSUM + ((upper ? 7 : 0) + q);
        if (todo && first) {
            lds_put(dst, old0 + v0);
            if (two) lds_put(dst + 4, old1 + v1);
        }
        __builtin_amdgcn_wave_barrier();
        if (todo && !first) {
            unsafeAtomicAdd(dst, v0);
            if (two) unsafeAtomicAdd(dst + 4, v1);
        }
        __builtin_amdgcn_wave_barrier();
    }
};

// ---------------------------------------------------------------------------
// Backward: __raygen__rg of cuda_train/backward/gaussians_aabb.cu:209-497.
//
// Per blended slab: (1) per-sample density s_k and e_k = g.c_k/s_k over the hit
// list (accumulateChunk_backw, 113-184); (2) the prefix loop (330-352) giving,
// per sample, T_k (transmittance before the sample) and D_k = g.(C_final - C
// accumulated before k); (3) per hit, the sum over its in-range samples
// (353-442).  Writing w = exp(-power/2), a_k = T_k (1 - exp(-s_k dt)) / s_k,
// X_k = (T_k e_k - D_k) dt + a_k (g.c_i - e_k), every accumulator of the
// reference's per-hit loop is a moment of y_k = X_k w_k over the slab:
//   ddensity      = sum y_k
//   drgb          = g * rho * sum w_k a_k
//   dscale, dpos, dR: sums of y_k times polynomials of degree <= 2 in k, because
//   the sample point x_k = x_c + u_k dt dir (u_k = k - 15.5) is affine in k.
// So the inner loop carries three moments (sum y, sum y u, sum y u^2) instead of
// nineteen running sums; the `power < k^2` mask follows the forward's 32-step recurrence, i.e. it
// is the mask the forward blended with.  Per Gaussian the moments turn into 13 sums in its whitened
// frame (RGX_NSUM); those are summed over the rays of a group of lanes (a row of 16 in the walk by rows, half a
// row in a replay) with DPP adds and carried on by one lane per group (all eight in a replay: GroupAdd); the
// change of variables to the 14 gradient words comes after all sums.
// ORDER: how a search of the tree descends.  RAYS: of a tile, in a replay, as the forward had them; their copies share the gradient trips.  (A search of parts
// goes by the launch's part_bits, and has lanes to spare.)
template <bool REPLAY, bool SUMS, bool STATS, bool HALF = false, int ORDER = BY_NODES, int RAYS = 64>
__device__ __forceinline__ void march_bwd(const MarchParams &P)
{
    static_assert(REPLAY || !SUMS, "sample sums come with a record");
    static_assert(!REPLAY || ORDER == BY_NODES, "a replay searches no tree");
    static_assert(SUMS || !HALF, "the colour sums' format is a property of the sample sums");
    static_assert(REPLAY || RAYS == 64, "a search goes by part_bits");
    using Pt = Part<RAYS>;
    // A search in the place of a replay by parts has a grid for the parts, then one for the whole tiles.
    const unsigned of_parts = REPLAY || P.part_bits == 0 ? 0u : (gridDim.x / ((1u << P.part_bits) + 1u)) << P.part_bits;
    const int bits = REPLAY ? Pt::BITS : blockIdx.x < of_parts ? P.part_bits : 0;
    int px0, py0, tile, part = 0;
    // A launch that replays sample sums has a grid for every piece of the tiles' records, the last (longest) pieces first.
    const unsigned grid = SUMS ? gridDim.x / (unsigned)P.rec_pieces : gridDim.x;
    const int turn = P.rec_turn ? (int)(blockIdx.x & 7) : 0; // (the workgroup's XCD)
    const int piece = SUMS ? (2 * P.rec_pieces - 1 - (int)(blockIdx.x / grid) - turn) % P.rec_pieces : 0;
    if (!tile_origin(P, SUMS ? blockIdx.x % grid : REPLAY || bits > 0 ? blockIdx.x : blockIdx.x - of_parts, px0, py0, &tile, bits, &part)) return; // whole wave
    const uint32_t *reg = P.records ? P.records + (((int64_t)tile << (REPLAY ? bits : P.rec_bits)) + part) * P.rec_tile_words : nullptr;
    [[maybe_unused]] bool mine = true; // (a search)
    const int rays = REPLAY ? RAYS : 64 >> bits, width = bits > 1 ? 4 : 8, height = bits == 0 ? 8 : bits == 3 ? 2 : 4;
    px0 += bits > 1 ? 4 * (part & 1) : 0;
    py0 += height * (bits > 1 ? part >> 1 : part);
    if (REPLAY) {
        // overflowed, not this launch's, or with / without sample sums: another kernel handles the tile
        if (record_status(P, reg) != (SUMS ? RGX_REC_COMPLETE_SUMS : RGX_REC_COMPLETE)) return;
        if (SUMS && HALF != (P.m.record_format == 1)) return; // (the launcher picks the variant of the record's format)
        if (SUMS && piece > (int)(uni_u32(reg[4]) & 0xffu)) return; // the record has fewer pieces
    } else if (P.only_overflow && bits == P.rec_bits) {
        if (record_usable(P, reg) || (bits > 0 && record_uncut(P, reg))) return; // replayed, or the tile's
    } else if (P.only_overflow) {
        // The tile, for those of its parts whose lists a search in any order finds again: one for all of them costs less than one for each.
        mine = record_uncut(P, reg + ((int)threadIdx.x >> (6 - P.rec_bits)) * P.rec_tile_words);
        if (!__any(mine)) return;
    }
    const int lane = threadIdx.x;
    __shared__ float s_acc[REPLAY ? RGX_NSUM * RGX_CCAP : 1];
    __shared__ uint32_t s_pid[REPLAY ? RGX_CCAP : 1];
    __shared__ float s_frame[REPLAY ? 9 * RGX_CCAP : 1];
    __shared__ __align__(4) uint8_t s_rowlist[REPLAY ? 4 * RGX_CCAP : 4];
    __shared__ uint32_t s_stage[REPLAY && SUMS ? RGX_STAGE_WORDS : 1];
    __shared__ uint8_t s_mark[REPLAY ? RGX_CCAP : 1];
    const ReplayLds RL = {s_acc, s_pid, s_mark, s_frame, s_rowlist};
    if constexpr (REPLAY) {
        for (int i = lane; i < RGX_NSUM * RGX_CCAP; i += 64) s_acc[i] = 0.f;
        for (int i = lane; i < RGX_CCAP; i += 64) {
            s_pid[i] = 0u;
            s_mark[i] = 0;
        }
        __syncthreads();
    }
    int px, py;
    lane_pixel(px0, py0, Pt::ray(threadIdx.x), px, py);
    const int copy = REPLAY ? Pt::copy(threadIdx.x) : 0;
    const bool valid = px < P.cam.width && py < P.cam.height && (REPLAY || ((int)threadIdx.x < rays && mine));
    CountersFor<STATS> cn;
    RGX_SEC_START(cn, 1);
    RayState R;
    // a replay follows the forward's iteration sequence, so it takes the forward's conventions
    // (reciprocal multiply in the bbox test, clipped slab bounds); so does the search in the place of a replay
    const bool as_forward = REPLAY || P.only_overflow;
    ray_begin(P, px, py, valid, !as_forward, R);
    const f3 dir = R.dir;
    f3 g = mk3(0.f, 0.f, 0.f);
    float D = 0.f;
    if (valid) {
        const int64_t ray = (int64_t)py * P.cam.width + px;
        g = mk3(P.dloss[3 * ray], P.dloss[3 * ray + 1], P.dloss[3 * ray + 2]);
        D = dot3(g, mk3(P.fwd_colors[3 * ray], P.fwd_colors[3 * ray + 1], P.fwd_colors[3 * ray + 2]));
    }
    const bool any_odd = REPLAY && __any(!(fabsf(g.x) < INFINITY && fabsf(g.y) < INFINITY && fabsf(g.z) < INFINITY));

    // A replay of lists alone, by parts, adds a ray's hits up one after the other where its forward's copies each had some: its transmittance is the forward's up to
    // rounding, some 1e-6 of it.  So that no ray ends before the forward's did its floor lies below that; one that goes on for it finds no hit, and the
    // record's end is its own.
    constexpr bool LOOSE = REPLAY && !SUMS && RAYS < 64;
    const float t_floor = LOOSE ? P.m.t_eps * (1.0f - 0x1p-16f) : P.m.t_eps;

    // one slab iteration; `drive(need, tlo, thi, p0, ov, found, searched_to, body_a, mid, body_b)` supplies the hit lists
    auto iteration = [&](auto drive) {
        float tlo, thi;
        const bool need = slab_begin(P, as_forward, t_floor, R, tlo, thi);
        int p0 = 0;
        bool ov = false;
        float found = -1.0f, searched_to = 0.f;
        RGX_SEC(cn, RGX_SEC_TOP);
        if (__any(need || (R.active && R.searching))) {
            // (a ray that is not marching may be at no finite place)
            const float dt = R.dt, tbuffer = need ? R.tbuffer : 0.0f;
            // (1) s_k and g.c~_k  -> PA, PB
            float PA[RGX_BUFFER_SIZE], PB[RGX_BUFFER_SIZE];
#pragma unroll
            for (int i = 0; i < RGX_BUFFER_SIZE; ++i) PA[i] = PB[i] = 0.f;
            const f3 rdt0 = dir * fmaf(dt, 0.5f, tbuffer);
            const f3 rdt1 = dir * fmaf(dt, 16.5f, tbuffer);
            auto densities = [&](const auto &e, bool hit, bool, auto half) {
                if (hit) {
                    const float4 col = e.prim->rgba4, pos4 = e.prim->pos4;
                    const float rho = col.w;
                    const float ddc = dot3(g, mk3(col.x, col.y, col.z));
                    f3 U, V, W, inv;
                    float k;
                    e.frame(U, V, W, inv, k);
                    constexpr int base = decltype(half)::value * RGX_CHUNK_SIZE;
                    HitSetup hs = hit_setup(U, V, W, inv, k, pos4, dir, base ? rdt1 : rdt0, dt);
#pragma unroll
                    for (int i = base; i < base + RGX_CHUNK_SIZE; ++i) {
                        const float gw = hs.power < hs.cut ? gauss_weight(hs.power) : 0.0f;
                        PA[i] = fmaf(rho, gw, PA[i]);
                        PB[i] = fmaf(ddc, gw, PB[i]);
                        hs.power += hs.inc;
                        hs.inc += hs.inc_st;
                    }
                }
            };
            // (1') the same from the forward's sample sums: PA = sum rho w, PB = g . sum rgb rho w
            auto load_sums = [&](const float4 *slot) {
                RGX_SEC(cn, RGX_SEC_WALK);
                // Through a buffer descriptor: one register of address for all of them.  Six of the eight groups of four samples' colours are
                // in flight with the densities; with all of them the kernel has no register left, and the compiler makes
                // them wait for each other.
                constexpr int QUADS = RGX_BUFFER_SIZE / 4;
                const auto desc = __builtin_amdgcn_make_buffer_rsrc((void *)slot, 0, P.sum_slot_words * 4, 0x00020000);
                // A ray without a hit in the iteration asks past the end of the slot: the descriptor's check returns zeros, which is what the forward
                // stored, and reads nothing (150 k Gaussians 619x411, rays that leave the scene early beside rays that do not: 1.48 -> 1.37 ms).
                // (The stores of the zeros stay: lines written in part cost the forward more, 2.01 -> 2.30 there.)
                const int mine = need && p0 > 0 ? (RAYS == 64 ? lane : copy * (QUADS / Pt::COPIES) * RAYS + Pt::ray(lane)) * 16 : P.sum_slot_words * 4;
                auto load = [&](int i) { return __builtin_bit_cast(quad, __builtin_amdgcn_raw_buffer_load_b128(desc, mine, i * (RAYS * 16), 2)); };
                if constexpr (RAYS < 64) { // each copy its run of the samples, in the first places (prefix)
                    constexpr int OWN = RGX_BUFFER_SIZE / Pt::COPIES, OWN_QUADS = OWN / 4;
                    quad d[OWN_QUADS], r[OWN_QUADS], gr[OWN_QUADS], b[OWN_QUADS];
#pragma unroll
                    for (int i = 0; i < OWN_QUADS; ++i) {
                        d[i] = load(i);
                        if constexpr (!HALF) {
                            r[i] = load(QUADS + i);
                            gr[i] = load(2 * QUADS + i);
                            b[i] = load(3 * QUADS + i);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < OWN_QUADS; ++i)
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            PA[4 * i + k] = d[i][k];
                            if constexpr (!HALF) PB[4 * i + k] = fmaf(g.x, r[i][k], fmaf(g.y, gr[i][k], g.z * b[i][k]));
                        }
                    if constexpr (HALF) {
                        const int chunk = copy * OWN / RGX_CHUNK_SIZE, first = copy * OWN % RGX_CHUNK_SIZE;
                        const uint32_t *col = (const uint32_t *)slot + RGX_BUFFER_SIZE * RAYS + (chunk * 24 + 3 * first / 2) * RAYS + Pt::ray(lane);
                        const f3 gs = g * __builtin_nontemporal_load((const float *)slot + RGX_BUFFER_SIZE * RAYS + 2 * 24 * RAYS + chunk * RAYS + Pt::ray(lane));
                        float v[3 * OWN];
#pragma unroll
                        for (int j = 0; j < 3 * OWN / 2; ++j) {
                            const uint32_t w = __builtin_nontemporal_load(col + j * RAYS);
                            const float2 two = __half22float2(*(const __half2 *)&w);
                            v[2 * j] = two.x;
                            v[2 * j + 1] = two.y;
                        }
#pragma unroll
                        for (int i = 0; i < OWN; ++i) PB[i] = fmaf(gs.x, v[3 * i], fmaf(gs.y, v[3 * i + 1], gs.z * v[3 * i + 2]));
                    }
                    RGX_SEC(cn, RGX_SEC_SUMS);
                    return;
                }
#pragma unroll
                for (int i = 0; i < QUADS; ++i) {
                    const quad d = load(i);
#pragma unroll
                    for (int k = 0; k < 4; ++k) PA[4 * i + k] = d[k];
                }
                if constexpr (!HALF) {
                    quad r[QUADS], gr[QUADS], b[QUADS];
                    auto ask = [&](int i) {
                        r[i] = load(QUADS + i);
                        gr[i] = load(2 * QUADS + i);
                        b[i] = load(3 * QUADS + i);
                        __builtin_amdgcn_sched_barrier(0);
                    };
#pragma unroll
                    for (int i = 0; i < 6; ++i) ask(i);
#pragma unroll
                    for (int i = 0; i < QUADS; ++i) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) PB[4 * i + k] = fmaf(g.x, r[i][k], fmaf(g.y, gr[i][k], g.z * b[i][k]));
                        __builtin_amdgcn_sched_barrier(0);
                        if (i + 6 < QUADS) ask(i + 6);
                    }
                } else {
#pragma unroll
                    for (int chunk = 0; chunk < 2; ++chunk) {
                        const uint32_t *col = (const uint32_t *)slot + RGX_BUFFER_SIZE * RAYS + chunk * (24 * RAYS) + Pt::ray(lane);
                        const float up = __builtin_nontemporal_load((const float *)slot + RGX_BUFFER_SIZE * RAYS + 2 * 24 * RAYS + chunk * RAYS + Pt::ray(lane));
                        const f3 gs = g * up; // the chunk's power of two goes into dL/dC once instead of into 48 sums
                        float v[48];
#pragma unroll
                        for (int j = 0; j < 24; ++j) {
                            const uint32_t w = __builtin_nontemporal_load(col + j * RAYS);
                            const float2 two = __half22float2(*(const __half2 *)&w);
                            v[2 * j] = two.x;
                            v[2 * j + 1] = two.y;
                        }
#pragma unroll
                        for (int i = 0; i < RGX_CHUNK_SIZE; ++i)
                            PB[chunk * RGX_CHUNK_SIZE + i] = fmaf(gs.x, v[3 * i], fmaf(gs.y, v[3 * i + 1], gs.z * v[3 * i + 2]));
                    }
                }
                RGX_SEC(cn, RGX_SEC_SUMS);
            };
            // (2) prefix: PA <- a_k, PB <- (T_k e_k - D_k) dt - a_k e_k   (so X_k = PB + PA * g.c_i);
            // it always covers all 32 samples (330-352)
            float T_after = R.T, D_after = D;
            bool use_second = true; // transmittance at the chunk boundary gates the second chunk (398)
            auto prefix = [&](bool) {
                RGX_SEC(cn, RGX_SEC_WALK);
                const bool has = need && p0 > 0;
                if constexpr (SUMS && RAYS < 64) {
                    // Each copy goes through its run of the samples, and has the others' results handed over (a ray without a hit goes through zeros).
                    // (All samples in every copy: a step of 4 k Gaussians 256x256 0.83 instead of 0.79 ms, 100 k in a ball 1.17 instead of 1.14.)
                    constexpr int OWN = RGX_BUFFER_SIZE / Pt::COPIES;
                    float w[OWN], e[OWN], inv_d[OWN], all[Pt::COPIES], T = R.T, T_mid = R.T, sum = 0.f, before[OWN];
                    T_after = R.T;
#pragma unroll
                    for (int i = 0; i < OWN; ++i) {
                        const float sd = PA[i];
                        inv_d[i] = sd > 0.0f ? __builtin_amdgcn_rcpf(sd) : 0.0f;
                        e[i] = PB[i] * inv_d[i];
                        w[i] = __expf(-sd * dt);
                    }
                    // the transmittance one sample after the other, as the forward rounded it
                    float ws[OWN][Pt::COPIES];
#pragma unroll
                    for (int i = 0; i < OWN; ++i) Pt::of_all(w[i], ws[i]);
#pragma unroll
                    for (int k = 0; k < Pt::COPIES; ++k) {
                        T = copy == k ? T_after : T;
                        if (k * OWN == RGX_CHUNK_SIZE) T_mid = T_after;
#pragma unroll
                        for (int i = 0; i < OWN; ++i) T_after *= ws[i][k];
                    }
#pragma unroll
                    for (int i = 0; i < OWN; ++i) {
                        const float a = T * (1.0f - w[i]) * inv_d[i];
                        before[i] = sum;
                        sum += T * (1.0f - w[i]) * e[i];
                        PA[i] = a;
                        PB[i] = T * e[i];
                        T *= w[i];
                    }
                    Pt::of_all(sum, all);
                    float D_own = D;
#pragma unroll
                    for (int k = 0; k < Pt::COPIES; ++k) {
                        D_own = copy == k ? D_after : D_own;
                        D_after -= all[k];
                    }
#pragma unroll
                    for (int i = 0; i < OWN; ++i) PB[i] = (PB[i] - (D_own - before[i])) * dt - PA[i] * e[i];
#pragma unroll
                    for (int i = 0; i < OWN; ++i) {
                        float a[Pt::COPIES], b[Pt::COPIES];
                        Pt::of_all(PA[i], a);
                        Pt::of_all(PB[i], b);
#pragma unroll
                        for (int k = 0; k < Pt::COPIES; ++k) { // (the run itself last: it lies in the first places)
                            w[i] = a[0];
                            e[i] = b[0];
                            if (k > 0) {
                                PA[k * OWN + i] = a[k];
                                PB[k * OWN + i] = b[k];
                            }
                        }
                    }
#pragma unroll
                    for (int i = 0; i < OWN; ++i) {
                        PA[i] = w[i];
                        PB[i] = e[i];
                    }
                    use_second = T_mid > P.m.t_eps;
                    RGX_SEC(cn, RGX_SEC_BLEND);
                    return has;
                }
                if (has) {
                    float T_mid = R.T;
#pragma unroll
                    for (int i = 0; i < RGX_BUFFER_SIZE; ++i) {
                        if (i == RGX_CHUNK_SIZE) T_mid = T_after;
                        const float sd = PA[i];
                        const float inv_d = sd > 0.0f ? __builtin_amdgcn_rcpf(sd) : 0.0f;
                        const float e = PB[i] * inv_d;
                        const float w = __expf(-sd * dt);
                        const float a = T_after * (1.0f - w) * inv_d;
                        PA[i] = a;
                        PB[i] = (T_after * e - D_after) * dt - a * e;
                        D_after -= T_after * (1.0f - w) * e;
                        T_after *= w;
                    }
                    use_second = T_mid > P.m.t_eps;
                }
                RGX_SEC(cn, RGX_SEC_BLEND);
                return has;
            };
            // (3) per table entry: moments per lane, row sum, one set of atomics per row
            auto gradients = [&](const auto &e, bool hit, bool live, auto which) {
                constexpr int GROUP = decltype(which)::group; // lanes that share this trip's entry
                static_assert(!REPLAY || GROUP == 8, "a replay walks by half rows");
                RGX_SEC(cn, RGX_SEC_WALK);
                const uint64_t bal = __ballot(hit);
                GroupAdd add;
                float out[RGX_NSUM];
                // In a replay all lanes go through the trip, those without a hit with a Gaussian of no extent (k = 0: no sample
                // is inside its cut-off, and its whitened frame is zero): their sums come out as zeros, and neither those
                // nor a branch have to be made for them (3 M 1237x822 7.56 -> 7.44 ms, 4 k 128x128 0.161 -> 0.157).
                // (Where dL/dC is no number, zero times that is not zero: any_odd.)
                if constexpr (!REPLAY) {
#pragma unroll
                    for (int c = 0; c < RGX_NSUM; ++c) out[c] = 0.f;
                }
                const int32_t pid = e.pid;
                if (REPLAY || hit) {
                    const float4 col = e.colour(), e5 = e.position();
                    f3 U, V, W, inv;
                    float k;
                    e.frame(U, V, W, inv, k);
                    if constexpr (REPLAY) k = hit ? k : 0.0f;
                    const float rho = col.w;
                    const float dcg = dot3(mk3(col.x, col.y, col.z), g) * __builtin_amdgcn_rcpf(rho);
                    // the forward's sample recurrence (the mask is the one the forward blended with)
                    HitSetup hs = hit_setup(U, V, W, inv, k, e5, dir, rdt0, dt);
                    const f3 Mx0 = hs.Mx0, Md = hs.Md;
                    const float cut0 = hs.cut, cut1 = use_second ? cut0 : -1.0f; // (the second chunk's gate is in its cut-off)
                    float s0 = 0.f, s1 = 0.f, s2 = 0.f, gc = 0.f;
#pragma unroll
                    for (int b = 0; b < RGX_BUFFER_SIZE; b += RGX_SAMPLE_BLOCK) {
                        SampleBlock S;
                        S.step(hs, b < RGX_CHUNK_SIZE ? cut0 : cut1);
                        if (!__builtin_amdgcn_inverse_ballot_w64(S.any)) continue;
#pragma unroll
                        for (int j = 0; j < RGX_SAMPLE_BLOCK; ++j) {
                            const int i = b + j;
                            const float wd = gauss_weight(S.power[j]);
                            const float y = fmaf(PA[i], dcg, PB[i]) * wd;
                            const float u = (float)i - 15.5f;
                            // (see accumulate_samples; here only scalar moves write the mask, and s0 to gc next go through
                            // the moments' arithmetic)
                            asm("s_mov_b64 exec, %[in]\n\tv_add_f32_e32 %[s0], %[y], %[s0]\n\tv_fmac_f32_e32 %[s1], %[u], %[y]\n\t"
                                "v_fmac_f32_e32 %[s2], %[uu], %[y]\n\tv_fmac_f32_e32 %[gc], %[a], %[w]\n\ts_mov_b64 exec, %[l]"
                                : [s0] "+&v"(s0), [s1] "+&v"(s1), [s2] "+&v"(s2), [gc] "+&v"(gc)
                                : [in] "s"(S.in[j]), [y] "v"(y), [a] "v"(PA[i]), [w] "v"(wd), [u] "i"(__builtin_bit_cast(uint32_t, u)),
                                  [uu] "i"(__builtin_bit_cast(uint32_t, u * u)), [l] "s"(S.any));
                        }
                    }
                    if constexpr (REPLAY) add.begin(s_acc, s_mark, e.slot, live && ((bal >> (lane & ~7)) & 0xffull) != 0);
                    // moments -> sums in the whitened frame.  (Mx)_k = Mxc + u_k dt Md, Mxc at the slab centre (u = 0)
                    const f3 Mxc = Mx0 + Md * (15.5f * dt);
                    const float m1 = s1 * dt, m2 = s2 * (dt * dt);
                    // sum y (Mx) = B;  sum y (Mx)_a (Mx)_b = Mxc_a B_b + Md_a E_b
                    const f3 B = Mxc * s0 + Md * m1, E = Mxc * m1 + Md * m2;
                    const float gcol = gc * rho;
                    out[0] = s0;
                    out[1] = g.x * gcol; out[2] = g.y * gcol; out[3] = g.z * gcol;
                    if (REPLAY && __builtin_expect(any_odd, 0)) {
#pragma unroll
                        for (int c = 1; c < 4; ++c) out[c] = hit ? out[c] : 0.f;
                    }
                    out[4] = B.x; out[5] = B.y; out[6] = B.z;
                    out[7] = fmaf(Mxc.x, B.x, Md.x * E.x);
                    out[8] = fmaf(Mxc.y, B.y, Md.y * E.y);
                    out[9] = fmaf(Mxc.z, B.z, Md.z * E.z);
                    out[10] = fmaf(Mxc.x, B.y, Md.x * E.y);
                    out[11] = fmaf(Mxc.x, B.z, Md.x * E.z);
                    out[12] = fmaf(Mxc.y, B.z, Md.y * E.z);
                }
                // summed over the group's rays; one lane per group carries the sums on
                if constexpr (REPLAY) {
                    float r[7];
                    group_sums_split(out, r);
                    add.end(s_acc, r, e.slot);
                    RGX_SEC(cn, RGX_SEC_SHADE);
                    return;
                }
#pragma unroll
                for (int c = 0; c < RGX_NSUM; ++c) out[c] = group_sum<GROUP>(out[c]);
                if ((lane & (GROUP - 1)) == 0 && live && ((bal >> lane) & ((1ull << GROUP) - 1ull))) {
                    // to memory
                    float grad[14];
                    sums_to_gradients(e.prim, out, grad);
                    float *dst = P.gbuf + (int64_t)pid * 16;
#pragma unroll
                    for (int c = 0; c < 14; ++c) unsafeAtomicAdd(dst + c, grad[c]);
                    cn.grad_atomics += 14;
                }
                RGX_SEC(cn, RGX_SEC_SHADE);
            };
            bool has;
            if constexpr (SUMS) has = drive(need, tlo, thi, p0, ov, found, searched_to, load_sums, prefix, gradients);
            else has = drive(need, tlo, thi, p0, ov, found, searched_to, densities, prefix, gradients);
            if (has) {
                D = D_after;
                R.T = T_after;
                if (copy == 0) {
                    cn.slabs++;
                    cn.hit_pairs += p0;
                }
            }
            if (ov) cn.overflow++;
        }
        RGX_SEC(cn, RGX_SEC_WALK);
        if constexpr (STATS && RAYS < 64) {
            Counters mine = {};
            slab_end(R, need, p0, found, searched_to, mine);
            if (copy == 0) {
                cn.rays_hit += mine.rays_hit;
                cn.empty += mine.empty;
            }
        } else {
            slab_end(R, need, p0, found, searched_to, cn);
        }
        RGX_SEC(cn, RGX_SEC_END);
    };

    RGX_SEC(cn, RGX_SEC_SETUP);
    if constexpr (REPLAY) {
        // (a part's stream may go on in a slot of the pool)
        const int most = P.rec_tile_words + (RAYS < 64 && uni_u32(reg[RGX_REC_MORE + 1]) != 0u ? P.sum_slot_words * Pt::COPIES : 0);
        int used = min((int)uni_u32(reg[1]), most), start = RGX_REC_HEAD;
        if constexpr (SUMS) {
            const int states = (int)(uni_u32(reg[4]) & 0xffu);
            if (piece < states && piece + 1 < P.rec_pieces) used = min((int)uni_u32(reg[5 + piece]), used);
            const uint32_t state_slot = uni_u32(reg[4]) >> 8;
            if (piece > 0 && state_slot < (uint32_t)P.sum_slots) {
                // the piece starts with the state the forward had there; what the loss's gradient still sees of the ray's
                // colour is what the forward had not yet added to it
                start = min((int)uni_u32(reg[5 + piece - 1]), used);
                const float *st = (const float *)(P.sum_pool + (int64_t)state_slot * (P.sum_slot_words / 4)) + (piece - 1) * (8 * RAYS) + Pt::ray(lane);
                R.T = st[0];
                R.tbuffer = st[RAYS];
                R.tenter = st[2 * RAYS];
                R.dt = st[3 * RAYS];
                R.slab_spacing = R.dt * RGX_BUFFER_SIZE;
                D -= dot3(g, mk3(st[4 * RAYS], st[5 * RAYS], st[6 * RAYS]));
                const uint32_t flags = ((const uint32_t *)st)[7 * RAYS];
                R.active = flags & 1u;
                R.searching = flags & 2u;
                R.first = flags & 4u;
            }
        }
        const uint32_t *more = reg;
        int share = 0, more_from = -1;
        if constexpr (RAYS < 64) {
            share = P.rec_tile_words;
            const uint32_t slot1 = uni_u32(reg[RGX_REC_MORE + 1]);
            if (slot1 != 0u && slot1 - 1u + (uint32_t)Pt::COPIES <= (uint32_t)P.sum_slots) {
                more_from = (int)uni_u32(reg[RGX_REC_MORE]);
                more = (const uint32_t *)(P.sum_pool + (int64_t)(slot1 - 1u) * (P.sum_slot_words / 4)) - share;
            }
        }
        Replayer<SUMS, RAYS> rp = {RecordView<SUMS, (RAYS < 64)>{reg, s_stage, -(1 << 30), used, more, share, more_from}, start, -1, false, RL};
        while (__any(R.active) && !rp.lost && (!(SUMS || LOOSE) || rp.at < used)) {
            iteration([&](bool need, float, float, int &p0, bool &, float &found, float &searched_to, auto a, auto mid, auto b) {
                return rp.template slab<SUMS>(P, R, need, p0, found, searched_to, cn, a, mid, b);
            });
        }
        replay_flush(P, RL, cn);
        if ((rp.lost || rp.at != rp.rv.used) && lane == 0) {
            cn.replay_lost = 1;
            if (P.faults) atomicAdd(&P.faults[0], 1u); // counted with or without a statistics block
        }
    } else {
        RGX_TILE_LDS(ORDER);
        Frustum F;
        frustum_planes(P.cam, px0, py0, F, width, height);
        {
            const float t_far = wave_max_all(R.active && R.texit < 1e30f ? R.texit : 0.f);
            if constexpr (ORDER == BY_PAIRS) frustum_cut_pairs(P, F, t_far, L.queue);
            else frustum_cut(P, F, t_far, L.queue);
        }
        Window Wn = {0.f, 0, false, 4, false, false};
        NoRecorder rec;
        while (__any(R.active)) {
            iteration([&](bool need, float tlo, float thi, int &p0, bool &ov, float &found, float &searched_to, auto a, auto mid,
                          auto b) { return slab_tables<WALK_BACKWARD, ORDER>(P, L, F, Wn, R, need, tlo, thi, p0, ov, found, searched_to, cn, rec, a, mid, b); });
        }
    }
    flush_stats(P.stats, cn);
    RGX_SEC(cn, RGX_SEC_EPILOGUE);
    RGX_SEC_FLUSH(cn, REPLAY ? (SUMS ? RGX_SECK_BWD_SUMS : RGX_SECK_BWD_LISTS) : RGX_SECK_BWD_TREE);
}

// Launch order of the replaying backward.  A tile is one wavefront's work from start to end, so a
// launch ends with a tail in which ever fewer tiles are still running; the tail is as long as the
// tiles that start last.  The records say how much work each tile is (words used), so every XCD
// takes its tiles from the largest record to the smallest and the tail consists of the cheapest
// tiles.  One workgroup per XCD list: counting sort over 1024 size classes (order within a class
// does not matter); tiles outside the image and tiles without a usable record go last.
#define RGX_ORDER_BINS 1024
// the sum of the values of the threads before this one; s_wave: a word per wavefront
__device__ __forceinline__ uint32_t block_sum_before(uint32_t v, uint32_t *s_wave)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t upto = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(upto, o);
        if (lane >= o) upto += t;
    }
    if (lane == 63) s_wave[wave] = upto;
    __syncthreads();
    uint32_t before = upto - v;
    for (int w = 0; w < wave; ++w) before += s_wave[w];
    return before;
}
__global__ __launch_bounds__(256) void k_tile_order(const MarchParams P)
{
    __shared__ uint32_t s_bin[RGX_ORDER_BINS];
    __shared__ uint32_t s_part[4];
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    const int per_block = g.bw * g.bh, cnt = g.per_xcd * per_block, xcd = blockIdx.x;
    auto size_class = [&](int j) -> uint32_t {
        const int block = xcd + 8 * (j / per_block), within = j % per_block;
        const int tx = (block % g.blocks_x) * g.bw + within % g.bw;
        const int ty = (block / g.blocks_x) * g.bh + within / g.bw;
        if (tx >= P.tiles_x || ty >= P.tiles_y) return 0u;
        const uint32_t *reg = P.records + (int64_t)(ty * P.tiles_x + tx) * P.rec_tile_words;
        if (!record_usable(P, reg)) return 0u;
        const uint64_t used = min(reg[1], (uint32_t)P.rec_tile_words);
        return 1u + (uint32_t)(used * (RGX_ORDER_BINS - 2) / (uint32_t)P.rec_tile_words);
    };
    for (int i = threadIdx.x; i < RGX_ORDER_BINS; i += 256) s_bin[i] = 0u;
    __syncthreads();
    for (int j = threadIdx.x; j < cnt; j += 256) atomicAdd(&s_bin[size_class(j)], 1u);
    __syncthreads();
    // first position of each class, classes in descending order: thread t owns four
    const int c0 = RGX_ORDER_BINS - 4 - 4 * threadIdx.x;
    const uint32_t n0 = s_bin[c0], n1 = s_bin[c0 + 1], n2 = s_bin[c0 + 2], n3 = s_bin[c0 + 3];
    const uint32_t base = block_sum_before(n0 + n1 + n2 + n3, s_part); // tiles in heavier classes
    s_bin[c0 + 3] = base;
    s_bin[c0 + 2] = base + n3;
    s_bin[c0 + 1] = base + n3 + n2;
    s_bin[c0] = base + n3 + n2 + n1;
    __syncthreads();
    for (int j = threadIdx.x; j < cnt; j += 256) P.tile_order[xcd * cnt + atomicAdd(&s_bin[size_class(j)], 1u)] = (uint32_t)j;
}

// Launch order of the forward.  Nothing tells what a tile will cost before it is marched, but the
// number of Gaussians in front of it is a fair guess: k_block_cost counts, per block of tiles, the
// Gaussians whose centre projects into it (one pass over the primitive records, the adds of a
// wavefront combined per block first); k_block_order then sorts the blocks by that count, heaviest
// first, and deals them to the 8 XCDs in serpentine order, so that every XCD gets the same share of
// heavy and light blocks and starts with its heaviest.  A block's tiles still run next to each
// other on one XCD (what its L2 is shared for); only the order of the blocks changes.
// Layout of the list memory: order[8 * per_xcd], then cost[blocks].
// (A workgroup takes a run of consecutive Gaussians and counts in LDS first: the adds of all workgroups to the few
// blocks in the middle of the image, one after the other in memory, were three quarters of this kernel's time.)
#define RGX_COST_BINS 2048
__global__ __launch_bounds__(256) void k_block_cost(const MarchParams P, uint32_t *__restrict__ cost, int nb, int per_group)
{
    __shared__ uint32_t s_cost[RGX_COST_BINS];
    for (int b = threadIdx.x; b < nb; b += 256) s_cost[b] = 0u;
    __syncthreads();
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    const int64_t first = (int64_t)blockIdx.x * per_group;
    for (int64_t i = first + threadIdx.x; i < first + per_group; i += 256) { // (per_group is a multiple of 256: whole waves)
        int block = -1;
        if (i < P.n) {
            const float4 pos4 = P.prims[i].pos4;   // eye - centre
            const float k = P.prims[i].inv_inter4.w;
            const f3 c = mk3(-pos4.x, -pos4.y, -pos4.z);
            const float z = dot3(c, mk3(P.cam.w[0], P.cam.w[1], P.cam.w[2]));
            if (k == k && z > 1e-6f) { // visible at all, and in front of the camera
                const float x = dot3(c, mk3(P.cam.u[0], P.cam.u[1], P.cam.u[2])) / z, y = dot3(c, mk3(P.cam.v[0], P.cam.v[1], P.cam.v[2])) / z;
                const float fx = (x / (2.0f * P.cam.tan_half_fov_x) + P.cam.principal_x) * (float)P.cam.width;
                const float fy = (y / (2.0f * P.cam.tan_half_fov_y) + P.cam.principal_y) * (float)P.cam.height;
                if (fx >= 0.f && fx < (float)P.cam.width && fy >= 0.f && fy < (float)P.cam.height)
                    block = (((int)fy >> 3) / g.bh) * g.blocks_x + ((int)fx >> 3) / g.bw;
            }
        }
        // Gaussians are in Morton order, so a wavefront's mostly fall into a few blocks: one add per block
        uint64_t todo = __ballot(block >= 0);
        const int lane = threadIdx.x & 63;
        while (todo) {
            const int lead = __builtin_ctzll(todo);
            const int b = __builtin_amdgcn_readlane(block, lead);
            const uint64_t same = __ballot(block == b);
            if (lane == lead) atomicAdd(&s_cost[b], (uint32_t)__popcll(same));
            todo &= ~same;
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += 256)
        if (s_cost[b]) atomicAdd(&cost[b], s_cost[b]);
}

__global__ __launch_bounds__(1024) void k_block_order(const MarchParams P, const uint32_t *__restrict__ cost, uint32_t *__restrict__ order)
{
    __shared__ uint32_t s_bin[RGX_ORDER_BINS], s_wave[16];
    __shared__ uint32_t s_max;
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    const int nb = g.blocks_x * ((P.tiles_y + g.bh - 1) / g.bh), slots = 8 * g.per_xcd;
    for (int i = threadIdx.x; i < RGX_ORDER_BINS; i += blockDim.x) s_bin[i] = 0u;
    if (threadIdx.x == 0) s_max = 1u;
    for (int i = threadIdx.x; i < slots; i += blockDim.x) order[i] = (uint32_t)nb; // a block outside the image: nothing to do
    __syncthreads();
    uint32_t mx = 0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) mx = max(mx, cost[b]);
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor(mx, o));
    if ((threadIdx.x & 63) == 0) atomicMax(&s_max, mx);
    __syncthreads();
    const uint64_t top = s_max;
    auto bin = [&](int b) { return (uint32_t)(RGX_ORDER_BINS - 1) - (uint32_t)((uint64_t)cost[b] * (RGX_ORDER_BINS - 1) / top); }; // heaviest first
    for (int b = threadIdx.x; b < nb; b += blockDim.x) atomicAdd(&s_bin[bin(b)], 1u);
    __syncthreads();
    {
        static_assert(RGX_ORDER_BINS == 1024, "a bin per thread");
        const uint32_t before = block_sum_before(s_bin[threadIdx.x], s_wave);
        s_bin[threadIdx.x] = before;
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        const int r = (int)atomicAdd(&s_bin[bin(b)], 1u); // rank by weight (order within a bin does not matter)
        const int round = r >> 3, k = r & 7;
        order[((round & 1) ? 7 - k : k) * g.per_xcd + round] = (uint32_t)b;
    }
}

// The backward that searches the tree, and those that replay the forward's record: its lists, or its sample sums.
// (The replay of lists alone keeps the 64 density and colour sums it rebuilds across two walks, and spills 200 bytes a
// lane; it runs for the first view of a shape, and where memory is short.)
template <bool STATS, int ORDER>
__global__ __launch_bounds__(64) RGX_WAVES_ATTR void k_march_bwd(const MarchParams P) { march_bwd<false, false, STATS, false, ORDER>(P); }
template <bool STATS, int RAYS = 64>
__global__ __launch_bounds__(64) RGX_WAVES_ATTR void k_march_bwd_replay(const MarchParams P) { march_bwd<true, false, STATS, false, BY_NODES, RAYS>(P); }
template <bool STATS, bool HALF = false, int RAYS = 64>
#ifndef RGX_WAVES_ATTR_SUMS
#define RGX_WAVES_ATTR_SUMS RGX_WAVES_ATTR
#endif
__global__ __launch_bounds__(64) RGX_WAVES_ATTR_SUMS void k_march_bwd_replay_sums(const MarchParams P) { march_bwd<true, true, STATS, HALF, BY_NODES, RAYS>(P); }

enum { RGX_BWD_TREE, RGX_BWD_TREE_PAIRS, RGX_BWD_LISTS, RGX_BWD_SUMS };
template <int RAYS>
static void launch_replay(int which, bool stats, bool half, dim3 grid, hipStream_t s, const MarchParams &P)
{
    const dim3 wave(64);
    if (which == RGX_BWD_SUMS) {
        if (stats && half) hipLaunchKernelGGL((k_march_bwd_replay_sums<true, true, RAYS>), grid, wave, 0, s, P);
        else if (stats) hipLaunchKernelGGL((k_march_bwd_replay_sums<true, false, RAYS>), grid, wave, 0, s, P);
        else if (half) hipLaunchKernelGGL((k_march_bwd_replay_sums<false, true, RAYS>), grid, wave, 0, s, P);
        else hipLaunchKernelGGL((k_march_bwd_replay_sums<false, false, RAYS>), grid, wave, 0, s, P);
    } else {
        if (stats) hipLaunchKernelGGL((k_march_bwd_replay<true, RAYS>), grid, wave, 0, s, P);
        else hipLaunchKernelGGL((k_march_bwd_replay<false, RAYS>), grid, wave, 0, s, P);
    }
}
static void launch_march_bwd(int which, bool stats, bool half, dim3 grid, hipStream_t s, const MarchParams &P)
{
    const dim3 wave(64);
    if (which == RGX_BWD_SUMS || which == RGX_BWD_LISTS) {
        if (P.part_bits == 0) launch_replay<64>(which, stats, half, grid, s, P);
        else if (P.part_bits == 1) launch_replay<32>(which, stats, half, grid, s, P);
        else launch_replay<16>(which, stats, half, grid, s, P);
    } else if (which == RGX_BWD_TREE_PAIRS) {
        if (stats) hipLaunchKernelGGL((k_march_bwd<true, BY_PAIRS>), grid, wave, 0, s, P);
        else hipLaunchKernelGGL((k_march_bwd<false, BY_PAIRS>), grid, wave, 0, s, P);
    } else {
        if (stats) hipLaunchKernelGGL((k_march_bwd<true, BY_NODES>), grid, wave, 0, s, P);
        else hipLaunchKernelGGL((k_march_bwd<false, BY_NODES>), grid, wave, 0, s, P);
    }
}

// Test hook for the cooperative collect: per pixel a segment [tlo, thi] (thi < tlo = pixel idle);
// writes each ray's hit count (negated when cut at cap) and the INPUT indices of its hits.
// (Uncounted, over a tree that has pairs, by pairs: both ways of descending are held to the per-ray query.)
template <bool STATS, bool PAIRS>
__global__ __launch_bounds__(64) void k_collect_tiles(const MarchParams P, const float *__restrict__ seg_lo,
                                                      const float *__restrict__ seg_hi, int cap, int32_t *__restrict__ counts,
                                                      int32_t *__restrict__ ids)
{
    RGX_TILE_LDS(PAIRS);
    int px0, py0;
    if (!tile_origin(P, blockIdx.x, px0, py0)) return;
    const int lane = threadIdx.x;
    int px, py;
    lane_pixel(px0, py0, threadIdx.x, px, py);
    const bool valid = px < P.cam.width && py < P.cam.height;
    const int64_t ray = (int64_t)py * P.cam.width + px;
    CountersFor<STATS> cn; // with counters or without, as the march kernels
    Frustum F;
    frustum_planes(P.cam, px0, py0, F);
    const f3 dir = compute_ray(P.cam, (unsigned)px, (unsigned)py);
    const float tlo = valid ? seg_lo[ray] : 1.f, thi = valid ? seg_hi[ray] : 0.f;
    const bool need = valid && thi >= tlo;
    {
        const float t_far = wave_max_all(need && thi < 1e30f ? thi : 0.f);
        if constexpr (PAIRS) frustum_cut_pairs(P, F, t_far, L.queue);
        else frustum_cut(P, F, t_far, L.queue);
    }
    int p0 = 0, written = 0;
    bool ov = false;
    if (__any(need)) {
        RayState R;
        R.dir = dir;
        R.active = false; // not searching: the driver only sees the `need` lanes
        R.searching = false;
        R.tbuffer = tlo;
        R.texit = thi;
        R.slab_spacing = 0.f;
        Window Wn = {0.f, 0, false, 1, false, false};
        float found = -1.0f, searched_to = 0.f;
        MarchParams Pc = P;
        Pc.m.max_prim_slice = cap;
        auto record = [&](const auto &e, bool hit, bool, auto) {
            if (hit) ids[ray * cap + written++] = (int32_t)P.order[e.pid];
        };
        NoRecorder rec;
        slab_tables<WALK_ROWS, PAIRS>(Pc, L, F, Wn, R, need, tlo, thi, p0, ov, found, searched_to, cn, rec, record, [](bool) { return false; }, record);
    }
    if (valid) counts[ray] = ov ? -p0 : p0;
}

// gbuf (Morton order, 16 floats per Gaussian) -> the five gradient tensors in input order
__global__ __launch_bounds__(256) void k_unpermute_grads(const float4 *__restrict__ gbuf, const uint32_t *__restrict__ place,
                                                         int64_t n, float *__restrict__ ddens, float *__restrict__ drgb,
                                                         float *__restrict__ dpos, float *__restrict__ dscale,
                                                         float *__restrict__ dquat)
{
    // in input order (place: input index -> sorted position): one 64-byte read wherever it lies, whole lines written
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t j = place[i];
    const float4 a = gbuf[4 * j], b = gbuf[4 * j + 1], c = gbuf[4 * j + 2], d = gbuf[4 * j + 3];
    ddens[i] = a.x;
    drgb[3 * i] = a.y; drgb[3 * i + 1] = a.z; drgb[3 * i + 2] = a.w;
    dpos[3 * i] = b.x; dpos[3 * i + 1] = b.y; dpos[3 * i + 2] = b.z;
    dscale[3 * i] = b.w; dscale[3 * i + 1] = c.x; dscale[3 * i + 2] = c.y;
    dquat[4 * i] = c.z; dquat[4 * i + 1] = c.w; dquat[4 * i + 2] = d.x; dquat[4 * i + 3] = d.y;
}

// Clears what a launch starts from, in one kernel: a launch of its own for a few words takes 4.5 us (4 k Gaussians 128x128: two of 24 launches).
// A backward: the gradient block, and the count of this launch's replays that lost their record (or null).
__global__ __launch_bounds__(256) void k_clear_backward(float4 *p, int64_t n4, uint32_t *lost)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n4) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i == 0 && lost) *lost = 0u;
}

// A forward: the 16 bytes at a and at b (either may be null), the bump counter of the record's sample-sum pool and the
// workspace's fault counters; and n words at cost.
__global__ __launch_bounds__(256) void k_clear_forward(float4 *a, uint32_t first, float4 *b, uint32_t *cost, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0 && a) *a = make_float4(__uint_as_float(first), 0.f, 0.f, 0.f);
    if (i == 1 && b) *b = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < n) cost[i] = 0u;
}

// ---------------------------------------------------------------------------
// Test hooks: the two queries on caller-supplied segments.
__global__ __launch_bounds__(64) void k_first_hit(const MarchParams P, f3 o, int64_t n, const float *__restrict__ dirs,
                                                  const float *__restrict__ tlo, const float *__restrict__ thi,
                                                  float *__restrict__ out)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    Counters cn;
    out[r] = first_hit(P, o, mk3(dirs[3 * r], dirs[3 * r + 1], dirs[3 * r + 2]), tlo[r], thi[r], cn);
}

__global__ __launch_bounds__(64) void k_trace_segments(const MarchParams P, f3 o, int64_t n, const float *__restrict__ dirs,
                                                       const float *__restrict__ tlo, const float *__restrict__ thi, int cap,
                                                       int32_t *__restrict__ counts, int32_t *__restrict__ ids)
{
    __shared__ int32_t hits[RGX_LDS_HITS][64];
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    Counters cn;
    // the id row doubles as the spill area; LDS entries are copied out afterwards
    const HitList hl = {&hits[0][threadIdx.x], ids + r * cap + RGX_LDS_HITS};
    bool ov;
    const int p0 = collect(P, o, mk3(dirs[3 * r], dirs[3 * r + 1], dirs[3 * r + 2]), tlo[r], thi[r], cap, hl, ov, cn);
    for (int j = 0; j < p0; ++j) ids[r * cap + j] = (int32_t)P.order[hl.get(j)];
    counts[r] = ov ? -p0 : p0;
}


// ---------------------------------------------------------------------------
static inline dim3 grid_for(int64_t n, int block) { return dim3((unsigned)((n + block - 1) / block)); }

// March workspace: the gradient block (16 words per Gaussian, Morton order) and the tile order of
// the replaying backward.  The order's room is sized from the ray count alone (images of ordinary
// proportions fit; a launch whose tile grid needs more runs in launch order).
struct MarchWs {
    size_t gbuf, faults, order, order_words, total;
};
static inline MarchWs march_ws_layout(int64_t n, int64_t n_rays)
{
    MarchWs L;
    L.gbuf = 0;
    L.faults = rgx_align_up((size_t)(n > 0 ? n : 1) * 16 * sizeof(float), 256); // 256 bytes: the fault counters
    L.order = L.faults + 256;
    L.order_words = (size_t)(n_rays / 64) * 5 / 4 + 2048;
    L.total = L.order + rgx_align_up(L.order_words * sizeof(uint32_t), 256);
    return L;
}

extern "C" int rgx_march_workspace_bytes(int64_t n, int64_t n_rays, int32_t max_prim_slice, size_t *bytes)
{
    if (n < 0 || n_rays < 0 || max_prim_slice < 0 || !bytes) return RGX_EINVAL;
    *bytes = march_ws_layout(n, n_rays).total;
    return RGX_OK;
}

static int fill_params(MarchParams &P, const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims,
                       int64_t n, void *march_ws, size_t march_ws_bytes, RgxStats *stats)
{
    if (!ws || !cam || !march || n < 0 || (n > 0 && !prims) || cam->width <= 0 || cam->height <= 0 ||
        march->max_prim_slice < 0 || !(march->dt_step > 0.0f) || ((uintptr_t)prims & 15u))
        return RGX_EINVAL;
    const MarchWs M = march_ws_layout(n, 0);
    if (!march_ws || march_ws_bytes < M.faults || ((uintptr_t)march_ws & 255u)) return RGX_EWORKSPACE;
    const WsLayout L = rgx_ws_layout(n);
    const char *w = (const char *)ws;
    P.cam = *cam;
    P.m = *march;
    P.nodes = (const Node *)(w + L.nodes);
    P.right = (const int32_t *)(w + L.right);
    P.pairs = (const float4 *)(w + L.pairs);
    P.order = (const uint32_t *)(w + L.vals0);
    P.place = (const uint32_t *)(w + L.vals1);
    P.hdr = (const WsHeader *)(w + L.header);
    P.prims = (const Prim *)prims;
    P.n = n;
    P.ray_colors = nullptr;
    P.frame = nullptr;
    P.depth = nullptr;
    P.fwd_colors = nullptr;
    P.dloss = nullptr;
    P.gbuf = (float *)((char *)march_ws + M.gbuf);
    P.stats = stats;
    P.tiles_x = (cam->width + 7) / 8;
    P.tiles_y = (cam->height + 7) / 8;
    P.records = nullptr;
    P.rec_tile_words = 0;
    P.only_overflow = 0;
    P.rec_pieces = 1;
    P.rec_first = P.rec_equal = P.rec_turn = 0;
    // room for the tile order?  (a workspace sized for fewer rays, or an image of extreme proportions, goes without)
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    const size_t order_words = (size_t)8 * g.per_xcd * g.bw * g.bh;
    P.tile_order = M.order + order_words * sizeof(uint32_t) <= march_ws_bytes ? (uint32_t *)((char *)march_ws + M.order) : nullptr;
    P.use_tile_order = 0;
    P.part_bits = P.rec_bits = 0;
    P.faults = M.order <= march_ws_bytes ? (uint32_t *)((char *)march_ws + M.faults) : nullptr;
    P.ray_counts = nullptr;
    P.sum_pool = nullptr;
    P.sum_next = nullptr;
    P.sum_first = 0;
    P.sum_slots = 0;
    P.sum_slot_words = RGX_SUM_SLOT_WORDS;
    if (march->record_format != 0 && march->record_format != 1) return RGX_EINVAL;
    return RGX_OK;
}

#define RGX_REC_MIN_TILE_WORDS 1024

extern "C" int rgx_march_records_bytes(int32_t width, int32_t height, int32_t tile_words, size_t *bytes)
{
    if (width <= 0 || height <= 0 || tile_words < RGX_REC_MIN_TILE_WORDS || (tile_words & 3) || !bytes) return RGX_EINVAL;
    *bytes = (size_t)((width + 7) / 8) * (size_t)((height + 7) / 8) * (size_t)tile_words * sizeof(uint32_t);
    return RGX_OK;
}

static int part_bits(const MarchParams &P, bool image_only);
static int attach_records(MarchParams &P, void *records, size_t records_bytes)
{
    if (!records) return RGX_OK;
    const size_t ntiles = (size_t)P.tiles_x * P.tiles_y;
    const size_t words = records_bytes / sizeof(uint32_t) / ntiles;
    if (((uintptr_t)records & 15u) || words < RGX_REC_MIN_TILE_WORDS) return RGX_EWORKSPACE;
    P.records = (uint32_t *)records;
    P.sum_slot_words = P.m.record_format == 1 ? RGX_SUM_SLOT_WORDS_HALF : RGX_SUM_SLOT_WORDS;
    if (words >= RGX_REC_LIST_WORDS + RGX_SUM_SLOT_WORDS) {
        // room beyond the hit lists: RGX_REC_LIST_WORDS per tile, a 256-byte pool header, the sample-sum slots
        P.rec_tile_words = RGX_REC_LIST_WORDS;
        const size_t head = ntiles * (size_t)RGX_REC_LIST_WORDS * sizeof(uint32_t);
        const size_t slots = (records_bytes - head - 256) / ((size_t)P.sum_slot_words * sizeof(uint32_t));
        P.sum_next = (uint32_t *)((char *)records + head);
        P.sum_pool = (float4 *)((char *)records + head + 256);
        P.sum_slots = (int32_t)(slots > 0x7fffffff ? 0x7fffffff : slots);
    } else {
        P.rec_tile_words = (int32_t)words & ~3;
    }
    // By parts of tiles: each has its share of the region, and slots of its share of the size.
    const int bits = part_bits(P, false);
    P.part_bits = P.rec_bits = bits;
    P.rec_tile_words = P.rec_tile_words >> bits & ~3;
    if (bits > 0 && P.sum_slots >= (int64_t)(ntiles << bits) + (int64_t)ntiles) P.sum_first = (uint32_t)(ntiles << bits); // (one for each part)
    P.sum_slot_words >>= bits;
    P.sum_slots = (int32_t)std::min<int64_t>((int64_t)P.sum_slots << bits, 0x7fffffff);
    RecordPieces rp = record_pieces((int)std::min<int64_t>((int64_t)ntiles << bits, 0x7fffffff));
    if (bits > 0) rp.most = std::min(rp.most, RGX_REC_MORE - 4); // (what would be the last pieces' words say where a region goes on)
    P.rec_pieces = P.m.record_format == 1 ? min(rp.most, RGX_SUM_SLOT_WORDS_HALF / RGX_REC_STATE_WORDS + 1) : rp.most;
    P.rec_first = rp.first;
    P.rec_equal = rp.equal;
    P.rec_turn = rp.turn;
    return RGX_OK;
}

// A launch in which every wavefront starts at once lasts as long as its longest, and one with few tiles leaves most of the chip idle.  So an image of few
// tiles is marched by parts of tiles: halves (8x4 pixels), 4x4 blocks or 4x2 pixels, a wavefront for each, whose lanes hold each ray twice, four
// or eight times over (Part).  A part has a narrower frustum, whose tables hold fewer Gaussians, as many entries tested at a time as its rays have
// copies, and walks that are shorter by as much; what is done more often is the sweep.  Measured, ms of a frame by whole tiles / halves / 4x4 / 4x2,
// where not taken before by four wavefronts a tile that swept together, met at barriers and had the tile's 64 rays four times over (up to 768 tiles: in brackets) or
// by halves whose idle lanes did nothing (769 to 1 296: likewise):
//     tiles                                     64                  256                 625                 900
//     fixed step, 4 k Gaussians in a cube   [1.32] 0.58 0.45    [0.56] 0.49 0.41    [0.49] 0.42 0.41    [0.61] 0.41 0.44
//     fixed step, 30 k in a ball            [2.65] 1.19 0.57    [1.43] 0.60 0.41    [0.94] 0.47 0.41    [1.18] 0.46 0.40
//     fixed step, 100 k in a ball           [5.36] 2.23 1.22    [2.30] 1.11 0.54    [1.59] 0.88 0.55    [1.75] 0.76 0.49
//     fixed step, 1 M in a ball of radius 2 [13.3] 5.35 3.41    [5.47] 2.94 1.65    [4.77] 1.92 1.86    [3.38] 2.00 2.30
//     adaptive step, 60 k heavy-tailed      [2.28] 0.95 0.64    [1.18] 0.65 0.56    [0.97] 0.66 0.94    [0.80] 0.80 1.17
//     adaptive step, 3 M heavy-tailed       [8.46] 5.29 3.26    [3.68] 3.01 2.12    [4.07] 2.31 3.01    [3.67] 2.90 3.61
//     tiles                                    1 225                 1 600               2 025               3 025               4 056
//     fixed step, 4 k in a cube          [0.55] 0.47 0.40 0.53   0.67 0.49 0.42      0.67 0.46 0.44      0.62 0.48 0.61      0.55 0.61 0.93
//     fixed step, 100 k in a ball        [1.45] 1.24 0.63 0.62   2.17 1.04 0.60      1.88 0.89 0.62      1.24 0.71 0.70      1.06 0.83 1.01
//     fixed step, 1 M, radius 2          [3.03] 2.68 2.18 2.68   4.34 2.32 2.36      3.99 2.59 2.61      2.99 2.82 3.41      2.92 2.99 4.15
//     adaptive step, 60 k heavy-tailed   [0.81] 0.74 0.94 1.52   0.88 0.85 1.09      0.83 1.01 1.28      0.87 1.14 1.69      1.07 1.39 2.11
//     adaptive step, 3 M heavy-tailed    [3.59] 3.00 3.19 4.30   4.00 3.68 3.86      3.85 3.86 4.20      4.61 4.70 5.42      4.56 4.92 6.25
// Halves / 4x4 with the adaptive step, which the first columns leave out: 60 k heavy-tailed 625 tiles 0.76 / 0.68, 784 0.74 / 0.77, 900 0.73 / 0.81; 3 M heavy-tailed 2.90 / 2.19,
// 2.50 / 2.22, 2.63 / 2.35.
// The lines lie where a finer part stops gaining over the scenes of each step; the step stands for what else those scenes differ in: around an object half the tiles are
// empty, from within a scene all are heavy.  (Halves for the heaviest blocks only of an image with more tiles: 300 k 800x800 2.25 -> 2.73 ms
// for 512 tiles of 10 000.)  The sums of a ray's hits are added up in another order, and where max_prim_slice cuts a ray's list other hits are kept, equally exact both.
struct PartLines {
    int eighths, quarters, halves; // up to so many tiles
};
static inline PartLines image_part_lines(bool adaptive) { return adaptive ? PartLines{256, 800, 1600} : PartLines{768, 2048, 3200}; }

// Records by parts.  Which: those of the fixed step.
//   No record: the backward searches the tree again, one wavefront per tile, and has to meet the hits and the
//     transmittance of the forward: that is a march of whole tiles then, whatever the step, and every slab's list in one (slab_tables).
//   A record and the adaptive step: the next step's length depends on the last bit of the transmittance, and a sample that
//     so crosses a Gaussian's cut-off moves that Gaussian's gradient by a visible part (1e-3 of the norm at 150 k Gaussians):
//     no longer the gradients that larger images give.  Whole tiles.
//   A record and the fixed step: what the backward replays is what the parts recorded, and against 64 bits its gradients are as good (3 k Gaussians,
//     512 rays 240x320: 2.2e-6 to 3.0e-6 of their norm, whole tiles 4.8e-6 to 5.4e-6; where a sample lies at a cut-off both the same).  (A part whose region overflowed is
//     searched again, as it was marched: lists that max_prim_slice cut are cut to the same hits there.)
// Measured, ms of a training step by whole tiles / halves / 4x4, where not taken before by four wavefronts a tile (up to 1 024 tiles: in brackets):
//     tiles                               400                    784                  1 024                 1 156
//     4 k Gaussians in a cube     [0.87] 0.86 0.75       [0.83] 0.88 0.79      [0.80] 0.89 0.79
//     16 k in a cube              [1.43] 1.25 0.93       [1.24] 1.26 1.02      [1.15] 1.28 1.04       1.61 1.30 1.09
//     300 k in a ball             [16.2] 4.31 3.06 (625)
//     20 k in a ball of radius 2  [0.70] 0.75 0.66       [0.81] 0.79 0.76      [0.89] 0.80 0.84       0.93 0.80 0.90
//     100 k, radius 2             [7.99] 2.53 1.47       [2.35] 1.88 1.85      [2.30] 1.83 1.97       2.73 2.06 2.29
//     300 k, radius 2             [13.4] 3.79 2.14       [11.5] 3.13 2.69      [10.7] 3.13 2.96       10.1 3.32 3.29
//     tiles                             1 296                1 600                1 936                2 304           2 500
//     16 k in a cube                1.60 1.30 1.17       1.54 1.23 1.29       1.62 1.31            1.69 1.45
//     20 k, radius 2                0.92 0.81 0.96       1.00 0.89 1.07       0.95 0.94            1.00 1.02
//     100 k, radius 2               2.73 2.28 2.37       2.86 2.38 2.68       2.69 2.48            2.47 2.80      2.61 3.00
//     300 k, radius 2               9.51 3.58 3.52       10.1 3.50 3.88       4.20 3.72            4.58 4.43      4.05 4.50
// The line of halves lies where one of these scenes stops gaining.  That of 4x4 lies between what they gain and what they lose: from 784 to 1 156 tiles 4x4 are 10 to 20 % ahead of halves in the
// cubes, even in the ball with 300 k, 5 to 12 % behind with 20 k and 100 k.  (1 k Gaussians alone take 0.52 -> 0.54 at 900 to 1 024 tiles by parts.)  The large gains are
// those of scenes whose tiles' lists overflowed their regions: by parts these go on in slots.
// (Eighths gain with up to 144 tiles -- 64 tiles: 4 k 0.80 -> 0.67, 16 k 1.27 -> 0.92, 300 k in a ball 52.8 -> 3.78 -- and lose from 256 on: 20 k of radius 2
// 0.64 -> 0.70.  But their windows, eight times as many, add a Gaussian's sums to memory more often than a search for the whole tile would.)
static constexpr PartLines record_part_lines() { return {0, 1200, 2000}; }

// image_only: no backward follows this launch
static bool sums_in_any_order(const MarchParams &P, bool image_only) { return image_only || (P.records && !P.m.dynamic_sampling); }
static int part_bits(const MarchParams &P, bool image_only)
{
    if (!sums_in_any_order(P, image_only)) return 0;
    const PartLines L = image_only ? image_part_lines(P.m.dynamic_sampling) : record_part_lines();
    const int tiles = P.tiles_x * P.tiles_y;
    return tiles <= L.eighths ? 3 : tiles <= L.quarters ? 2 : tiles <= L.halves ? 1 : 0;
}

// What precedes a forward's march: counters cleared, and its launch order: blocks of tiles by their estimated weight (k_block_cost,
// k_block_order), when the workspace has room for the lists.
static void prepare_forward(MarchParams &P, bool image_only, hipStream_t s)
{
    // The order only matters for the end of a launch, where ever fewer tiles still run: with many
    // rounds of tiles per wave slot (3072 slots: 12 per CU) that end is a small part of the launch
    // and the pass over the primitive records takes what it brings (forward without -> with the order: 1 M Gaussians at
    // 800x800, 3.3 rounds: 5.51 -> 5.32 ms; 300 k there 2.84 -> 2.82; 3 M at 1237x822, 5.2 rounds: 9.71 -> 9.67; 3 M at
    // 1920x1080, 10.5 rounds: 17.12 -> 17.09).  Nor does it where every wavefront starts at once.
    const int64_t tiles = (int64_t)P.tiles_x * P.tiles_y;
    if (!P.records) P.part_bits = part_bits(P, image_only); // (else it is the record's)
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    const int nb = g.blocks_x * ((P.tiles_y + g.bh - 1) / g.bh);
    const bool at_once = P.part_bits > 0 && tiles << P.part_bits <= 3072;
    const bool ordered = P.tile_order && P.n > 0 && tiles <= 6 * 3072 && !at_once && nb <= RGX_COST_BINS; // (more blocks: a very long, thin image)
    uint32_t *order = P.tile_order, *cost = ordered ? P.tile_order + 8 * g.per_xcd : nullptr;
    if (P.sum_next || P.faults || ordered)
        hipLaunchKernelGGL(k_clear_forward, dim3(ordered ? (unsigned)((nb + 255) / 256) : 1u), dim3(256), 0, s, (float4 *)P.sum_next, P.sum_first, (float4 *)P.faults, cost, ordered ? nb : 0);
    if (!ordered) return;
    const int per_group = (int)((((P.n + 511) / 512) + 255) / 256 * 256); // 512 workgroups at most, whole waves
    hipLaunchKernelGGL(k_block_cost, dim3((unsigned)((P.n + per_group - 1) / per_group)), dim3(256), 0, s, P, cost, nb, per_group);
    hipLaunchKernelGGL(k_block_order, dim3(1), dim3(1024), 0, s, P, cost, order);
    P.use_tile_order = 2;
}

static inline dim3 march_grid(const MarchParams &P)
{
    const TileGrid g = tile_grid(P.tiles_x, P.tiles_y);
    return dim3((unsigned)(8 * g.per_xcd * g.bw * g.bh) << P.part_bits);
}

// Sweeps by pairs of nodes: the same launches, up to six rounds of tiles, over trees that have them.  A tile's own time gets shorter, which is what a launch with
// few rounds lasts; with many rounds the wavefronts hide each other's trips to memory (forward by nodes / by pairs: 300 k Gaussians
// 800x800 2.77 / 2.66 ms, its frame with lobes 2.38 / 2.27, 1 M 800x800 5.28 / 5.19, viewer 1 M 1280x720 6.08 / 6.06; 3 M
// 1920x1080, 10.5 rounds, 16.88 / 16.96).
// A backward that searches the tree for a tile whose record overflowed goes as the forward that wrote the record went (sweep_begin): with another
// order, where lists are cut, its gradient has little to do with the image.
#define RGX_PAIR_TILES (6 * 3072)
static bool by_pairs(const MarchParams &P, bool image_only)
{
    return sums_in_any_order(P, image_only) && P.n <= RGX_PAIR_BOXES && P.tiles_x * P.tiles_y <= RGX_PAIR_TILES;
}
// half: the record's colour sums are in half precision
static void launch_forward(const MarchParams &P, bool viewer, bool counting, bool half, bool image_only, hipStream_t s)
{
    const bool pairs = by_pairs(P, image_only);
    const dim3 grid = march_grid(P), block(64);
    // what: RECORD, VIEWER, STATS, HALF
#define RGX_FWD_OF(RAYS, RECORD, VIEWER, STATS, HALF)                                           \
    do {                                                                                        \
        if (pairs) hipLaunchKernelGGL((k_march_fwd<true, RECORD, VIEWER, STATS, HALF, false, RAYS>), grid, block, 0, s, P); \
        else hipLaunchKernelGGL((k_march_fwd<false, RECORD, VIEWER, STATS, HALF, false, RAYS>), grid, block, 0, s, P); \
    } while (0)
#define RGX_FWD(...)                                                                            \
    do {                                                                                        \
        if (P.part_bits == 0) RGX_FWD_OF(64, __VA_ARGS__);                                      \
        else if (P.part_bits == 1) RGX_FWD_OF(32, __VA_ARGS__);                                 \
        else RGX_FWD_OF(16, __VA_ARGS__);                                                       \
    } while (0)
#define RGX_FWD_IMAGE(...)                                                                      \
    do {                                                                                        \
        if (P.part_bits == 3) RGX_FWD_OF(8, __VA_ARGS__);                                       \
        else RGX_FWD(__VA_ARGS__);                                                              \
    } while (0)
    static_assert(record_part_lines().eighths == 0, "a record is of quarters at the finest");
    if (viewer) {
        if (counting) RGX_FWD_IMAGE(false, true, true, false);
        else RGX_FWD_IMAGE(false, true, false, false);
    } else if (P.records && half) {
        if (counting) RGX_FWD(true, false, true, true);
        else RGX_FWD(true, false, false, true);
    } else if (P.records) {
        if (counting) RGX_FWD(true, false, true, false);
        else RGX_FWD(true, false, false, false);
    } else if (!image_only) {
        if (counting) hipLaunchKernelGGL((k_march_fwd<false, false, false, true, false, true>), grid, block, 0, s, P);
        else hipLaunchKernelGGL((k_march_fwd<false, false, false, false, false, true>), grid, block, 0, s, P);
    } else {
        if (counting) RGX_FWD_IMAGE(false, false, true, false);
        else RGX_FWD_IMAGE(false, false, false, false);
    }
#undef RGX_FWD_IMAGE
#undef RGX_FWD
#undef RGX_FWD_OF
}

static int march_forward_launch(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                float *ray_colors, void *march_ws, size_t march_ws_bytes, void *records, size_t records_bytes,
                                RgxStats *stats, uint32_t *ray_counts, bool image_only, void *stream);

extern "C" int rgx_march_forward(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                 float *ray_colors, void *march_ws, size_t march_ws_bytes, void *records, size_t records_bytes,
                                 RgxStats *stats, void *stream)
{
    return march_forward_launch(ws, cam, march, prims, n, ray_colors, march_ws, march_ws_bytes, records, records_bytes, stats,
                                nullptr, false, stream);
}

extern "C" int rgx_march_test(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                              float *ray_colors, void *march_ws, size_t march_ws_bytes, RgxStats *stats, void *stream)
{
    return march_forward_launch(ws, cam, march, prims, n, ray_colors, march_ws, march_ws_bytes, nullptr, 0, stats, nullptr, true, stream);
}

extern "C" int rgx_march_forward_counts(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                        float *ray_colors, void *march_ws, size_t march_ws_bytes, void *records,
                                        size_t records_bytes, RgxStats *stats, uint32_t *ray_counts, void *stream)
{
    if (!ray_counts) return RGX_EINVAL;
    return march_forward_launch(ws, cam, march, prims, n, ray_colors, march_ws, march_ws_bytes, records, records_bytes, stats,
                                ray_counts, false, stream);
}

static int march_forward_launch(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                float *ray_colors, void *march_ws, size_t march_ws_bytes, void *records, size_t records_bytes,
                                RgxStats *stats, uint32_t *ray_counts, bool image_only, void *stream)
{
    const DeviceScope on_device(ws);
    MarchParams P;
    int rc = fill_params(P, ws, cam, march, prims, n, march_ws, march_ws_bytes, stats);
    if (rc) return rc;
    if (!ray_colors) return RGX_EINVAL;
    rc = attach_records(P, records, records_bytes);
    if (rc) return rc;
    P.ray_colors = ray_colors;
    P.ray_counts = ray_counts;
    const bool counting = stats != nullptr || ray_counts != nullptr;
    void *span = rgx_span_begin(RGX_T_MARCH_FWD, (hipStream_t)stream);
    prepare_forward(P, image_only, (hipStream_t)stream);
    const bool half = P.sum_pool && P.m.record_format == 1;
    launch_forward(P, false, counting, half, image_only, (hipStream_t)stream);
    rgx_span_end(span, (hipStream_t)stream);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

extern "C" int rgx_march_viewer(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                uint8_t *frame, float *depth, void *march_ws, size_t march_ws_bytes, RgxStats *stats, void *stream)
{
    const DeviceScope on_device(ws);
    MarchParams P;
    const int rc = fill_params(P, ws, cam, march, prims, n, march_ws, march_ws_bytes, stats);
    if (rc != RGX_OK) return rc;
    if (!frame || !depth || ((uintptr_t)frame & 3u)) return RGX_EINVAL;
    P.frame = frame;
    P.depth = depth;
    void *span = rgx_span_begin(RGX_T_MARCH_FWD, (hipStream_t)stream);
    prepare_forward(P, true, (hipStream_t)stream);
    launch_forward(P, true, stats != nullptr, false, true, (hipStream_t)stream);
    rgx_span_end(span, (hipStream_t)stream);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

// timed: record the event-timed spans (they may create events; the allocation-free entry point goes without)
static int march_backward_launch(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                 const float *ray_colors, const float *dloss, float *ddens, float *drgb, float *dpos,
                                 float *dscale, float *dquat, void *march_ws, size_t march_ws_bytes, const void *records,
                                 size_t records_bytes, RgxStats *stats, void *stream, bool timed);

extern "C" int rgx_march_backward(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                  const float *ray_colors, const float *dloss, float *ddens, float *drgb, float *dpos,
                                  float *dscale, float *dquat, void *march_ws, size_t march_ws_bytes, const void *records,
                                  size_t records_bytes, RgxStats *stats, void *stream)
{
    const DeviceScope on_device(ws);
    return march_backward_launch(ws, cam, march, prims, n, ray_colors, dloss, ddens, drgb, dpos, dscale, dquat, march_ws,
                                 march_ws_bytes, records, records_bytes, stats, stream, true);
}

// ---------------------------------------------------------------------------
// rgx_march_backward_noalloc: the backward whose scratch memory -- gradient block, fault counters,
// tile order: a march workspace for RGX_NOALLOC_MAX_GAUSSIANS Gaussians and RGX_NOALLOC_MAX_RAYS
// rays -- is a file-scope device array instead of a buffer of the caller's.  Every GPU the library
// runs on holds its own copy of the array, at its own address, until the process ends.  `scratch`
// is the host-side stand-in of that array, not a device address: the device address is asked for
// once per device (with that device current) and kept, and only that address goes to kernels.
static __device__ __align__(256) unsigned char scratch[RGX_NOALLOC_SCRATCH_BYTES];

#define RGX_NOALLOC_MAX_DEVICES 64
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[RGX_NOALLOC_MAX_DEVICES]; // per device: the device address of its `scratch`, or null

// The current device's copy of the array.
static int noalloc_scratch(void **out)
{
    int dev = -1;
    RGX_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= RGX_NOALLOC_MAX_DEVICES) return RGX_ELIMIT;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        RGX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return RGX_EHIP;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return RGX_OK;
}

extern "C" int rgx_march_backward_noalloc(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims,
                                          int64_t n, const float *ray_colors, const float *dloss, float *ddens, float *drgb,
                                          float *dpos, float *dscale, float *dquat, const void *records, size_t records_bytes,
                                          RgxStats *stats, void *stream)
{
    static_assert(RGX_NOALLOC_SCRATCH_BYTES % 256 == 0, "the array is a 256-byte aligned march workspace");
    if (!ws || !cam || n < 0 || cam->width <= 0 || cam->height <= 0) return RGX_EINVAL;
    if (n > RGX_NOALLOC_MAX_GAUSSIANS || (int64_t)cam->width * cam->height > RGX_NOALLOC_MAX_RAYS) return RGX_ELIMIT;
    if (march_ws_layout(RGX_NOALLOC_MAX_GAUSSIANS, RGX_NOALLOC_MAX_RAYS).total != RGX_NOALLOC_SCRATCH_BYTES) return RGX_EWORKSPACE;
    const DeviceScope on_device(ws);
    void *scr = nullptr;
    const int rc = noalloc_scratch(&scr);
    if (rc) return rc;
    // the launch clears what it reads of the array with a kernel (the gradient block of these n Gaussians; the tile
    // order is rewritten in full before use), so the previous call's contents do not matter
    return march_backward_launch(ws, cam, march, prims, n, ray_colors, dloss, ddens, drgb, dpos, dscale, dquat, scr,
                                 RGX_NOALLOC_SCRATCH_BYTES, records, records_bytes, stats, stream, false);
}

static int march_backward_launch(const void *ws, const RgxCamera *cam, const RgxMarch *march, const float *prims, int64_t n,
                                 const float *ray_colors, const float *dloss, float *ddens, float *drgb, float *dpos,
                                 float *dscale, float *dquat, void *march_ws, size_t march_ws_bytes, const void *records,
                                 size_t records_bytes, RgxStats *stats, void *stream, bool timed)
{
    MarchParams P;
    int rc = fill_params(P, ws, cam, march, prims, n, march_ws, march_ws_bytes, stats);
    if (rc) return rc;
    if (!ray_colors || !dloss || (n > 0 && (!ddens || !drgb || !dpos || !dscale || !dquat))) return RGX_EINVAL;
    rc = attach_records(P, (void *)records, records_bytes);
    if (rc) return rc;
    if (n == 0) return RGX_OK;
    P.fwd_colors = ray_colors;
    P.dloss = dloss;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_clear_backward, grid_for(4 * n, 256), dim3(256), 0, s, (float4 *)P.gbuf, 4 * n, P.faults);
    void *span = timed ? rgx_span_begin(RGX_T_MARCH_BWD, s) : nullptr;
    if (P.records) {
        // tiles with a complete record replay it; the few whose record overflowed are recomputed
        if (P.tile_order && P.part_bits == 0) {
            hipLaunchKernelGGL(k_tile_order, dim3(8), dim3(256), 0, s, P);
            P.use_tile_order = 1;
        }
        if (P.sum_pool)
            launch_march_bwd(RGX_BWD_SUMS, stats != nullptr, P.m.record_format == 1, dim3(march_grid(P).x * (unsigned)P.rec_pieces), s, P);
        launch_march_bwd(RGX_BWD_LISTS, stats != nullptr, false, march_grid(P), s, P);
        P.only_overflow = 1;
        P.use_tile_order = 0;
    }
    const int tree = by_pairs(P, false) ? RGX_BWD_TREE_PAIRS : RGX_BWD_TREE;
    const unsigned parts = march_grid(P).x;
    launch_march_bwd(tree, stats != nullptr, false, dim3(P.part_bits > 0 ? parts + (parts >> P.part_bits) : parts), s, P);
    rgx_span_end(span, s);
    span = timed ? rgx_span_begin(RGX_T_UNPERMUTE, s) : nullptr;
    hipLaunchKernelGGL(k_unpermute_grads, grid_for(n, 256), dim3(256), 0, s, (const float4 *)P.gbuf, P.place, n, ddens, drgb,
                       dpos, dscale, dquat);
    rgx_span_end(span, s);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

extern "C" int rgx_march_faults(const void *march_ws, size_t march_ws_bytes, int64_t n, uint64_t *host_out2, void *stream)
{
    if (!march_ws || n < 0 || !host_out2) return RGX_EINVAL;
    const DeviceScope on_device(march_ws);
    const MarchWs M = march_ws_layout(n, 0);
    host_out2[0] = host_out2[1] = 0;
    if (M.order > march_ws_bytes) return RGX_OK; // no room for the counters: none kept
    uint32_t words[2] = {0, 0};
    RGX_HIP(hipMemcpyAsync(words, (const char *)march_ws + M.faults, sizeof words, hipMemcpyDeviceToHost, (hipStream_t)stream));
    RGX_HIP(hipStreamSynchronize((hipStream_t)stream));
    host_out2[0] = words[0];
    host_out2[1] = words[1];
    return RGX_OK;
}

static int hook_params(MarchParams &P, const void *ws, const float *prims, int64_t n_prims)
{
    if (!ws || n_prims < 0 || (n_prims > 0 && !prims)) return RGX_EINVAL;
    const WsLayout L = rgx_ws_layout(n_prims);
    const char *w = (const char *)ws;
    P = MarchParams{};
    P.nodes = (const Node *)(w + L.nodes);
    P.right = (const int32_t *)(w + L.right);
    P.pairs = (const float4 *)(w + L.pairs);
    P.order = (const uint32_t *)(w + L.vals0);
    P.place = (const uint32_t *)(w + L.vals1);
    P.hdr = (const WsHeader *)(w + L.header);
    P.prims = (const Prim *)prims;
    P.n = n_prims;
    return RGX_OK;
}

extern "C" int rgx_first_hit(const void *ws, const float *prims, int64_t n_prims, const float *eye, int64_t n,
                             const float *dirs, const float *tlo, const float *thi, float *out_t, void *stream)
{
    const DeviceScope on_device(ws);
    MarchParams P;
    const int rc = hook_params(P, ws, prims, n_prims);
    if (rc) return rc;
    if (!eye || n < 0 || (n > 0 && (!dirs || !tlo || !thi || !out_t))) return RGX_EINVAL;
    if (n == 0) return RGX_OK;
    hipLaunchKernelGGL(k_first_hit, grid_for(n, 64), dim3(64), 0, (hipStream_t)stream, P, f3{eye[0], eye[1], eye[2]}, n, dirs,
                       tlo, thi, out_t);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

extern "C" int rgx_trace_segments(const void *ws, const float *prims, int64_t n_prims, const float *eye, int64_t n,
                                  const float *dirs, const float *tlo, const float *thi, int32_t cap, int32_t *counts,
                                  int32_t *ids, void *stream)
{
    const DeviceScope on_device(ws);
    MarchParams P;
    const int rc = hook_params(P, ws, prims, n_prims);
    if (rc) return rc;
    if (!eye || n < 0 || cap <= 0 || (n > 0 && (!dirs || !tlo || !thi || !counts || !ids))) return RGX_EINVAL;
    if (n == 0) return RGX_OK;
    hipLaunchKernelGGL(k_trace_segments, grid_for(n, 64), dim3(64), 0, (hipStream_t)stream, P, f3{eye[0], eye[1], eye[2]}, n,
                       dirs, tlo, thi, (int)cap, counts, ids);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

extern "C" int rgx_collect_tiles(const void *ws, const RgxCamera *cam, const float *prims, int64_t n_prims, const float *tlo,
                                 const float *thi, int32_t cap, int32_t *counts, int32_t *ids, int32_t uncounted, void *stream)
{
    const DeviceScope on_device(ws);
    MarchParams P;
    const int rc = hook_params(P, ws, prims, n_prims);
    if (rc) return rc;
    if (!cam || cam->width <= 0 || cam->height <= 0 || cap <= 0 || !tlo || !thi || !counts || !ids) return RGX_EINVAL;
    P.cam = *cam;
    P.tiles_x = (cam->width + 7) / 8;
    P.tiles_y = (cam->height + 7) / 8;
    if (uncounted && n_prims <= RGX_PAIR_BOXES)
        hipLaunchKernelGGL((k_collect_tiles<false, true>), march_grid(P), dim3(64), 0, (hipStream_t)stream, P, tlo, thi, (int)cap, counts, ids);
    else if (uncounted) hipLaunchKernelGGL((k_collect_tiles<false, false>), march_grid(P), dim3(64), 0, (hipStream_t)stream, P, tlo, thi, (int)cap, counts, ids);
    else hipLaunchKernelGGL((k_collect_tiles<true, false>), march_grid(P), dim3(64), 0, (hipStream_t)stream, P, tlo, thi, (int)cap, counts, ids);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

#ifdef RGX_SECTION_CLOCKS
// Diagnostic builds only: the section census since the last reset, summed over workgroups and launches per kernel:
// host_out[kernel][section] cycles and host_out[kernel][RGX_NSEC] waves (RGX_NSECK x (RGX_NSEC + 1) words).  Waits for the device.
extern "C" int rgx_debug_section_cycles(unsigned long long *host_out, int reset)
{
    RGX_HIP(hipDeviceSynchronize());
    if (host_out) {
        static unsigned host[2][RGX_SEC_ROWS][16];
        RGX_HIP(hipMemcpyFromSymbol(host, HIP_SYMBOL(g_section_cycles), sizeof(host)));
        for (int i = 0; i < RGX_NSECK * (RGX_NSEC + 1); ++i) host_out[i] = 0;
        for (int pass = 0; pass < 2; ++pass)
            for (int r = 0; r < RGX_SEC_ROWS; ++r) {
                const unsigned *row = host[pass][r];
                if (!row[RGX_NSEC] || row[RGX_NSEC + 1] >= RGX_NSECK) continue;
                for (int k = 0; k <= RGX_NSEC; ++k) host_out[row[RGX_NSEC + 1] * (RGX_NSEC + 1) + k] += row[k];
            }
    }
    if (reset) {
        void *p = nullptr;
        RGX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(g_section_cycles)));
        RGX_HIP(hipMemset(p, 0, sizeof(unsigned) * 2 * RGX_SEC_ROWS * 16));
    }
    return RGX_OK;
}
// The raw table: 2 x RGX_SEC_ROWS x 16 words (see g_section_cycles), for per-workgroup timelines.
extern "C" int rgx_debug_section_rows(unsigned *host_out)
{
    if (!host_out) return RGX_EINVAL;
    RGX_HIP(hipDeviceSynchronize());
    RGX_HIP(hipMemcpyFromSymbol(host_out, HIP_SYMBOL(g_section_cycles), sizeof(unsigned) * 2 * RGX_SEC_ROWS * 16));
    return RGX_OK;
}
#endif

// Test hook: counts the pairs for which the plain division or the plain square root differs in any
// bit from `/` or sqrtf() (expected: none, for operands inside the ranges plain_roots() grants).
__global__ __launch_bounds__(256) void k_check_plain_arith(const float *__restrict__ a, const float *__restrict__ b, int64_t n,
                                                           uint32_t *bad)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float x = a[i], y = b[i];
    const bool same = __float_as_uint(div_rn_plain(x, y)) == __float_as_uint(x / y) &&
                      __float_as_uint(div_rn_plain(1.0f, y)) == __float_as_uint(1.0f / y) &&
                      __float_as_uint(sqrt_rn_plain(fabsf(x))) == __float_as_uint(sqrtf(fabsf(x))) &&
                      __float_as_uint(sqrt_rn_plain(fabsf(x) * 0x1p-40f)) == __float_as_uint(sqrtf(fabsf(x) * 0x1p-40f));
    if (!same) atomicAdd(bad, 1u);
}

extern "C" int rgx_check_plain_arith(const float *a, const float *b, int64_t n, uint32_t *bad, void *stream)
{
    const DeviceScope on_device(a);
    if (n < 0 || (n > 0 && (!a || !b)) || !bad) return RGX_EINVAL;
    if (n > 0) hipLaunchKernelGGL(k_check_plain_arith, grid_for(n, 256), dim3(256), 0, (hipStream_t)stream, a, b, n, bad);
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}

// Measurement hook: one instruction repeated, sixteen independent registers per lane so that none waits for the one
// before, for the rate at which the card issues that class of VALU instruction (asm volatile: the compiler may
// neither fold nor reorder them).
#define RGX_PROBE_REP16(S) S(0) S(1) S(2) S(3) S(4) S(5) S(6) S(7) S(8) S(9) S(10) S(11) S(12) S(13) S(14) S(15)
template <int KIND>
__global__ __launch_bounds__(256) void k_probe_valu(int iters, float seed, float *sink)
{
    float a[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = seed + (float)(threadIdx.x + i);
    const float m = 1.0f - seed * 1e-9f, c = seed * 1e-9f;
    unsigned long long mask = __ballot(threadIdx.x & 1);
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#define RGX_P_FMA(i) asm volatile("v_fma_f32 %0, %0, %1, %2" : "+v"(a[i]) : "v"(m), "v"(c));
#define RGX_P_ADD(i) asm volatile("v_add_f32 %0, %0, %1" : "+v"(a[i]) : "v"(c));
#define RGX_P_MOV(i) asm volatile("v_mov_b32 %0, %1" : "=v"(a[i]) : "v"(m));
#define RGX_P_AND(i) asm volatile("v_and_b32 %0, %0, %1" : "+v"(a[i]) : "v"(m));
#define RGX_P_CMP(i) asm volatile("v_cmp_lt_f32 %0, %1, %2" : "=s"(mask) : "v"(a[i]), "v"(m));
#define RGX_P_CND(i) asm volatile("v_cndmask_b32 %0, %0, %1, %2" : "+v"(a[i]) : "v"(m), "s"(mask));
#define RGX_P_MAX(i) asm volatile("v_max_f32 %0, %0, %1" : "+v"(a[i]) : "v"(m));
#define RGX_P_DPP(i) asm volatile("v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:0" : "+v"(a[i]));
#define RGX_P_SHL(i) asm volatile("v_lshlrev_b32 %0, 1, %0" : "+v"(a[i]));
#define RGX_P_EXP(i) asm volatile("v_exp_f32 %0, %0" : "+v"(a[i]));
            if constexpr (KIND == 0) { RGX_PROBE_REP16(RGX_P_FMA) }
            else if constexpr (KIND == 1) { RGX_PROBE_REP16(RGX_P_ADD) }
            else if constexpr (KIND == 2) { RGX_PROBE_REP16(RGX_P_MOV) }
            else if constexpr (KIND == 3) { RGX_PROBE_REP16(RGX_P_AND) }
            else if constexpr (KIND == 4) { RGX_PROBE_REP16(RGX_P_CMP) }
            else if constexpr (KIND == 5) { RGX_PROBE_REP16(RGX_P_CND) }
            else if constexpr (KIND == 6) { RGX_PROBE_REP16(RGX_P_MAX) }
            else if constexpr (KIND == 7) { RGX_PROBE_REP16(RGX_P_DPP) }
            else if constexpr (KIND == 8) { RGX_PROBE_REP16(RGX_P_SHL) }
            else { RGX_PROBE_REP16(RGX_P_EXP) }
        }
    }
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += a[i];
    if (t == -1.2345f) *sink = t + (float)mask; // (practically never: keeps the registers live)
}

// The same with the registers named: what an instruction costs depends on where its operands live.  The register
// file has two banks, even and odd register numbers: a multiply-add whose three sources sit in one bank takes
// longer, and one that reads a register the previous instruction also read in that place takes shorter.  KIND 10:
// acc = x * k + acc with a fresh x from the other bank (the sample loops' form); 11: d = a * b + c, all fresh, banks
// mixed; 12: the same with a, b, c in one bank; 13: d = a * b, both fresh.
template <int KIND>
__global__ __launch_bounds__(256) void k_probe_valu_banks(int iters, float seed, float *sink)
{
    // v32..v47: destinations / accumulators; v64..v159: operands; v48: a constant
    asm volatile("v_mov_b32 v32, %0\n v_mov_b32 v33, %0\n v_mov_b32 v34, %0\n v_mov_b32 v35, %0\n v_mov_b32 v36, %0\n v_mov_b32 v37, %0\n v_mov_b32 v38, %0\n v_mov_b32 v39, %0\n v_mov_b32 v40, %0\n v_mov_b32 v41, %0\n v_mov_b32 v42, %0\n v_mov_b32 v43, %0\n v_mov_b32 v44, %0\n v_mov_b32 v45, %0\n v_mov_b32 v46, %0\n v_mov_b32 v47, %0" :: "v"(seed) : "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47");
    asm volatile("v_mov_b32 v64, %0\n v_mov_b32 v65, %0\n v_mov_b32 v66, %0\n v_mov_b32 v67, %0\n v_mov_b32 v68, %0\n v_mov_b32 v69, %0\n v_mov_b32 v70, %0\n v_mov_b32 v71, %0\n v_mov_b32 v72, %0\n v_mov_b32 v73, %0\n v_mov_b32 v74, %0\n v_mov_b32 v75, %0\n v_mov_b32 v76, %0\n v_mov_b32 v77, %0\n v_mov_b32 v78, %0\n v_mov_b32 v79, %0" :: "v"(seed) : "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79");
    asm volatile("v_mov_b32 v80, %0\n v_mov_b32 v81, %0\n v_mov_b32 v82, %0\n v_mov_b32 v83, %0\n v_mov_b32 v84, %0\n v_mov_b32 v85, %0\n v_mov_b32 v86, %0\n v_mov_b32 v87, %0\n v_mov_b32 v88, %0\n v_mov_b32 v89, %0\n v_mov_b32 v90, %0\n v_mov_b32 v91, %0\n v_mov_b32 v92, %0\n v_mov_b32 v93, %0\n v_mov_b32 v94, %0\n v_mov_b32 v95, %0" :: "v"(seed) : "v80", "v81", "v82", "v83", "v84", "v85", "v86", "v87", "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95");
    asm volatile("v_mov_b32 v96, %0\n v_mov_b32 v97, %0\n v_mov_b32 v98, %0\n v_mov_b32 v99, %0\n v_mov_b32 v100, %0\n v_mov_b32 v101, %0\n v_mov_b32 v102, %0\n v_mov_b32 v103, %0\n v_mov_b32 v104, %0\n v_mov_b32 v105, %0\n v_mov_b32 v106, %0\n v_mov_b32 v107, %0\n v_mov_b32 v108, %0\n v_mov_b32 v109, %0\n v_mov_b32 v110, %0\n v_mov_b32 v111, %0" :: "v"(seed) : "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111");
    asm volatile("v_mov_b32 v112, %0\n v_mov_b32 v113, %0\n v_mov_b32 v114, %0\n v_mov_b32 v115, %0\n v_mov_b32 v116, %0\n v_mov_b32 v117, %0\n v_mov_b32 v118, %0\n v_mov_b32 v119, %0\n v_mov_b32 v120, %0\n v_mov_b32 v121, %0\n v_mov_b32 v122, %0\n v_mov_b32 v123, %0\n v_mov_b32 v124, %0\n v_mov_b32 v125, %0\n v_mov_b32 v126, %0\n v_mov_b32 v127, %0" :: "v"(seed) : "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127");
    asm volatile("v_mov_b32 v128, %0\n v_mov_b32 v129, %0\n v_mov_b32 v130, %0\n v_mov_b32 v131, %0\n v_mov_b32 v132, %0\n v_mov_b32 v133, %0\n v_mov_b32 v134, %0\n v_mov_b32 v135, %0\n v_mov_b32 v136, %0\n v_mov_b32 v137, %0\n v_mov_b32 v138, %0\n v_mov_b32 v139, %0\n v_mov_b32 v140, %0\n v_mov_b32 v141, %0\n v_mov_b32 v142, %0\n v_mov_b32 v143, %0" :: "v"(seed) : "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", "v137", "v138", "v139", "v140", "v141", "v142", "v143");
    asm volatile("v_mov_b32 v144, %0\n v_mov_b32 v145, %0\n v_mov_b32 v146, %0\n v_mov_b32 v147, %0\n v_mov_b32 v148, %0\n v_mov_b32 v149, %0\n v_mov_b32 v150, %0\n v_mov_b32 v151, %0\n v_mov_b32 v152, %0\n v_mov_b32 v153, %0\n v_mov_b32 v154, %0\n v_mov_b32 v155, %0\n v_mov_b32 v156, %0\n v_mov_b32 v157, %0\n v_mov_b32 v158, %0\n v_mov_b32 v159, %0" :: "v"(seed) : "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159");
    asm volatile("v_mov_b32 v48, %0" :: "v"(seed) : "v48");
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (KIND == 10) { // x from the bank the accumulator is not in
                asm volatile("v_fma_f32 v32, v65, v48, v32\n" "v_fma_f32 v33, v66, v48, v33\n" "v_fma_f32 v34, v69, v48, v34\n" "v_fma_f32 v35, v70, v48, v35\n" "v_fma_f32 v36, v73, v48, v36\n" "v_fma_f32 v37, v74, v48, v37\n" "v_fma_f32 v38, v77, v48, v38\n" "v_fma_f32 v39, v78, v48, v39\n" "v_fma_f32 v40, v81, v48, v40\n" "v_fma_f32 v41, v82, v48, v41\n" "v_fma_f32 v42, v85, v48, v42\n" "v_fma_f32 v43, v86, v48, v43\n" "v_fma_f32 v44, v89, v48, v44\n" "v_fma_f32 v45, v90, v48, v45\n" "v_fma_f32 v46, v93, v48, v46\n" "v_fma_f32 v47, v94, v48, v47\n" ::: "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47");
            } else if constexpr (KIND == 11) {
                asm volatile("v_fma_f32 v32, v64, v97, v128\n" "v_fma_f32 v33, v66, v99, v130\n" "v_fma_f32 v34, v68, v101, v132\n" "v_fma_f32 v35, v70, v103, v134\n" "v_fma_f32 v36, v72, v105, v136\n" "v_fma_f32 v37, v74, v107, v138\n" "v_fma_f32 v38, v76, v109, v140\n" "v_fma_f32 v39, v78, v111, v142\n" "v_fma_f32 v40, v80, v113, v144\n" "v_fma_f32 v41, v82, v115, v146\n" "v_fma_f32 v42, v84, v117, v148\n" "v_fma_f32 v43, v86, v119, v150\n" "v_fma_f32 v44, v88, v121, v152\n" "v_fma_f32 v45, v90, v123, v154\n" "v_fma_f32 v46, v92, v125, v156\n" "v_fma_f32 v47, v94, v127, v158\n" ::: "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47");
            } else if constexpr (KIND == 12) {
                asm volatile("v_fma_f32 v32, v64, v96, v128\n" "v_fma_f32 v33, v66, v98, v130\n" "v_fma_f32 v34, v68, v100, v132\n" "v_fma_f32 v35, v70, v102, v134\n" "v_fma_f32 v36, v72, v104, v136\n" "v_fma_f32 v37, v74, v106, v138\n" "v_fma_f32 v38, v76, v108, v140\n" "v_fma_f32 v39, v78, v110, v142\n" "v_fma_f32 v40, v80, v112, v144\n" "v_fma_f32 v41, v82, v114, v146\n" "v_fma_f32 v42, v84, v116, v148\n" "v_fma_f32 v43, v86, v118, v150\n" "v_fma_f32 v44, v88, v120, v152\n" "v_fma_f32 v45, v90, v122, v154\n" "v_fma_f32 v46, v92, v124, v156\n" "v_fma_f32 v47, v94, v126, v158\n" ::: "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47");
            } else {
                asm volatile("v_mul_f32 v32, v64, v97\n" "v_mul_f32 v33, v66, v99\n" "v_mul_f32 v34, v68, v101\n" "v_mul_f32 v35, v70, v103\n" "v_mul_f32 v36, v72, v105\n" "v_mul_f32 v37, v74, v107\n" "v_mul_f32 v38, v76, v109\n" "v_mul_f32 v39, v78, v111\n" "v_mul_f32 v40, v80, v113\n" "v_mul_f32 v41, v82, v115\n" "v_mul_f32 v42, v84, v117\n" "v_mul_f32 v43, v86, v119\n" "v_mul_f32 v44, v88, v121\n" "v_mul_f32 v45, v90, v123\n" "v_mul_f32 v46, v92, v125\n" "v_mul_f32 v47, v94, v127\n" ::: "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47");
            }
        }
    }
    float t;
    asm volatile("v_add_f32 %0, v32, v47" : "=v"(t));
    if (t == -1.2345f) *sink = t; // (practically never: keeps the result observable)
}

extern "C" int rgx_probe_valu_rate(int32_t waves, int32_t iters, int32_t kind, float *sink, uint64_t *instructions, void *stream)
{
    if (waves <= 0 || iters <= 0 || kind < 0 || kind > 13 || !sink || !instructions) return RGX_EINVAL;
    const DeviceScope on_device(sink);
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    hipStream_t s = (hipStream_t)stream;
    switch (kind) {
    case 0: hipLaunchKernelGGL(k_probe_valu<0>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 1: hipLaunchKernelGGL(k_probe_valu<1>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 2: hipLaunchKernelGGL(k_probe_valu<2>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 3: hipLaunchKernelGGL(k_probe_valu<3>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 4: hipLaunchKernelGGL(k_probe_valu<4>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 5: hipLaunchKernelGGL(k_probe_valu<5>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 6: hipLaunchKernelGGL(k_probe_valu<6>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 7: hipLaunchKernelGGL(k_probe_valu<7>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 8: hipLaunchKernelGGL(k_probe_valu<8>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 9: hipLaunchKernelGGL(k_probe_valu<9>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 10: hipLaunchKernelGGL(k_probe_valu_banks<10>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 11: hipLaunchKernelGGL(k_probe_valu_banks<11>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    case 12: hipLaunchKernelGGL(k_probe_valu_banks<12>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    default: hipLaunchKernelGGL(k_probe_valu_banks<13>, grid, block, 0, s, (int)iters, 1.0f, sink); break;
    }
    *instructions = (uint64_t)grid.x * 4u * (uint64_t)iters * 64u;
    RGX_LAUNCH_CHECK();
    return RGX_OK;
}
