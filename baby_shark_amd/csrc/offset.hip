// Volume::offset on the device (src/voxel/volume/mod.rs:95-108): remove_if
// |v| > 2h, fast sweeping (src/voxel/fast_sweep.rs), removal of empty leaves,
// v -= D on the active values.
//
// Parallel schedule with the reference's exact result.  A sweep in direction
// (sx, sy, sz) pops leaves in lexicographic order with each axis ascending or
// descending by its sign (fast_sweep.rs:612-684), and a leaf reads only its
// six face neighbours: the three upwind ones are already swept, the three
// downwind ones are not.  With K = sx*lx + sy*ly + sz*lz over leaf
// coordinates, face neighbours sit on planes K - 1 and K + 1, so every leaf on
// one plane can be swept at once once plane K - 1 is done.  Inside a leaf the
// x-y-z loop order has the same structure over voxel planes u + v + w
// (u, v, w the voxel coordinates counted in the sweep direction): a voxel
// reads updated values on plane - 1 and old ones on plane + 1.  So a sweep is
// a sequence of plane launches, and inside each leaf a wavefront walks the 22
// voxel planes.
//
// The leaf queue.  Every leaf in the grid at the start of a sweep is in its
// queue (sweep 1 collects every leaf; sweep s + 1 takes the leaves popped in
// sweep s), and a leaf joins when a swept upwind neighbour pushes it
// (fast_sweep.rs:186-273).  The reference also creates empty leaves at the
// other faces of every stencil; they stay empty unless pushed and are removed
// at the end, so only pushed leaves are created here.  A pushed leaf lies on
// the next plane and is swept there.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

#include "common.hpp"
#include "leafmap.hpp"

namespace bs {

namespace {

constexpr float FS_FAR = 3.40282347e+38f;

struct OffsetState {
    uint32_t fail;        // bit 0: a leaf outside the reachable box (bit 2: past the last plane,
                          // bit 3: a pool leaf off the planes, else off the map), bit 1: pool or hash full
    uint32_t nan;         // some active value is NaN
    uint32_t live;        // leaves of the result
};

// Per pool leaf: bit 0, the leaf must be swept; bits 1..6, the face towards -x,
// +x, -y, +y, -z, +z holds a voxel that can be pushed (fast_sweep.rs:186-273);
// bit 7, it has an active voxel.
// A sweep that changes no voxel of a leaf has found each one at the value its
// neighbours give, in whatever order, so the next sweeps leave the leaf as it
// is until one of the six layers next to it changes: bit 0 is set where a voxel
// of the leaf or of such a layer changed since the leaf was last swept, and a
// leaf without it only pushes.
constexpr uint32_t WORK_SWEEP = 1u, WORK_LIVE = 128u;

// The sweeps work on a pool of leaves.  A voxel of it is one word: the bits of
// its magnitude shifted left, bit 0 set when its sign is not the sweeps' (a
// voxel they set has theirs), or NONE when it is inactive.  NONE is +inf's
// word, which no active voxel has: a band value beyond 2h was removed and a
// swept one is at most the limit.  Magnitudes order like their bits.  They are
// held times `scale`, a power of two that puts h at 1 or above (exact), so that
// the march's square roots stay in the range of sqrt_normal.
constexpr uint32_t INF_BITS = 0x7F800000u, FAR_BITS = 0x7F7FFFFFu, NONE = INF_BITS << 1;

struct SweepArgs {
    LeafMap map;
    int4* origins;
    uint64_t* frozen;  // active after remove_if: 8 words per leaf
    uint32_t* words;   // 512 per leaf
    uint32_t* work;    // see WORK_SWEEP
    uint32_t capacity;
    int sx, sy, sz;
    int neg;  // the sweeps' sign
    float h, limit;       // in the words' units
    float unscale;        // the caller's units per unit of the words
    uint32_t past_limit;  // bits of the first float above the limit
    int normal;           // this h and limit, and no NaN: the fast marches serve
};

// ---------------------------------------------------------------- remove_if
// leaf_node/tree_node.rs:151-160: active entries with |v| > 2h become
// inactive.  keep[leaf] = the leaf still has an active entry.
__global__ __launch_bounds__(256) void k_remove_if(uint64_t n, const uint64_t* __restrict__ masks,
                                                    const float* __restrict__ values, float two_h,
                                                    uint64_t* __restrict__ out_masks, uint32_t* __restrict__ keep) {
    const uint64_t leaf = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (leaf >= n) return;
    const int lane = threadIdx.x & 63;
    const int w = lane >> 3;
    const uint64_t word = masks[leaf * 8 + w];
    const float4* vp = reinterpret_cast<const float4*>(values + leaf * 512 + (uint64_t)lane * 8);
    const float4 q0 = vp[0], q1 = vp[1];
    const float v[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    uint32_t drop = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) drop |= (uint32_t)(fabsf(v[k]) > two_h) << k;
    const uint64_t bits = (word >> ((lane & 7) * 8)) & 0xFFull;
    uint64_t part = (bits & ~(uint64_t)drop) << ((lane & 7) * 8);
    part |= shfl_xor_u64(part, 1);
    part |= shfl_xor_u64(part, 2);
    part |= shfl_xor_u64(part, 4);
    if ((lane & 7) == 0) out_masks[leaf * 8 + w] = part;
    const uint64_t any = __ballot(part != 0);
    if (lane == 0) keep[leaf] = any != 0;
}

// Brings the kept leaves into the pool (frozen = mask after remove_if) and
// registers them in the leaf map; src[slot] = the input leaf.
__global__ __launch_bounds__(256) void k_pool_init(uint64_t n, const uint32_t* __restrict__ keep,
                                                    const uint32_t* __restrict__ dst, const int32_t* __restrict__ origins,
                                                    const uint64_t* __restrict__ rm_masks,
                                                    const float* __restrict__ values, float scale, SweepArgs a,
                                                    uint32_t* __restrict__ src, OffsetState* st) {
    const uint64_t leaf = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (leaf >= n || !keep[leaf]) return;
    const int lane = threadIdx.x & 63;
    const uint32_t s = dst[leaf];
    const float4* p = reinterpret_cast<const float4*>(values + leaf * 512 + (uint64_t)lane * 8);
    const float4 q0 = p[0], q1 = p[1];
    const float v[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    const uint32_t act = reinterpret_cast<const uint8_t*>(rm_masks)[leaf * 64 + lane];
    uint32_t w[8];
    bool nan = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const bool on = (act >> k) & 1u;
        w[k] = on ? __float_as_uint(fabsf(v[k]) * scale) << 1 | ((__float_as_uint(v[k]) >> 31) ^ (uint32_t)a.neg) : NONE;
        nan |= on && v[k] != v[k];
    }
    uint4* out = reinterpret_cast<uint4*>(a.words + (uint64_t)s * 512 + (uint64_t)lane * 8);
    out[0] = make_uint4(w[0], w[1], w[2], w[3]);
    out[1] = make_uint4(w[4], w[5], w[6], w[7]);
    if (lane < 8) a.frozen[(uint64_t)s * 8 + lane] = rm_masks[leaf * 8 + lane];
    if (nan) atomicOr(&st->nan, 1u);
    if (lane == 0) {
        const int4 o = make_int4(origins[leaf * 4], origins[leaf * 4 + 1], origins[leaf * 4 + 2], 0);
        a.origins[s] = o;
        a.work[s] = WORK_SWEEP | WORK_LIVE;
        src[s] = (uint32_t)leaf;
        if (!a.map.put(o.x >> 3, o.y >> 3, o.z >> 3, (int32_t)s)) atomicOr(&st->fail, 1u);
    }
}

// ---------------------------------------------------------------- plane buckets
__device__ inline int32_t leaf_plane(const int4 o, int sx, int sy, int sz) {
    return sx * (o.x >> 3) + sy * (o.y >> 3) + sz * (o.z >> 3);
}

// Leaves per plane.  A block counts its run of leaves in LDS (the planes of a
// run fit PLANE_LDS bins in every box up to 1300 leaves a side; past that the
// bins are in memory) and adds each plane's count once: with an atomic per leaf
// on a few hundred words, 567 k leaves took 0.26 ms, and 0.30 ms to scatter.
constexpr uint32_t PLANE_LDS = 4096;
constexpr int PLANE_BLOCK = 256;
constexpr uint32_t PLANE_RUN = 4096;  // leaves per block
__global__ __launch_bounds__(PLANE_BLOCK) void k_plane_hist(uint32_t n, const int4* __restrict__ origins, int sx, int sy,
                                                            int sz, int32_t kmin, uint32_t n_planes,
                                                            uint32_t* __restrict__ hist, uint32_t* fail) {
    __shared__ uint32_t bin[PLANE_LDS];
    const bool lds = n_planes <= PLANE_LDS;
    const uint32_t i0 = blockIdx.x * PLANE_RUN, i1 = min(n, i0 + PLANE_RUN);
    for (uint32_t k = threadIdx.x; lds && k < n_planes; k += PLANE_BLOCK) bin[k] = 0;
    __syncthreads();
    for (uint32_t i = i0 + threadIdx.x; i < i1; i += PLANE_BLOCK) {
        const int32_t k = leaf_plane(origins[i], sx, sy, sz) - kmin;
        if (k < 0 || (uint32_t)k >= n_planes)
            atomicOr(fail, 1u | 8u);
        else
            atomicAdd(lds ? &bin[k] : &hist[k], 1u);
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; lds && k < n_planes; k += PLANE_BLOCK)
        if (bin[k]) atomicAdd(&hist[k], bin[k]);
}

// order[] = the pool's leaves bucketed by plane, each with its origin and, in
// w, its pool slot.  Counted per block first, so a block takes each plane's
// range at once.
__global__ __launch_bounds__(PLANE_BLOCK) void k_plane_scatter(uint32_t n, const int4* __restrict__ origins, int sx,
                                                               int sy, int sz, int32_t kmin, uint32_t n_planes,
                                                               uint32_t* __restrict__ cursor, int4* __restrict__ order) {
    __shared__ uint32_t bin[PLANE_LDS];
    const bool lds = n_planes <= PLANE_LDS;
    const uint32_t i0 = blockIdx.x * PLANE_RUN, i1 = min(n, i0 + PLANE_RUN);
    if (lds) {
        for (uint32_t k = threadIdx.x; k < n_planes; k += PLANE_BLOCK) bin[k] = 0;
        __syncthreads();
        for (uint32_t i = i0 + threadIdx.x; i < i1; i += PLANE_BLOCK) {
            const int32_t k = leaf_plane(origins[i], sx, sy, sz) - kmin;
            if (k >= 0 && (uint32_t)k < n_planes) atomicAdd(&bin[k], 1u);
        }
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < n_planes; k += PLANE_BLOCK)
            if (bin[k]) bin[k] = atomicAdd(&cursor[k], bin[k]);
        __syncthreads();
    }
    for (uint32_t i = i0 + threadIdx.x; i < i1; i += PLANE_BLOCK) {
        int4 o = origins[i];
        const int32_t k = leaf_plane(o, sx, sy, sz) - kmin;
        if (k < 0 || (uint32_t)k >= n_planes) continue;
        o.w = (int32_t)i;
        order[atomicAdd(lds ? &bin[k] : &cursor[k], 1u)] = o;
    }
}

// ---------------------------------------------------------------- sweep
// The leaf and the six neighbour layers touching it in one padded block,
// leaf-local -1..8 per axis (edge and corner cells are never written or used),
// a z-row every 16 words with z = 0 on a 16-byte border.
constexpr int PB = 10, PY = 16, PX = PB * PY;
__device__ inline int pidx(int x, int y, int z) { return (x + 1) * PX + (y + 1) * PY + 4 + z; }

// f32 square root, correctly rounded for 0 and from 2^-96 up (NaN below 0):
// the hardware's is within one ulp, and the signs of two residuals say
// whether the float below or above it is the rounded one.
__device__ inline float sqrt_normal(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float below = __uint_as_float(__float_as_uint(s) - 1u), above = __uint_as_float(__float_as_uint(s) + 1u);
    float r = __builtin_fmaf(-below, s, x) <= 0.0f ? below : s;
    r = __builtin_fmaf(-above, s, x) > 0.0f ? above : r;
    return r;
}

// fast_sweep.rs:509-537 for sorted a1 <= a2 <= a3 (sort3, helpers/utils.rs:4-16),
// f32 throughout; the three candidate solutions are all computed and one is
// selected, which yields the same value as the reference's early returns.
// NORMAL: h is at least 1.  A radicand is then 0, negative or at least 2^-72: each
// of up to three subtractions from 2h^2 or 3h^2 leaves at least an ulp of what
// it subtracted from, so sqrt_normal serves.
template <bool NORMAL>
__device__ inline float solve_sorted(float a1, float a2, float a3, float h, float two_h_sq, float three_h_sq) {
    auto root = [](float x) { return NORMAL ? sqrt_normal(x) : sqrt_rn(x); };
    const float s1 = a1 + h;
    const float a1a2_sum = a1 + a2;
    const float a1a2_diff = a1 - a2;
    const float a1a2_diff_sq = a1a2_diff * a1a2_diff;
    const float s2 = (a1a2_sum + root(two_h_sq - a1a2_diff_sq)) * 0.5f;
    const float a1a2a3_sum = a1a2_sum + a3;
    const float a1a3_diff = a1 - a3;
    const float a1a3_diff_sq = a1a3_diff * a1a3_diff;
    const float a2a3_diff = a2 - a3;
    const float a2a3_diff_sq = a2a3_diff * a2a3_diff;
    const float s3 = (a1a2a3_sum + root(three_h_sq - a1a2_diff_sq - a1a3_diff_sq - a2a3_diff_sq)) * (1.0f / 3.0f);
    float r = fabsf(s2) <= a3 ? s2 : s3;
    asm volatile("" : "+v"(r));  // no branch around s2 and s3: nearly every plane of voxels needs them
    return fabsf(s1) <= a2 ? s1 : r;
}

// How a leaf is marched.  On one axis the reference takes option_min_by(at(+),
// at(-), cmp_abs) (utils.rs:64-73, fast_sweep.rs:137-140): the + value unless the
// - value has the strictly smaller magnitude; the sign of the first axis with a
// neighbour decides whether the voxel is updated.
// MARCH_ONE_SIGN  every voxel of the block has the sweeps' sign: an axis takes
//                 the smaller word, and without any neighbour the solve gives
//                 more than the limit;
// MARCH_SIGNED    both signs: that rule on words;
// MARCH_GENERAL   any h and limit, and NaN: that rule on floats.
enum MarchKind : int { MARCH_ONE_SIGN = 0, MARCH_SIGNED = 1, MARCH_GENERAL = 2 };

// The wavefront over the leaf's 22 voxel planes (fast_sweep.rs:120-184 for each
// voxel): plane p holds the voxels u + v + w = p (u, v, w the voxel's coordinates
// counted along the sweep), which do not depend on each other; lane (u, v) takes
// w = p - u - v.  A voxel reads the new values of its three upwind neighbours,
// written on plane p - 1, and the old ones of the downwind neighbours, all
// through one address that moves a word per plane.
//
// One wave issues an instruction every 4 to 5 cycles and a leaf is one wave, so
// the march costs its instruction count: about 75 a plane of voxels (95 with two
// signs), 4.8 us a leaf; 7.5 us with 150, from float compares, activity bytes and
// the full range's square root.
template <int KIND>
__device__ inline void march(const SweepArgs& a, uint32_t* word, int lane, uint32_t frozen) {
    const int x = lane >> 3, y = lane & 7;
    const int first_w = -(a.sx > 0 ? x : 7 - x) - (a.sy > 0 ? y : 7 - y);
    uint32_t* row = word + pidx(x, y, 0);
    const float h = a.h, h_sq = h * h, two_h_sq = h_sq + h_sq, three_h_sq = two_h_sq + h_sq;
    for (int p = 0; p < 22; ++p) {
        const int w = first_w + p;
        if ((uint32_t)w < 8u) {
            const int z = a.sz > 0 ? w : 7 - w;
            uint32_t* c = row + z;
            const uint32_t xp = c[PX], xm = c[-PX], yp = c[PY], ym = c[-PY], zp = c[1], zm = c[-1], own = c[0];
            const bool fixed = (frozen >> z) & 1u;
            if constexpr (KIND != MARCH_GENERAL) {
                uint32_t bx, by, bz;  // the axes' neighbours
                if constexpr (KIND == MARCH_ONE_SIGN) {
                    bx = min(xp, xm), by = min(yp, ym), bz = min(zp, zm);
                } else {
                    auto pick = [](uint32_t plus, uint32_t minus) { return (minus | 1u) < (plus & ~1u) ? minus : plus; };
                    bx = pick(xp, xm), by = pick(yp, ym), bz = pick(zp, zm);
                }
                const uint32_t mx = min(bx >> 1, FAR_BITS), my = min(by >> 1, FAR_BITS), mz = min(bz >> 1, FAR_BITS);
                const uint32_t lo = min(min(mx, my), mz), hi = max(max(mx, my), mz),
                               mid = max(min(mx, my), min(max(mx, my), mz));
                const float d = solve_sorted<true>(__uint_as_float(lo), __uint_as_float(mid), __uint_as_float(hi), h,
                                                   two_h_sq, three_h_sq);
                const uint32_t first = KIND == MARCH_ONE_SIGN ? 0u : (bx < NONE ? bx : (by < NONE ? by : bz));
                if (d < __uint_as_float(min(own >> 1, a.past_limit)) && !fixed && !(first & 1u))
                    *c = __float_as_uint(d) << 1;
            } else {
                const uint32_t plus[3] = {xp, yp, zp}, minus[3] = {xm, ym, zm};
                bool has[3];
                uint32_t q[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const bool hp = plus[k] != NONE, hm = minus[k] != NONE;
                    has[k] = hp || hm;
                    q[k] = (hp && hm) ? (__uint_as_float(plus[k] >> 1) > __uint_as_float(minus[k] >> 1) ? minus[k] : plus[k])
                                      : (hp ? plus[k] : minus[k]);
                }
                const uint32_t first = has[0] ? q[0] : (has[1] ? q[1] : q[2]);
                float a1 = has[0] ? __uint_as_float(q[0] >> 1) : FS_FAR, a2 = has[1] ? __uint_as_float(q[1] >> 1) : FS_FAR,
                      a3 = has[2] ? __uint_as_float(q[2] >> 1) : FS_FAR, t;
                if (a1 > a3) t = a1, a1 = a3, a3 = t;
                if (a1 > a2) t = a1, a1 = a2, a2 = t;
                if (a2 > a3) t = a2, a2 = a3, a3 = t;
                const float d = fabsf(solve_sorted<false>(a1, a2, a3, h, two_h_sq, three_h_sq));
                const float old = own != NONE ? __uint_as_float(own >> 1) : FS_FAR;
                if (!fixed && (has[0] || has[1] || has[2]) && !(first & 1u) && !(d > a.limit) && d < old)
                    *c = __float_as_uint(d) << 1;
            }
        }
        // the wave's LDS operations complete in order: the compiler alone must keep the next plane's reads below
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// Claims the missing neighbours that a leaf pushes: lanes 0..2, the sweep's
// +direction face of each axis.  A created slot is published without a fence:
// in this plane a lookup of the new leaf reads only its words, which hold the
// empty leaf already, and its origin and work bits are read only in a later
// plane.
__device__ inline void push_neighbours(const SweepArgs& a, int4 org, uint32_t faces, uint32_t plane, uint32_t n_planes,
                                       uint32_t start, uint2* counts, OffsetState* st, int lane, bool there) {
    const int s = lane == 0 ? a.sx : (lane == 1 ? a.sy : a.sz);
    if (lane >= 3 || !((faces >> (2 * lane + (s > 0 ? 2 : 1))) & 1u)) return;
    if (plane + 1 >= n_planes) atomicOr(&st->fail, 1u | 4u);
    if (there) return;
    const int32_t nx = (org.x >> 3) + (lane == 0 ? s : 0), ny = (org.y >> 3) + (lane == 1 ? s : 0),
                  nz = (org.z >> 3) + (lane == 2 ? s : 0);
    int32_t* cell = a.map.claim(nx, ny, nz, &st->fail);
    if (!cell) return;
    const uint32_t slot = start + atomicAdd(&counts[plane + 1].y, 1u);
    if (slot < a.capacity) {
        a.origins[slot] = make_int4(nx * 8, ny * 8, nz * 8, 0);
        a.work[slot] = WORK_SWEEP;
        atomicExch(cell, (int32_t)slot);
    } else {
        atomicOr(&st->fail, 2u);  // pool overflow: retried with a larger pool
    }
}

// a word with its sign bit on top: below INF_BITS exactly when the voxel is
// active with the sweeps' sign
__device__ inline uint32_t sign_first(uint32_t w) { return w >> 1 | w << 31; }

// One leaf plane of one sweep: entries [b0, b0 + n_old) of `order` (origin and,
// in w, pool slot) plus the leaves created while the previous plane was swept.
// counts[p + 1] holds the pool size when plane p begins (x) and the leaves plane
// p creates (y, all on plane p + 1), so this plane sweeps the pool range [x, x + y)
// of counts[plane] after its bucket and allocates its own new leaves from x + y
// on; the sweep's first plane has no leaves created before it and begins with
// `pool` leaves.  One wavefront per leaf, looping over the plane's leaves.
//
// A sweep is a chain of these launches, so what counts is the time of one leaf
// from end to end: three dependent rounds of loads (the leaf's entry; its
// words, work bits and six map cells; the six neighbour layers), the march, the
// write-back of what changed, and the pushes.  Code that runs once per leaf
// costs most of its time in instruction fetch (a launch starts with a cold
// instruction cache: about 15 cycles an instruction), so the pool holds words
// that go to LDS as they are; from values and masks, coding and decoding
// them took 2.5 us of a leaf's 11.5.
__global__ __launch_bounds__(64) void k_sweep_plane(SweepArgs a, const int4* __restrict__ order, uint32_t b0,
                                                     uint32_t n_old, uint32_t plane, uint32_t first,
                                                     uint32_t n_planes, uint32_t pool, uint2* counts, OffsetState* st) {
    __shared__ __align__(16) uint32_t word[PB * PX];
    const int lane = threadIdx.x, x = lane >> 3, y = lane & 7;
    int4 entry = order[b0 + min(blockIdx.x, max(n_old, 1u) - 1)];  // before the counts arrive
    const uint2 before = counts[plane];
    const uint32_t new_lo = plane == first ? pool : before.x;
    const uint32_t start = plane == first ? pool : min(new_lo + before.y, a.capacity);
    const uint32_t n_new = start - new_lo;
    if (blockIdx.x == 0 && lane == 0) counts[plane + 1].x = start;
    for (uint32_t item = blockIdx.x; item < n_old + n_new; item += gridDim.x) {
        if (item >= n_old) {
            entry = a.origins[new_lo + (item - n_old)];
            entry.w = (int32_t)(new_lo + (item - n_old));
        } else if (item != blockIdx.x) {
            entry = order[b0 + item];
        }
        const uint32_t slot = (uint32_t)entry.w;
        const uint32_t work = a.work[slot];
        uint4* mine = reinterpret_cast<uint4*>(a.words + (uint64_t)slot * 512 + lane * 8);
        const uint4 w0 = mine[0], w1 = mine[1];
        // byte y of a frozen word x holds row (x, y)
        const uint32_t frozen = reinterpret_cast<const uint8_t*>(a.frozen)[(uint64_t)slot * 64 + lane];
        // lanes 0..5: the neighbour slots (-1: none, or a leaf being created, which has no active voxel)
        int32_t nb = -1;
        if (lane < 6) {
            const int ax = lane >> 1, dir = (lane & 1) ? 1 : -1;
            nb = a.map.find((entry.x >> 3) + (ax == 0 ? dir : 0), (entry.y >> 3) + (ax == 1 ? dir : 0),
                            (entry.z >> 3) + (ax == 2 ? dir : 0));
        }
        int32_t n[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) n[k] = __builtin_amdgcn_readlane(nb, k);
        const bool there = (lane == 0 ? (a.sx > 0 ? n[1] : n[0])
                                      : (lane == 1 ? (a.sy > 0 ? n[3] : n[2]) : (a.sz > 0 ? n[5] : n[4]))) >= 0;
        if (!(work & WORK_SWEEP)) {
            push_neighbours(a, entry, work, plane, n_planes, start, counts, st, lane, there);
            continue;
        }
        // the six layers next to the leaf, a voxel per lane and face (slot 0 in place of a missing neighbour)
        uint32_t f[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int far = (k & 1) ? 0 : 7;  // -side neighbour: its layer 7; +side: layer 0
            const int off = k < 2 ? (far << 6 | lane) : (k < 4 ? (x << 6 | far << 3 | y) : (lane << 3 | far));
            f[k] = a.words[(n[k] >= 0 ? (uint64_t)n[k] : 0) * 512 + off];
        }
        uint4* own = reinterpret_cast<uint4*>(word + pidx(x, y, 0));
        own[0] = w0;
        own[1] = w1;
        const uint32_t old[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
        uint32_t least = NONE, either = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) least = min(least, sign_first(old[k])), either |= old[k];
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            f[k] = n[k] >= 0 ? f[k] : NONE;
            least = min(least, sign_first(f[k])), either |= f[k];
            const int g = (k & 1) ? 8 : -1;
            word[k < 2 ? pidx(g, x, y) : (k < 4 ? pidx(x, g, y) : pidx(x, y, g))] = f[k];
        }
        __syncthreads();
        if (!a.normal)
            march<MARCH_GENERAL>(a, word, lane, frozen);
        else if (__ballot(least < INF_BITS)) {
            if (__ballot(either & 1u))
                march<MARCH_SIGNED>(a, word, lane, frozen);
            else
                march<MARCH_ONE_SIGN>(a, word, lane, frozen);
        }  // else no voxel has the sweeps' sign: none is set, and none can be pushed
        __syncthreads();
        // what changed, what can be pushed
        const uint4 r0 = own[0], r1 = own[1];
        const uint32_t now[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
        uint32_t diff = 0;
        least = NONE;
#pragma unroll
        for (int k = 0; k < 8; ++k) diff |= now[k] ^ old[k], least = min(least, sign_first(now[k]));
        const uint32_t limit_bits = __float_as_uint(a.limit);
        const uint64_t FX0 = 0xFFull, FX7 = FX0 << 56, FY0 = 0x0101010101010101ull, FY7 = FY0 << 7;  // rows of the faces
        const uint64_t can = __ballot(least < limit_bits);
        uint32_t faces = (uint32_t)((can & FX0) != 0) << 1 | (uint32_t)((can & FX7) != 0) << 2 |
                         (uint32_t)((can & FY0) != 0) << 3 | (uint32_t)((can & FY7) != 0) << 4 |
                         (uint32_t)(__ballot(sign_first(now[0]) < limit_bits) != 0) << 5 |
                         (uint32_t)(__ballot(sign_first(now[7]) < limit_bits) != 0) << 6 | (work & WORK_LIVE);
        const uint64_t set = __ballot(diff != 0);
        if (set) {
            faces |= WORK_SWEEP | WORK_LIVE;
            mine[0] = r0;
            mine[1] = r1;
            const uint32_t moved = (uint32_t)((set & FX0) != 0) | (uint32_t)((set & FX7) != 0) << 1 |
                                   (uint32_t)((set & FY0) != 0) << 2 | (uint32_t)((set & FY7) != 0) << 3 |
                                   (uint32_t)(__ballot(now[0] != old[0]) != 0) << 4 |
                                   (uint32_t)(__ballot(now[7] != old[7]) != 0) << 5;
            if (lane < 6 && nb >= 0 && (moved >> lane & 1u)) atomicOr(&a.work[nb], WORK_SWEEP);
        }
        if (lane == 0) a.work[slot] = faces;
        push_neighbours(a, entry, faces, plane, n_planes, start, counts, st, lane, there);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- output
// Sort keys of the final pool: empty leaves (fast_sweep.rs:61-64
// remove_empty_branches) sort last.
__global__ __launch_bounds__(256) void k_final_keys(uint32_t n, const int4* __restrict__ origins,
                                                     const uint32_t* __restrict__ work, uint64_t* __restrict__ keys,
                                                     uint32_t* __restrict__ idx, OffsetState* st) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n && (work[i] & WORK_LIVE);
    if (i < n) {
        const int4 o = origins[i];
        keys[i] = live ? leaf_key(o.x >> 3, o.y >> 3, o.z >> 3) : ~0ull;
        idx[i] = i;
    }
    const uint64_t b = __ballot(live);
    if ((threadIdx.x & 63) == 0 && b) atomicAdd(&st->live, (uint32_t)__popcll(b));
}

// Gathers the live leaves in key order and applies v -= D to active values
// (visitors/value_mut_visitor.rs:4-32 visits active values only): a frozen
// voxel has its input value, a swept one its word's, an inactive one what the
// input held (0 in a created leaf).
__global__ __launch_bounds__(256) void k_final_gather(uint64_t n_out, const uint32_t* __restrict__ src_idx, SweepArgs a,
                                                       uint32_t n_keep, const uint32_t* __restrict__ src,
                                                       const float* __restrict__ in_values, float distance,
                                                       int4* __restrict__ origins, uint64_t* __restrict__ masks,
                                                       float* __restrict__ values) {
    const uint64_t leaf = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (leaf >= n_out) return;
    const int lane = threadIdx.x & 63;
    const uint32_t s = src_idx[leaf];
    const uint4* wp = reinterpret_cast<const uint4*>(a.words + (uint64_t)s * 512 + lane * 8);
    const uint4 w0 = wp[0], w1 = wp[1];
    const uint32_t frozen = reinterpret_cast<const uint8_t*>(a.frozen)[(uint64_t)s * 64 + lane];
    float4 q0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), q1 = q0;
    if (s < n_keep) {
        const float4* vp = reinterpret_cast<const float4*>(in_values + (uint64_t)src[s] * 512 + lane * 8);
        q0 = vp[0];
        q1 = vp[1];
    }
    const uint32_t w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
    float v[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    uint32_t row = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (w[k] == NONE) continue;
        row |= 1u << k;
        if (!((frozen >> k) & 1u))
            v[k] = __uint_as_float(__float_as_uint(__uint_as_float(w[k] >> 1) * a.unscale) | (uint32_t)a.neg << 31);
        v[k] = v[k] - distance;
    }
    float4* op = reinterpret_cast<float4*>(values + leaf * 512 + (uint64_t)lane * 8);
    op[0] = make_float4(v[0], v[1], v[2], v[3]);
    op[1] = make_float4(v[4], v[5], v[6], v[7]);
    const uint64_t m = gather_word(row, lane & 7);
    if ((lane & 7) == 0) masks[leaf * 8 + (lane >> 3)] = m;
    if (lane == 0) origins[leaf] = a.origins[s];
}

constexpr int kDirs[8][3] = {{1, 1, 1},  {-1, 1, 1},  {1, -1, 1},  {-1, -1, 1},
                             {1, 1, -1}, {-1, 1, -1}, {1, -1, -1}, {-1, -1, -1}};  // fast_sweep.rs:36-57

template <class K, class V>
void sort_pairs_u64(bs_ctx* ctx, const K* k, K* ks, const V* v, V* vs, uint64_t n) {
    size_t bytes = 0;
    BS_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k, ks, v, vs, (int)n, 0, 64, ctx->stream));
    void* tmp = ctx->scratch.get(S_CUB, bytes);
    BS_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, bytes, k, ks, v, vs, (int)n, 0, 64, ctx->stream));
}

void exclusive_scan_u32(bs_ctx* ctx, const uint32_t* in, uint32_t* out, uint64_t n) {
    size_t bytes = 0;
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, ctx->stream));
    void* tmp = ctx->scratch.get(S_CUB, bytes);
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, (int)n, ctx->stream));
}

// Device buffers of an offset, back to the pool on every exit path once the
// stream is done with them.  All that grows with the volume or the leaf pool is
// here (2.2 KB per pool leaf), so that nothing of that size stays with the
// context.
struct OffsetBuffers {
    hipStream_t st;
    std::vector<void*> ptrs;
    explicit OffsetBuffers(hipStream_t s) : st(s) { ptrs.reserve(8); }
    template <class T> T* alloc(uint64_t count) {
        ptrs.push_back(alloc_block(std::max<uint64_t>(count, 1) * sizeof(T)));
        return static_cast<T*>(ptrs.back());
    }
    // several arrays in one block: f lays them out from p on (see take), first from null to find the size
    template <class F> void carve(F&& f) {
        uint8_t* p = nullptr;
        f(p);
        p = alloc<uint8_t>((uint64_t)(uintptr_t)p);
        f(p);
    }
    ~OffsetBuffers() {
        const bool done = hipStreamSynchronize(st) == hipSuccess;
        for (void* p : ptrs) free_block(p, !done);
    }
};

}  // namespace

Topology& ensure_topology(bs_ctx* ctx, bs_volume* v);

namespace {

// An array at p on a 256-byte border; p moves past it.
template <class T> void take(uint8_t*& p, T*& array, uint64_t count) {
    array = reinterpret_cast<T*>(p);
    p += (count * sizeof(T) + 255) / 256 * 256;
}

// What remove_if leaves of the volume, the same for every attempt.
struct KeptLeaves {
    uint64_t* masks = nullptr;  // per input leaf: 8 words
    uint32_t *keep = nullptr, *dst = nullptr;
};

struct OffsetResult {
    uint64_t n_out = 0;
    bool retry = false;
};

// One attempt with a pool of `capacity` leaves; retry = the pool or the leaf
// map was too small (nothing of `vol` was modified).
OffsetResult offset_attempt(bs_ctx* ctx, bs_volume* vol, float distance, uint64_t capacity, bool force_hash,
                            const KeptLeaves& kept, bs_volume& out, bs_offset_stats* stats) {
    hipStream_t st = ctx->stream;
    OffsetResult res;
    const uint64_t n = vol->n_leaves;
    const float h = vol->voxel_size;
    const float two_h = h * 2.0f;  // volume/mod.rs:96
    float ext = fabsf(distance) + h + h;  // volume/mod.rs:98-99
    ext = std::copysign(ext, std::signbit(distance) ? -1.0f : 1.0f);
    const float limit_abs = fabsf(ext);
    const int neg = std::signbit(ext) ? 1 : 0;

    if (stats) stats->n_kept = 0;
    if (n == 0) return res;
    Scratch& S = ctx->scratch;
    OffsetBuffers B(st);
    // remove_if and compaction of the surviving leaves
    uint64_t* rm_masks = kept.masks;
    uint32_t *keep = kept.keep, *dst = kept.dst;
    int32_t* dbox = S.as<int32_t>(S_LEAF_BOX, 6);
    k_remove_if<<<div_up(n, 4), 256, 0, st>>>(n, vol->masks, vol->values, two_h, rm_masks, keep);
    BS_HIP(hipGetLastError());
    exclusive_scan_u32(ctx, keep, dst, n);
    k_leaf_box_init<<<1, 64, 0, st>>>(dbox);
    BS_HIP(hipGetLastError());
    k_leaf_box<<<(unsigned)std::min<uint64_t>(div_up(n, 256), 256), 256, 0, st>>>(
        n, reinterpret_cast<const int4*>(vol->origins), dbox, keep);
    BS_HIP(hipGetLastError());
    uint32_t* first = static_cast<uint32_t*>(pinned_words(ctx, 8));
    BS_HIP(hipMemcpyAsync(first, dst + n - 1, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipMemcpyAsync(first + 1, keep + n - 1, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipMemcpyAsync(first + 2, dbox, 6 * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipStreamSynchronize(st));
    const uint64_t n_keep = (uint64_t)first[0] + first[1];
    int32_t box[6];
    std::memcpy(box, first + 2, sizeof(box));
    if (stats) stats->n_kept = n_keep;
    if (n_keep == 0) return res;
    int32_t lo[3] = {box[0], box[1], box[2]}, hi[3] = {box[3], box[4], box[5]};
    BS_REQUIRE(capacity >= n_keep && capacity < (1ull << 31), BS_ERR_INVALID_ARG, "offset leaf pool too large");

    // Reach of the extension: a value grows by at least h/sqrt(3) per voxel
    // step (the three-term Godunov update is the smallest increment), so no
    // leaf beyond limit*sqrt(3)/h + 2 voxels of the band is ever pushed.
    const int32_t margin = (int32_t)std::ceil(((double)limit_abs / (double)h * 1.7320508075688772 + 4.0) / 8.0) + 1;
    LeafMap map{};
    uint64_t cells = 1;
    for (int k = 0; k < 3; ++k) {
        lo[k] -= margin;
        hi[k] += margin;
        cells *= (uint64_t)(hi[k] - lo[k] + 1);
    }
    map.dense = !force_hash && cells <= (1ull << 28);
    if (map.dense) {
        map.x0 = lo[0], map.y0 = lo[1], map.z0 = lo[2];
        map.nx = hi[0] - lo[0] + 1, map.ny = hi[1] - lo[1] + 1, map.nz = hi[2] - lo[2] + 1;
        map.cells = B.alloc<int32_t>(cells);
        BS_HIP(hipMemsetAsync(map.cells, 0xFF, sizeof(int32_t) * cells, st));
    } else {
        uint64_t cap = 1024;
        while (cap < 2 * capacity) cap <<= 1;
        map.cap_mask = (uint32_t)(cap - 1);
        map.keys = B.alloc<uint64_t>(cap);
        map.cells = B.alloc<int32_t>(cap);
        BS_HIP(hipMemsetAsync(map.keys, 0xFF, sizeof(uint64_t) * cap, st));
        BS_HIP(hipMemsetAsync(map.cells, 0xFF, sizeof(int32_t) * cap, st));
    }
    if (stats) stats->used_hash = !map.dense;
    if (stats) stats->n_capacity = capacity;

    SweepArgs a{};
    a.map = map;
    a.capacity = (uint32_t)capacity;
    int4* order = nullptr;
    uint32_t* src = nullptr;
    B.carve([&](uint8_t*& p) {
        take(p, a.origins, capacity);
        take(p, a.frozen, 8 * capacity);
        take(p, a.work, capacity);
        take(p, order, capacity + 1);  // a plane past the last bucket reads an entry that it does not use
        take(p, src, n_keep);
    });
    a.words = B.alloc<uint32_t>(512 * capacity);
    a.neg = neg;
    // the words' units (see NONE): scaling up by a power of two is exact, and nothing overflows with h within
    // 2^+-60 and the limit within 2^59 of it
    int h_exp = 0;
    std::frexp(h, &h_exp);
    const bool in_range = h_exp >= -60 && h_exp <= 60 && limit_abs / h <= 5.0e17f;
    const int up = in_range && h_exp < 1 ? 1 - h_exp : 0;
    const float scale = std::ldexp(1.0f, up);
    a.unscale = std::ldexp(1.0f, -up);
    a.h = h * scale;
    a.limit = limit_abs * scale;
    const float past_limit = std::nextafter(a.limit, INFINITY);
    std::memcpy(&a.past_limit, &past_limit, sizeof(float));
    // leaves created by the sweep start empty (Leaf::empty)
    BS_HIP(hipMemsetD32Async(a.words + 512 * n_keep, (int)NONE, 512 * (capacity - n_keep), st));
    BS_HIP(hipMemsetAsync(a.frozen + 8 * n_keep, 0, sizeof(uint64_t) * 8 * (capacity - n_keep), st));
    // the planes of the map box, as many in every direction; their leaf counts and bucket starts, the state (read
    // back with the starts in one copy) and the pool counts
    const uint32_t n_planes = (uint32_t)(hi[0] - lo[0] + hi[1] - lo[1] + hi[2] - lo[2] + 1);
    constexpr uint32_t STATE_WORDS = sizeof(OffsetState) / sizeof(uint32_t);
    uint32_t* hist = S.as<uint32_t>(S_OFF_PLANES, 4 * (uint64_t)(n_planes + 2) + STATE_WORDS + 2);
    uint32_t* off = hist + n_planes + 1;
    OffsetState* dstate = reinterpret_cast<OffsetState*>(off + n_planes + 1);
    uint2* counts = reinterpret_cast<uint2*>(hist + (2 * (n_planes + 1) + STATE_WORDS + 1) / 2 * 2);
    uint32_t* back = static_cast<uint32_t*>(pinned_words(ctx, n_planes + 1 + STATE_WORDS));
    const uint32_t* hoff = back;
    OffsetState cur{};
    auto read_state = [&] { std::memcpy(&cur, back + n_planes + 1, sizeof(cur)); };
    BS_HIP(hipMemsetAsync(dstate, 0, sizeof(OffsetState), st));
    k_pool_init<<<div_up(n, 4), 256, 0, st>>>(n, keep, dst, vol->origins, rm_masks, vol->values, scale, a, src, dstate);
    BS_HIP(hipGetLastError());

    uint64_t planes_total = 0, swept = 0;
    uint32_t pool = (uint32_t)n_keep;  // pool size at the start of the sweep
    auto check = [&](int s) {
        BS_REQUIRE(!(cur.fail & 1u), BS_ERR_INTERNAL,
                   "offset: a pushed leaf left the reachable box (flags " + std::to_string(cur.fail) + ", sweep " +
                       std::to_string(s) + ", pool " + std::to_string(pool) + ")");
        return cur.fail == 0;
    };
    for (int s = 0; s < 8; ++s) {
        a.sx = kDirs[s][0], a.sy = kDirs[s][1], a.sz = kDirs[s][2];
        const int32_t kmin = (a.sx > 0 ? lo[0] : -hi[0]) + (a.sy > 0 ? lo[1] : -hi[1]) + (a.sz > 0 ? lo[2] : -hi[2]);
        BS_HIP(hipMemsetAsync(hist, 0, sizeof(uint32_t) * (n_planes + 1), st));
        BS_HIP(hipMemsetAsync(counts, 0, sizeof(uint2) * (n_planes + 1), st));
        k_plane_hist<<<div_up(pool, PLANE_RUN), PLANE_BLOCK, 0, st>>>(pool, a.origins, a.sx, a.sy, a.sz, kmin, n_planes,
                                                                      hist, &dstate->fail);
        BS_HIP(hipGetLastError());
        exclusive_scan_u32(ctx, hist, off, n_planes + 1);
        BS_HIP(hipMemcpyAsync(back, off, sizeof(uint32_t) * (n_planes + 1 + STATE_WORDS), hipMemcpyDeviceToHost, st));
        k_plane_scatter<<<div_up(pool, PLANE_RUN), PLANE_BLOCK, 0, st>>>(pool, a.origins, a.sx, a.sy, a.sz, kmin,
                                                                         n_planes, off, order);
        BS_HIP(hipGetLastError());
        BS_HIP(hipStreamSynchronize(st));
        read_state();
        res.retry = !check(s);
        if (res.retry) return res;
        a.normal = in_range && !cur.nan;
        // the first and the last plane holding a leaf (the pool is never empty)
        uint32_t first = 0, last = n_planes - 1;
        while (hoff[first + 1] == 0) ++first;
        while (hoff[last] == hoff[n_planes]) --last;
        auto launch = [&](uint32_t p) {
            // enough blocks for the bucket and the leaves the previous plane may have created
            const uint32_t bucket = hoff[p + 1] - hoff[p], prev = p > first ? hoff[p] - hoff[p - 1] : 0;
            const unsigned grid = (unsigned)std::min<uint64_t>((uint64_t)bucket + prev + 64, 4096);
            k_sweep_plane<<<grid, 64, 0, st>>>(a, order, hoff[p], bucket, p, first, n_planes, pool, counts, dstate);
            BS_HIP(hipGetLastError());
            ++planes_total;
        };
        uint32_t p = first;
        while (p <= last) launch(p++);
        // past the last bucket: on while the planes create leaves, a few planes for each look
        uint32_t* tail = back + n_planes + 1;
        for (;;) {
            for (uint32_t e = std::min(n_planes, p + 4); p < e; ++p) launch(p);
            BS_HIP(hipMemcpyAsync(tail, counts + p, sizeof(uint2), hipMemcpyDeviceToHost, st));
            BS_HIP(hipStreamSynchronize(st));
            if (p == n_planes || tail[1] == 0) break;
        }
        // the pool's size after the last plane swept
        if ((uint64_t)tail[0] + tail[1] > capacity) {
            res.retry = true;
            return res;
        }
        pool = tail[0] + tail[1];
        swept += pool;  // every leaf in the pool at the end of a sweep was swept in it
    }
    const uint32_t n_pool = pool;
    if (stats) {
        stats->n_swept = swept;
        stats->n_pool = n_pool;
        stats->n_planes = planes_total;
        stats->n_launches = planes_total;
    }

    // empty leaves go, the rest sorted by origin, shifted by -D
    uint64_t *keys = nullptr, *keys_s = nullptr;
    uint32_t *idx = nullptr, *idx_s = nullptr;
    B.carve([&](uint8_t*& p) {
        take(p, keys, n_pool);
        take(p, keys_s, n_pool);
        take(p, idx, n_pool);
        take(p, idx_s, n_pool);
    });
    k_final_keys<<<div_up(n_pool, 256), 256, 0, st>>>(n_pool, a.origins, a.work, keys, idx, dstate);
    BS_HIP(hipGetLastError());
    BS_HIP(hipMemcpyAsync(back + n_planes + 1, dstate, sizeof(cur), hipMemcpyDeviceToHost, st));
    sort_pairs_u64(ctx, keys, keys_s, idx, idx_s, n_pool);
    BS_HIP(hipStreamSynchronize(st));
    read_state();
    res.retry = !check(8);
    if (res.retry) return res;
    const uint32_t n_out = cur.live;
    alloc_leaves(&out, n_out);
    if (n_out) {
        k_final_gather<<<div_up(n_out, 4), 256, 0, st>>>(n_out, idx_s, a, (uint32_t)n_keep, src, vol->values, distance,
                                                         reinterpret_cast<int4*>(out.origins), out.masks, out.values);
        BS_HIP(hipGetLastError());
    }
    BS_HIP(hipStreamSynchronize(st));
    res.n_out = n_out;
    return res;
}

}  // namespace

// Volume::offset (volume/mod.rs:95-108) of `vol` in place.
void volume_offset(bs_ctx* ctx, bs_volume* vol, float distance, bs_offset_stats* stats) {
    BS_REQUIRE(std::isfinite(distance), BS_ERR_INVALID_ARG, "offset distance must be finite");
    const auto t_wall = std::chrono::steady_clock::now();
    EventPair ev;
    ev.start(ctx->stream);
    BS_REQUIRE(vol->device == ctx->device, BS_ERR_INVALID_ARG, "volume lives on another device");
    require_tree(vol);
    const float two_h = vol->voxel_size * 2.0f;
    // fast_sweep.rs:100 unwraps the leaf at every queued origin, and the queue
    // holds every active tile that survives remove_if: the reference panics.
    for (const TileRec& t : vol->tiles)
        BS_REQUIRE(fabsf(t.value) > two_h, BS_ERR_INTERNAL,
                   "offset: an active tile lies within the band; the reference panics (fast_sweep.rs:100)");
    if (stats) *stats = bs_offset_stats{};
    uint64_t capacity = std::max<uint64_t>(4 * vol->n_leaves + 4096, 8192);
    // the result's leaf arrays, given back unless they have moved into the volume
    struct Result {
        hipStream_t st;
        bs_volume v;
        ~Result() { free_leaves(&v, st); }
    } result{ctx->stream, {}};
    bs_volume& out = result.v;
    out.device = vol->device;
    OffsetBuffers kept_block(ctx->stream);
    KeptLeaves kept;
    kept_block.carve([&](uint8_t*& p) {
        take(p, kept.masks, 8 * vol->n_leaves);
        take(p, kept.keep, vol->n_leaves);
        take(p, kept.dst, vol->n_leaves);
    });
    OffsetResult r;
    for (int attempt = 0;; ++attempt) {
        r = offset_attempt(ctx, vol, distance, capacity, (ctx->paths & BS_PATH_FORCE_HASH) != 0, kept, out, stats);
        if (!r.retry) break;
        BS_REQUIRE(attempt < 6, BS_ERR_INTERNAL, "offset: leaf pool kept overflowing");
        capacity *= 4;
    }
    // the tree: remove_if (tiles, emptied leaves, empty nodes), the new leaves, empty nodes again.  A volume
    // without one has the tree that its leaves give (no tile survives), and so has the result.
    std::unique_ptr<Topology> t2;
    std::unique_ptr<DeviceTree> d2;
    if (vol->topo || vol->tree || !vol->tiles.empty()) {
        if (const DeviceTree* d = ensure_tree(ctx, vol))
            d2 = tree_after_offset(ctx, *d, reinterpret_cast<const int4*>(vol->origins), kept.keep, vol->n_leaves,
                                   reinterpret_cast<const int4*>(out.origins), out.n_leaves);
        if (!d2) {
            std::vector<uint32_t> keep(vol->n_leaves);
            std::vector<int32_t> o4(4 * out.n_leaves);
            if (!keep.empty())
                BS_HIP(hipMemcpy(keep.data(), kept.keep, sizeof(uint32_t) * keep.size(), hipMemcpyDeviceToHost));
            if (!o4.empty())
                BS_HIP(hipMemcpy(o4.data(), out.origins, sizeof(int32_t) * o4.size(), hipMemcpyDeviceToHost));
            std::vector<std::array<int32_t, 3>> out_origins(out.n_leaves);
            for (uint64_t i = 0; i < out.n_leaves; ++i) out_origins[i] = {o4[4 * i], o4[4 * i + 1], o4[4 * i + 2]};
            t2 = ensure_topology(ctx, vol).after_offset(keep, out_origins, two_h);
        }
    }
    const uint64_t n_out = out.n_leaves;
    free_leaves(vol);
    vol->n_leaves = n_out;
    vol->origins = out.origins;
    vol->masks = out.masks;
    vol->values = out.values;
    out.origins = nullptr;
    out.masks = nullptr;
    out.values = nullptr;
    vol->tiles.clear();  // remove_if deactivated every tile (checked above)
    vol->topo = std::move(t2);
    vol->tree = std::move(d2);
    ev.stop(ctx->stream);
    if (stats) {
        stats->n_out = n_out;
        stats->ms_device = ev.ms();
        stats->ms_wall = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_wall).count();
    }
}

}  // namespace bs
