// Mesh -> narrow-band signed distance volume on one MI355X.
//
// Replaces MeshToVolume::convert (src/voxel/mesh_to_volume.rs:52-73):
//   subdivide     mesh_to_volume.rs:75-116   one thread per (triangle, row)
//   leaves        :118-168 active set        dilated boxes -> dense leaf grid or GPU hash -> compact
//   distance      :118-196 min over pairs    one workgroup per 8^3 leaf, box/leaf regions scattered
//                                            into an LDS arg-min, reference arithmetic for the winner
//   winding       aabb_tree.rs:571-817       LBVH + order-2 dipoles, wave-coherent traversal
//   sign          mesh_to_volume.rs:238-292  wn < threshold => +|d| else -|d|
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <type_traits>

#include "common.hpp"
#include "surrogate.hpp"
#include "m2v_kernels.hpp"

namespace bs {

namespace {

constexpr float INV_4PI = 0.0795774715459476678844f;
constexpr int BVH_LEAF_SIZE = 2;     // a node covering <= 2 triangles is evaluated as a leaf
constexpr int WN_STACK = 128;        // per-wave traversal stack depth
constexpr int WN_BLOCK = 256;

enum Counter : int {
    C_ERR = 0, C_LEAVES, C_RECHECK, C_NEAR_INTERNAL, C_FAR, C_LEAF_VISITS, C_LEAF_TRIS, C_BOX_LO, C_BOX_HI = C_BOX_LO + 3,
    C_PAIRS = C_BOX_HI + 3, C_SG_TILES, C_SG_CULLED, C_SG_MISS, C_SG_FALLBACK, C_COUNT
};
enum ErrBits : unsigned { E_RANGE = 1, E_TOO_MANY_SUBS = 2, E_STACK = 4, E_HASH = 8, E_TREE = 16 };

// ---------------------------------------------------------------------------
// subdivision (mesh_to_volume.rs:75-116)

__device__ inline void load_tri(const float* t, F3& a, F3& b, F3& c) {
    a = {t[0], t[1], t[2]};
    b = {t[3], t[4], t[5]};
    c = {t[6], t[7], t[8]};
}

__global__ void k_subdiv_count(const float* __restrict__ tris, uint64_t n, float h, uint32_t* rows, uint64_t* subs,
                               unsigned* err) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    F3 a, b, c;
    load_tri(tris + 9 * i, a, b, c);
    float num_subs = floorf(div_rn(tri_max_side(a, b, c), h));
    if (num_subs < 2.0f) {
        rows[i] = 1;
        subs[i] = 1;
        return;
    }
    // `for i in 0..num_subs as usize` (NaN -> 0 rows)
    float lim = 65536.0f;
    if (!(num_subs < lim)) {
        if (num_subs == num_subs) atomicOr(err, E_TOO_MANY_SUBS);
        rows[i] = 0;
        subs[i] = 0;
        return;
    }
    uint32_t ns = (uint32_t)num_subs;
    rows[i] = ns;
    subs[i] = (uint64_t)ns * ns;
}

// One thread per (triangle, row i): a_i is p1 + s1 accumulated i times, then the
// row emits (a_prev, b_s, a_s), (a_s, b_s, c_s) i times and (a, b, c), exactly
// as the reference's sequential loop does.
__global__ void k_subdiv_emit(const float* __restrict__ tris, uint64_t n, float h, const uint32_t* __restrict__ row_off,
                              const uint64_t* __restrict__ sub_off, uint64_t total_rows, float* __restrict__ out) {
    uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= total_rows) return;
    // triangle t: row_off[t] <= r < row_off[t+1]
    uint64_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint64_t mid = (lo + hi) >> 1;
        if (row_off[mid] <= r) lo = mid;
        else hi = mid;
    }
    uint64_t t = lo;
    uint32_t i = (uint32_t)(r - row_off[t]);
    F3 p1, p2, p3;
    load_tri(tris + 9 * t, p1, p2, p3);
    float* o = out + 9 * sub_off[t];
    auto put = [&](uint64_t k, F3 a, F3 b, F3 c) {
        float* q = o + 9 * k;
        q[0] = a.x; q[1] = a.y; q[2] = a.z;
        q[3] = b.x; q[4] = b.y; q[5] = b.z;
        q[6] = c.x; q[7] = c.y; q[8] = c.z;
    };
    float num_subs = floorf(div_rn(tri_max_side(p1, p2, p3), h));
    if (num_subs < 2.0f) {
        put(0, p1, p2, p3);
        return;
    }
    float inv = div_rn(1.0f, num_subs);
    F3 s1 = f3_muls(f3_sub(p2, p1), inv);
    F3 s2 = f3_muls(f3_sub(p3, p2), inv);
    F3 a = p1;
    for (uint32_t k = 0; k < i; ++k) a = f3_add(a, s1);
    F3 b = f3_add(a, s1);
    F3 c = f3_add(b, s2);
    F3 a_s = f3_add(a, s2), b_s = f3_add(b, s2), c_s = f3_add(c, s2);
    F3 a_prev = a;
    uint64_t k0 = (uint64_t)i * i;
    for (uint32_t k = 0; k < i; ++k) {
        put(k0 + 2 * k, a_prev, b_s, a_s);
        put(k0 + 2 * k + 1, a_s, b_s, c_s);
        a_prev = a_s;
        a_s = f3_add(a_s, s2);
        b_s = f3_add(b_s, s2);
        c_s = f3_add(c_s, s2);
    }
    put(k0 + 2 * (uint64_t)i, a, b, c);
}

// ---------------------------------------------------------------------------
// dilated boxes (mesh_to_volume.rs:124-141) and distance records

__device__ inline int floor_div8(int v) { return v >> 3; }

// per-block partial sums/bounds, reduced by k_reduce_partials (no same-address
// atomics in the bulk kernels)
struct Partial {
    unsigned long long pairs;
    int lo[3], hi[3];
};

template <int BLOCK>
__device__ inline void block_reduce_partial(Partial mine, Partial* out) {
    __shared__ Partial sp[BLOCK / 64];
    for (int s = 32; s >= 1; s >>= 1) {
        mine.pairs += __shfl_xor(mine.pairs, s);
        for (int k = 0; k < 3; ++k) {
            mine.lo[k] = min(mine.lo[k], __shfl_xor(mine.lo[k], s));
            mine.hi[k] = max(mine.hi[k], __shfl_xor(mine.hi[k], s));
        }
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sp[w] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        Partial r = sp[0];
        for (int i = 1; i < BLOCK / 64; ++i) {
            r.pairs += sp[i].pairs;
            for (int k = 0; k < 3; ++k) {
                r.lo[k] = min(r.lo[k], sp[i].lo[k]);
                r.hi[k] = max(r.hi[k], sp[i].hi[k]);
            }
        }
        out[blockIdx.x] = r;
    }
}

__global__ __launch_bounds__(1024) void k_reduce_partials(const Partial* __restrict__ in, unsigned n,
                                                          unsigned long long* counters) {
    Partial mine{0, {INT32_MAX, INT32_MAX, INT32_MAX}, {INT32_MIN, INT32_MIN, INT32_MIN}};
    for (unsigned i = threadIdx.x; i < n; i += blockDim.x) {
        const Partial& p = in[i];
        mine.pairs += p.pairs;
        for (int k = 0; k < 3; ++k) {
            mine.lo[k] = min(mine.lo[k], p.lo[k]);
            mine.hi[k] = max(mine.hi[k], p.hi[k]);
        }
    }
    __shared__ Partial sp[16];
    for (int s = 32; s >= 1; s >>= 1) {
        mine.pairs += __shfl_xor(mine.pairs, s);
        for (int k = 0; k < 3; ++k) {
            mine.lo[k] = min(mine.lo[k], __shfl_xor(mine.lo[k], s));
            mine.hi[k] = max(mine.hi[k], __shfl_xor(mine.hi[k], s));
        }
    }
    if ((threadIdx.x & 63) == 0) sp[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        Partial r = sp[0];
        for (unsigned i = 1; i < blockDim.x / 64; ++i) {
            r.pairs += sp[i].pairs;
            for (int k = 0; k < 3; ++k) {
                r.lo[k] = min(r.lo[k], sp[i].lo[k]);
                r.hi[k] = max(r.hi[k], sp[i].hi[k]);
            }
        }
        counters[C_PAIRS] = r.pairs;
        for (int k = 0; k < 3; ++k) {
            counters[C_BOX_LO + k] = (unsigned long long)(long long)r.lo[k];
            counters[C_BOX_HI + k] = (unsigned long long)(long long)r.hi[k];
        }
    }
}

constexpr int SETUP_BLOCK = 256;

__global__ __launch_bounds__(SETUP_BLOCK) void k_subtri_setup(const float* __restrict__ sub, uint64_t n_sub, float inv_h,
                                                              int band, DistRec* __restrict__ recs,
                                                              uint32_t* __restrict__ cov, Partial* partials,
                                                              unsigned* err) {
    uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    Partial mine{0, {INT32_MAX, INT32_MAX, INT32_MAX}, {INT32_MIN, INT32_MIN, INT32_MIN}};
    if (t < n_sub) {
        F3 a, b, c;
        load_tri(sub + 9 * t, a, b, c);
        F3 mn = f3_min2(c, f3_min2(a, b));
        F3 mx = f3_max2(c, f3_max2(a, b));
        float fl[3] = {floorf(mn.x * inv_h), floorf(mn.y * inv_h), floorf(mn.z * inv_h)};
        float cl[3] = {ceilf(mx.x * inv_h), ceilf(mx.y * inv_h), ceilf(mx.z * inv_h)};
        int lo[3], hi[3];
        bool ok = true;
        for (int k = 0; k < 3; ++k) {
            ok &= fabsf(fl[k]) < 8.0e6f && fabsf(cl[k]) < 8.0e6f;
            lo[k] = ok ? (int)fl[k] - band : 0;
            hi[k] = ok ? (int)cl[k] + band : 0;
        }
        if (!ok) atomicOr(err, E_RANGE);
        if (hi[0] == lo[0] || hi[1] == lo[1] || hi[2] == lo[2])
            for (int k = 0; k < 3; ++k) { lo[k] -= 1; hi[k] += 1; }
        DistRec r;
        r.a[0] = a.x; r.a[1] = a.y; r.a[2] = a.z;
        const F3 e0 = f3_sub(b, a), ec = f3_sub(c, a);
        const F3 nn = {e0.y * ec.z - e0.z * ec.y, e0.z * ec.x - e0.x * ec.z, e0.x * ec.y - e0.y * ec.x};
        const float nl2 = nn.x * nn.x + nn.y * nn.y + nn.z * nn.z;
        const float l0sq = e0.x * e0.x + e0.y * e0.y + e0.z * e0.z;
        bool degenerate = !(nl2 > 0.0f) || !(l0sq > 0.0f);
        if (!degenerate) {
            const float l0 = sqrtf(l0sq), inl = 1.0f / sqrtf(nl2);
            const F3 U = {e0.x / l0, e0.y / l0, e0.z / l0};
            const F3 N = {nn.x * inl, nn.y * inl, nn.z * inl};
            const F3 V = {N.y * U.z - N.z * U.y, N.z * U.x - N.x * U.z, N.x * U.y - N.y * U.x};
            r.U[0] = U.x; r.U[1] = U.y; r.U[2] = U.z;
            r.V[0] = V.x; r.V[1] = V.y; r.V[2] = V.z;
            r.N[0] = N.x; r.N[1] = N.y; r.N[2] = N.z;
            const float cu = U.x * ec.x + U.y * ec.y + U.z * ec.z;
            const float cv = V.x * ec.x + V.y * ec.y + V.z * ec.z;
            const float fx = cu - l0;
            r.L0 = l0;
            r.L1 = sqrtf(fx * fx + cv * cv);
            r.L2 = sqrtf(cu * cu + cv * cv);
            // c on b or on a within rounding: no direction to project on
            degenerate = !(r.L1 > 0.0f) || !(r.L2 > 0.0f);
            r.e1x = fx / r.L1;
            r.e1y = cv / r.L1;
            r.e2x = cu / r.L2;
            r.e2y = cv / r.L2;
            r.flags = 0;
        }
        if (degenerate) {
            for (int k = 0; k < 3; ++k) r.U[k] = r.V[k] = r.N[k] = 0.0f;
            r.L0 = r.e1x = r.e1y = r.L1 = r.e2x = r.e2y = r.L2 = 0.0f;
            r.flags = 1;
        }
        r.pad[0] = r.pad[1] = 0;
        for (int k = 0; k < 3; ++k) { r.box[k] = lo[k]; r.box[3 + k] = hi[k]; }
        recs[t] = r;
        uint32_t nl = 1;
        for (int k = 0; k < 3; ++k) nl *= (uint32_t)(floor_div8(hi[k]) - floor_div8(lo[k]) + 1);
        cov[t] = nl;
        mine.pairs = (unsigned long long)(hi[0] - lo[0] + 1) * (hi[1] - lo[1] + 1) * (hi[2] - lo[2] + 1);
        for (int k = 0; k < 3; ++k) { mine.lo[k] = lo[k]; mine.hi[k] = hi[k]; }
    }
    block_reduce_partial<SETUP_BLOCK>(mine, partials);
}

// ---------------------------------------------------------------------------
// leaf allocation: a dense leaf grid over the boxes' bounding box when that
// grid is small, else an open-addressing hash; both end in the same sorted
// leaf list (lexicographic origin order) and a key -> leaf id lookup.

struct LeafIndex {
    // dense grid
    uint32_t* grid = nullptr;
    int gx0 = 0, gy0 = 0, gz0 = 0, gny = 0, gnz = 0;
    uint64_t gsize = 0;
    // hash
    uint64_t* hkeys = nullptr;
    uint32_t* hvals = nullptr;
    uint32_t cap_mask = 0;
    bool dense = true;

    __device__ uint64_t dense_index(int lx, int ly, int lz) const {
        return ((uint64_t)(lx - gx0) * gny + (uint64_t)(ly - gy0)) * gnz + (uint64_t)(lz - gz0);
    }
    __device__ uint32_t find(int lx, int ly, int lz) const {
        if (dense) return grid[dense_index(lx, ly, lz)];
        uint32_t slot = hash_find(hkeys, cap_mask, leaf_key(lx, ly, lz));
        return slot == NOT_FOUND ? NOT_FOUND : hvals[slot];
    }
};

template <class F>
__device__ inline void for_each_leaf(const DistRec& r, F&& f) {
    int x0 = floor_div8(r.box[0]), y0 = floor_div8(r.box[1]), z0 = floor_div8(r.box[2]);
    int x1 = floor_div8(r.box[3]), y1 = floor_div8(r.box[4]), z1 = floor_div8(r.box[5]);
    uint32_t j = 0;
    for (int x = x0; x <= x1; ++x)
        for (int y = y0; y <= y1; ++y)
            for (int z = z0; z <= z1; ++z) f(j++, x, y, z);
}

__global__ void k_leaf_mark(const DistRec* __restrict__ recs, uint64_t n_sub, LeafIndex ix, unsigned* err) {
    uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_sub) return;
    const DistRec& r = recs[t];
    bool ok = true;
    for_each_leaf(r, [&](uint32_t, int x, int y, int z) {
        if (ix.dense) ix.grid[ix.dense_index(x, y, z)] = 1u;
        else ok &= hash_insert(ix.hkeys, ix.cap_mask, leaf_key(x, y, z));
    });
    if (!ok) atomicOr(err, E_HASH);
}

struct DenseOccupied {
    const uint32_t* grid;
    __device__ bool operator()(uint32_t i) const { return grid[i] != 0u; }
};
struct HashOccupied {
    __device__ bool operator()(uint64_t k) const { return k != EMPTY_KEY; }
};

// leaf ids and origins, from dense grid indices (already in lexicographic order)
__global__ void k_leaf_assign_dense(const uint32_t* __restrict__ idx, uint64_t n_leaves, LeafIndex ix,
                                    int32_t* origins) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_leaves) return;
    uint64_t d = idx[i];
    ix.grid[d] = (uint32_t)i;
    const int lz = (int)(d % (uint64_t)ix.gnz) + ix.gz0;
    d /= (uint64_t)ix.gnz;
    const int ly = (int)(d % (uint64_t)ix.gny) + ix.gy0;
    const int lx = (int)(d / (uint64_t)ix.gny) + ix.gx0;
    origins[4 * i + 0] = lx * 8;
    origins[4 * i + 1] = ly * 8;
    origins[4 * i + 2] = lz * 8;
    origins[4 * i + 3] = 0;
}

__global__ void k_leaf_assign_hash(const uint64_t* __restrict__ sorted, uint64_t n_leaves, LeafIndex ix,
                                   int32_t* origins, unsigned* err) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_leaves) return;
    uint64_t k = sorted[i];
    uint32_t slot = hash_find(ix.hkeys, ix.cap_mask, k);
    if (slot == NOT_FOUND) atomicOr(err, E_HASH);
    else ix.hvals[slot] = (uint32_t)i;
    int lx, ly, lz;
    leaf_key_decode(k, lx, ly, lz);
    origins[4 * i + 0] = lx * 8;
    origins[4 * i + 1] = ly * 8;
    origins[4 * i + 2] = lz * 8;
    origins[4 * i + 3] = 0;
}

// candidate lists: (leaf id, sub-triangle) for every box/leaf overlap,
// radix-sorted by leaf id (stable, so sub-triangle order within a leaf).
// A block's sub-triangles own one contiguous range of the output: it is
// assembled in LDS and written out coalesced (directly when it is longer than
// CP_LDS entries).
constexpr int CP_BLOCK = 256;
constexpr uint32_t CP_LDS = 4096;
__global__ __launch_bounds__(CP_BLOCK) void k_cand_pairs(const DistRec* __restrict__ recs, uint64_t n_sub,
                                                         const uint32_t* __restrict__ cov_off, LeafIndex ix,
                                                         uint32_t n_leaves, uint32_t* keys, uint32_t* vals,
                                                         unsigned* err) {
    __shared__ uint32_t sk[CP_LDS], sv[CP_LDS];
    const uint64_t t0 = (uint64_t)blockIdx.x * CP_BLOCK;
    const uint64_t t = t0 + threadIdx.x;
    const uint32_t b0 = cov_off[t0], b1 = cov_off[min<uint64_t>(t0 + CP_BLOCK, n_sub)];
    const bool staged = b1 - b0 <= CP_LDS;  // the same for the whole block
    if (t < n_sub) {
        const DistRec& r = recs[t];
        const uint32_t base = cov_off[t];
        bool ok = true;
        for_each_leaf(r, [&](uint32_t j, int x, int y, int z) {
            uint32_t lid = ix.find(x, y, z);
            if (lid >= n_leaves) {
                ok = false;
                lid = n_leaves;  // sorts past every real leaf; never read
            }
            if (staged) {
                sk[base - b0 + j] = lid;
                sv[base - b0 + j] = (uint32_t)t;
            } else {
                keys[base + j] = lid;
                vals[base + j] = (uint32_t)t;
            }
        });
        if (!ok) atomicOr(err, E_HASH);
    }
    if (staged) {
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < b1 - b0; i += CP_BLOCK) {
            keys[b0 + i] = sk[i];
            vals[b0 + i] = sv[i];
        }
    }
}

// off[k] = first entry whose key is >= k, for k = 0..n_leaves (keys sorted;
// keys >= n_leaves are failed lookups and end the lists), by a binary search
// per leaf.  Every slot is written: a leaf without candidates gets an empty list.
__global__ void k_cand_offsets(const uint32_t* __restrict__ keys, uint32_t n, uint32_t n_leaves, uint32_t* off) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k > n_leaves) return;
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if (keys[mid] < k) lo = mid + 1;
        else hi = mid;
    }
    off[k] = lo;
}

// ---------------------------------------------------------------------------
// distance: one workgroup per leaf, LDS best[512] of (d^2 bits << 32 | t).
// Wave w takes candidates w, w+4, ...; for a candidate it walks the box/leaf
// intersection with lanes packed as (x-slice, y, z): the y,z part of the local
// frame coordinates is computed once per candidate, a step in x costs one FMA
// per coordinate.  Merging is a 64-bit LDS atomic min, so equal squared
// distances resolve to the lower sub-triangle index whatever the order.
// The arg-min is re-evaluated with the reference's closest-point arithmetic.

// floor(65536 / d) + 1: (i * m) >> 16 == i / d for i < 1024, d <= 64
__constant__ uint32_t kMagic[65] = {
    0, 65537, 32769, 21846, 16385, 13108, 10923, 9363, 8193, 7282, 6554, 5958, 5462, 5042, 4682, 4370, 4097,
    3856, 3641, 3450, 3277, 3121, 2979, 2850, 2731, 2622, 2521, 2428, 2341, 2260, 2185, 2115, 2049, 1986, 1928,
    1873, 1821, 1772, 1725, 1681, 1639, 1599, 1561, 1525, 1490, 1457, 1425, 1395, 1366, 1338, 1311, 1286, 1261,
    1237, 1214, 1192, 1171, 1150, 1130, 1111, 1093, 1075, 1058, 1041, 1025};

// Union-find over a leaf's voxels in LDS, for the shared-sign groups (see the
// shared-sign kernels further down for the argument).
__device__ inline int uf_find(int* par, int x) {
    int p = __hip_atomic_load(&par[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (p != x) {
        x = p;
        p = __hip_atomic_load(&par[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return x;
}

__device__ inline void uf_unite(int* par, int a, int b) {
    // every failed exchange means another lane hooked b first: the loop ends
    for (;;) {
        a = uf_find(par, a);
        b = uf_find(par, b);
        if (a == b) return;
        if (a > b) {
            const int t = a;
            a = b;
            b = t;
        }
        if (atomicCAS(&par[b], b, a) == b) return;
    }
}

constexpr int DIST_BLOCK = 256;

// Workgroups go to the 8 XCDs in turn; renumbered, each XCD works through runs
// of `run` consecutive workgroups (compact parts of the volume) that share
// records in its L2, and the runs interleave across XCDs for balance.  The last
// partial round keeps its numbering.
__device__ inline uint32_t xcd_workgroup(uint32_t run) {
    const uint32_t full = gridDim.x / (8 * run) * (8 * run);
    const uint32_t wg = blockIdx.x;
    if (wg >= full) return wg;
    const uint32_t xcd = wg & 7, i = wg >> 3;
    return ((i / run) * 8 + xcd) * run + i % run;
}

// Neighbouring leaves share most of their candidates, so an XCD takes runs of
// this many: 8.96 -> 8.80 ms at 150 k leaves, 336 -> 315 us at 1.6 k.  (One eighth
// of the leaves per XCD, without interleaving, had been slower: the XCDs finish
// unevenly.)
constexpr uint32_t DIST_RUN = 32;

// GROUPS: the leaf's shared-sign groups are formed here too, from the
// distances still in the workgroup: face-adjacent active voxels whose
// distances sum above group_thr are united (LDS union-find, root = smallest
// offset), roots[leaf * 512 + v] = root offset (0xFFFF inactive), rep_cnt[leaf]
// = number of groups.
template <bool GROUPS>
__global__ __launch_bounds__(DIST_BLOCK) void k_distance(const int32_t* __restrict__ origins,
                                                         const uint32_t* __restrict__ cand_off,
                                                         const uint32_t* __restrict__ cand_list,
                                                         const DistRec* __restrict__ recs,
                                                         const float* __restrict__ sub, float h, uint32_t n_cand,
                                                         float* __restrict__ values, uint64_t* __restrict__ masks,
                                                         float group_thr, uint16_t* __restrict__ roots,
                                                         uint32_t* __restrict__ rep_cnt) {
    __shared__ unsigned long long best[LEAF_VOX];
    const int leaf = (int)xcd_workgroup(DIST_RUN);
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    for (int i = tid; i < LEAF_VOX; i += DIST_BLOCK) best[i] = ~0ull;
    const int ox = origins[4 * leaf], oy = origins[4 * leaf + 1], oz = origins[4 * leaf + 2];
    const uint32_t c1 = min(cand_off[leaf + 1], n_cand), c0 = min(cand_off[leaf], c1);
    __syncthreads();
    constexpr uint32_t WAVES = DIST_BLOCK / 64;
    for (uint32_t cb = c0 + wave; cb < c1; cb += 64 * WAVES) {
        // the wave's next 64 candidates, one index per lane: one vector load
        // instead of a dependent load per candidate
        const uint32_t cl = cb + (uint32_t)lane * WAVES;
        const int tl = cl < c1 ? (int)cand_list[cl] : 0;
        const int nk = (int)min(64u, (c1 - cb + WAVES - 1) / WAVES);
        for (int k = 0; k < nk; ++k) {
            const uint32_t t = (uint32_t)__builtin_amdgcn_readlane(tl, k);
            const DistRec r = recs[t];
            pin_dist_rec(r);  // the whole record in one round of scalar loads
            const int x0 = max(r.box[0], ox), x1 = min(r.box[3], ox + 7);
            const int y0 = max(r.box[1], oy), y1 = min(r.box[4], oy + 7);
            const int z0 = max(r.box[2], oz), z1 = min(r.box[5], oz + 7);
            const int nz = z1 - z0 + 1, ny = y1 - y0 + 1, nyz = ny * nz;
            if (x1 < x0 || ny <= 0 || nz <= 0) continue;  // box misses the leaf: never for a listed candidate
            const uint32_t m_yz = kMagic[nyz], m_z = kMagic[nz];
            asm volatile("" ::"s"(m_yz), "s"(m_z));  // both table reads in one round trip
            const int spp = (int)((64u * m_yz) >> 16);  // x-slices per pass, 64 / nyz
            // 24-bit multiplies (full rate; every operand is below 2^17)
            const int s = (int)(__umul24((uint32_t)lane, m_yz) >> 16);
            const int rr = lane - (int)__umul24((uint32_t)s, (uint32_t)nyz);
            const int yq = (int)(__umul24((uint32_t)rr, m_z) >> 16);
            const int zq = rr - (int)__umul24((uint32_t)yq, (uint32_t)nz);
            const float py = (float)(y0 + yq) * h, pz = (float)(z0 + zq) * h;
            // the lane's first voxel in the leaf; a step in x is spp slices on
            int vo = ((x0 - ox) << 6) + ((y0 - oy) << 3) + (z0 - oz) + (s << 6) + (yq << 3) + zq;
            // x runs as a float: whole numbers below 2^24, so every step is exact
            float x = (float)(x0 + s);
            const float xe = (float)x1, xs = (float)spp;
            if (s < spp) {
                if (r.flags == 0) {
                    const float dy = py - r.a[1], dz = pz - r.a[2];
                    const float bu = __builtin_fmaf(r.U[1], dy, r.U[2] * dz);
                    const float bv = __builtin_fmaf(r.V[1], dy, r.V[2] * dz);
                    const float bw = __builtin_fmaf(r.N[1], dy, r.N[2] * dz);
                    // the fields the x loop reads, in scalar registers before it
                    // starts (else their loads sink into the loop body)
                    const PlaneRec q = plane_rec(r);
                    unsigned long long* slot = best + vo;
                    for (; x <= xe; x += xs, slot += spp << 6) {
                        const float dx = x * h - q.a0;
                        const float pu = __builtin_fmaf(q.U0, dx, bu);
                        const float pv = __builtin_fmaf(q.V0, dx, bv);
                        const float pw = __builtin_fmaf(q.N0, dx, bw);
                        const float d2 = __builtin_fmaf(pw, pw, plane_dist2(q, pu, pv));
                        const unsigned long long key = ((unsigned long long)__float_as_uint(d2) << 32) | t;
                        atomicMin(slot, key);
                    }
                } else {
                    const float* v = sub + 9 * (uint64_t)t;
                    for (; x <= xe; x += xs, vo += spp << 6) {
                        const float d = ericson_distance({v[0], v[1], v[2]}, {v[3], v[4], v[5]}, {v[6], v[7], v[8]},
                                                         {x * h, py, pz});
                        if (d == d) {  // a NaN distance never enters the field (`dist < cur` is false)
                            const unsigned long long key = ((unsigned long long)__float_as_uint(d * d) << 32) | t;
                            atomicMin(&best[vo], key);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    constexpr int PER = LEAF_VOX / DIST_BLOCK;
    float vk[PER];
    bool ak[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int off = tid + DIST_BLOCK * k;
        const unsigned long long key = best[off];
        const bool active = key != ~0ull;
        float v = 0.0f;
        if (active) {
            const float* tv = sub + 9 * (uint64_t)(uint32_t)key;
            const float px = (float)(ox + (off >> 6)) * h, py = (float)(oy + ((off >> 3) & 7)) * h,
                        pz = (float)(oz + (off & 7)) * h;
            v = ericson_distance({tv[0], tv[1], tv[2]}, {tv[3], tv[4], tv[5]}, {tv[6], tv[7], tv[8]}, {px, py, pz});
        }
        values[(uint64_t)leaf * LEAF_VOX + off] = v;
        const unsigned long long m = __ballot(active);
        if (lane == 0) masks[(uint64_t)leaf * 8 + (off >> 6)] = m;
        vk[k] = v;
        ak[k] = active;
    }
    if constexpr (GROUPS) {
        // best[] is free once every key has been read: 512 distances (-1 for an
        // inactive voxel) and 512 union-find parents take its place
        __shared__ uint32_t n_roots;
        float* d = reinterpret_cast<float*>(best);
        int* par = reinterpret_cast<int*>(best) + LEAF_VOX;
        __syncthreads();
        if (tid == 0) n_roots = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int off = tid + DIST_BLOCK * k;
            d[off] = ak[k] ? vk[k] : -1.0f;
            par[off] = off;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int v = tid + DIST_BLOCK * k;
            if (!ak[k]) continue;
            const float dv = vk[k];
            if ((v >> 6) < 7 && d[v + 64] >= 0.0f && dv + d[v + 64] > group_thr) uf_unite(par, v, v + 64);
            if (((v >> 3) & 7) < 7 && d[v + 8] >= 0.0f && dv + d[v + 8] > group_thr) uf_unite(par, v, v + 8);
            if ((v & 7) < 7 && d[v + 1] >= 0.0f && dv + d[v + 1] > group_thr) uf_unite(par, v, v + 1);
        }
        __syncthreads();
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int v = tid + DIST_BLOCK * k;
            const int r = ak[k] ? uf_find(par, v) : -1;
            roots[(uint64_t)leaf * LEAF_VOX + v] = ak[k] ? (uint16_t)r : (uint16_t)0xFFFF;
            mine += (uint32_t)__popcll(__ballot(ak[k] && r == v));
        }
        if (lane == 0) atomicAdd(&n_roots, mine);
        __syncthreads();
        if (tid == 0) rep_cnt[leaf] = n_roots;
    }
}

// 21 bits spread to every third bit (Morton codes)
__device__ inline uint64_t spread21(uint64_t v) {
    v &= 0x1FFFFF;
    v = (v | v << 32) & 0x1F00000000FFFFull;
    v = (v | v << 16) & 0x1F0000FF0000FFull;
    v = (v | v << 8) & 0x100F00F00F00F00Full;
    v = (v | v << 4) & 0x10C30C30C30C30C3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}

// Active voxel list, slot = leaf * 512 + offset.  The leaves are listed in the
// order perm gives (identity when perm is null): count per listed leaf here.
__global__ void k_leaf_popcount(const uint64_t* __restrict__ masks, uint64_t n_leaves,
                                const uint32_t* __restrict__ perm, uint32_t* cnt) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_leaves) return;
    const uint64_t leaf = perm ? perm[i] : i;
    uint32_t c = 0;
    for (int w = 0; w < 8; ++w) c += __popcll(masks[8 * leaf + w]);
    cnt[i] = c;
}

// Z-order key of each leaf's coordinates (in leaves, relative to the lowest
// leaf of the grid, 21 bits per axis) with the leaf id as its value: sorted,
// consecutive leaves are neighbours in space far more often than in the
// lexicographic order, where the end of one row of leaves jumps to the other
// side of the surface.
__global__ void k_leaf_morton(const int32_t* __restrict__ origins, uint64_t n_leaves, int lx0, int ly0, int lz0,
                              uint64_t* keys, uint32_t* ids) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_leaves) return;
    const uint64_t x = (uint64_t)(uint32_t)((origins[4 * i] >> 3) - lx0);
    const uint64_t y = (uint64_t)(uint32_t)((origins[4 * i + 1] >> 3) - ly0);
    const uint64_t z = (uint64_t)(uint32_t)((origins[4 * i + 2] >> 3) - lz0);
    keys[i] = (spread21(x) << 2) | (spread21(y) << 1) | spread21(z);
    ids[i] = (uint32_t)i;
}

// Within a leaf the voxels are listed in Morton order, so 64 consecutive
// entries (one winding-number wave) form compact 4x4x4 blocks rather than 8x8
// slabs.  One wave per listed leaf: wave b lists leaf perm[b] (b when perm is
// null) at act_off[b], 64 Morton indices per step.
constexpr int AL_BLOCK = 256;
__global__ __launch_bounds__(AL_BLOCK) void k_active_list(const uint64_t* __restrict__ masks,
                                                          const uint32_t* __restrict__ perm,
                                                          const uint32_t* __restrict__ act_off, uint64_t n_leaves,
                                                          uint32_t* out) {
    const uint64_t b = (uint64_t)blockIdx.x * (AL_BLOCK / 64) + (threadIdx.x >> 6);
    if (b >= n_leaves) return;
    const int lane = threadIdx.x & 63;
    const uint32_t leaf = perm ? perm[b] : (uint32_t)b;
    const uint64_t* mk = masks + (uint64_t)leaf * 8;
    uint32_t pos = act_off[b];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int m = (c << 6) | lane;  // Morton index of the voxel in the leaf
        const int x = ((m >> 2) & 1) | ((m >> 4) & 2) | ((m >> 6) & 4);
        const int y = ((m >> 1) & 1) | ((m >> 3) & 2) | ((m >> 5) & 4);
        const int z = (m & 1) | ((m >> 2) & 2) | ((m >> 4) & 4);
        const int off = (x << 6) | (y << 3) | z;
        const bool act = (mk[off >> 6] >> (off & 63)) & 1ull;
        const unsigned long long bl = __ballot(act);
        if (act) out[pos + __popcll(bl & ((1ull << lane) - 1))] = leaf * 512u + (uint32_t)off;
        pos += (uint32_t)__popcll(bl);
    }
}

// ---------------------------------------------------------------------------
// LBVH over the original triangles + order-2 dipole data (aabb_tree.rs:711-816)

__device__ inline unsigned ordered_bits(float f) {
    unsigned u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float from_ordered_bits(unsigned u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

// centroid bounds per block (ordered-int encoding), reduced by k_bounds_final
__global__ __launch_bounds__(256) void k_centroid_bounds(const float* __restrict__ tris, uint64_t n, uint4* part) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned lo[3] = {~0u, ~0u, ~0u}, hi[3] = {0, 0, 0};
    if (i < n) {
        F3 a, b, c;
        load_tri(tris + 9 * i, a, b, c);
        F3 mn = f3_min2(c, f3_min2(a, b)), mx = f3_max2(c, f3_max2(a, b));
        float ce[3] = {(mn.x + mx.x) * 0.5f, (mn.y + mx.y) * 0.5f, (mn.z + mx.z) * 0.5f};
        for (int k = 0; k < 3; ++k) lo[k] = hi[k] = ordered_bits(ce[k]);
    }
    for (int s = 32; s >= 1; s >>= 1)
        for (int k = 0; k < 3; ++k) {
            lo[k] = min(lo[k], (unsigned)__shfl_xor((int)lo[k], s));
            hi[k] = max(hi[k], (unsigned)__shfl_xor((int)hi[k], s));
        }
    __shared__ unsigned sl[4][3], sh[4][3];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 3; ++k) { sl[w][k] = lo[k]; sh[w][k] = hi[k]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; ++q)
            for (int k = 0; k < 3; ++k) { lo[k] = min(lo[k], sl[q][k]); hi[k] = max(hi[k], sh[q][k]); }
        part[2 * blockIdx.x] = make_uint4(lo[0], lo[1], lo[2], 0);
        part[2 * blockIdx.x + 1] = make_uint4(hi[0], hi[1], hi[2], 0);
    }
}

__global__ __launch_bounds__(1024) void k_bounds_final(const uint4* __restrict__ part, unsigned nb, unsigned* bounds) {
    unsigned lo[3] = {~0u, ~0u, ~0u}, hi[3] = {0, 0, 0};
    for (unsigned b = threadIdx.x; b < nb; b += blockDim.x) {
        uint4 l = part[2 * b], u = part[2 * b + 1];
        lo[0] = min(lo[0], l.x); lo[1] = min(lo[1], l.y); lo[2] = min(lo[2], l.z);
        hi[0] = max(hi[0], u.x); hi[1] = max(hi[1], u.y); hi[2] = max(hi[2], u.z);
    }
    for (int s = 32; s >= 1; s >>= 1)
        for (int k = 0; k < 3; ++k) {
            lo[k] = min(lo[k], (unsigned)__shfl_xor((int)lo[k], s));
            hi[k] = max(hi[k], (unsigned)__shfl_xor((int)hi[k], s));
        }
    __shared__ unsigned sl[16][3], sh[16][3];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 3; ++k) { sl[w][k] = lo[k]; sh[w][k] = hi[k]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned q = 1; q < blockDim.x / 64; ++q)
            for (int k = 0; k < 3; ++k) { lo[k] = min(lo[k], sl[q][k]); hi[k] = max(hi[k], sh[q][k]); }
        for (int k = 0; k < 3; ++k) { bounds[k] = lo[k]; bounds[3 + k] = hi[k]; }
    }
}

__global__ void k_morton(const float* __restrict__ tris, uint64_t n, const unsigned* __restrict__ bounds,
                         uint64_t* codes, uint32_t* idx) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    F3 a, b, c;
    load_tri(tris + 9 * i, a, b, c);
    F3 mn = f3_min2(c, f3_min2(a, b)), mx = f3_max2(c, f3_max2(a, b));
    float ce[3] = {(mn.x + mx.x) * 0.5f, (mn.y + mx.y) * 0.5f, (mn.z + mx.z) * 0.5f};
    uint64_t q[3];
    for (int k = 0; k < 3; ++k) {
        float lo = from_ordered_bits(bounds[k]), hi = from_ordered_bits(bounds[3 + k]);
        float ext = hi - lo;
        float u = ext > 0.0f ? (ce[k] - lo) / ext : 0.0f;
        u = fminf(fmaxf(u, 0.0f), 1.0f);
        q[k] = (uint64_t)fminf(u * 2097152.0f, 2097151.0f);
    }
    codes[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    idx[i] = (uint32_t)i;
}

__device__ inline int lbvh_delta(const uint64_t* __restrict__ k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clz((unsigned)(i ^ j));
    return __clzll(a ^ b);
}

// Node record, 64 B = one s_load_dwordx16: A = (c.xyz, (radius*acc)^2),
// B = (awn.xyz, trace O2), C = (S00, S11, S22, 2 S01), D = (2 S02, 2 S12) with
// S the symmetric part of order2 = sum a c n^T - c_d awn^T (only S enters
// r^T O2 r), and links L = (left, right) for an internal node or
// (first triangle, -count) for a node evaluated as a leaf (count <= BVH_LEAF_SIZE).
struct alignas(16) NodeRec {
    float4 A, B, C;
    float2 D;
    int2 L;
};
static_assert(sizeof(NodeRec) == 64, "NodeRec layout");

// Karras 2012: internal node i of n-1; leaves are n-1+k.  links = (left, right,
// first, count) over the sorted order.
__global__ void k_lbvh_build(const uint64_t* __restrict__ keys, int n, NodeRec* nodes, int2* kids, int* parent) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int d = (lbvh_delta(keys, n, i, i + 1) - lbvh_delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = lbvh_delta(keys, n, i, i - d);
    int lmax = 2;
    while (lbvh_delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (lbvh_delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = lbvh_delta(keys, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (lbvh_delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + min(d, 0);
    int first = min(i, j), last = max(i, j);
    int left = (first == gamma) ? (n - 1 + gamma) : gamma;
    int right = (last == gamma + 1) ? (n - 1 + gamma + 1) : gamma + 1;
    const int count = last - first + 1;
    nodes[i].L = count <= BVH_LEAF_SIZE ? make_int2(first, -count) : make_int2(left, right);
    kids[i] = make_int2(left, right);
    parent[left] = i;
    parent[right] = i;
}

// Per-node accumulation of aabb_tree.rs:711-801 (InitData): area-weighted
// normal, area-weighted centre, sum of a*c*n^T, total area, plus the bbox.
struct NodeAcc {
    float awn[3], awc[3], o1[9], area;
    float bmin[3], bmax[3];
};

__device__ inline void acc_add(NodeAcc& r, const NodeAcc& a, const NodeAcc& b) {
    for (int k = 0; k < 3; ++k) {
        r.awn[k] = a.awn[k] + b.awn[k];
        r.awc[k] = a.awc[k] + b.awc[k];
        r.bmin[k] = fminf(a.bmin[k], b.bmin[k]);
        r.bmax[k] = fmaxf(a.bmax[k], b.bmax[k]);
    }
    for (int k = 0; k < 9; ++k) r.o1[k] = a.o1[k] + b.o1[k];
    r.area = a.area + b.area;
}

__device__ inline void acc_finalize(const NodeAcc& a, float acc, NodeRec* rec) {
    float4* node = &rec->A;
    float c[3];
    for (int k = 0; k < 3; ++k) c[k] = a.awc[k] / a.area;
    float o2[9];
    for (int r = 0; r < 3; ++r)
        for (int q = 0; q < 3; ++q) o2[3 * r + q] = a.o1[3 * r + q] - c[r] * a.awn[q];
    float dmin = 0.0f, dmax = 0.0f;
    for (int k = 0; k < 3; ++k) {
        dmin += (a.bmin[k] - c[k]) * (a.bmin[k] - c[k]);
        dmax += (a.bmax[k] - c[k]) * (a.bmax[k] - c[k]);
    }
    float radius = sqrtf(fmaxf(dmin, dmax));
    float ra = radius * acc;
    float far2 = (a.area > 0.0f) ? ra * ra : INFINITY;  // all-degenerate: never far
    // order-1 and trace terms scaled by 1/(4 pi), quadratic form by 3/(4 pi):
    // w = (B.r + B.w - (r^T S r) / |r|^2) / |r|^3 (aabb_tree.rs:803-816, factored)
    const float k1 = INV_4PI, k3 = 3.0f * INV_4PI;
    node[0] = make_float4(c[0], c[1], c[2], far2);
    node[1] = make_float4(k1 * a.awn[0], k1 * a.awn[1], k1 * a.awn[2], k1 * (o2[0] + o2[4] + o2[8]));
    node[2] = make_float4(k3 * o2[0], k3 * o2[4], k3 * o2[8], k3 * (o2[1] + o2[3]));
    rec->D = make_float2(k3 * (o2[2] + o2[6]), k3 * (o2[5] + o2[7]));
}

// Traversal copy of triangle k, 3 x float4 (48 B) per triangle.
__device__ inline void store_btri(float* btris, uint64_t k, const F3& a, const F3& b, const F3& c) {
    float4* bt = reinterpret_cast<float4*>(btris) + 3 * k;
    bt[0] = make_float4(a.x, a.y, a.z, b.x);
    bt[1] = make_float4(b.y, b.z, c.x, c.y);
    bt[2] = make_float4(c.z, 0.0f, 0.0f, 0.0f);
}

// InitData of one triangle (aabb_tree.rs:711-801) and its bbox.
__device__ inline NodeAcc tri_acc(const F3& a, const F3& b, const F3& c) {
    NodeAcc d;
    F3 e0 = f3_sub(b, a), e1 = f3_sub(c, a);
    F3 cr = {e0.y * e1.z - e0.z * e1.y, e0.z * e1.x - e0.x * e1.z, e0.x * e1.y - e0.y * e1.x};
    float cl2 = cr.x * cr.x + cr.y * cr.y + cr.z * cr.z;
    F3 mn = f3_min2(c, f3_min2(a, b)), mx = f3_max2(c, f3_max2(a, b));
    d.bmin[0] = mn.x; d.bmin[1] = mn.y; d.bmin[2] = mn.z;
    d.bmax[0] = mx.x; d.bmax[1] = mx.y; d.bmax[2] = mx.z;
    for (int q = 0; q < 3; ++q) { d.awn[q] = 0.0f; d.awc[q] = 0.0f; }
    for (int q = 0; q < 9; ++q) d.o1[q] = 0.0f;
    d.area = 0.0f;
    if (cl2 > 0.0f) {  // degenerate triangles are skipped (aabb_tree.rs:757-759)
        float cl = sqrtf(cl2);
        float area = cl * 0.5f;
        float nrm[3] = {cr.x / cl, cr.y / cl, cr.z / cl};
        float ce[3] = {(a.x + b.x + c.x) / 3.0f, (a.y + b.y + c.y) / 3.0f, (a.z + b.z + c.z) / 3.0f};
        d.area = area;
        for (int q = 0; q < 3; ++q) {
            d.awn[q] = area * nrm[q];
            d.awc[q] = area * ce[q];
        }
        for (int r = 0; r < 3; ++r)
            for (int q = 0; q < 3; ++q) d.o1[3 * r + q] = (area * ce[r]) * nrm[q];
    }
    return d;
}

// Leaf data, then node heights bottom-up with one 32-bit atomicMax per step:
// the first child to arrive stores its height + 1 and stops, the second reads
// it back from the same atomic and carries on.  No data other than the atomic
// word crosses threads, so no memory fences are needed; node data is then
// combined level by level (k_lbvh_level), one launch per height.
__global__ void k_lbvh_leaves(const float* __restrict__ tris, int n, const uint32_t* __restrict__ order, float acc,
                              const int* __restrict__ parent, unsigned* hword, uint32_t* height, NodeAcc* accs,
                              NodeRec* nodes, float* btris, unsigned* err) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    F3 a, b, c;
    load_tri(tris + 9 * (uint64_t)order[k], a, b, c);
    // traversal copy of the triangle in Morton order
    store_btri(btris, k, a, b, c);
    const NodeAcc d = tri_acc(a, b, c);
    int node = n - 1 + k;
    accs[node] = d;
    acc_finalize(d, acc, nodes + node);
    nodes[node].L = make_int2(k, -1);
    unsigned hgt = 0;
    int p = parent[node];
    for (int level = 0; p >= 0; ++level) {
        if (level > 250) {  // deeper than the 8-bit height sort allows: corrupt parent links
            atomicOr(err, E_TREE);
            return;
        }
        unsigned old = atomicMax(&hword[p], hgt + 1);
        if (old == 0) return;  // the sibling finishes this node
        hgt = max(old, hgt + 1);
        height[p] = hgt;
        p = parent[p];
    }
}

__global__ void k_lbvh_level(const uint32_t* __restrict__ level_nodes, uint32_t count, float acc,
                             const int2* __restrict__ kids, NodeAcc* accs, NodeRec* nodes) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int p = (int)level_nodes[i];
    const int2 L = kids[p];
    NodeAcc s;
    acc_add(s, accs[L.x], accs[L.y]);
    accs[p] = s;
    acc_finalize(s, acc, nodes + p);
}

__global__ void k_iota(uint32_t* out, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = i;
}

__global__ void k_level_starts(const uint32_t* __restrict__ hs, uint32_t n, uint32_t* starts) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t h = hs[i];
    if (h < 256 && (i == 0 || hs[i - 1] != h)) starts[h] = i;
}

// ---------------------------------------------------------------------------
// Clustered build (PLOC: Meister and Bittner, "Parallel Locally-Ordered
// Clustering for Bounding Volume Hierarchy Construction", IEEE TVCG 2018).
// The clusters start as the triangles in Morton order.  In each iteration
// every cluster finds, among the clusters within PLOC_R places of it, the one
// whose union with it has the smallest box surface (ties to the lower place);
// mutual pairs merge into a new node at the lower place and the array is
// compacted in order.  Boxes built from nearby clusters this way are tighter
// than the Morton-split boxes, so fewer voxels find a node near.  The finished
// tree is laid out depth-first with the two children of every node side by
// side, 128-byte aligned (one cache line for the sibling pair the traversal
// reads together), and the triangles in the same depth-first order.
constexpr int PLOC_R = 16;
constexpr int PLOC_BLOCK = 256;
constexpr uint64_t PLOC_MIN_TRIS = 1u << 18;  // smaller meshes take the Morton split

// Per temporary node: triangles below it, child pairs its subtree allocates
// in the traversal layout (0 when it is evaluated as a leaf), its height in
// that layout, and (parent << 1 | side), -1 while it has no parent.
struct PlocInfo {
    int tris, pairs, height, parent;
};

// Temporary ids: triangle k of the Morton order is node k, merged nodes are
// n, n + 1, ... in the order merges take them.  ring[0] = cluster count,
// ring[2] = next merged id.
__global__ void k_ploc_leaves(const float* __restrict__ tris, int n, const uint32_t* __restrict__ order,
                              NodeAcc* __restrict__ accs, float4* __restrict__ box, PlocInfo* __restrict__ info,
                              int* __restrict__ clus, uint32_t* __restrict__ keep, uint32_t* __restrict__ ring) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) {
        ring[0] = (uint32_t)n;
        ring[2] = 0;
        keep[n] = 0;  // the scan runs over n + 1 entries: the last one gives the count
    }
    if (k >= n) return;
    F3 a, b, c;
    load_tri(tris + 9 * (uint64_t)order[k], a, b, c);
    const NodeAcc d = tri_acc(a, b, c);
    accs[k] = d;
    box[2 * k] = make_float4(d.bmin[0], d.bmin[1], d.bmin[2], 0.0f);
    box[2 * k + 1] = make_float4(d.bmax[0], d.bmax[1], d.bmax[2], 0.0f);
    info[k] = PlocInfo{1, 0, 0, -1};
    clus[k] = k;
}

// Nearest neighbour of every cluster within PLOC_R places, by union box
// surface (a NaN surface counts as infinite, so a neighbour is always found
// when the cluster has one).
__global__ __launch_bounds__(PLOC_BLOCK) void k_ploc_nn(const int* __restrict__ clus, const float4* __restrict__ box,
                                                        const uint32_t* __restrict__ count, int* __restrict__ nn) {
    __shared__ float4 slo[PLOC_BLOCK + 2 * PLOC_R], shi[PLOC_BLOCK + 2 * PLOC_R];
    const int N = (int)*count;
    const int base = blockIdx.x * PLOC_BLOCK;
    if (base >= N) return;  // the whole block: no barrier is skipped by part of it
    for (int t = threadIdx.x; t < PLOC_BLOCK + 2 * PLOC_R; t += PLOC_BLOCK) {
        const int j = base - PLOC_R + t;
        if (j >= 0 && j < N) {
            const int c = clus[j];
            slo[t] = box[2 * c];
            shi[t] = box[2 * c + 1];
        }
    }
    __syncthreads();
    const int i = base + (int)threadIdx.x;
    if (i >= N) return;
    const float4 a0 = slo[threadIdx.x + PLOC_R], a1 = shi[threadIdx.x + PLOC_R];
    float best = INFINITY;
    int bj = -1;
    const int jlo = max(i - PLOC_R, 0), jhi = min(i + PLOC_R, N - 1);
    for (int j = jlo; j <= jhi; ++j) {
        if (j == i) continue;
        const float4 b0 = slo[j - base + PLOC_R], b1 = shi[j - base + PLOC_R];
        const float dx = fmaxf(a1.x, b1.x) - fminf(a0.x, b0.x);
        const float dy = fmaxf(a1.y, b1.y) - fminf(a0.y, b0.y);
        const float dz = fmaxf(a1.z, b1.z) - fminf(a0.z, b0.z);
        float d2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
        d2 = (d2 == d2) ? d2 : INFINITY;
        if (bj < 0 || d2 < best) {
            best = d2;
            bj = j;
        }
    }
    nn[i] = bj;
}

// Mutual nearest neighbours i < j merge into a new node at place i; place j
// is dropped.  keep[i] = 1 for every place that stays (0 past the count).
__global__ void k_ploc_merge(int* __restrict__ clus, const int* __restrict__ nn, const uint32_t* __restrict__ count,
                             int n, uint32_t* __restrict__ keep, uint32_t* __restrict__ next_id,
                             NodeAcc* __restrict__ accs, float4* __restrict__ box, PlocInfo* __restrict__ info,
                             int2* __restrict__ kids) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int N = (int)*count;
    if (i >= N) {
        keep[i] = 0;
        return;
    }
    const int j = nn[i];
    const bool mutual = j >= 0 && nn[j] == i;
    keep[i] = (mutual && j < i) ? 0u : 1u;
    if (!mutual || j < i) return;
    const int a = clus[i], b = clus[j];
    const int id = n + (int)atomicAdd(next_id, 1u);
    NodeAcc s;
    acc_add(s, accs[a], accs[b]);
    accs[id] = s;
    box[2 * id] = make_float4(s.bmin[0], s.bmin[1], s.bmin[2], 0.0f);
    box[2 * id + 1] = make_float4(s.bmax[0], s.bmax[1], s.bmax[2], 0.0f);
    const PlocInfo ia = info[a], ib = info[b];
    const int t = ia.tris + ib.tris;
    const bool leaf = t <= BVH_LEAF_SIZE;
    info[id] = PlocInfo{t, leaf ? 0 : 1 + ia.pairs + ib.pairs, leaf ? 0 : 1 + max(ia.height, ib.height), -1};
    info[a].parent = 2 * id;
    info[b].parent = 2 * id + 1;
    kids[id - n] = make_int2(a, b);
    clus[i] = id;
}

// In-order compaction of the kept places; thread 0 writes the new count.
__global__ void k_ploc_compact(const int* __restrict__ clus, const uint32_t* __restrict__ keep,
                               const uint32_t* __restrict__ pos, const uint32_t* __restrict__ count, int n,
                               uint32_t* __restrict__ count_next, int* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *count_next = pos[n];
    if (i >= (int)*count) return;
    if (keep[i]) out[pos[i]] = clus[i];
}

// The root (place 0 once one cluster is left) and the tree height.
__global__ void k_ploc_root(const int* __restrict__ clus, const PlocInfo* __restrict__ info, uint32_t* out) {
    const int r = clus[0];
    out[0] = (uint32_t)r;
    out[1] = (uint32_t)info[r].height;
}

// Depth-first layout.  The child pair of node X goes to records (2 P(X),
// 2 P(X) + 1), P(root) = 1, and P(child) = P(X) + 1 (+ the pairs of the left
// sibling's subtree for a right child); the triangles of X start at the
// number of triangles in the left subtrees along its path.  Each node walks
// its path to the root to sum these.  Record 0 is the root, record 1 unused.
__global__ void k_ploc_place(const uint32_t* __restrict__ root_buf, const PlocInfo* __restrict__ info,
                             const int2* __restrict__ kids, const NodeAcc* __restrict__ accs,
                             const float* __restrict__ tris, const uint32_t* __restrict__ order, int n, float acc,
                             NodeRec* __restrict__ nodes, float* __restrict__ btris, unsigned* err) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= 2 * n - 1) return;
    const PlocInfo me = info[x];
    bool rec = true;  // x has a record of its own: its parent is not evaluated as a leaf
    if (me.parent >= 0)
        rec = info[me.parent >> 1].tris > BVH_LEAF_SIZE;
    else if (x != (int)root_buf[0])
        return;  // never merged: the clustering ran to one cluster, so only the root
    if (!rec && x >= n) return;
    int first = 0, q = 1, side0 = 0, left_pairs0 = 0, depth = 0;
    for (int pw = me.parent; pw >= 0; ++depth) {
        if (depth > 1024) {  // longer than any path of a tree over 2^30 triangles built by merges
            atomicOr(err, E_TREE);
            return;
        }
        const int p = pw >> 1, side = pw & 1;
        int lt = 0, lp = 0;
        if (side) {
            const PlocInfo l = info[kids[p - n].x];
            lt = l.tris;
            lp = l.pairs;
        }
        first += lt;
        if (depth == 0) {
            side0 = side;
            left_pairs0 = lp;
        } else {
            q += 1 + lp;
        }
        pw = info[p].parent;
    }
    if (x < n) {
        F3 a, b, c;
        load_tri(tris + 9 * (uint64_t)order[x], a, b, c);
        store_btri(btris, (uint64_t)first, a, b, c);
    }
    if (!rec) return;
    NodeRec* r = nodes + (me.parent < 0 ? 0 : 2 * q + side0);
    acc_finalize(accs[x], acc, r);
    if (me.tris <= BVH_LEAF_SIZE) {
        r->L = make_int2(first, -me.tris);
    } else {
        const int P = me.parent < 0 ? 1 : q + 1 + left_pairs0;
        r->L = make_int2(2 * P, 2 * P + 1);
    }
}

// ---------------------------------------------------------------------------
// Top-down binned build, the default for meshes of 2^18 triangles or more.
// Each node is cut where  d2(L) nL + d2(R) nR  is smallest over TD_BINS
// centroid bins per axis, d2 being the squared diagonal of a side's box and n
// its triangle count: a voxel finds a node near in proportion to the node's
// squared radius, and a near node costs visits in proportion to the triangles
// below it.  Over band voxels of a 1.3 M-triangle mesh this tree needs about
// 17% fewer node evaluations than the clustered one, about as many near and
// far visits as the reference's 12-bucket SAH tree (aabb_tree.rs:419-514) and
// fewer triangle evaluations.
//
// The tree is cut level by level; each level moves the triangles of the nodes
// it cuts, in order, to their side in the other of two buffers.  A node of
// more than TD_SMALL triangles is split into tasks of TD_CHUNK triangles; each
// task bins its triangles in LDS and merges them into the node's bins
// (k_td_bin), one wave per node picks the cut and creates the children with
// their tasks (k_td_select), and each task moves its triangles and gathers
// the children's centroid bounds (k_td_partition).
// A node of 2..TD_SMALL triangles is built down to single triangles by one
// wave (k_td_small), four independent waves per block.  The level kernels
// loop over their work with grids sized to the level.
// Node ids follow the clustered build (the triangle at position k is node k,
// internal nodes are n, n+1, ...), so the depth-first layout (k_ploc_place)
// is shared with it.  A node of at most TD_SMALL triangles takes the ids of
// its whole subtree when it is created (its left child's subtree first), so
// only large nodes take ids with atomics: ids vary from run to run, the tree,
// the triangle order and the layout do not.
constexpr int TD_BINS = 16;
constexpr int TD_SMALL = 64;       // nodes of at most this many triangles: one wave, one triangle per lane
constexpr int TD_CHUNK = 2048;     // triangles per task
constexpr int TD_BLOCK = 256;
constexpr int TD_GRID_MAX = 4096;  // blocks of the looping level kernels, at most
constexpr int TD_DEPTH_CAP = 64;   // deeper nodes are cut at the middle of their range
constexpr int TD_BW = 7;           // words per bin: count, box lo xyz, box hi xyz (ordered bits)
constexpr int TD_NODE_WORDS = 3 * TD_BINS * TD_BW;
// counter words: [0], [1] frontier sizes and [2], [3] task counts of the two
// level buffers, then the small-node list size, next id, root, (root, height)
constexpr int TD_C_FR = 0, TD_C_TASKS = 2, TD_C_SMALL = 4, TD_C_NEXT = 5, TD_C_ROOT = 6, TD_C_OUT = 7;
constexpr int TD_C_WORDS = 16;

struct TdNode {  // a node of more than TD_SMALL triangles at the current level
    int begin, end, id, depth;
    uint32_t clo[3], chi[3];  // bounds of its triangles' box centres (ordered bits)
    int task0, pad;           // its first task
};
struct TdSmall {  // a node of 2..TD_SMALL triangles; its subtree's ids are id .. id + (end - begin) - 2
    int begin, end, id, depth_buf;  // depth << 1 | the triangle buffer that holds its range
};
struct TdSplit {
    int axis, bin, nleft;  // bin < 0: cut at the middle of the range
    int slot[2];           // the children's frontier slots (-1: not a large node)
    int pad[3];
};

// Triangle records in the level buffers: (box lo, triangle index bits), (box hi, 0).
__device__ inline float td_centre(float lo, float hi) { return (lo + hi) * 0.5f; }
__device__ inline float td_scale(float lo, float hi) {
    const float ext = hi - lo;
    return ext > 0.0f ? (float)TD_BINS / ext : 0.0f;
}
__device__ inline int td_bin(float c, float lo, float scale) {
    return (int)fminf(fmaxf((c - lo) * scale, 0.0f), (float)(TD_BINS - 1));
}
__device__ inline bool td_is_min(int f) { return f >= 1 && f <= 3; }
__device__ inline uint32_t td_identity(int w) {
    const int f = w % TD_BW;
    return f == 0 ? 0u : (td_is_min(f) ? 0xFFFFFFFFu : 0u);
}
__device__ inline uint32_t td_merge(int f, uint32_t a, uint32_t b) {
    return f == 0 ? a + b : (td_is_min(f) ? min(a, b) : max(a, b));
}
__device__ inline float td_diag2(const uint32_t* w) {  // w[1..3] box lo, w[4..6] box hi (ordered bits)
    float d2 = 0.0f;
    for (int k = 0; k < 3; ++k) {
        const float d = from_ordered_bits(w[4 + k]) - from_ordered_bits(w[1 + k]);
        d2 += d * d;
    }
    return d2;
}

// Lane moves within rows of 16 lanes through DPP (no LDS round trip): a lane
// whose source lies outside its row keeps `old`.  Controls: quad_perm [1,0,3,2]
// and [2,3,0,1], row_half_mirror, row_mirror, row_shl:S (0x100 + S) and
// row_shr:S (0x110 + S).
template <int CTRL>
__device__ inline uint32_t td_dpp(uint32_t old, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, 0xF, 0xF, false);
}
__device__ inline uint32_t td_readlane(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }

// Minimum (MAX: maximum) of an ordered-bits word over the wave, in every lane.
template <bool MAX>
__device__ inline uint32_t td_wave_ext(uint32_t x) {
    auto f = [](uint32_t a, uint32_t b) { return MAX ? max(a, b) : min(a, b); };
    x = f(x, td_dpp<0xB1>(x, x));
    x = f(x, td_dpp<0x4E>(x, x));
    x = f(x, td_dpp<0x141>(x, x));
    x = f(x, td_dpp<0x140>(x, x));
    return f(f(td_readlane(x, 0), td_readlane(x, 16)), f(td_readlane(x, 32), td_readlane(x, 48)));
}

// The lowest lane of those with the smallest cost; -1 when no lane offers a cut.
__device__ inline int td_best(bool valid, float cost) {
    const uint32_t key = valid ? ordered_bits(cost) : 0xFFFFFFFFu;
    const uint32_t m = td_wave_ext<false>(key);
    const uint64_t hit = __ballot(valid && key == m);
    return hit ? __ffsll((unsigned long long)hit) - 1 : -1;
}

// Prefix (left) and suffix (right) of the 16 bins of each axis held by lanes
// 0..47 (lane = axis * 16 + bin, one DPP row per axis), W words per bin merged
// as td_merge does; Rn[] is the right side of a cut after the lane's bin.
// Returns the lane of the cheapest cut as td_best does.
template <int W>
__device__ inline int td_choose(uint32_t (&L)[W], uint32_t (&Rn)[W], int lane, bool allowed) {
    const int bin = lane & (TD_BINS - 1);
    uint32_t R[W];
    for (int f = 0; f < W; ++f) R[f] = L[f];
#define TD_SCAN_STEP(S)                                                        \
    for (int f = 0; f < W; ++f) {                                              \
        L[f] = td_merge(f, L[f], td_dpp<0x110 + (S)>(td_identity(f), L[f]));   \
        R[f] = td_merge(f, R[f], td_dpp<0x100 + (S)>(td_identity(f), R[f]));   \
    }
    TD_SCAN_STEP(1)
    TD_SCAN_STEP(2)
    TD_SCAN_STEP(4)
    TD_SCAN_STEP(8)
#undef TD_SCAN_STEP
    for (int f = 0; f < W; ++f) Rn[f] = td_dpp<0x101>(td_identity(f), R[f]);
    const bool valid = allowed && lane < 3 * TD_BINS && bin < TD_BINS - 1 && L[0] > 0 && Rn[0] > 0;
    const float cost = valid ? td_diag2(L) * (float)L[0] + td_diag2(Rn) * (float)Rn[0] : 0.0f;
    return td_best(valid, cost);
}

// Exclusive prefix of x over the block (TD_BLOCK threads); *total gets the sum.
__device__ inline uint32_t td_block_scan(uint32_t x, uint32_t* wsum, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = x;
    for (int s = 1; s < 64; s <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)inc, s);
        if (lane >= s) inc += y;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int q = 0; q < TD_BLOCK / 64; ++q) {
        if (q < w) before += wsum[q];
        all += wsum[q];
    }
    __syncthreads();
    *total = all;
    return before + inc - x;
}

// The root: triangles as records in buffer 0, the level-0 frontier and its
// tasks, counters.
__global__ void k_td_init(const float* __restrict__ tris, int n, const unsigned* __restrict__ bounds,
                          float4* __restrict__ prims, TdNode* __restrict__ fr, int2* __restrict__ tasks,
                          uint32_t* __restrict__ bins, uint32_t* __restrict__ ctr, PlocInfo* __restrict__ info,
                          uint8_t* __restrict__ ndepth, uint32_t* __restrict__ hist) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int n_tasks = (n + TD_CHUNK - 1) / TD_CHUNK;
    if (i < n) {
        F3 a, b, c;
        load_tri(tris + 9 * (uint64_t)i, a, b, c);
        const F3 mn = f3_min2(c, f3_min2(a, b)), mx = f3_max2(c, f3_max2(a, b));
        prims[2 * (uint64_t)i] = make_float4(mn.x, mn.y, mn.z, __uint_as_float((uint32_t)i));
        prims[2 * (uint64_t)i + 1] = make_float4(mx.x, mx.y, mx.z, 0.0f);
    }
    if (i < n_tasks) tasks[i] = make_int2(0, i * TD_CHUNK);
    if (blockIdx.x != 0) return;
    for (int w = threadIdx.x; w < TD_NODE_WORDS; w += blockDim.x) bins[w] = td_identity(w);
    for (int w = threadIdx.x; w < 256; w += blockDim.x) hist[w] = 0;
    if (threadIdx.x == 0) {
        for (int k = 0; k < TD_C_WORDS; ++k) ctr[k] = 0;
        TdNode r;
        r.begin = 0;
        r.end = n;
        r.id = n;
        r.depth = 0;
        for (int k = 0; k < 3; ++k) {
            r.clo[k] = bounds[k];
            r.chi[k] = bounds[3 + k];
        }
        r.task0 = 0;
        r.pad = 0;
        fr[0] = r;
        ctr[TD_C_FR] = 1;  // the root is large: n >= 2^18
        ctr[TD_C_TASKS] = (uint32_t)n_tasks;
        ctr[TD_C_NEXT] = 1;  // the root is internal node n
        ctr[TD_C_ROOT] = (uint32_t)n;
        info[n] = PlocInfo{n, 0, 0, -1};
        ndepth[0] = 0;
    }
}

// Per task: its triangles' centroid bins on the three axes (count and box),
// in LDS, then merged into the node's bins; the task's bin counts are kept
// for the partition.  Block 0 clears the next level's frontier and task counts.
__global__ __launch_bounds__(TD_BLOCK) void k_td_bin(const float4* __restrict__ prims, const TdNode* __restrict__ fr,
                                                     const int2* __restrict__ tasks, uint32_t* __restrict__ ctr, int in,
                                                     uint32_t* __restrict__ gbins, uint32_t* __restrict__ tcnt) {
    __shared__ uint32_t sb[TD_NODE_WORDS];
    const uint32_t n_tasks = ctr[TD_C_TASKS + in];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctr[TD_C_FR + (in ^ 1)] = 0;
        ctr[TD_C_TASKS + (in ^ 1)] = 0;
    }
    for (uint32_t t = blockIdx.x; t < n_tasks; t += gridDim.x) {  // uniform over the block
        const int2 task = tasks[t];
        const TdNode nd = fr[task.x];
        for (int w = threadIdx.x; w < TD_NODE_WORDS; w += TD_BLOCK) sb[w] = td_identity(w);
        float lo[3], sc[3];
        for (int k = 0; k < 3; ++k) {
            lo[k] = from_ordered_bits(nd.clo[k]);
            sc[k] = td_scale(lo[k], from_ordered_bits(nd.chi[k]));
        }
        __syncthreads();
        const int e = min(task.y + TD_CHUNK, nd.end);
        for (int p = task.y + (int)threadIdx.x; p < e; p += TD_BLOCK) {
            const float4 a = prims[2 * (uint64_t)p], b = prims[2 * (uint64_t)p + 1];
            const float c[3] = {td_centre(a.x, b.x), td_centre(a.y, b.y), td_centre(a.z, b.z)};
            const unsigned bl[3] = {ordered_bits(a.x), ordered_bits(a.y), ordered_bits(a.z)};
            const unsigned bh[3] = {ordered_bits(b.x), ordered_bits(b.y), ordered_bits(b.z)};
            for (int k = 0; k < 3; ++k) {
                uint32_t* bb = sb + (k * TD_BINS + td_bin(c[k], lo[k], sc[k])) * TD_BW;
                atomicAdd(bb, 1u);
                for (int q = 0; q < 3; ++q) {
                    atomicMin(bb + 1 + q, bl[q]);
                    atomicMax(bb + 4 + q, bh[q]);
                }
            }
        }
        __syncthreads();
        if (threadIdx.x < 3 * TD_BINS) tcnt[(uint64_t)t * 3 * TD_BINS + threadIdx.x] = sb[threadIdx.x * TD_BW];
        uint32_t* g = gbins + (uint64_t)task.x * TD_NODE_WORDS;
        for (int w = threadIdx.x; w < TD_NODE_WORDS; w += TD_BLOCK) {
            const int f = w % TD_BW;
            if (sb[w - f] == 0) continue;  // empty bin
            const uint32_t v = sb[w];
            if (f == 0)
                atomicAdd(g + w, v);
            else if (td_is_min(f))
                atomicMin(g + w, v);
            else
                atomicMax(g + w, v);
        }
        __syncthreads();  // sb is reset for the next task
    }
}

// Children of a cut node: a single triangle becomes a leaf at its final
// position; a node of 2..TD_SMALL triangles goes to the small list with the
// ids of its subtree (`ids` .. `ids` + size - 2); a larger one takes one id
// and goes to the frontier (the caller fills its record).  *x: the next id.
__device__ inline int td_child(int cb, int ce, int parent, int depth, int n, uint32_t id, uint8_t* ndepth,
                               PlocInfo* info) {
    const int cs = ce - cb;
    if (cs == 1) {
        info[cb] = PlocInfo{1, 0, 0, parent};
        return cb;
    }
    info[n + (int)id] = PlocInfo{cs, 0, 0, parent};
    ndepth[id] = (uint8_t)min(depth, 255);
    return n + (int)id;
}

// One wave per large node of the level: the cheapest cut, its children
// (small ones to the small list, larger ones to the next frontier with their
// tasks; their centroid bounds are gathered by k_td_partition).  Ids, list
// slots and tasks are counted per block in LDS and taken with one global
// atomic per counter and block.
__global__ __launch_bounds__(TD_BLOCK) void k_td_select(
    const TdNode* __restrict__ fr, uint32_t* __restrict__ ctr, int in, const uint32_t* __restrict__ gbins, int n,
    int fr_cap, int small_cap, int task_cap, TdSplit* __restrict__ split, TdNode* __restrict__ fr_out,
    uint32_t* __restrict__ gbins_out, int2* __restrict__ tasks_out, TdSmall* __restrict__ small_out,
    PlocInfo* __restrict__ info, int2* __restrict__ kids, uint8_t* __restrict__ ndepth, unsigned* err) {
    __shared__ uint32_t cnt[4], base[4];  // ids, small-list slots, frontier slots, tasks of the block
    const uint32_t count = min(ctr[TD_C_FR + in], (uint32_t)fr_cap);
    const int lane = threadIdx.x & 63;
    for (uint32_t r0 = blockIdx.x * (TD_BLOCK / 64); r0 < count; r0 += gridDim.x * (TD_BLOCK / 64)) {
        const int i = (int)r0 + (int)(threadIdx.x >> 6);
        const bool active = i < (int)count;
        if (threadIdx.x < 4) cnt[threadIdx.x] = 0;
        __syncthreads();
        TdNode nd{};
        int axis = 0, sbin = -1, nleft = 0;
        uint32_t off[4] = {0, 0, 0, 0};
        if (active) {
            nd = fr[i];
            const uint32_t* g = gbins + (uint64_t)i * TD_NODE_WORDS;
            uint32_t L[TD_BW], Rn[TD_BW];
            for (int f = 0; f < TD_BW; ++f) L[f] = lane < 3 * TD_BINS ? g[lane * TD_BW + f] : td_identity(f);
            const int wl = td_choose<TD_BW>(L, Rn, lane, nd.depth < TD_DEPTH_CAP);
            nleft = (nd.end - nd.begin) >> 1;
            if (wl >= 0) {
                axis = wl / TD_BINS;
                sbin = wl % TD_BINS;
                nleft = (int)td_readlane(L[0], wl);
            }
            if (lane == 0) {
                uint32_t need[4] = {0, 0, 0, 0};
                for (int side = 0; side < 2; ++side) {
                    const int cs = side ? nd.end - nd.begin - nleft : nleft;
                    if (cs >= 2 && cs <= TD_SMALL) {
                        need[0] += (uint32_t)(cs - 1);  // the small node and its subtree
                        need[1] += 1;
                    } else if (cs > TD_SMALL) {
                        need[0] += 1;
                        need[2] += 1;
                        need[3] += (uint32_t)((cs + TD_CHUNK - 1) / TD_CHUNK);
                    }
                }
                for (int c = 0; c < 4; ++c) off[c] = need[c] ? atomicAdd(&cnt[c], need[c]) : 0u;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            base[0] = cnt[0] ? atomicAdd(ctr + TD_C_NEXT, cnt[0]) : 0u;
            base[1] = cnt[1] ? atomicAdd(ctr + TD_C_SMALL, cnt[1]) : 0u;
            base[2] = cnt[2] ? atomicAdd(ctr + TD_C_FR + (in ^ 1), cnt[2]) : 0u;
            base[3] = cnt[3] ? atomicAdd(ctr + TD_C_TASKS + (in ^ 1), cnt[3]) : 0u;
        }
        __syncthreads();
        int slot[2] = {-1, -1}, t0[2] = {0, 0}, nt[2] = {0, 0}, cb0[2] = {0, 0};
        if (active && lane == 0) {
            uint32_t nid = base[0] + off[0], ns = base[1] + off[1], nf = base[2] + off[2], ntk = base[3] + off[3];
            int kid[2];
            for (int side = 0; side < 2; ++side) {
                const int cb = side ? nd.begin + nleft : nd.begin, ce = side ? nd.end : nd.begin + nleft;
                const int cs = ce - cb, parent = 2 * nd.id + side;
                const uint32_t take = cs == 1 ? 0u : (cs <= TD_SMALL ? (uint32_t)(cs - 1) : 1u);
                if (nid + take > (uint32_t)(n - 1)) {  // a binary tree over n triangles has n - 1 internal nodes
                    atomicOr(err, E_TREE);
                    kid[side] = n;
                    continue;
                }
                kid[side] = td_child(cb, ce, parent, nd.depth + 1, n, nid, ndepth, info);
                const uint32_t id = nid;
                nid += take;
                if (cs == 1) continue;
                if (cs <= TD_SMALL) {
                    const uint32_t j = ns++;
                    if (j >= (uint32_t)small_cap) {
                        atomicOr(err, E_TREE);
                        continue;
                    }
                    small_out[j] = TdSmall{cb, ce, n + (int)id, (nd.depth + 1) << 1 | (in ^ 1)};
                } else {
                    const uint32_t j = nf++, tn = (uint32_t)((cs + TD_CHUNK - 1) / TD_CHUNK), tb = ntk;
                    ntk += tn;
                    if (j >= (uint32_t)fr_cap || tb + tn > (uint32_t)task_cap) {
                        atomicOr(err, E_TREE);
                        continue;
                    }
                    TdNode c;
                    c.begin = cb;
                    c.end = ce;
                    c.id = n + (int)id;
                    c.depth = nd.depth + 1;
                    for (int q = 0; q < 3; ++q) {
                        c.clo[q] = 0xFFFFFFFFu;  // k_td_partition gathers them
                        c.chi[q] = 0u;
                    }
                    c.task0 = (int)tb;
                    c.pad = 0;
                    fr_out[j] = c;
                    slot[side] = (int)j;
                    t0[side] = (int)tb;
                    nt[side] = (int)tn;
                    cb0[side] = cb;
                }
            }
            kids[nd.id - n] = make_int2(kid[0], kid[1]);
            split[i] = TdSplit{axis, sbin, nleft, {slot[0], slot[1]}, {0, 0, 0}};
        }
        for (int side = 0; side < 2; ++side) {
            const int j = __shfl(slot[side], 0);
            if (j < 0) continue;
            for (int w = lane; w < TD_NODE_WORDS; w += 64) gbins_out[(uint64_t)j * TD_NODE_WORDS + w] = td_identity(w);
            const int tb = __shfl(t0[side], 0), tn = __shfl(nt[side], 0), cb = __shfl(cb0[side], 0);
            for (int u = lane; u < tn; u += 64) tasks_out[tb + u] = make_int2(j, cb + u * TD_CHUNK);
        }
        __syncthreads();  // cnt and base are reset for the next round
    }
}

// Per task: its triangles to their side of the cut in the other buffer, in
// order: rounds of TD_BLOCK consecutive triangles, placed by a block scan of
// the side flags.  A triangle that becomes a leaf writes its index to `order`;
// the centroid bounds of each side that is a large node are reduced over the
// task and merged into its frontier record.
__global__ __launch_bounds__(TD_BLOCK) void k_td_partition(const float4* __restrict__ pin, float4* __restrict__ pout,
                                                           const TdNode* __restrict__ fr, const int2* __restrict__ tasks,
                                                           const uint32_t* __restrict__ ctr, int in,
                                                           const TdSplit* __restrict__ split,
                                                           const uint32_t* __restrict__ tcnt,
                                                           TdNode* __restrict__ fr_out, uint32_t* __restrict__ order,
                                                           unsigned* err) {
    __shared__ uint32_t wsum[TD_BLOCK / 64], wl[TD_BLOCK / 64], wr[TD_BLOCK / 64];
    __shared__ uint32_t wb[TD_BLOCK / 64][12];
    const uint32_t n_tasks = ctr[TD_C_TASKS + in];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    for (uint32_t t = blockIdx.x; t < n_tasks; t += gridDim.x) {  // uniform over the block
        const int2 task = tasks[t];
        const TdNode nd = fr[task.x];
        const TdSplit sp = split[task.x];
        const int size = nd.end - nd.begin;
        const int cb = task.y, ce = min(cb + TD_CHUNK, nd.end);
        uint32_t before;
        if (sp.bin >= 0) {  // left triangles of the node's earlier tasks
            uint32_t part = 0;
            for (int u = nd.task0 + (int)threadIdx.x; u < (int)t; u += TD_BLOCK) {
                const uint32_t* c = tcnt + (uint64_t)u * 3 * TD_BINS + sp.axis * TD_BINS;
                for (int b = 0; b <= sp.bin; ++b) part += c[b];
            }
            (void)td_block_scan(part, wsum, &before);
        } else {
            before = (uint32_t)min(cb - nd.begin, sp.nleft);
        }
        // the cut axis's bounds by selects (a run-time index would send nd to LDS)
        const uint32_t clo_a = sp.axis == 0 ? nd.clo[0] : (sp.axis == 1 ? nd.clo[1] : nd.clo[2]);
        const uint32_t chi_a = sp.axis == 0 ? nd.chi[0] : (sp.axis == 1 ? nd.chi[1] : nd.chi[2]);
        const float lo = from_ordered_bits(clo_a);
        const float sc = td_scale(lo, from_ordered_bits(chi_a));
        const uint32_t l0 = (uint32_t)nd.begin + before;
        const uint32_t r0 = (uint32_t)(nd.begin + sp.nleft) + ((uint32_t)(cb - nd.begin) - before);
        const uint32_t lend = (uint32_t)(nd.begin + sp.nleft), rend = (uint32_t)nd.end;
        const bool leaf_l = sp.nleft == 1, leaf_r = size - sp.nleft == 1;
        uint32_t run_l = 0, run_r = 0;
        // centroid bounds of the sides (ordered bits), lo xyz then hi xyz; the
        // side is picked by selects (an array indexed by it would go to LDS)
        uint32_t cl0[3], ch0[3], cl1[3], ch1[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            cl0[q] = cl1[q] = 0xFFFFFFFFu;
            ch0[q] = ch1[q] = 0u;
        }
        bool bad = false;
        for (int base = cb; base < ce; base += TD_BLOCK) {
            const int p = base + (int)threadIdx.x;
            const bool act = p < ce;
            float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
            bool left = false;
            if (act) {
                a = pin[2 * (uint64_t)p];
                b = pin[2 * (uint64_t)p + 1];
                const float c[3] = {td_centre(a.x, b.x), td_centre(a.y, b.y), td_centre(a.z, b.z)};
                if (sp.bin >= 0) {
                    const float ca = sp.axis == 0 ? c[0] : (sp.axis == 1 ? c[1] : c[2]);
                    left = td_bin(ca, lo, sc) <= sp.bin;
                } else {
                    left = p - nd.begin < sp.nleft;
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const uint32_t o = ordered_bits(c[q]);
                    cl0[q] = left ? min(cl0[q], o) : cl0[q];
                    ch0[q] = left ? max(ch0[q], o) : ch0[q];
                    cl1[q] = left ? cl1[q] : min(cl1[q], o);
                    ch1[q] = left ? ch1[q] : max(ch1[q], o);
                }
            }
            const uint64_t bl = __ballot(act && left), br = __ballot(act && !left);
            if (lane == 0) {
                wl[w] = (uint32_t)__popcll(bl);
                wr[w] = (uint32_t)__popcll(br);
            }
            __syncthreads();
            uint32_t pl = 0, pr = 0, tl = 0, tr = 0;
            for (int q = 0; q < TD_BLOCK / 64; ++q) {
                if (q < w) {
                    pl += wl[q];
                    pr += wr[q];
                }
                tl += wl[q];
                tr += wr[q];
            }
            __syncthreads();  // wl and wr are rewritten next round
            if (act) {
                const uint32_t d = left ? l0 + run_l + pl + (uint32_t)__popcll(bl & below)
                                        : r0 + run_r + pr + (uint32_t)__popcll(br & below);
                if (d >= (left ? lend : rend)) {
                    bad = true;
                } else {
                    pout[2 * (uint64_t)d] = a;
                    pout[2 * (uint64_t)d + 1] = b;
                    if (left ? leaf_l : leaf_r) order[d] = __float_as_uint(a.w);
                }
            }
            run_l += tl;
            run_r += tr;
        }
#pragma unroll
        for (int sd = 0; sd < 2; ++sd) {
            if (sp.slot[sd] < 0) continue;  // uniform over the block
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const uint32_t mn = td_wave_ext<false>(sd ? cl1[q] : cl0[q]);
                const uint32_t mx = td_wave_ext<true>(sd ? ch1[q] : ch0[q]);
                if (lane == 0) {
                    wb[w][q] = mn;
                    wb[w][3 + q] = mx;
                }
            }
            __syncthreads();
            if (threadIdx.x < 6) {
                const int q = threadIdx.x;
                uint32_t v = wb[0][q];
                for (int x = 1; x < TD_BLOCK / 64; ++x) v = q < 3 ? min(v, wb[x][q]) : max(v, wb[x][q]);
                TdNode* c = fr_out + sp.slot[sd];
                if (q < 3)
                    atomicMin(&c->clo[q], v);
                else
                    atomicMax(&c->chi[q - 3], v);
            }
            __syncthreads();  // wb is rewritten for the other side
        }
        if (sp.bin >= 0) {  // the cut must agree with the bins it was chosen from
            uint32_t want = 0;
            const uint32_t* c = tcnt + (uint64_t)t * 3 * TD_BINS + sp.axis * TD_BINS;
            for (int q = 0; q <= sp.bin; ++q) want += c[q];
            bad = bad || want != run_l;
        }
        if (bad) atomicOr(err, E_TREE);
    }
}

// One wave per node of 2..TD_SMALL triangles, four independent waves per
// block: the whole subtree, cut by the same rule over each range's own
// centroid bounds (the middle of the range when bins cannot cut it), with the
// triangles' boxes in LDS and their order permuted between two index buffers.
// The node took the ids of its subtree when it was created; its internal
// nodes take them in the order they are created.
__device__ inline void td_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(TD_BLOCK) void k_td_small(const float4* __restrict__ prims, int n,
                                                       const TdSmall* __restrict__ small, const uint32_t* __restrict__ ctr,
                                                       int small_cap, PlocInfo* __restrict__ info,
                                                       int2* __restrict__ kids, uint32_t* __restrict__ order,
                                                       uint8_t* __restrict__ ndepth, unsigned* err) {
    constexpr int WAVES = TD_BLOCK / 64;
    __shared__ float4 srl[WAVES][TD_SMALL], srh[WAVES][TD_SMALL];
    __shared__ uint8_t sperm[WAVES][2][TD_SMALL];
    __shared__ uint32_t ssb[WAVES][3 * TD_BINS * TD_BW];
    __shared__ int4 sstk[WAVES][TD_SMALL / 2];  // pending ranges are disjoint and hold >= 2 triangles
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t i = blockIdx.x * WAVES + w;
    if (i >= min(ctr[TD_C_SMALL], (uint32_t)small_cap)) return;  // whole waves; no block barrier follows
    float4* rl = srl[w];
    float4* rh = srh[w];
    uint32_t* sb = ssb[w];
    int4* stk = sstk[w];
    const TdSmall sm = small[i];
    const int s = sm.end - sm.begin;
    if (s < 2 || s > TD_SMALL || sm.id < n || sm.id - n + (s - 1) > n - 1) {
        if (lane == 0) atomicOr(err, E_TREE);
        return;
    }
    const float4* src = prims + (uint64_t)(sm.depth_buf & 1) * 2 * (uint64_t)n;
    if (lane < s) {
        rl[lane] = src[2 * (uint64_t)(sm.begin + lane)];
        rh[lane] = src[2 * (uint64_t)(sm.begin + lane) + 1];
        sperm[w][0][lane] = (uint8_t)lane;
    }
    int id_next = sm.id + 1;  // used by lane 0
    if (lane == 0) stk[0] = make_int4(0, s, sm.id, sm.depth_buf & ~1);
    int sp = 1;
    td_wave_sync();
    const uint64_t below = (1ull << lane) - 1ull;
    while (sp > 0) {
        --sp;
        const int4 e = stk[sp];
        const int b = e.x, en = e.y, id = e.z, depth = e.w >> 1;
        int buf = e.w & 1;
        const int sz = en - b;
        int nleft = sz >> 1;
        if (sz > 2) {
            const bool mine = lane < sz;
            float4 l = make_float4(0.0f, 0.0f, 0.0f, 0.0f), h = l;
            int q = 0;
            if (mine) {
                q = sperm[w][buf][b + lane];
                l = rl[q];
                h = rh[q];
            }
            const float c[3] = {td_centre(l.x, h.x), td_centre(l.y, h.y), td_centre(l.z, h.z)};
            float mn[3], mx[3], sc[3];
            for (int k = 0; k < 3; ++k) {
                mn[k] = mine ? c[k] : INFINITY;
                mx[k] = mine ? c[k] : -INFINITY;
            }
            for (int k = 0; k < 3; ++k) {
                mn[k] = from_ordered_bits(td_wave_ext<false>(ordered_bits(mn[k])));
                mx[k] = from_ordered_bits(td_wave_ext<true>(ordered_bits(mx[k])));
                sc[k] = td_scale(mn[k], mx[k]);
            }
            int axis = 0, sbin = -1;
            if (depth < TD_DEPTH_CAP && (sc[0] > 0.0f || sc[1] > 0.0f || sc[2] > 0.0f)) {
                for (int x = lane; x < 3 * TD_BINS * TD_BW; x += 64) {
                    const int f = x % TD_BW;
                    sb[x] = f == 0 ? 0u : (f <= 3 ? 0xFFFFFFFFu : 0u);
                }
                td_wave_sync();
                if (mine) {
                    const unsigned bl[3] = {ordered_bits(l.x), ordered_bits(l.y), ordered_bits(l.z)};
                    const unsigned bh[3] = {ordered_bits(h.x), ordered_bits(h.y), ordered_bits(h.z)};
                    for (int k = 0; k < 3; ++k) {
                        uint32_t* bb = sb + (k * TD_BINS + td_bin(c[k], mn[k], sc[k])) * TD_BW;
                        atomicAdd(bb, 1u);
                        for (int q3 = 0; q3 < 3; ++q3) {
                            atomicMin(bb + 1 + q3, bl[q3]);
                            atomicMax(bb + 4 + q3, bh[q3]);
                        }
                    }
                }
                td_wave_sync();
                uint32_t L[TD_BW], Rn[TD_BW];
                for (int f = 0; f < TD_BW; ++f) {
                    const uint32_t id0 = f == 0 ? 0u : (f <= 3 ? 0xFFFFFFFFu : 0u);
                    L[f] = lane < 3 * TD_BINS ? sb[lane * TD_BW + f] : id0;
                }
                const int wl = td_choose<TD_BW>(L, Rn, lane, true);
                if (wl >= 0) {
                    axis = wl / TD_BINS;
                    sbin = wl % TD_BINS;
                    nleft = (int)td_readlane(L[0], wl);
                }
                td_wave_sync();  // sb is read before the next range clears it
            }
            // stable partition of the range into the other index buffer
            bool lf;
            if (sbin >= 0) {
                const float ca = axis == 0 ? c[0] : (axis == 1 ? c[1] : c[2]);
                lf = mine && td_bin(ca, mn[axis], sc[axis]) <= sbin;
            } else {
                lf = lane < nleft;
            }
            const uint64_t BL = __ballot(mine && lf), BR = __ballot(mine && !lf);
            if (__popcll(BL) != nleft) {  // the bins and the partition disagree: never expected
                if (lane == 0) atomicOr(err, E_TREE);
                return;  // the whole wave
            }
            if (mine) {
                const int d = lf ? b + __popcll(BL & below) : b + nleft + __popcll(BR & below);
                sperm[w][buf ^ 1][d] = (uint8_t)q;
            }
            buf ^= 1;
            td_wave_sync();
        }
        if (lane == 0) {
            int kid[2];
            for (int side = 0; side < 2; ++side) {
                const int cb = side ? b + nleft : b, ce = side ? en : b + nleft, cs = ce - cb;
                const int parent = 2 * id + side;
                if (cs == 1) {
                    const int pos = sm.begin + cb;
                    kid[side] = pos;
                    info[pos] = PlocInfo{1, 0, 0, parent};
                    order[pos] = __float_as_uint(rl[sperm[w][buf][cb]].w);
                } else {
                    kid[side] = td_child(sm.begin + cb, sm.begin + ce, parent, depth + 1, n, (uint32_t)(id_next - n),
                                         ndepth, info);
                    ++id_next;
                    stk[sp++] = make_int4(cb, ce, kid[side], (depth + 1) << 1 | buf);
                }
            }
            kids[id - n] = make_int2(kid[0], kid[1]);
        }
        sp = __shfl(sp, 0);
        td_wave_sync();
    }
}

// Leaf data at every position.
__global__ void k_td_leaves(const float* __restrict__ tris, int n, const uint32_t* __restrict__ order,
                            NodeAcc* __restrict__ accs, unsigned* err) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t o = order[k];
    if (o >= (uint32_t)n) {  // a position no leaf wrote
        atomicOr(err, E_TREE);
        return;
    }
    F3 a, b, c;
    load_tri(tris + 9 * (uint64_t)o, a, b, c);
    accs[k] = tri_acc(a, b, c);
}

// Internal nodes grouped by depth, a counting sort: per-block LDS counts and
// one global atomic per depth and block.  hist[0, 256) counts, hist[256, 512)
// cursors, hist[512, 769) group starts.
__global__ __launch_bounds__(256) void k_td_depth_hist(const uint8_t* __restrict__ ndepth, int m, uint32_t* hist) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int i = blockIdx.x * 256 + (int)threadIdx.x;
    if (i < m) atomicAdd(&h[ndepth[i]], 1u);
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

__global__ __launch_bounds__(256) void k_td_depth_scan(uint32_t* hist) {
    __shared__ uint32_t wsum[4];
    const uint32_t x = hist[threadIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = x;
    for (int s = 1; s < 64; s <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)inc, s);
        if (lane >= s) inc += y;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int q = 0; q < 4; ++q) {
        if (q < w) before += wsum[q];
        all += wsum[q];
    }
    hist[256 + threadIdx.x] = before + inc - x;
    hist[512 + threadIdx.x] = before + inc - x;
    if (threadIdx.x == 0) hist[768] = all;
}

__global__ __launch_bounds__(256) void k_td_depth_scatter(const uint8_t* __restrict__ ndepth, int m, uint32_t* hist,
                                                          uint32_t* __restrict__ out) {
    __shared__ uint32_t h[256], b[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int i = blockIdx.x * 256 + (int)threadIdx.x;
    uint32_t d = 0, r = 0;
    if (i < m) {
        d = ndepth[i];
        r = atomicAdd(&h[d], 1u);
    }
    __syncthreads();
    if (h[threadIdx.x]) b[threadIdx.x] = atomicAdd(&hist[256 + threadIdx.x], h[threadIdx.x]);
    __syncthreads();
    if (i < m) out[b[d] + r] = (uint32_t)i;
}

// Node data of one depth level (internal nodes n + inode[i]; the next level
// down is complete) and the traversal-layout counts k_ploc_place needs.
__global__ void k_td_level(const uint32_t* __restrict__ inode, uint32_t count, int n, const int2* __restrict__ kids,
                           NodeAcc* accs, PlocInfo* info) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int x = (int)inode[i], p = n + x;
    const int2 L = kids[x];
    NodeAcc s;
    acc_add(s, accs[L.x], accs[L.y]);
    accs[p] = s;
    const PlocInfo il = info[L.x], ir = info[L.y];
    PlocInfo me = info[p];
    const bool leaf = me.tris <= BVH_LEAF_SIZE;
    me.pairs = leaf ? 0 : 1 + il.pairs + ir.pairs;
    me.height = leaf ? 0 : 1 + max(il.height, ir.height);
    info[p] = me;
}

// ---------------------------------------------------------------------------
// winding numbers at active voxels, wave-coherent traversal

// Solid angle of triangle (a, b, c) seen from the origin (a, b, c already
// relative to the query), aabb_tree.rs:582-615 in the Van Oosterom-Strackee
// form: tan(W/2) = det[a b c] / (|a||b||c| + (a.b)|c| + (a.c)|b| + (b.c)|a|),
// which equals the reference's normalised expression.  Zero when a vertex
// coincides with the query or the triple product vanishes.
// The triple product keeps the reference's unfused f32 arithmetic: for a
// point a few ulps off a triangle's plane, whether it rounds to zero decides
// between a zero solid angle and +-2 pi, as in the reference.  The lengths and
// the denominator only scale the angle and are written with explicit FMAs
// (the library is built without contraction, for the distance arithmetic).
__device__ inline float solid_angle_rel(float ax, float ay, float az, float bx, float by, float bz, float cx, float cy,
                                        float cz) {
    const float la = fast_sqrt(__builtin_fmaf(ax, ax, __builtin_fmaf(ay, ay, az * az)));
    const float lb = fast_sqrt(__builtin_fmaf(bx, bx, __builtin_fmaf(by, by, bz * bz)));
    const float lc = fast_sqrt(__builtin_fmaf(cx, cx, __builtin_fmaf(cy, cy, cz * cz)));
    const float det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx);
    const float ab = __builtin_fmaf(ax, bx, __builtin_fmaf(ay, by, az * bz));
    const float ac = __builtin_fmaf(ax, cx, __builtin_fmaf(ay, cy, az * cz));
    const float bc = __builtin_fmaf(bx, cx, __builtin_fmaf(by, cy, bz * cz));
    const float den = __builtin_fmaf(la * lb, lc, __builtin_fmaf(ab, lc, __builtin_fmaf(ac, lb, bc * la)));
    const float w = 2.0f * fast_atan2(det, den);
    return (la == 0.0f || lb == 0.0f || lc == 0.0f || det == 0.0f) ? 0.0f : w;
}

__device__ inline double solid_angle_rel64(double ax, double ay, double az, double bx, double by, double bz, double cx,
                                           double cy, double cz) {
    double la = sqrt(ax * ax + ay * ay + az * az);
    double lb = sqrt(bx * bx + by * by + bz * bz);
    double lc = sqrt(cx * cx + cy * cy + cz * cz);
    double det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx);
    double den = la * lb * lc + (ax * bx + ay * by + az * bz) * lc + (ax * cx + ay * cy + az * cz) * lb +
                 (bx * cx + by * cy + bz * cz) * la;
    if (la == 0.0 || lb == 0.0 || lc == 0.0 || det == 0.0) return 0.0;
    return 2.0 * atan2(det, den);
}


// order-2 far-field term of a node at query offset r = c - p, with the node's
// coefficients pre-scaled (acc_finalize): 17 VALU operations
__device__ inline float dipole_term(const float4& B, const float4& C, const float2& D, float rx, float ry, float rz,
                                   float r2) {
    const float inv_r = fast_rsq(r2);
    const float inv_r2 = inv_r * inv_r;
    const float u = __builtin_fmaf(C.x, rx, __builtin_fmaf(C.w, ry, D.x * rz));
    const float v = __builtin_fmaf(C.y, ry, D.y * rz);
    const float rsr = __builtin_fmaf(rx, u, __builtin_fmaf(ry, v, rz * (C.z * rz)));
    const float lin = __builtin_fmaf(B.x, rx, __builtin_fmaf(B.y, ry, __builtin_fmaf(B.z, rz, B.w)));
    return (inv_r * inv_r2) * __builtin_fmaf(-rsr, inv_r2, lin);
}

// Per-wave traversal stacks.  An entry is a pair of sibling nodes and the lanes
// for which their parent was near; the stack never holds more entries than the
// tree is high.  LaneStack keeps entry k in lane k of four VGPRs (written by a
// per-lane select, read with v_readlane: no memory round trip) and serves trees
// lower than 64; LdsStack serves any height up to 256 from LDS.
struct LaneStack {
    static constexpr int DEPTH = 64;
    int a0 = 0, b0 = 0, l0 = 0, h0 = 0;
    __device__ void push(int sp, int a, int b, unsigned long long m, int lane) {
        const bool mine = lane == sp;
        a0 = mine ? a : a0;
        b0 = mine ? b : b0;
        l0 = mine ? (int)(unsigned)m : l0;
        h0 = mine ? (int)(unsigned)(m >> 32) : h0;
    }
    __device__ void pop(int sp, int& a, int& b, unsigned long long& m) const {
        a = __builtin_amdgcn_readlane(a0, sp);
        b = __builtin_amdgcn_readlane(b0, sp);
        m = ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(h0, sp) << 32) |
            (unsigned)__builtin_amdgcn_readlane(l0, sp);
    }
};

struct LdsStack {
    static constexpr int DEPTH = 256;
    int4* e;  // this wave's DEPTH entries: (a, b, mask lo, mask hi)
    __device__ void push(int sp, int a, int b, unsigned long long m, int lane) {
        if (lane == 0) e[sp] = make_int4(a, b, (int)(unsigned)m, (int)(unsigned)(m >> 32));
    }
    __device__ void pop(int sp, int& a, int& b, unsigned long long& m) const {
        const int4 v = e[sp];
        a = __builtin_amdgcn_readfirstlane(v.x);
        b = __builtin_amdgcn_readfirstlane(v.y);
        m = ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane(v.w) << 32) |
            (unsigned)__builtin_amdgcn_readfirstlane(v.z);
    }
};


// Empty asm that consumes every word of a node record as a scalar register:
// the record's loads must all be issued before it (one memory round trip
// instead of one per use site).
__device__ inline void pin_record(const NodeRec& r) {
    asm volatile("" ::"s"(r.A.x), "s"(r.A.y), "s"(r.A.z), "s"(r.A.w), "s"(r.B.x), "s"(r.B.y), "s"(r.B.z),
                 "s"(r.B.w), "s"(r.C.x), "s"(r.C.y), "s"(r.C.z), "s"(r.C.w), "s"(r.D.x), "s"(r.D.y), "s"(r.L.x),
                 "s"(r.L.y));
}

// Per-lane winding sum (plain f32: its rounding, ~1e-6 over a few hundred
// terms, is far below the FP64 re-check band, which has to cover the cut-off of
// a chunk's polynomial too where one is used: see WN_FAR_BAND) and, when
// counting, per-wave visit counters for the work accounting.
template <bool COUNT>
struct WnAcc {
    float s = 0.0f;
    unsigned long long near_int = 0, far = 0, leaf = 0, tri = 0;
};

// A wave's near leaves waiting for their exact solid angles, one (lane, leaf)
// pair per entry.  A leaf is near for a quarter of the lanes that reach it
// (5.5 of the 22.7 leaves that a wave meets, at 1.3 M triangles on a grid of
// 1050 voxels), so the pairs of several leaves are collected and taken 64 at a
// time, every lane working: a lane evaluates a leaf for the voxel of any lane
// and adds the angle to that lane's sum in LDS.
struct LeafQueue {
    static constexpr int BATCH = 64;
    static constexpr int CAP = BATCH - 1 + 2 * 64;  // what is left plus one visited pair of nodes
    int2* e;     // (first triangle, lane | count << 8)
    float* sum;  // per lane
    int n = 0;   // wave-uniform
};

// Evaluates the queue's last `count` entries (the same for every lane).
__device__ inline void wn_leaves(LeafQueue& q, int count, float px, float py, float pz, int lane,
                                 const float* __restrict__ btris) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    q.n -= count;
    const bool mine = lane < count;
    const int2 en = q.e[q.n + (mine ? lane : 0)];
    const int owner = en.y & 63, cnt = en.y >> 8;
    const float x = __shfl(px, owner, 64), y = __shfl(py, owner, 64), z = __shfl(pz, owner, 64);
    // all BVH_LEAF_SIZE triangles requested at once (btris is padded)
    const float4* tp = reinterpret_cast<const float4*>(btris) + 3 * (uint64_t)(uint32_t)en.x;
    float4 t4[3 * BVH_LEAF_SIZE];
#pragma unroll
    for (int k = 0; k < 3 * BVH_LEAF_SIZE; ++k) t4[k] = tp[k];
    const float* t = reinterpret_cast<const float*>(t4);
    float om = 0.0f;
#pragma unroll
    for (int k = 0; k < BVH_LEAF_SIZE; ++k) {
        const float* tr = t + 12 * k;
        const float sa = solid_angle_rel(tr[0] - x, tr[1] - y, tr[2] - z, tr[3] - x, tr[4] - y, tr[5] - z, tr[6] - x,
                                         tr[7] - y, tr[8] - z);
        om += (k < cnt) ? sa : 0.0f;
    }
    if (mine) atomicAdd(&q.sum[owner], om * INV_4PI);
}

// One node for the lanes in m.  Lane sets stay in scalar registers (ballot
// results combined with SALU ops, turned back into per-lane conditions by
// inverse_ballot): far lanes add the order-2 term, near lanes either queue a
// leaf for its triangles' exact solid angles or ask for the node's children.
// Returns the mask of lanes that need the children (0 for a leaf).
template <bool COUNT>
__device__ inline unsigned long long wn_visit(const NodeRec& r, unsigned long long m, float px, float py, float pz,
                                              int lane, LeafQueue& q, WnAcc<COUNT>& a) {
    const float rx = r.A.x - px, ry = r.A.y - py, rz = r.A.z - pz;
    const float r2 = __builtin_fmaf(rx, rx, __builtin_fmaf(ry, ry, rz * rz));
    const unsigned long long far_all = __ballot(r2 > r.A.w);
    const unsigned long long farm = m & far_all;
    const unsigned long long nm = m & ~far_all;
    if (COUNT) a.far += __popcll(farm);
    if (farm) {
        if (__builtin_amdgcn_inverse_ballot_w64(farm)) a.s += dipole_term(r.B, r.C, r.D, rx, ry, rz, r2);
    }
    if (nm == 0) return 0;
    if (r.L.y < 0) {  // leaf: triangles [L.x, L.x - L.y)
        const int cnt = -r.L.y;
        if (COUNT) {
            a.leaf += __popcll(nm);
            a.tri += (unsigned long long)__popcll(nm) * cnt;
        }
        const int at = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(nm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)nm, 0u));
        if (__builtin_amdgcn_inverse_ballot_w64(nm)) q.e[q.n + at] = make_int2(r.L.x, lane | cnt << 8);
        q.n += __popcll(nm);
        return 0;
    }
    if (COUNT) a.near_int += __popcll(nm);
    return nm;
}

// consecutive workgroups of the winding-number list that one XCD takes in a row
constexpr uint32_t WN_CHUNK = 512;

// What lies far from a whole chunk (64 consecutive entries of the winding
// number list, one wave of k_winding) is summed once for the chunk: the order-2
// terms of such nodes are smooth there, and their sum is kept as its Taylor
// polynomial of degree 3 about the chunk's centre (the method of local
// expansions, Greengard and Rokhlin, "A Fast Algorithm for Particle
// Simulations", 1987).  A node joins it when it is far, by the traversal's own
// criterion, from every point of the ball (centre, rho) around the chunk, and
// its distance from the centre is above wn_kappa(accuracy) * rho, which keeps
// the cut-off terms below those that the order-2 term leaves out.  Everything
// else ends in the chunk's list: k_winding visits the listed nodes per voxel.
// A node near for every voxel, or still outside kappa * rho, is opened here, so
// the list holds what the voxels have to look at themselves.  A workgroup's lists
// lie in its own part of the list memory, one behind the other; a chunk whose list
// reaches past that part, or whose list or stack outgrows its share of LDS, has
// no polynomial and no list: its voxels walk the whole tree.  Which chunks these
// are depends on the mesh alone, not on the order in which workgroups run.
//
// 16 lanes per chunk: a tree level leaves about 15 nodes to look at, one per
// lane, so four chunks keep a wave busy where one would leave three lanes of
// four idle.
//
// Bound by vector issue (about 110 instructions per node that joins).  With the
// list, k_winding meets 99 nodes per wave instead of about 300: at 42 M voxels
// and 1.3 M triangles k_winding took 12.5 ms alone; the two take 7.8 ms, 6.8
// with the queued leaves (LeafQueue).  Shared-sign group roots, 64 of which lie
// across dozens of leaves, keep the walk from the root.
constexpr int FF_BLOCK = 256;
constexpr int FF_LANES = 16;                     // lanes per chunk
constexpr int FF_CHUNKS = FF_BLOCK / FF_LANES;   // chunks per workgroup
constexpr int FF_STACK = 192, FF_LIST = 128;     // LDS entries per chunk
constexpr uint32_t FF_PART = 64 * FF_CHUNKS;     // a workgroup's list entries
constexpr int FF_COEF = 24;                      // floats per chunk: centre, then 20 coefficients

struct FarChunk {
    uint32_t off, cnt;  // list entries [off, off + cnt); cnt == 0xFFFFFFFF: walk from the root
};

__device__ inline float ff_row_sum(float v) {
    auto add = [](float a, uint32_t b) { return a + __uint_as_float(b); };
    v = add(v, td_dpp<0xB1>(0u, __float_as_uint(v)));
    v = add(v, td_dpp<0x4E>(0u, __float_as_uint(v)));
    v = add(v, td_dpp<0x141>(0u, __float_as_uint(v)));
    return add(v, td_dpp<0x140>(0u, __float_as_uint(v)));
}
template <bool MAX>
__device__ inline int ff_row_ext(int v) {
    auto f = [](int a, uint32_t b) { return MAX ? max(a, (int)b) : min(a, (int)b); };
    v = f(v, td_dpp<0xB1>((uint32_t)v, (uint32_t)v));
    v = f(v, td_dpp<0x4E>((uint32_t)v, (uint32_t)v));
    v = f(v, td_dpp<0x141>((uint32_t)v, (uint32_t)v));
    return f(v, td_dpp<0x140>((uint32_t)v, (uint32_t)v));
}

// Taylor coefficients of a node's order-2 term about R = c - centre, in voxel
// units: with r = R - d, b = B.r, s = r.S.r and t the trace term,
//   (b + t) r^-3 - s r^-5
// and its first two derivatives, and the third derivative of b r^-3 (that of the
// quadratic part is one order smaller and left out).
struct FarSum {
    float c0 = 0.0f, gx = 0.0f, gy = 0.0f, gz = 0.0f;
    float hxx = 0.0f, hyy = 0.0f, hzz = 0.0f, hxy = 0.0f, hxz = 0.0f, hyz = 0.0f;
    float zx = 0.0f, zy = 0.0f, zz = 0.0f;  // |d|^2 (z.d)
    float kxxx = 0.0f, kyyy = 0.0f, kzzz = 0.0f, kxxy = 0.0f, kxxz = 0.0f, kxyy = 0.0f, kyyz = 0.0f, kxzz = 0.0f,
          kyzz = 0.0f, kxyz = 0.0f;

    __device__ void add(const float4& B, const float4& C, const float2& D, float x, float y, float z, float r2,
                        float inv_h, float inv_h2, float inv_h3) {
        const float inv = fast_rsq(r2), inv2 = inv * inv;
        const float a3 = inv * inv2, a5 = a3 * inv2, a7 = a5 * inv2, a9 = a7 * inv2;
        const float Bx = B.x * inv_h2, By = B.y * inv_h2, Bz = B.z * inv_h2, t = B.w * inv_h3;
        const float Sxx = C.x * inv_h3, Syy = C.y * inv_h3, Szz = C.z * inv_h3;
        const float Sxy2 = C.w * inv_h3, Sxz2 = D.x * inv_h3, Syz2 = D.y * inv_h3;  // twice the off-diagonals
        auto fma = [](float a, float b, float c) { return __builtin_fmaf(a, b, c); };
        const float b = fma(Bx, x, fma(By, y, Bz * z));
        const float vx = fma(Sxx, x, 0.5f * fma(Sxy2, y, Sxz2 * z));
        const float vy = fma(Syy, y, 0.5f * fma(Sxy2, x, Syz2 * z));
        const float vz = fma(Szz, z, 0.5f * fma(Sxz2, x, Syz2 * y));
        const float s = fma(vx, x, fma(vy, y, vz * z));
        const float bt = b + t;
        c0 += fma(bt, a3, -(s * a5));
        const float e = fma(5.0f * s, a7, -3.0f * bt * a5);
        gx -= fma(Bx, a3, fma(x, e, -2.0f * vx * a5));
        gy -= fma(By, a3, fma(y, e, -2.0f * vy * a5));
        gz -= fma(Bz, a3, fma(z, e, -2.0f * vz * a5));
        const float wr = 0.5f * fma(15.0f * bt, a7, -35.0f * s * a9), w5 = -3.0f * a5, w7 = 10.0f * a7;
        const float wx = fma(w5, Bx, fma(w7, vx, wr * x));
        const float wy = fma(w5, By, fma(w7, vy, wr * y));
        const float wz = fma(w5, Bz, fma(w7, vz, wr * z));
        const float eh = 0.5f * e;
        hxx += fma(wx, x, fma(-a5, Sxx, eh));
        hyy += fma(wy, y, fma(-a5, Syy, eh));
        hzz += fma(wz, z, fma(-a5, Szz, eh));
        hxy += fma(wx, y, fma(wy, x, -a5 * Sxy2));
        hxz += fma(wx, z, fma(wz, x, -a5 * Sxz2));
        hyz += fma(wy, z, fma(wz, y, -a5 * Syz2));
        const float z5 = 1.5f * a5, z7 = -7.5f * a7 * b;
        zx += fma(z5, Bx, z7 * x);
        zy += fma(z5, By, z7 * y);
        zz += fma(z5, Bz, z7 * z);
        const float q7 = -7.5f * a7, q9 = 17.5f * b * a9;
        const float qx = fma(q7, Bx, q9 * x), qy = fma(q7, By, q9 * y), qz = fma(q7, Bz, q9 * z);
        const float xx = x * x, yy = y * y, zz2 = z * z, xy = 2.0f * x * y, xz = 2.0f * x * z, yz = 2.0f * y * z;
        kxxx = fma(qx, xx, kxxx);
        kyyy = fma(qy, yy, kyyy);
        kzzz = fma(qz, zz2, kzzz);
        kxxy = fma(qy, xx, fma(qx, xy, kxxy));
        kxxz = fma(qz, xx, fma(qx, xz, kxxz));
        kxyy = fma(qx, yy, fma(qy, xy, kxyy));
        kyyz = fma(qz, yy, fma(qy, yz, kyyz));
        kxzz = fma(qx, zz2, fma(qz, xz, kxzz));
        kyzz = fma(qy, zz2, fma(qz, yz, kyzz));
        kxyz = fma(qx, yz, fma(qy, xz, fma(qz, xy, kxyz)));
    }
};

__global__ __launch_bounds__(FF_BLOCK) void k_far_field(const uint32_t* __restrict__ act, uint32_t n_act,
                                                        uint32_t n_chunks, const int32_t* __restrict__ origins, float h,
                                                        float inv_h, float kappa, const NodeRec* __restrict__ nodes,
                                                        int n_nodes, uint32_t* __restrict__ list,
                                                        FarChunk* __restrict__ chunks, float* __restrict__ coef) {
    __shared__ int s_stack[FF_CHUNKS][FF_STACK];
    __shared__ uint32_t s_list[FF_CHUNKS][FF_LIST];
    __shared__ uint32_t s_cnt[FF_CHUNKS];
    const int grp = threadIdx.x / FF_LANES, gl = threadIdx.x % FF_LANES, sh = threadIdx.x & 48;
    // a workgroup covers FF_CHUNKS / 4 workgroups of k_winding: the same runs on the same XCD
    const uint32_t group = xcd_workgroup(WN_CHUNK * (WN_BLOCK / 64) / FF_CHUNKS), chunk = group * FF_CHUNKS + grp;
    const bool valid = chunk < n_chunks;
    // the chunk's voxels, four per lane; past the end of the list the last one again
    int v[4][3], lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint64_t i = (uint64_t)chunk * 64 + (uint32_t)(gl * 4 + j);
        const uint32_t slot = act[i < n_act ? (uint32_t)i : n_act - 1];
        const int4 o = reinterpret_cast<const int4*>(origins)[slot >> 9];
        v[j][0] = o.x + (int)((slot >> 6) & 7);
        v[j][1] = o.y + (int)((slot >> 3) & 7);
        v[j][2] = o.z + (int)(slot & 7);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = min(lo[k], v[j][k]);
            hi[k] = max(hi[k], v[j][k]);
        }
    }
    float ctr[3], rho2 = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lo[k] = ff_row_ext<false>(lo[k]);
        hi[k] = ff_row_ext<true>(hi[k]);
        ctr[k] = 0.5f * (float)lo[k] + 0.5f * (float)hi[k];  // whole or half voxels: exact
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float d2 = 0.0f;
#pragma unroll
        for (int k = 0; k < 3; ++k) d2 = __builtin_fmaf((float)v[j][k] - ctr[k], (float)v[j][k] - ctr[k], d2);
        rho2 = fmaxf(rho2, d2);
    }
    rho2 = __int_as_float(ff_row_ext<true>(__float_as_int(rho2)));  // >= 0: ordered as integers
    const float rho = fmaxf(sqrtf(rho2) * 1.0001f, 1.0f);           // in voxels
    const float zone2 = kappa * rho * kappa * rho;
    const float cx = ctr[0] * h, cy = ctr[1] * h, cz = ctr[2] * h;
    const float inv_h2 = inv_h * inv_h, inv_h3 = inv_h2 * inv_h;

    FarSum f;
    int sp = valid ? 1 : 0;
    uint32_t cnt = 0;
    bool bad = false;
    if (gl == 0) s_stack[grp][0] = 0;
    // one pass takes up to 16 nodes off each chunk's stack; a tree's nodes are
    // taken once each, so more passes than nodes means corrupt links
    for (int pass = 0; __any(sp > 0); ++pass) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int take = min(sp, FF_LANES);
        sp -= take;
        const int node = gl < take ? s_stack[grp][sp + gl] : -1;
        bool open = false, listed = false;
        int2 L = make_int2(0, 0);
        if (node >= 0) {
            const NodeRec r = nodes[node];
            L = r.L;
            const float x = (r.A.x - cx) * inv_h, y = (r.A.y - cy) * inv_h, z = (r.A.z - cz) * inv_h;
            const float r2 = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
            const float fr = sqrtf(r.A.w) * inv_h;  // the node is far beyond this distance
            const float out = fr + rho, in = fr - rho;
            const bool leaf = L.y < 0;
            if (r2 > out * out && r2 > zone2) {
                f.add(r.B, r.C, r.D, x, y, z, r2, inv_h, inv_h2, inv_h3);
            } else if (!leaf && ((in > 0.0f && r2 <= in * in) || r2 > zone2)) {
                open = true;
            } else {
                listed = true;
            }
        }
        const uint32_t below = (1u << gl) - 1;
        const uint32_t om = (uint32_t)(__ballot(open) >> sh) & 0xFFFFu, lm = (uint32_t)(__ballot(listed) >> sh) & 0xFFFFu;
        const int n_open = __popc(om), n_list = __popc(lm);
        if (sp + 2 * n_open > FF_STACK || cnt + n_list > FF_LIST || pass > n_nodes) {
            bad = true;
            sp = 0;
        } else {
            if (open) {
                const int at = sp + 2 * __popc(om & below);
                s_stack[grp][at] = L.x;
                s_stack[grp][at + 1] = L.y;
            }
            if (listed) s_list[grp][cnt + __popc(lm & below)] = (uint32_t)node;
            sp += 2 * n_open;
            cnt += n_list;
        }
    }
    // the chunk's place in the workgroup's part of the list memory
    if (gl == 0) s_cnt[grp] = bad || !valid ? 0u : cnt;
    __syncthreads();
    if (!valid) return;
    uint32_t before = 0;
#pragma unroll
    for (int g = 0; g < FF_CHUNKS; ++g) before += g < grp ? s_cnt[g] : 0u;
    const uint32_t base = group * FF_PART;
    if (bad || before + cnt > FF_PART) {
        if (gl == 0) chunks[chunk] = FarChunk{0u, 0xFFFFFFFFu};
        return;
    }
    if (gl == 0) chunks[chunk] = FarChunk{base + before, cnt};
    for (uint32_t i = gl; i < cnt; i += FF_LANES) list[base + before + i] = s_list[grp][i];
    float4* out = reinterpret_cast<float4*>(coef + (uint64_t)chunk * FF_COEF);
    float w[FF_COEF] = {f.c0, f.gx, f.gy, f.gz, f.hxx, f.hyy, f.hzz, f.hxy, f.hxz, f.hyz, f.kxxx + f.zx, f.kyyy + f.zy,
                        f.kzzz + f.zz, f.kxxy + f.zy, f.kxxz + f.zz, f.kxyy + f.zx, f.kyyz + f.zz, f.kxzz + f.zx,
                        f.kyzz + f.zy, f.kxyz, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 20; ++k) w[k] = ff_row_sum(w[k]);
    w[20] = ctr[0];
    w[21] = ctr[1];
    w[22] = ctr[2];
    if (gl == 0)
#pragma unroll
        for (int k = 0; k < FF_COEF / 4; ++k) out[k] = make_float4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
}

// the chunk's polynomial at voxel (vx, vy, vz)
__device__ inline float far_value(const float* __restrict__ w, int vx, int vy, int vz) {
    const float x = (float)vx - w[20], y = (float)vy - w[21], z = (float)vz - w[22];
    auto fma = [](float a, float b, float c) { return __builtin_fmaf(a, b, c); };
    const float px = fma(x, fma(x, w[10], fma(y, w[13], fma(z, w[14], w[4]))),
                         fma(y, fma(y, w[15], fma(z, w[19], w[7])), fma(z, fma(z, w[17], w[8]), w[1])));
    const float py = fma(y, fma(y, w[11], fma(z, w[16], w[5])), fma(z, fma(z, w[18], w[9]), w[2]));
    const float pz = fma(z, fma(z, w[12], w[6]), w[3]);
    return fma(x, px, fma(y, py, fma(z, pz, w[0])));
}

template <class Stack, bool COUNT>
__global__ __launch_bounds__(WN_BLOCK) void k_winding(const uint32_t* __restrict__ act, uint32_t n_act,
                                                      const int32_t* __restrict__ origins, float h,
                                                      const NodeRec* __restrict__ nodes, int n_nodes,
                                                      const float* __restrict__ btris, float thr, float fp64_band,
                                                      const FarChunk* __restrict__ chunks,
                                                      const uint32_t* __restrict__ list,
                                                      const float* __restrict__ coef, float* __restrict__ values,
                                                      uint32_t* __restrict__ recheck, unsigned long long* counters,
                                                      unsigned* err) {
    const int lane = threadIdx.x & 63;
    const uint32_t gid = xcd_workgroup(WN_CHUNK) * WN_BLOCK + threadIdx.x;
    const bool valid = gid < n_act;
    const uint32_t slot = valid ? act[gid] : 0u;
    const uint32_t leaf = slot >> 9, off = slot & 511u;
    int vx = 0, vy = 0, vz = 0;
    if (valid) {
        vx = origins[4 * leaf] + (int)(off >> 6);
        vy = origins[4 * leaf + 1] + (int)((off >> 3) & 7);
        vz = origins[4 * leaf + 2] + (int)(off & 7);
    }
    const float px = (float)vx * h, py = (float)vy * h, pz = (float)vz * h;
    const unsigned long long init = __ballot(valid);
    if (init == 0) return;
    WnAcc<COUNT> a;
    Stack stk;
    if constexpr (!std::is_same<Stack, LaneStack>::value) {
        __shared__ int4 lds_stack[WN_BLOCK / 64][LdsStack::DEPTH];
        stk.e = lds_stack[threadIdx.x >> 6];
    }
    __shared__ int2 leaf_queue[WN_BLOCK / 64][LeafQueue::CAP];
    __shared__ float leaf_sum[WN_BLOCK / 64][64];
    LeafQueue q;
    q.e = leaf_queue[threadIdx.x >> 6];
    q.sum = leaf_sum[threadIdx.x >> 6];
    q.sum[lane] = 0.0f;
    // the nodes to start from: the chunk's list, or the root (internal node 0, or
    // the only leaf when n == 1); 64 of them at a time, one per lane
    uint32_t start_off = 0, starts = 1;
    bool listed = false;
    if (chunks) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gid >> 6));
        const FarChunk fc = chunks[c];
        listed = fc.cnt != 0xFFFFFFFFu;
        if (listed) {
            start_off = fc.off;
            starts = fc.cnt;
            a.s = far_value(coef + (uint64_t)c * FF_COEF, vx, vy, vz);
        }
    }
    int ids = listed && (uint32_t)lane < starts ? (int)list[start_off + lane] : 0;
    uint32_t next = 0;
    int sp = 0;
    bool overflow = false;
    // the pair to visit next (wave-uniform); the first child pair of a visit
    // is taken here directly instead of through the stack, which only holds
    // the second ones: the visiting order is the same depth-first order
    int c0 = 0, c1 = 0;
    unsigned long long m = 0;
    bool have = false;
    // every sibling pair is visited at most once per wave in a tree: more
    // visits than nodes means corrupt links, and the walk stops
    for (int pops = 0;; ++pops) {
        unsigned long long m1 = m;
        if (!have) {
            if (sp > 0) {
                --sp;
                stk.pop(sp, c0, c1, m);
                m1 = m;
            } else {
                if (next >= starts) break;
                // two start nodes as one pair
                if (next && (next & 63) == 0) ids = next + lane < starts ? (int)list[start_off + next + lane] : 0;
                c0 = __builtin_amdgcn_readlane(ids, (int)(next & 63));
                c1 = __builtin_amdgcn_readlane(ids, (int)((next + 1) & 63));
                m = init;
                m1 = next + 1 < starts ? init : 0;
                next += 2;
            }
        }
        if (pops > n_nodes) {
            overflow = true;
            break;
        }
        const NodeRec r0 = nodes[c0];
        const NodeRec r1 = nodes[c1];
        pin_record(r0);
        pin_record(r1);
        const unsigned long long n0 = wn_visit(r0, m, px, py, pz, lane, q, a);
        const unsigned long long n1 = wn_visit(r1, m1, px, py, pz, lane, q, a);
        while (q.n >= LeafQueue::BATCH) wn_leaves(q, LeafQueue::BATCH, px, py, pz, lane, btris);
        if (sp + 1 > Stack::DEPTH) {
            overflow = true;
            break;
        }
        have = (n0 | n1) != 0;
        if (n0) {
            if (n1) stk.push(sp++, r1.L.x, r1.L.y, n1, lane);
            c0 = r0.L.x, c1 = r0.L.y, m = n0;
        } else if (n1) {
            c0 = r1.L.x, c1 = r1.L.y, m = n1;
        }
    }
    if (q.n > 0) wn_leaves(q, q.n, px, py, pz, lane, btris);
    if (overflow && lane == 0) atomicOr(err, E_STACK);
    if (COUNT && lane == 0) {
        atomicAdd(&counters[C_NEAR_INTERNAL], a.near_int);
        atomicAdd(&counters[C_FAR], a.far);
        atomicAdd(&counters[C_LEAF_VISITS], a.leaf);
        atomicAdd(&counters[C_LEAF_TRIS], a.tri);
    }
    if (!valid) return;
    const float w = a.s + q.sum[lane];
    float* vp = values + slot;
    const float d = *vp;
    *vp = (w < thr) ? copysignf(d, 1.0f) : copysignf(d, -1.0f);
    if (fabsf(w - thr) < fp64_band) {
        uint32_t k = (uint32_t)atomicAdd(&counters[C_RECHECK], 1ull);
        recheck[k] = slot;
    }
}

// FP64 re-evaluation of the voxels whose f32 winding number fell inside the
// ambiguity band around the threshold: same tree, every term in double.
__global__ void k_winding_fp64(const uint32_t* __restrict__ list, uint32_t n, const int32_t* __restrict__ origins, float h,
                               const NodeRec* __restrict__ nodes, int n_nodes, const float* __restrict__ btris,
                               float thr, float* __restrict__ values, unsigned* err) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t slot = list[i];
    const uint32_t leaf = slot >> 9, off = slot & 511u;
    const int vx = origins[4 * leaf] + (int)(off >> 6);
    const int vy = origins[4 * leaf + 1] + (int)((off >> 3) & 7);
    const int vz = origins[4 * leaf + 2] + (int)(off & 7);
    const double px = (float)vx * h, py = (float)vy * h, pz = (float)vz * h;
    int stack[WN_STACK];
    int sp = 0;
    stack[sp++] = 0;
    double w = 0.0;
    for (int pops = 0; sp > 0; ++pops) {
        if (pops > n_nodes) {
            atomicOr(err, E_STACK);
            return;
        }
        const int node = stack[--sp];
        const float4 A = nodes[node].A, B = nodes[node].B, C = nodes[node].C;
        const float2 D = nodes[node].D;
        const double rx = A.x - px, ry = A.y - py, rz = A.z - pz;
        const double r2 = rx * rx + ry * ry + rz * rz;
        if (r2 > (double)A.w) {  // coefficients carry 1/(4 pi) and 3/(4 pi) (acc_finalize)
            double inv_r = 1.0 / sqrt(r2), inv_r2 = inv_r * inv_r;
            double rsr = C.x * rx * rx + C.y * ry * ry + C.z * rz * rz + C.w * rx * ry + D.x * rx * rz + D.y * ry * rz;
            double lin = B.x * rx + B.y * ry + B.z * rz + B.w;
            w += inv_r * inv_r2 * (lin - rsr * inv_r2);
            continue;
        }
        const int2 L = nodes[node].L;
        if (L.y < 0) {
            double om = 0.0;
            for (int k = 0; k < -L.y; ++k) {
                const float* t = btris + 12 * (uint64_t)(L.x + k);
                om += solid_angle_rel64(t[0] - px, t[1] - py, t[2] - pz, t[3] - px, t[4] - py, t[5] - pz, t[6] - px,
                                        t[7] - py, t[8] - pz);
            }
            w += om / (4.0 * M_PI);
        } else {
            if (sp + 2 > WN_STACK) {
                atomicOr(err, E_STACK);
                return;
            }
            stack[sp++] = L.y;
            stack[sp++] = L.x;
        }
    }
    float* vp = values + slot;
    const float d = *vp;
    *vp = (w < (double)thr) ? copysignf(d, 1.0f) : copysignf(d, -1.0f);
}

// ---------------------------------------------------------------------------
// Shared signs.  For face neighbours v, u of one leaf with |d_v| + |d_u| > thr
// (thr bounds the sample spacing plus the distance and sub-triangle rounding),
// no point of the surface lies on the segment between them: a crossing point s
// would give |d_v| + |d_u| <= |v - s| + |s - u| = |v - u|.  A closed mesh's
// winding number is constant off the surface, so such voxels share their sign.
// Each leaf's voxels are grouped by a union-find over those links; the root of
// a group is its smallest offset (a larger root is always hooked under a
// smaller one), its winding number is evaluated and its sign is copied to the
// group.  Groups never span leaves.

// the group roots of every leaf, slot = leaf * 512 + offset, in offset order
// One wave per listed leaf: wave b lists the group roots of leaf perm[b] (b
// when perm is null) at rep_off[b], in voxel order.
__global__ __launch_bounds__(AL_BLOCK) void k_sign_reps(const uint16_t* __restrict__ roots,
                                                        const uint32_t* __restrict__ perm,
                                                        const uint32_t* __restrict__ rep_off, uint64_t n_leaves,
                                                        uint32_t* __restrict__ reps) {
    const uint64_t b = (uint64_t)blockIdx.x * (AL_BLOCK / 64) + (threadIdx.x >> 6);
    if (b >= n_leaves) return;
    const int lane = threadIdx.x & 63;
    const uint32_t leaf = perm ? perm[b] : (uint32_t)b;
    const uint16_t* rt = roots + (uint64_t)leaf * LEAF_VOX;
    uint32_t pos = rep_off[b];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int v = (c << 6) | lane;
        const bool rep = rt[v] == (uint16_t)v;
        const unsigned long long bl = __ballot(rep);
        if (rep) reps[pos + __popcll(bl & ((1ull << lane) - 1))] = leaf * 512u + (uint32_t)v;
        pos += (uint32_t)__popcll(bl);
    }
}

// out[i] = in[perm[i]]
__global__ void k_gather_u32(const uint32_t* __restrict__ in, const uint32_t* __restrict__ perm, uint64_t n,
                             uint32_t* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[perm[i]];
}

// every non-root voxel takes the sign of its (already signed) root
__global__ __launch_bounds__(512) void k_sign_broadcast(const uint16_t* __restrict__ roots, float* __restrict__ values) {
    const uint64_t leaf = blockIdx.x;
    const int v = threadIdx.x;
    const uint16_t r = roots[leaf * LEAF_VOX + v];
    if (r == (uint16_t)0xFFFF || r == (uint16_t)v) return;
    float* vp = values + leaf * LEAF_VOX;
    vp[v] = copysignf(vp[v], vp[r]);
}

// ---------------------------------------------------------------------------
// host driver

template <class T>
T read_scalar(bs_ctx* ctx, const T* dptr) {
    T v;
    BS_HIP(hipMemcpyAsync(&v, dptr, sizeof(T), hipMemcpyDeviceToHost, ctx->stream));
    BS_HIP(hipStreamSynchronize(ctx->stream));
    return v;
}

// Several device scalars back in one round trip: asynchronous copies into the
// context's pinned buffer (words [320, 512); the side stream's BVH readback
// uses [0, 259)), one synchronisation of the main stream, then a host copy.
class Readback {
    bs_ctx* ctx_;
    uint8_t* base_;
    struct Item {
        size_t off, size;
        void* dst;
    };
    Item items_[8];
    int n_ = 0;
    size_t used_ = 0;

public:
    static constexpr size_t BYTES = 4 * (512 - 320);
    explicit Readback(bs_ctx* c) : ctx_(c), base_(reinterpret_cast<uint8_t*>(c->host_pinned + 320)) {}
    template <class T>
    void add(const T* dptr, T* host, size_t count = 1) {
        const size_t off = (used_ + 7) & ~size_t(7), bytes = sizeof(T) * count;
        if (n_ == 8 || off + bytes > BYTES) throw Error(BS_ERR_INTERNAL, "readback batch too large");
        BS_HIP(hipMemcpyAsync(base_ + off, dptr, bytes, hipMemcpyDeviceToHost, ctx_->stream));
        items_[n_++] = {off, bytes, host};
        used_ = off + bytes;
    }
    void wait() {
        BS_HIP(hipStreamSynchronize(ctx_->stream));
        for (int i = 0; i < n_; ++i) std::memcpy(items_[i].dst, base_ + items_[i].off, items_[i].size);
        n_ = 0;
        used_ = 0;
    }
};

template <class TIn, class TOut>
void exclusive_scan(bs_ctx* ctx, const TIn* in, TOut* out, uint64_t n) {
    BS_REQUIRE(n < (1ull << 31), BS_ERR_INVALID_ARG, "scan longer than 2^31 elements");
    size_t bytes = 0;
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, ctx->stream));
    void* tmp = ctx->scratch.get(S_CUB, bytes);
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, (int)n, ctx->stream));
}

template <class K, class V>
void sort_pairs_on(bs_ctx* ctx, hipStream_t stream, int cub_slot, const K* k, K* ks, const V* v, V* vs, uint64_t n,
                   int end_bit) {
    BS_REQUIRE(n < (1ull << 31), BS_ERR_INVALID_ARG, "sort longer than 2^31 elements");
    size_t bytes = 0;
    BS_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k, ks, v, vs, (int)n, 0, end_bit, stream));
    void* tmp = ctx->scratch.get(cub_slot, bytes);
    BS_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, bytes, k, ks, v, vs, (int)n, 0, end_bit, stream));
}

template <class K, class V>
void sort_pairs(bs_ctx* ctx, const K* k, K* ks, const V* v, V* vs, uint64_t n, int end_bit) {
    sort_pairs_on(ctx, ctx->stream, S_CUB, k, ks, v, vs, n, end_bit);
}

// The context's second stream, its fork/join events and pinned readback
// buffer, created on first use.
void ensure_side_stream(bs_ctx* ctx) {
    if (!ctx->stream2) BS_HIP(hipStreamCreateWithFlags(&ctx->stream2, hipStreamNonBlocking));
    if (!ctx->ev_fork) BS_HIP(hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming));
    if (!ctx->ev_join) BS_HIP(hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming));
    if (!ctx->ev_leaves) BS_HIP(hipEventCreateWithFlags(&ctx->ev_leaves, hipEventDisableTiming));
    if (!ctx->host_pinned) BS_HIP(hipHostMalloc((void**)&ctx->host_pinned, sizeof(uint32_t) * 512, hipHostMallocDefault));
}

// Waits for the second stream when a call leaves early, so that no kernel of
// it still uses the scratch arena afterwards.
struct SideJoin {
    hipStream_t s;
    ~SideJoin() { (void)hipStreamSynchronize(s); }
};

template <class It, class Out, class Pred>
void select_if(bs_ctx* ctx, It in, Out out, uint32_t* d_count, uint64_t n, Pred pred) {
    BS_REQUIRE(n < (1ull << 31), BS_ERR_INVALID_ARG, "selection over more than 2^31 elements");
    size_t bytes = 0;
    BS_HIP(hipcub::DeviceSelect::If(nullptr, bytes, in, out, d_count, (int)n, pred, ctx->stream));
    void* tmp = ctx->scratch.get(S_CUB, bytes);
    BS_HIP(hipcub::DeviceSelect::If(tmp, bytes, in, out, d_count, (int)n, pred, ctx->stream));
}

int bits_for(uint64_t v) {
    int b = 1;
    while ((1ull << b) <= v) ++b;
    return b;
}

struct PhaseTimer {
    bs_ctx* ctx;
    hipEvent_t ev[8];
    int n = 0;
    explicit PhaseTimer(bs_ctx* c) : ctx(c) {
        if (ctx->profiling)
            for (auto& e : ev) BS_HIP(hipEventCreate(&e));
    }
    ~PhaseTimer() {
        if (ctx->profiling)
            for (auto& e : ev) (void)hipEventDestroy(e);
    }
    void mark() {
        if (ctx->profiling && n < 8) BS_HIP(hipEventRecord(ev[n++], ctx->stream));
    }
    double ms(int a, int b) {
        if (!ctx->profiling || b >= n) return 0.0;
        float f = 0;
        BS_HIP(hipEventSynchronize(ev[b]));
        BS_HIP(hipEventElapsedTime(&f, ev[a], ev[b]));
        return f;
    }
};

uint32_t next_pow2(uint64_t v) {
    uint64_t p = 1024;
    while (p < v) p <<= 1;
    if (p > (1ull << 31)) throw Error(BS_ERR_INVALID_ARG, "leaf hash table would exceed 2^31 slots");
    return (uint32_t)p;
}

// Least distance, in radii of the chunk, of a node whose term is expanded about
// the chunk's centre.  The expansion cuts off terms of (1 / kappa)^4, the order-2
// term of a node at the traversal's limit those of (1 / accuracy)^2: the limit
// grows with the square root of the accuracy.  A lower kappa takes more, and
// smaller, nodes into the polynomial, which lowers the whole error: against
// exact sums in 64 bits (rms over 600 voxels, eight meshes) 1.2e-2 to 2.6e-2 at 2
// and 1.2e-2 to 2.9e-2 at 5, where the walk from the root has 1.4e-2 to 3.1e-2;
// both kernels take 7.8 ms at 2, 8.7 at 3 and 9.3 at 4 (42 M voxels).
//
// How far a voxel's sum is then from the walk's depends on which voxels share its
// chunk.  Voxels within fp64_band of the threshold take the FP64 walk's sign
// whatever their sum, so a band above that difference leaves every sign the
// walk's.  On eight open meshes and soups, three grids each, seven thresholds, no
// sign differed with the default band at accuracies of 2, 3 and 4, nor with one of
// 0.05; without one up to 23,321 did, over the thresholds, on 478,748 voxels; at
// accuracy 1, where terms are taken a node's radius from the node, some still did
// with 0.3.  So the far field is for the default accuracy
// and band upwards; below either, every voxel walks from the root.
//
// Upwards to an accuracy of 4: the lists grow with its square, and from 5 on most
// chunks have none and their time is lost.  Conversions of 42 M, 3.5 M, 14 M and
// 0.7 M voxels with and without: 19.0 / 26.6, 2.7 / 3.2, 6.3 / 8.2 and 1.08 / 1.08 ms
// at 2, 54 / 60, 5.1 / 6.1, 11.6 / 15.8 and 1.69 / 1.61 at 4, 83 / 83, 7.9 / 8.1,
// 22.3 / 21.1 and 2.08 / 1.90 at 5, 115 / 110, 10.9 / 10.4, 27.8 / 26.9 and 2.43 / 2.28
// at 6.
constexpr float WN_FAR_BAND = 0.1f, WN_FAR_ACCURACY = 2.0f, WN_FAR_ACCURACY_MAX = 4.0f;
float wn_kappa(float accuracy) { return sqrtf(2.0f * accuracy); }

}  // namespace

// Dense leaf grids up to this many cells (4 B each); larger extents hash.
constexpr uint64_t DENSE_LEAF_GRID_MAX = 1ull << 28;
// volumes of at least this many leaves list their active voxels in the leaves'
// Z order for the winding-number pass (smaller ones keep the leaf order)
constexpr uint64_t LEAF_Z_MIN = 4096;

void mesh_to_volume_device(bs_ctx* ctx, const float* d_tris, uint64_t n, const bs_m2v_params& prm, bs_volume** out) {
    *out = nullptr;
    BS_REQUIRE(prm.voxel_size > 0.0f && std::isfinite(prm.voxel_size), BS_ERR_INVALID_ARG, "voxel_size must be > 0");
    BS_REQUIRE(prm.band >= 0 && prm.band < (1 << 20), BS_ERR_INVALID_ARG, "band must be in [0, 2^20)");
    BS_REQUIRE(prm.sign_mode == BS_SIGN_PER_VOXEL || prm.sign_mode == BS_SIGN_SHARED ||
                   prm.sign_mode == BS_SIGN_SURROGATE,
               BS_ERR_INVALID_ARG, "sign_mode must be BS_SIGN_PER_VOXEL, BS_SIGN_SHARED or BS_SIGN_SURROGATE");
    if (n == 0) throw Error(BS_ERR_EMPTY, "empty mesh: the reference returns None");
    BS_REQUIRE(n < (1ull << 30), BS_ERR_INVALID_ARG, "more than 2^30 triangles");
    hipStream_t st = ctx->stream;
    auto& S = ctx->scratch;
    const float h = prm.voxel_size;
    const float inv_h = 1.0f / h;  // MeshToVolume::set_voxel_size (mesh_to_volume.rs:48)
    const int band = (int)prm.band;
    PhaseTimer tm(ctx);
    auto wall0 = std::chrono::steady_clock::now();
    tm.mark();

    unsigned long long* counters = S.as<unsigned long long>(S_COUNTERS, C_COUNT);
    unsigned* err = reinterpret_cast<unsigned*>(S.get(S_MISC3, 64));
    BS_HIP(hipMemsetAsync(counters, 0, sizeof(unsigned long long) * C_COUNT, st));
    BS_HIP(hipMemsetAsync(err, 0, 64, st));
    const unsigned TB = 256;

    // ---- 0. LBVH + dipoles over the original mesh, on the second stream: it
    // needs only the triangles, so it is built beside the subdivision, leaf
    // allocation and distance passes; the winding pass waits for it
    ensure_side_stream(ctx);
    hipStream_t sb = ctx->stream2;
    BS_HIP(hipEventRecord(ctx->ev_fork, st));
    BS_HIP(hipStreamWaitEvent(sb, ctx->ev_fork, 0));
    SideJoin side_join{sb};
    const int nt = (int)n;
    const int n_int = nt - 1;
    int H = 0;  // tree height (root level)
    bool use_lds = false;
    const int n_nodes = 2 * nt - 1;
    // large meshes: the top-down binned tree (the clustered one when asked),
    // whose few dozen launches pay off where the winding pass is long, laid out
    // depth-first; smaller ones or BS_PATH_LBVH: the Morton split (2 * id must
    // fit an int)
    const bool big = !(ctx->paths & BS_PATH_LBVH) && n >= PLOC_MIN_TRIS && n < (1ull << 28);
    const bool ploc = big && (ctx->paths & BS_PATH_PLOC);
    const bool topdown = big && !ploc;
    const bool dfs = ploc || topdown;
    const int n_rec = dfs ? 2 * nt : n_nodes;  // records of the traversal layout
    int ploc_iters = 0;  // clustering iterations or top-down levels
    unsigned* bounds = reinterpret_cast<unsigned*>(S.get(S_BVH_MISC, 64));
    const unsigned nb = div_up(n, 256);
    uint4* bparts = S.as<uint4>(S_BVH_BOX, 2 * (uint64_t)nb);
    const uint64_t n_mort = topdown ? 1 : n;  // the top-down build needs no Morton order
    uint64_t* codes = S.as<uint64_t>(S_MORTON, n_mort);
    uint64_t* codes_s = S.as<uint64_t>(S_MORTON_SORTED, n_mort);
    uint32_t* idx = S.as<uint32_t>(S_IDX, n_mort);
    uint32_t* idx_s = S.as<uint32_t>(S_IDX_SORTED, n);  // the triangle order of the tree
    // Morton split: parent links, height words and the height sort; top-down
    // build: node depths (in `height`) and the nodes grouped by depth (inode_s)
    const int n_lb = dfs ? 1 : std::max(n_int, 1);
    const int n_td = topdown ? std::max(n_int, 1) : n_lb;
    int* parent = S.as<int>(S_BVH_PARENT, dfs ? 1 : n_nodes);
    unsigned* hword = S.as<unsigned>(S_BVH_FLAGS, n_lb);
    uint32_t* height = S.as<uint32_t>(S_BVH_HEIGHT, n_td);
    uint32_t* height_s = S.as<uint32_t>(S_BVH_HEIGHT_S, n_lb);
    uint32_t* inode = S.as<uint32_t>(S_BVH_INODE, n_lb);
    uint32_t* inode_s = S.as<uint32_t>(S_BVH_INODE_S, n_td);
    NodeAcc* accs = S.as<NodeAcc>(S_BVH_INIT, n_nodes);
    NodeRec* nodes = S.as<NodeRec>(S_BVH_NODES, (uint64_t)n_rec);
    float* btris = S.as<float>(S_BVH_TRIS, 12 * (n + BVH_LEAF_SIZE));  // padded: leaves read BVH_LEAF_SIZE triangles
    int2* kids = S.as<int2>(S_BVH_KIDS, std::max(n_int, 1));  // binary children of internal nodes
    uint32_t* starts = reinterpret_cast<uint32_t*>(S.get(S_BVH_STARTS, sizeof(uint32_t) * 258));
    // Morton order, binary tree, leaves and the height grouping run while the
    // host drives the subdivision and leaf allocation below (mostly scalar
    // readbacks, so the device is largely idle there); only the per-level
    // combination, which needs the level starts on the host, waits for the
    // distance launch
    k_centroid_bounds<<<nb, 256, 0, sb>>>(d_tris, n, bparts);
    k_bounds_final<<<1, 1024, 0, sb>>>(bparts, nb, bounds);
    if (!topdown) {
        k_morton<<<div_up(n, TB), TB, 0, sb>>>(d_tris, n, bounds, codes, idx);
        sort_pairs_on(ctx, sb, S_CUB_B, codes, codes_s, idx, idx_s, n, 63);
    }
    uint32_t* hs = ctx->host_pinned;  // level starts [0, 258) (clustered: count ring, root, height), error word
    // clustered build: the iterations the common case needs run here without
    // a host round trip; the count is read back after the distance launch
    float4* pbox = nullptr;
    PlocInfo* pinfo = nullptr;
    int *cl0 = nullptr, *cl1 = nullptr, *pnn = nullptr;
    uint32_t *keep = nullptr, *kpos = nullptr, *ring = nullptr;
    void* scan_tmp = nullptr;
    size_t scan_bytes = 0;
    float4* td_prims = nullptr;
    TdNode* td_fr = nullptr;
    uint32_t *td_bins = nullptr, *td_tcnt = nullptr, *td_ctr = nullptr;
    int2* td_tasks = nullptr;
    TdSplit* td_split = nullptr;
    TdSmall* td_small = nullptr;
    uint32_t* td_hist = nullptr;
    uint8_t* td_depth = nullptr;
    int td_fr_cap = 0, td_task_cap = 0, td_small_cap = 0;
    // one level of the top-down build: triangles in buffer l & 1, lists l & 1
    auto td_level = [&](int l) {
        const int in = l & 1, out = in ^ 1;
        const uint64_t pw = 2 * (uint64_t)n, bw = (uint64_t)td_fr_cap * TD_NODE_WORDS;
        // level l holds at most 2^l nodes: grids sized to that, looping past TD_GRID_MAX blocks
        const uint64_t reach = l < 40 ? (1ull << l) : ~0ull;
        const uint64_t nfr = std::min<uint64_t>(reach, (uint64_t)td_fr_cap);
        const unsigned g_task = (unsigned)std::min<uint64_t>(
            {(uint64_t)td_task_cap, n / TD_CHUNK + nfr + 1, (uint64_t)TD_GRID_MAX});
        const unsigned g_sel = (unsigned)std::min<uint64_t>(div_up(nfr, TD_BLOCK / 64), TD_GRID_MAX);
        const int2* tin = td_tasks + (uint64_t)in * td_task_cap;
        int2* tout = td_tasks + (uint64_t)out * td_task_cap;
        k_td_bin<<<g_task, TD_BLOCK, 0, sb>>>(td_prims + in * pw, td_fr + (uint64_t)in * td_fr_cap, tin, td_ctr, in,
                                              td_bins + in * bw, td_tcnt);
        k_td_select<<<g_sel, TD_BLOCK, 0, sb>>>(td_fr + (uint64_t)in * td_fr_cap, td_ctr, in, td_bins + in * bw, nt,
                                                td_fr_cap, td_small_cap, td_task_cap, td_split,
                                                td_fr + (uint64_t)out * td_fr_cap, td_bins + out * bw, tout, td_small,
                                                pinfo, kids, td_depth, err);
        k_td_partition<<<g_task, TD_BLOCK, 0, sb>>>(td_prims + in * pw, td_prims + out * pw,
                                                    td_fr + (uint64_t)in * td_fr_cap, tin, td_ctr, in, td_split,
                                                    td_tcnt, td_fr + (uint64_t)out * td_fr_cap, idx_s, err);
    };
    auto ploc_iteration = [&](int it) {
        const uint32_t* cnt = ring + (it & 1);
        int* cin = (it & 1) ? cl1 : cl0;
        int* cout = (it & 1) ? cl0 : cl1;
        k_ploc_nn<<<div_up(n, PLOC_BLOCK), PLOC_BLOCK, 0, sb>>>(cin, pbox, cnt, pnn);
        k_ploc_merge<<<div_up(n, TB), TB, 0, sb>>>(cin, pnn, cnt, nt, keep, ring + 2, accs, pbox,
                                                    pinfo, kids);
        BS_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp, scan_bytes, keep, kpos, nt + 1, sb));
        k_ploc_compact<<<div_up(n, TB), TB, 0, sb>>>(cin, keep, kpos, cnt, nt, ring + ((it + 1) & 1), cout);
    };
    auto ploc_result = [&](int iters) {
        k_ploc_root<<<1, 1, 0, sb>>>((iters & 1) ? cl1 : cl0, pinfo, ring + 3);
        BS_HIP(hipMemcpyAsync(hs, ring, sizeof(uint32_t) * 5, hipMemcpyDeviceToHost, sb));
        BS_HIP(hipMemcpyAsync(hs + 258, err, sizeof(uint32_t), hipMemcpyDeviceToHost, sb));
    };
    if (ploc) {
        // buffers now; the launches follow the distance launch (below), so the
        // host enqueues the subdivision and leaf passes without waiting behind them
        pbox = S.as<float4>(S_PLOC_BOX, 2 * (uint64_t)n_nodes);
        pinfo = S.as<PlocInfo>(S_PLOC_INFO, n_nodes);
        cl0 = S.as<int>(S_PLOC_C0, n);
        cl1 = S.as<int>(S_PLOC_C1, n);
        pnn = S.as<int>(S_PLOC_NN, n);
        keep = S.as<uint32_t>(S_PLOC_KEEP, n + 1);
        kpos = S.as<uint32_t>(S_PLOC_POS, n + 1);
        ring = S.as<uint32_t>(S_PLOC_RING, 8);
        BS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, keep, kpos, nt + 1, sb));
        scan_tmp = S.get(S_CUB_B, scan_bytes);
    } else if (topdown) {
        td_fr_cap = nt / TD_SMALL + 2;
        td_task_cap = nt / TD_CHUNK + td_fr_cap + 1;
        td_small_cap = nt / 2 + 1;
        td_prims = S.as<float4>(S_TD_PRIMS, 4 * (uint64_t)n);  // two buffers of two float4 per triangle
        td_fr = S.as<TdNode>(S_TD_FR, 2 * (uint64_t)td_fr_cap);
        td_bins = S.as<uint32_t>(S_TD_BINS, 2 * (uint64_t)td_fr_cap * TD_NODE_WORDS);
        td_tasks = S.as<int2>(S_TD_TASKS, 2 * (uint64_t)td_task_cap);  // the task lists of two levels
        td_tcnt = S.as<uint32_t>(S_TD_TCNT, (uint64_t)td_task_cap * 3 * TD_BINS);
        td_split = S.as<TdSplit>(S_TD_SPLIT, (uint64_t)td_fr_cap);
        td_small = S.as<TdSmall>(S_TD_SMALL, (uint64_t)td_small_cap);
        td_ctr = S.as<uint32_t>(S_PLOC_RING, TD_C_WORDS);
        td_hist = S.as<uint32_t>(S_TD_HIST, 1024);
        td_depth = reinterpret_cast<uint8_t*>(height);  // one byte per internal node
        pinfo = S.as<PlocInfo>(S_PLOC_INFO, n_nodes);
        // the level passes follow the distance launch (below) and run beside
        // the candidate sort and the distance pass: run in the subdivision and
        // leaf passes instead, between the host's readbacks, they lengthened
        // that part by more than they slow the distance pass.  A balanced cut
        // halves a node: log2(n / TD_SMALL) levels, a few more for uneven cuts;
        // levels past the last large node cost a few empty launches
        k_td_init<<<div_up(n, TB), TB, 0, sb>>>(d_tris, nt, bounds, td_prims, td_fr, td_tasks, td_bins, td_ctr, pinfo,
                                                td_depth, td_hist);
        ploc_iters = (int)std::ceil(std::log2((double)n / TD_SMALL)) + 4;
    } else {
        BS_HIP(hipMemsetAsync(parent, 0xFF, sizeof(int) * n_nodes, sb));
        BS_HIP(hipMemsetAsync(hword, 0, sizeof(unsigned) * std::max(n_int, 1), sb));
        if (n_int > 0) k_lbvh_build<<<div_up(n_int, TB), TB, 0, sb>>>(codes_s, nt, nodes, kids, parent);
        k_lbvh_leaves<<<div_up(n, TB), TB, 0, sb>>>(d_tris, nt, idx_s, prm.wn_accuracy, parent, hword, height, accs,
                                                    nodes, btris, err);
    }
    if (!dfs && n_int > 0) {
        // internal nodes grouped by height; combined level by level further down
        k_iota<<<div_up(n_int, TB), TB, 0, sb>>>(inode, (uint32_t)n_int);
        sort_pairs_on(ctx, sb, S_CUB_B, height, height_s, inode, inode_s, (uint64_t)n_int, 8);
        BS_HIP(hipMemsetAsync(starts, 0xFF, sizeof(uint32_t) * 258, sb));
        k_level_starts<<<div_up(n_int, TB), TB, 0, sb>>>(height_s, (uint32_t)n_int, starts);
        BS_HIP(hipMemcpyAsync(hs, starts, sizeof(uint32_t) * 258, hipMemcpyDeviceToHost, sb));
        BS_HIP(hipMemcpyAsync(hs + 258, err, sizeof(uint32_t), hipMemcpyDeviceToHost, sb));
    }

    // ---- 1. subdivision
    uint32_t* rows = S.as<uint32_t>(S_ROWS, n + 1);
    uint64_t* subs = S.as<uint64_t>(S_SUBS, n + 1);
    uint32_t* row_off = S.as<uint32_t>(S_ROW_OFF, n + 1);
    uint64_t* sub_off = S.as<uint64_t>(S_SUB_OFF, n + 1);
    BS_HIP(hipMemsetAsync(rows + n, 0, sizeof(uint32_t), st));
    BS_HIP(hipMemsetAsync(subs + n, 0, sizeof(uint64_t), st));
    k_subdiv_count<<<div_up(n, TB), TB, 0, st>>>(d_tris, n, h, rows, subs, err);
    exclusive_scan(ctx, rows, row_off, n + 1);
    exclusive_scan(ctx, subs, sub_off, n + 1);
    const bool shared_signs = prm.sign_mode == BS_SIGN_SHARED;
    const bool surrogate_signs = prm.sign_mode == BS_SIGN_SURROGATE;
    uint32_t max_rows = 1;  // largest subdivision count: bounds the sub-triangle rounding
    uint32_t* d_max = nullptr;
    if (shared_signs || surrogate_signs) {
        d_max = reinterpret_cast<uint32_t*>(S.get(S_MISC2, 64));
        size_t bytes = 0;
        BS_HIP(hipcub::DeviceReduce::Max(nullptr, bytes, rows, d_max, (int)n, st));
        void* tmp = S.get(S_CUB, bytes);
        BS_HIP(hipcub::DeviceReduce::Max(tmp, bytes, rows, d_max, (int)n, st));
    }
    Readback rb(ctx);
    uint32_t h_max_rows = 1, h_rows = 0, h_err = 0;
    uint64_t n_sub = 0;
    if (d_max) rb.add(d_max, &h_max_rows);
    rb.add(row_off + n, &h_rows);
    rb.add(sub_off + n, &n_sub);
    rb.add(err, &h_err);
    rb.wait();
    max_rows = std::max<uint32_t>(1u, h_max_rows);
    const uint64_t total_rows = h_rows;
    if (h_err & E_TOO_MANY_SUBS)
        throw Error(BS_ERR_INVALID_ARG, "a triangle is subdivided into more than 2^32 sub-triangles");
    if (n_sub == 0) throw Error(BS_ERR_EMPTY, "no sub-triangles: the reference returns None");
    BS_REQUIRE(n_sub < (1ull << 31) - 1, BS_ERR_INVALID_ARG, "more than 2^31 sub-triangles");
    float* sub = S.as<float>(S_SUBTRIS, 9 * n_sub);
    k_subdiv_emit<<<div_up(total_rows, TB), TB, 0, st>>>(d_tris, n, h, row_off, sub_off, total_rows, sub);
    tm.mark();

    // ---- 2. boxes, records, leaf allocation, candidate lists
    DistRec* recs = S.as<DistRec>(S_RECS, n_sub);
    uint32_t* cov = S.as<uint32_t>(S_LEAFCNT, n_sub + 1);
    uint32_t* cov_off = S.as<uint32_t>(S_LEAFOFF, n_sub + 1);
    const unsigned setup_blocks = div_up(n_sub, SETUP_BLOCK);
    Partial* partials = S.as<Partial>(S_MISC0, setup_blocks);
    BS_HIP(hipMemsetAsync(cov + n_sub, 0, sizeof(uint32_t), st));
    k_subtri_setup<<<setup_blocks, SETUP_BLOCK, 0, st>>>(sub, n_sub, inv_h, band, recs, cov, partials, err);
    k_reduce_partials<<<1, 1024, 0, st>>>(partials, setup_blocks, counters);
    exclusive_scan(ctx, cov, cov_off, n_sub + 1);
    unsigned long long hc[C_COUNT];
    uint32_t h_cov = 0;
    rb.add(counters, hc, C_COUNT);
    rb.add(cov_off + n_sub, &h_cov);
    rb.add(err, &h_err);
    rb.wait();
    const uint64_t n_cov = h_cov;
    if (h_err & E_RANGE)
        throw Error(BS_ERR_INVALID_ARG, "mesh extent exceeds 8e6 voxels from the origin");
    BS_REQUIRE(n_cov < (1ull << 31), BS_ERR_INVALID_ARG, "more than 2^31 box/leaf overlaps");
    const uint64_t n_pairs = hc[C_PAIRS];
    LeafIndex ix;
    long long glo[3], ghi[3];
    uint64_t bbox_leaves = 1;
    for (int k = 0; k < 3; ++k) {
        glo[k] = (long long)hc[C_BOX_LO + k] >> 3;
        ghi[k] = (long long)hc[C_BOX_HI + k] >> 3;
        bbox_leaves *= (uint64_t)(ghi[k] - glo[k] + 1);
        if (bbox_leaves > (1ull << 40)) bbox_leaves = 1ull << 40;
    }
    ix.dense = bbox_leaves <= DENSE_LEAF_GRID_MAX && !(ctx->paths & BS_PATH_FORCE_HASH);
    uint32_t* leaf_idx = nullptr;
    uint64_t* hkeys_sorted = nullptr;
    uint32_t* d_count = reinterpret_cast<uint32_t*>(S.get(S_MISC1, 64));
    if (ix.dense) {
        ix.gx0 = (int)glo[0];
        ix.gy0 = (int)glo[1];
        ix.gz0 = (int)glo[2];
        ix.gny = (int)(ghi[1] - glo[1] + 1);
        ix.gnz = (int)(ghi[2] - glo[2] + 1);
        ix.gsize = bbox_leaves;
        ix.grid = S.as<uint32_t>(S_HASH_VALS, bbox_leaves);
        BS_HIP(hipMemsetAsync(ix.grid, 0, sizeof(uint32_t) * bbox_leaves, st));
        k_leaf_mark<<<div_up(n_sub, TB), TB, 0, st>>>(recs, n_sub, ix, err);
        leaf_idx = S.as<uint32_t>(S_KEYS, std::min<uint64_t>(n_cov, bbox_leaves));
        select_if(ctx, hipcub::CountingInputIterator<uint32_t>(0), leaf_idx, d_count, bbox_leaves,
                  DenseOccupied{ix.grid});
    } else {
        uint32_t cap = next_pow2(2 * std::min<uint64_t>(n_cov, bbox_leaves));
        ix.cap_mask = cap - 1;
        ix.hkeys = S.as<uint64_t>(S_HASH_KEYS, cap);
        ix.hvals = S.as<uint32_t>(S_HASH_VALS, cap);
        BS_HIP(hipMemsetAsync(ix.hkeys, 0xFF, sizeof(uint64_t) * cap, st));
        k_leaf_mark<<<div_up(n_sub, TB), TB, 0, st>>>(recs, n_sub, ix, err);
        uint64_t* keys = S.as<uint64_t>(S_KEYS, std::min<uint64_t>(n_cov, cap));
        select_if(ctx, ix.hkeys, keys, d_count, cap, HashOccupied{});
        const uint32_t nl = read_scalar(ctx, d_count);
        hkeys_sorted = S.as<uint64_t>(S_KEYS_SORTED, nl);
        size_t bytes = 0;
        BS_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, bytes, keys, hkeys_sorted, (int)nl, 0, 63, st));
        void* tmp = S.get(S_CUB, bytes);
        BS_HIP(hipcub::DeviceRadixSort::SortKeys(tmp, bytes, keys, hkeys_sorted, (int)nl, 0, 63, st));
    }
    uint32_t h_leaves = 0;
    rb.add(d_count, &h_leaves);
    rb.add(err, &h_err);
    rb.wait();
    const uint64_t n_leaves = h_leaves;
    if (h_err & E_HASH) throw Error(BS_ERR_INTERNAL, "leaf hash table overflow");
    // output volume
    auto* vol = new bs_volume();
    vol->device = ctx->device;
    vol->voxel_size = h;
    vol->n_leaves = n_leaves;
    // on failure both streams may still run kernels on the volume's arrays
    struct Release {
        hipStream_t a, b;
        void operator()(bs_volume* v) const {
            if (b) (void)hipStreamSynchronize(b);
            free_leaves(v, a);
            delete v;
        }
    };
    std::unique_ptr<bs_volume, Release> guard(vol, Release{st, ctx->stream2});
    alloc_leaves(vol, n_leaves);
    if (ix.dense)
        k_leaf_assign_dense<<<div_up(n_leaves, TB), TB, 0, st>>>(leaf_idx, n_leaves, ix, vol->origins);
    else
        k_leaf_assign_hash<<<div_up(n_leaves, TB), TB, 0, st>>>(hkeys_sorted, n_leaves, ix, vol->origins, err);
    // the winding-number list takes the leaves in Z order (sorted on the
    // second stream once the origins are written)
    const bool leaf_z = n_leaves >= LEAF_Z_MIN;
    if (leaf_z) BS_HIP(hipEventRecord(ctx->ev_leaves, st));
    // candidate lists
    uint32_t* ckeys = S.as<uint32_t>(S_CAND_LEAF, n_cov);
    uint32_t* cvals = S.as<uint32_t>(S_CAND_CNT, n_cov);
    uint32_t* ckeys_s = S.as<uint32_t>(S_CURSOR, n_cov);
    uint32_t* cand_list = S.as<uint32_t>(S_CAND_LIST, n_cov);
    uint32_t* cand_off = S.as<uint32_t>(S_CAND_OFF, n_leaves + 1);
    k_cand_pairs<<<div_up(n_sub, CP_BLOCK), CP_BLOCK, 0, st>>>(recs, n_sub, cov_off, ix, (uint32_t)n_leaves, ckeys,
                                                              cvals, err);
    sort_pairs(ctx, ckeys, ckeys_s, cvals, cand_list, n_cov, bits_for(n_leaves));
    k_cand_offsets<<<div_up(n_leaves + 1, TB), TB, 0, st>>>(ckeys_s, (uint32_t)n_cov, (uint32_t)n_leaves, cand_off);
    // a failed lookup (E_HASH) is reported with the other error bits at the
    // end: its pairs sort past every list and its leaf's list is empty, so
    // the passes below never read them
    tm.mark();

    // ---- 3. distance
    // shared signs: the link threshold and the group buffers, filled by the distance pass
    uint16_t* roots = nullptr;
    uint32_t* rep_cnt = nullptr;
    float group_thr = 0.0f;
    if (shared_signs || surrogate_signs) {
        double maxc = 0.0;
        for (int k = 0; k < 3; ++k)
            maxc = std::max({maxc, std::fabs((double)(long long)hc[C_BOX_LO + k]),
                             std::fabs((double)(long long)hc[C_BOX_HI + k])});
        maxc = (maxc + 1.0) * (double)h;
        // sample spacing, sub-triangle vertex drift (two roundings per
        // accumulation step) and distance rounding, each bounded in ulps of
        // the largest coordinate
        const double ulp = maxc * 0x1p-23;
        group_thr = (float)((double)h * (1.0 + 0x1p-10) + (4.0 * max_rows + 200.0) * ulp);
        roots = S.as<uint16_t>(S_SIGN_ROOTS, n_leaves * LEAF_VOX);
        rep_cnt = S.as<uint32_t>(S_REP_CNT, n_leaves + 1);
        BS_HIP(hipMemsetAsync(rep_cnt + n_leaves, 0, sizeof(uint32_t), st));
    }
    if (shared_signs) {
        k_distance<true><<<(unsigned)n_leaves, DIST_BLOCK, 0, st>>>(vol->origins, cand_off, cand_list, recs, sub, h,
                                                                    (uint32_t)n_cov, vol->values, vol->masks,
                                                                    group_thr, roots, rep_cnt);
    } else {
        k_distance<false><<<(unsigned)n_leaves, DIST_BLOCK, 0, st>>>(vol->origins, cand_off, cand_list, recs, sub, h,
                                                                     (uint32_t)n_cov, vol->values, vol->masks,
                                                                     0.0f, nullptr, nullptr);
    }
    tm.mark();

    // ---- BVH levels (clustered build: its layout) on the second stream, beside the distance pass
    if (ploc) {
        k_ploc_leaves<<<div_up(n, TB), TB, 0, sb>>>(d_tris, nt, idx_s, accs, pbox, pinfo, cl0, keep, ring);
        // a fifth to a third of the clusters merge per iteration: 3 log2(n)
        // iterations cover it; those past one cluster cost a few launches each
        ploc_iters = (int)std::ceil(3.0 * std::log2((double)n + 1.0));
        for (int it = 0; it < ploc_iters; ++it) ploc_iteration(it);
        ploc_result(ploc_iters);
        BS_HIP(hipStreamSynchronize(sb));
        uint32_t N = hs[ploc_iters & 1];
        // rare: more iterations than estimated, one at a time (each merges at
        // least the closest pair, so the count falls every time)
        while (N > 1) {
            ploc_iteration(ploc_iters++);
            BS_HIP(hipMemcpyAsync(hs, ring, sizeof(uint32_t) * 2, hipMemcpyDeviceToHost, sb));
            BS_HIP(hipStreamSynchronize(sb));
            const uint32_t N2 = hs[ploc_iters & 1];
            if (N2 >= N) throw Error(BS_ERR_INTERNAL, "BVH clustering made no progress");
            N = N2;
        }
        ploc_result(ploc_iters);
        BS_HIP(hipStreamSynchronize(sb));
        H = (int)hs[4];
        BS_REQUIRE(H < 250, BS_ERR_INTERNAL, "BVH deeper than the traversal stack");
        k_ploc_place<<<div_up(n_nodes, TB), TB, 0, sb>>>(ring + 3, pinfo, kids, accs, d_tris, idx_s, nt,
                                                        prm.wn_accuracy, nodes, btris, err);
    } else if (topdown) {
        for (int l = 0; l < ploc_iters; ++l) td_level(l);
        auto td_read = [&]() {
            BS_HIP(hipMemcpyAsync(hs, td_ctr, sizeof(uint32_t) * TD_C_WORDS, hipMemcpyDeviceToHost, sb));
            BS_HIP(hipMemcpyAsync(hs + 258, err, sizeof(uint32_t), hipMemcpyDeviceToHost, sb));
            BS_HIP(hipStreamSynchronize(sb));
            if (hs[258] & E_TREE) throw Error(BS_ERR_INTERNAL, "BVH build failed");
        };
        td_read();
        // rare: deeper than estimated, one level at a time (each level cuts
        // every large node, so the depth is at most TD_DEPTH_CAP + log2 n)
        while (hs[TD_C_FR + (ploc_iters & 1)] > 0) {
            BS_REQUIRE(ploc_iters < TD_DEPTH_CAP + 64, BS_ERR_INTERNAL, "BVH build did not finish");
            td_level(ploc_iters++);
            td_read();
        }
        const uint32_t n_small = hs[TD_C_SMALL];
        if (n_small > 0)
            k_td_small<<<div_up(n_small, TD_BLOCK / 64), TD_BLOCK, 0, sb>>>(td_prims, nt, td_small, td_ctr,
                                                                           td_small_cap, pinfo, kids, idx_s, td_depth,
                                                                           err);
        k_td_leaves<<<div_up(n, TB), TB, 0, sb>>>(d_tris, nt, idx_s, accs, err);
        k_td_depth_hist<<<div_up(n_int, 256), 256, 0, sb>>>(td_depth, n_int, td_hist);
        k_td_depth_scan<<<1, 256, 0, sb>>>(td_hist);
        k_td_depth_scatter<<<div_up(n_int, 256), 256, 0, sb>>>(td_depth, n_int, td_hist, inode_s);
        BS_HIP(hipMemcpyAsync(hs, td_hist + 512, sizeof(uint32_t) * 257, hipMemcpyDeviceToHost, sb));
        BS_HIP(hipMemcpyAsync(hs + 258, err, sizeof(uint32_t), hipMemcpyDeviceToHost, sb));
        BS_HIP(hipMemcpyAsync(hs + 259, td_ctr + TD_C_NEXT, sizeof(uint32_t), hipMemcpyDeviceToHost, sb));
        BS_HIP(hipStreamSynchronize(sb));
        if (hs[258] & E_TREE) throw Error(BS_ERR_INTERNAL, "BVH build failed");
        BS_REQUIRE(hs[259] == (uint32_t)n_int && hs[256] == (uint32_t)n_int, BS_ERR_INTERNAL,
                   "BVH build left internal nodes unused");
        BS_REQUIRE(hs[255] == hs[256], BS_ERR_INTERNAL, "BVH deeper than 254 levels");
        // deepest level first: a node's children are one level down
        for (int d = 254; d >= 0; --d) {
            const uint32_t b = hs[d], e = hs[d + 1];
            if (e > b) k_td_level<<<div_up(e - b, TB), TB, 0, sb>>>(inode_s + b, e - b, nt, kids, accs, pinfo);
        }
        k_ploc_root<<<1, 1, 0, sb>>>(reinterpret_cast<const int*>(td_ctr + TD_C_ROOT), pinfo, td_ctr + TD_C_OUT);
        BS_HIP(hipMemcpyAsync(hs, td_ctr + TD_C_OUT, sizeof(uint32_t) * 2, hipMemcpyDeviceToHost, sb));
        BS_HIP(hipStreamSynchronize(sb));
        H = (int)hs[1];
        BS_REQUIRE(H < 250, BS_ERR_INTERNAL, "BVH deeper than the traversal stack");
        k_ploc_place<<<div_up(n_nodes, TB), TB, 0, sb>>>(td_ctr + TD_C_OUT, pinfo, kids, accs, d_tris, idx_s, nt,
                                                        prm.wn_accuracy, nodes, btris, err);
    } else if (n_int > 0) {
        BS_HIP(hipStreamSynchronize(sb));
        if (hs[258] & E_TREE) throw Error(BS_ERR_INTERNAL, "BVH parent links are corrupt");
        // heights run 1..H contiguously in the sorted order
        H = 0;
        for (int k = 1; k < 256; ++k)
            if (hs[k] != 0xFFFFFFFFu) H = k;
        for (int k = 1; k <= H; ++k) {
            BS_REQUIRE(hs[k] != 0xFFFFFFFFu, BS_ERR_INTERNAL, "BVH height levels are not contiguous");
            const uint32_t b = hs[k], e = (k == H) ? (uint32_t)n_int : hs[k + 1];
            k_lbvh_level<<<div_up(e - b, TB), TB, 0, sb>>>(inode_s + b, e - b, prm.wn_accuracy, kids, accs, nodes);
        }
    }
    // the leaves' Z order, after the BVH on the second stream (still beside the distance pass)
    uint32_t* leaf_perm = nullptr;
    if (leaf_z) {
        uint64_t* mk = S.as<uint64_t>(S_LEAF_MKEY, n_leaves);
        uint64_t* mk_s = S.as<uint64_t>(S_LEAF_MKEY_S, n_leaves);
        uint32_t* ids = S.as<uint32_t>(S_LEAF_IDS, n_leaves);
        leaf_perm = S.as<uint32_t>(S_LEAF_PERM, n_leaves);
        int bits = 1;  // key bits per axis (at most 21; wider grids only sort coarser)
        for (int k = 0; k < 3; ++k)
            while (bits < 21 && (1ll << bits) < ghi[k] - glo[k] + 1) ++bits;
        BS_HIP(hipStreamWaitEvent(sb, ctx->ev_leaves, 0));
        k_leaf_morton<<<div_up(n_leaves, TB), TB, 0, sb>>>(vol->origins, n_leaves, (int)glo[0], (int)glo[1],
                                                           (int)glo[2], mk, ids);
        sort_pairs_on(ctx, sb, S_CUB_B, mk, mk_s, ids, leaf_perm, n_leaves, 3 * bits);
    }
    BS_HIP(hipEventRecord(ctx->ev_join, sb));

    // ---- 4. the BVH and the leaves' Z order (second stream) must be complete; active list
    BS_HIP(hipStreamWaitEvent(st, ctx->ev_join, 0));
    uint32_t* act_cnt = S.as<uint32_t>(S_ACT_CNT, n_leaves + 1);
    uint32_t* act_off = S.as<uint32_t>(S_ACT_OFF, n_leaves + 1);
    BS_HIP(hipMemsetAsync(act_cnt + n_leaves, 0, sizeof(uint32_t), st));
    k_leaf_popcount<<<div_up(n_leaves, TB), TB, 0, st>>>(vol->masks, n_leaves, leaf_perm, act_cnt);
    exclusive_scan(ctx, act_cnt, act_off, n_leaves + 1);
    const uint32_t n_act = read_scalar(ctx, act_off + n_leaves);
    uint32_t* act = S.as<uint32_t>(S_ACT_LIST, n_act);
    k_active_list<<<div_up(n_leaves, AL_BLOCK / 64), AL_BLOCK, 0, st>>>(vol->masks, leaf_perm, act_off, n_leaves,
                                                                       act);
    tm.mark();

    // ---- 6. group roots (shared and surrogate signs): the winding number is evaluated
    // at one voxel per group
    const uint32_t* wn_list = act;
    uint32_t n_wn = n_act;
    if ((shared_signs || surrogate_signs) && n_act > 0) {
        // surrogate signs: tile gate and star groups on the finished distances
        // (the same rounding margin as the shared-sign links, beyond h)
        if (surrogate_signs)
            surrogate_groups(ctx, st, vol, h, group_thr - (float)((double)h * (1.0 + 0x1p-10)), roots, rep_cnt,
                             counters + C_SG_TILES);
        // the roots in the leaves' Z order too (the counts gathered into the
        // active-list count buffer, whose last word is still 0)
        const uint32_t* cnt = rep_cnt;
        if (leaf_perm) {
            k_gather_u32<<<div_up(n_leaves, TB), TB, 0, st>>>(rep_cnt, leaf_perm, n_leaves, act_cnt);
            cnt = act_cnt;
        }
        uint32_t* rep_off = S.as<uint32_t>(S_REP_OFF, n_leaves + 1);
        exclusive_scan(ctx, cnt, rep_off, n_leaves + 1);
        n_wn = read_scalar(ctx, rep_off + n_leaves);
        uint32_t* reps = S.as<uint32_t>(S_REPS, std::max<uint32_t>(n_wn, 1));
        k_sign_reps<<<div_up(n_leaves, AL_BLOCK / 64), AL_BLOCK, 0, st>>>(roots, leaf_perm, rep_off, n_leaves, reps);
        wn_list = reps;
    }
    tm.mark();

    // ---- 7. winding numbers and signs
    uint32_t* recheck = S.as<uint32_t>(S_RECHECK, std::max<uint32_t>(n_wn, 1));
    if (n_wn > 0)
    {
        // a tree of height H needs at most H stack entries
        use_lds = !(H + 2 < LaneStack::DEPTH) || (ctx->paths & BS_PATH_FORCE_LDS_STACK);
        // the visit counters feed the work accounting of profiled runs only
        auto kern = use_lds ? (ctx->counting ? k_winding<LdsStack, true> : k_winding<LdsStack, false>)
                            : (ctx->counting ? k_winding<LaneStack, true> : k_winding<LaneStack, false>);
        FarChunk* chunks = nullptr;
        uint32_t* far_list = nullptr;
        float* coef = nullptr;
        // the polynomials are in voxel units: 1 / h^3 has to be a normal float
        if (wn_list == act && prm.wn_accuracy >= WN_FAR_ACCURACY && prm.wn_accuracy <= WN_FAR_ACCURACY_MAX &&
            prm.fp64_band >= WN_FAR_BAND && h > 1e-12f && h < 1e12f) {
            const uint32_t n_chunks = (uint32_t)div_up(n_wn, 64);
            const unsigned groups = div_up(n_chunks, FF_CHUNKS);
            try {  // 5.6 B a voxel, which the walk from the root does without
                far_list = S.as<uint32_t>(S_WN_LIST, (uint64_t)groups * FF_PART);
                coef = S.as<float>(S_WN_COEF, (uint64_t)n_chunks * FF_COEF);
                chunks = S.as<FarChunk>(S_WN_CHUNKS, n_chunks);
            } catch (const Error& e) {
                if (!e.out_of_memory) throw;
            }
            if (chunks)
                k_far_field<<<groups, FF_BLOCK, 0, st>>>(act, n_act, n_chunks, vol->origins, h, inv_h,
                                                         wn_kappa(prm.wn_accuracy), nodes, n_rec, far_list, chunks, coef);
        }
        kern<<<div_up(n_wn, WN_BLOCK), WN_BLOCK, 0, st>>>(wn_list, n_wn, vol->origins, h, nodes, n_rec, btris,
                                                          prm.sign_threshold, prm.fp64_band, chunks, far_list, coef,
                                                          vol->values, recheck, counters, err);
    }
    tm.mark();
    rb.add(counters, hc, C_COUNT);
    rb.add(err, &h_err);
    rb.wait();
    if (h_err & E_HASH) throw Error(BS_ERR_INTERNAL, "leaf lookup failed");
    const uint32_t n_re = (uint32_t)hc[C_RECHECK];
    if (n_re > 0)
        k_winding_fp64<<<div_up(n_re, 64), 64, 0, st>>>(recheck, n_re, vol->origins, h, nodes, n_rec, btris,
                                                        prm.sign_threshold, vol->values, err);
    if (roots) k_sign_broadcast<<<(unsigned)n_leaves, 512, 0, st>>>(roots, vol->values);
    tm.mark();
    // the error word again only when kernels ran after the last readback
    const unsigned e = (n_re > 0 || roots) ? read_scalar(ctx, err) : h_err;
    if (e & E_STACK) throw Error(BS_ERR_INTERNAL, "winding-number traversal stack overflow");
    if (e & E_TREE) throw Error(BS_ERR_INTERNAL, "BVH parent links are corrupt");
    auto wall1 = std::chrono::steady_clock::now();

    bs_m2v_stats& stt = ctx->last_m2v;
    stt = {};
    stt.n_tris = n;
    stt.n_sub = n_sub;
    stt.n_pairs = n_pairs;
    stt.n_leaves = n_leaves;
    stt.n_active = n_act;
    stt.n_candidates = n_cov;
    stt.n_bvh_nodes = (uint64_t)n_nodes;
    stt.wn_node_visits = hc[C_NEAR_INTERNAL];
    stt.wn_far_evals = hc[C_FAR];
    stt.wn_leaf_visits = hc[C_LEAF_VISITS];
    stt.wn_leaf_tris = hc[C_LEAF_TRIS];
    stt.n_fp64_rechecks = n_re;
    stt.used_hash = ix.dense ? 0 : 1;
    stt.used_lds_stack = use_lds ? 1 : 0;
    stt.bvh_height = (uint64_t)H;
    stt.ms_total = std::chrono::duration<double, std::milli>(wall1 - wall0).count();
    stt.ms_subdivide = tm.ms(0, 1);
    stt.ms_leaves = tm.ms(1, 2);
    stt.ms_distance = tm.ms(2, 3);
    stt.ms_bvh = tm.ms(3, 4);
    stt.ms_winding = tm.ms(5, 6);
    stt.n_sign_evals = n_wn;
    stt.ms_sign_share = (shared_signs || surrogate_signs) ? tm.ms(4, 5) + tm.ms(6, 7) : 0.0;
    stt.n_sg_tiles = hc[C_SG_TILES];
    stt.n_sg_culled = hc[C_SG_CULLED];
    stt.n_sg_misclassified = hc[C_SG_MISS];
    stt.n_sg_fallback = hc[C_SG_FALLBACK];
    stt.n_bvh_iterations = (uint64_t)ploc_iters;
    *out = guard.release();
}

void init_context_streams(bs_ctx* ctx) { ensure_side_stream(ctx); }

}  // namespace bs
