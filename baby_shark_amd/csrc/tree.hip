// The upper levels of a volume's grid on the device (see tree.hpp): building
// them from leaves, flood fill, CSG, offset and the visit order.
//
// Every rule works on single slots, node by node: a thread per slot, or per
// z-row of slots where a rule scans, a block per 16^3 node.  These passes stream
// 9 bytes a slot (40 MB per operand of 570 k leaves).  On the host, with the
// ordering of the leaf references and their transfer, they took 20 ms of a CSG
// call at that size; here about 0.5 ms, most of it launches and three looks at
// counts, and a call takes 2.3 ms (21.0 before) against 1.3 ms of leaf kernels.
// Small volumes gain too (0.9 -> 0.55 ms for 1,400 leaves): a 32^3 node is 295 KB
// whatever it holds, and a volume around the origin has eight.
#include "tree.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>

#include "common.hpp"
#include "leafmap.hpp"

namespace bs {

namespace {

constexpr uint64_t MAX_BLOCKS = 1ull << 24, MAX_ROOTS = 256, MAX_N2 = 1ull << 16;
constexpr int32_t SPAN1 = 4096, SPAN2 = 128;
constexpr float FAR = F32_MAX_V;

inline unsigned blocks(uint64_t n, unsigned per = 256) { return std::max(1u, div_up(n, per)); }

template <class T>
T* carve(uint8_t*& p, uint64_t n) {
    T* r = reinterpret_cast<T*>(p);
    p += (n * sizeof(T) + 255) / 256 * 256;
    return r;
}

std::unique_ptr<DeviceTree> new_tree(bs_ctx* ctx, uint32_t n1, uint32_t n2) {
    auto t = std::make_unique<DeviceTree>();
    auto lay = [&](uint8_t* p) {
        uint8_t* p0 = p;
        TreeView& v = t->v;
        v.kind1 = carve<uint8_t>(p, (uint64_t)n1 * N1_SLOTS);
        v.tile1 = carve<float>(p, (uint64_t)n1 * N1_SLOTS);
        v.child1 = carve<int32_t>(p, (uint64_t)n1 * N1_SLOTS);
        v.org1 = carve<int4>(p, n1);
        v.kind2 = carve<uint8_t>(p, (uint64_t)n2 * N2_SLOTS);
        v.tile2 = carve<float>(p, (uint64_t)n2 * N2_SLOTS);
        v.child2 = carve<int32_t>(p, (uint64_t)n2 * N2_SLOTS);
        v.org2 = carve<int4>(p, n2);
        v.n1 = n1;
        v.n2 = n2;
        return (uint64_t)(p - p0);
    };
    const uint64_t bytes = lay(nullptr);
    t->block = alloc_block(bytes);
    t->pending = ctx ? ctx->stream : nullptr;
    lay(static_cast<uint8_t*>(t->block));
    return t;
}

uint64_t tree_bytes(const DeviceTree& t) { return (uint64_t)((uint8_t*)(t.v.org2 + t.v.n2) - (uint8_t*)t.block); }

// A copy of a tree's slots, without its root map, made on the context's stream.
std::unique_ptr<DeviceTree> copy_slots(bs_ctx* ctx, const DeviceTree& s) {
    auto t = new_tree(ctx, s.v.n1, s.v.n2);
    if (s.v.n1) BS_HIP(hipMemcpyAsync(t->block, s.block, tree_bytes(s), hipMemcpyDeviceToDevice, ctx->stream));
    return t;
}

void scan_u32(bs_ctx* ctx, const uint32_t* in, uint32_t* out, uint64_t n) {
    size_t bytes = 0;
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, ctx->stream));
    void* tmp = ctx->scratch.get(S_CUB, bytes);
    BS_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, (int)n, ctx->stream));
}

__host__ __device__ inline uint32_t slot1(int32_t x, int32_t y, int32_t z) {  // of the 128^3 block holding a voxel
    return (uint32_t)((x >> 7 & 31) << 10 | (y >> 7 & 31) << 5 | (z >> 7 & 31));
}
__device__ inline uint32_t slot2(int32_t x, int32_t y, int32_t z) {  // of the leaf holding a voxel
    return (uint32_t)((x >> 3 & 15) << 8 | (y >> 3 & 15) << 4 | (z >> 3 & 15));
}
__device__ inline bool neg(float v) { return __float_as_uint(v) >> 31; }

// ------------------------------------------------------------------ build
// The 128^3 blocks of a box as a grid (x, y, z), and its 4096^3 blocks.
struct BlockGrid {
    int32_t x0, y0, z0, X0, Y0, Z0;  // first block, first root block
    uint32_t ny, nz, NY, NZ;
    uint64_t n, N;
    __host__ __device__ uint64_t cell(int32_t x, int32_t y, int32_t z) const {  // of a voxel
        return ((uint64_t)((x >> 7) - x0) * ny + (uint64_t)((y >> 7) - y0)) * nz + (uint64_t)((z >> 7) - z0);
    }
    __host__ __device__ uint32_t root(int32_t x, int32_t y, int32_t z) const {
        return ((uint32_t)((x >> 12) - X0) * NY + (uint32_t)((y >> 12) - Y0)) * NZ + (uint32_t)((z >> 12) - Z0);
    }
};

__global__ void k_mark_blocks(uint64_t n, const int4* __restrict__ origins, BlockGrid g, uint32_t* mark, uint32_t* rmark) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 o = origins[i];
    const uint64_t c = g.cell(o.x, o.y, o.z);
    if (!mark[c]) mark[c] = 1;
    const uint32_t r = g.root(o.x, o.y, o.z);
    if (!rmark[r]) rmark[r] = 1;
}

// tiles: (x, y, z, size) per tile; an 8^3 tile needs its block's node
__global__ void k_mark_tiles(uint32_t n, const int4* __restrict__ tiles, BlockGrid g, uint32_t* mark, uint32_t* rmark) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 o = tiles[i];
    if (o.w != SPAN2) mark[g.cell(o.x, o.y, o.z)] = 1;
    rmark[g.root(o.x, o.y, o.z)] = 1;
}

__global__ void k_link_blocks(BlockGrid g, const uint32_t* __restrict__ mark, const uint32_t* __restrict__ id,
                              const uint32_t* __restrict__ root_id, TreeView t) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= g.n || !mark[c]) return;
    const int32_t z = ((int32_t)(c % g.nz) + g.z0) * SPAN2, y = ((int32_t)(c / g.nz % g.ny) + g.y0) * SPAN2,
                  x = ((int32_t)(c / g.nz / g.ny) + g.x0) * SPAN2;
    t.org2[id[c]] = make_int4(x, y, z, 0);
    const uint64_t s = (uint64_t)root_id[g.root(x, y, z)] * N1_SLOTS + slot1(x, y, z);
    t.kind1[s] = SLOT_BRANCH;
    t.child1[s] = (int32_t)id[c];
}

__global__ void k_put_leaves(uint64_t n, const int4* __restrict__ origins, BlockGrid g, const uint32_t* __restrict__ id,
                             TreeView t) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 o = origins[i];
    const uint64_t s = (uint64_t)id[g.cell(o.x, o.y, o.z)] * N2_SLOTS + slot2(o.x, o.y, o.z);
    t.kind2[s] = SLOT_BRANCH;
    t.child2[s] = (int32_t)i;
}

__global__ void k_put_tiles(uint32_t n, const int4* __restrict__ tiles, const float* __restrict__ value, BlockGrid g,
                            const uint32_t* __restrict__ id, const uint32_t* __restrict__ root_id, TreeView t) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 o = tiles[i];
    if (o.w == SPAN2) {
        const uint64_t s = (uint64_t)root_id[g.root(o.x, o.y, o.z)] * N1_SLOTS + slot1(o.x, o.y, o.z);
        t.kind1[s] = SLOT_TILE;
        t.tile1[s] = value[i];
    } else {
        const uint64_t s = (uint64_t)id[g.cell(o.x, o.y, o.z)] * N2_SLOTS + slot2(o.x, o.y, o.z);
        t.kind2[s] = SLOT_TILE;
        t.tile2[s] = value[i];
    }
}

bool root_gap(const Topology::Key& a, const Topology::Key& b) {  // of two keys next to each other in order
    return a[0] == b[0] && a[1] == b[1] && b[2] != a[2] + SPAN1;
}
bool has_root_gap(const std::map<Topology::Key, int32_t>& root) {
    return std::adjacent_find(root.begin(), root.end(), [](const auto& a, const auto& b) {
               return root_gap(a.first, b.first);
           }) != root.end();
}

std::unique_ptr<DeviceTree> tree_from_leaves(bs_ctx* ctx, const int4* origins, uint64_t n,
                                             const std::vector<TileRec>& tiles, bool no_gap = false) {
    hipStream_t st = ctx->stream;
    Scratch& S = ctx->scratch;
    if (!n && tiles.empty()) return new_tree(ctx, 0, 0);
    int32_t lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
    if (n) {
        leaf_box(ctx, reinterpret_cast<const int32_t*>(origins), n, lo, hi);
        for (int k = 0; k < 3; ++k) lo[k] *= 8, hi[k] *= 8;
    }
    for (const TileRec& t : tiles) {
        const int32_t o[3] = {t.x, t.y, t.z};
        for (int k = 0; k < 3; ++k) lo[k] = std::min(lo[k], o[k]), hi[k] = std::max(hi[k], o[k]);
    }
    BlockGrid g{};
    g.x0 = lo[0] >> 7, g.y0 = lo[1] >> 7, g.z0 = lo[2] >> 7;
    g.X0 = lo[0] >> 12, g.Y0 = lo[1] >> 12, g.Z0 = lo[2] >> 12;
    g.ny = (uint32_t)((hi[1] >> 7) - g.y0 + 1), g.nz = (uint32_t)((hi[2] >> 7) - g.z0 + 1);
    g.NY = (uint32_t)((hi[1] >> 12) - g.Y0 + 1), g.NZ = (uint32_t)((hi[2] >> 12) - g.Z0 + 1);
    const uint64_t nx = (uint64_t)((hi[0] >> 7) - g.x0 + 1), NX = (uint64_t)((hi[0] >> 12) - g.X0 + 1);
    if (nx > MAX_BLOCKS || (uint64_t)g.ny * g.nz > MAX_BLOCKS || nx * g.ny * g.nz > MAX_BLOCKS) return nullptr;
    g.n = nx * g.ny * g.nz;
    g.N = NX * g.NY * g.NZ;
    if (g.N > MAX_ROOTS) return nullptr;
    uint32_t* mark = S.as<uint32_t>(S_TREE_MARK, 2 * (g.n + 1) + 2 * g.N);
    uint32_t *id = mark + g.n + 1, *rmark = id + g.n + 1, *root_id = rmark + g.N;
    BS_HIP(hipMemsetAsync(mark, 0, sizeof(uint32_t) * (g.n + 1), st));
    BS_HIP(hipMemsetAsync(rmark, 0, sizeof(uint32_t) * g.N, st));
    if (n) k_mark_blocks<<<blocks(n), 256, 0, st>>>(n, origins, g, mark, rmark);
    BS_HIP(hipGetLastError());
    int4* d_tiles = nullptr;
    float* d_tile_val = nullptr;
    std::vector<int4> h_tiles;  // read by the copies until the synchronisation below
    std::vector<float> h_val;
    if (!tiles.empty()) {
        for (const TileRec& t : tiles) h_tiles.push_back(make_int4(t.x, t.y, t.z, t.size)), h_val.push_back(t.value);
        d_tiles = S.as<int4>(S_TREE_TILES, tiles.size());
        d_tile_val = S.as<float>(S_TREE_TILE_VAL, tiles.size());
        BS_HIP(hipMemcpyAsync(d_tiles, h_tiles.data(), sizeof(int4) * tiles.size(), hipMemcpyHostToDevice, st));
        BS_HIP(hipMemcpyAsync(d_tile_val, h_val.data(), sizeof(float) * tiles.size(), hipMemcpyHostToDevice, st));
        k_mark_tiles<<<blocks(tiles.size()), 256, 0, st>>>((uint32_t)tiles.size(), d_tiles, g, mark, rmark);
        BS_HIP(hipGetLastError());
    }
    scan_u32(ctx, mark, id, g.n + 1);
    uint32_t* back = static_cast<uint32_t*>(pinned_words(ctx, 1 + 2 * g.N));
    BS_HIP(hipMemcpyAsync(back, id + g.n, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipMemcpyAsync(back + 1, rmark, sizeof(uint32_t) * g.N, hipMemcpyDeviceToHost, st));
    BS_HIP(hipStreamSynchronize(st));
    const uint32_t n2 = back[0];
    if (n2 > MAX_N2) return nullptr;
    std::vector<Topology::Key> keys;
    uint32_t* ids = back + 1 + g.N;
    for (uint32_t r = 0; r < g.N; ++r) {
        ids[r] = (uint32_t)keys.size();
        if (!back[1 + r]) continue;
        keys.push_back({((int32_t)(r / g.NZ / g.NY) + g.X0) * SPAN1, ((int32_t)(r / g.NZ % g.NY) + g.Y0) * SPAN1,
                        ((int32_t)(r % g.NZ) + g.Z0) * SPAN1});
    }
    if (no_gap && std::adjacent_find(keys.begin(), keys.end(), root_gap) != keys.end()) return nullptr;
    auto t = new_tree(ctx, (uint32_t)keys.size(), n2);
    std::vector<int4> org1;
    for (size_t i = 0; i < keys.size(); ++i) {
        t->root[keys[i]] = (int32_t)i;
        org1.push_back(make_int4(keys[i][0], keys[i][1], keys[i][2], 0));
    }
    // kinds, tile values and children of all slots: empty, 0, 0 (a child of a slot that is no branch is never
    // followed)
    BS_HIP(hipMemsetAsync(t->block, 0, (uint64_t)((uint8_t*)t->v.org2 - (uint8_t*)t->block), st));
    BS_HIP(hipMemcpyAsync(root_id, ids, sizeof(uint32_t) * g.N, hipMemcpyHostToDevice, st));
    BS_HIP(hipMemcpyAsync(t->v.org1, org1.data(), sizeof(int4) * org1.size(), hipMemcpyHostToDevice, st));
    k_link_blocks<<<blocks(g.n), 256, 0, st>>>(g, mark, id, root_id, t->v);
    if (n) k_put_leaves<<<blocks(n), 256, 0, st>>>(n, origins, g, id, t->v);
    if (!tiles.empty())
        k_put_tiles<<<blocks(tiles.size()), 256, 0, st>>>((uint32_t)tiles.size(), d_tiles, d_tile_val, g, id, root_id, t->v);
    BS_HIP(hipGetLastError());
    BS_HIP(hipStreamSynchronize(st));
    return t;
}

std::unique_ptr<DeviceTree> upload_tree(bs_ctx* ctx, const Topology& topo) {
    if (topo.n2.size() > MAX_N2 || topo.n1.size() > MAX_ROOTS) return nullptr;
    auto t = new_tree(ctx, (uint32_t)topo.n1.size(), (uint32_t)topo.n2.size());
    t->root = topo.root;
    const uint64_t bytes = tree_bytes(*t);
    std::vector<uint8_t> host(bytes);
    auto at = [&](void* p) { return host.data() + ((uint8_t*)p - (uint8_t*)t->block); };
    auto put = [&](const auto& nodes, uint64_t slots, uint8_t* kind, float* tile, int32_t* child, int4* org) {
        host_parallel_for(nodes.size(), [&](size_t i) {
            const auto& n = nodes[i];
            std::memcpy(at(kind + i * slots), n.kind.data(), slots);
            std::memcpy(at(tile + i * slots), n.tile.data(), slots * sizeof(float));
            std::memcpy(at(child + i * slots), n.child.data(), slots * sizeof(int32_t));
            const int4 o = make_int4(n.ox, n.oy, n.oz, 0);
            std::memcpy(at(org + i), &o, sizeof(o));
        });
    };
    put(topo.n1, N1_SLOTS, t->v.kind1, t->v.tile1, t->v.child1, t->v.org1);
    put(topo.n2, N2_SLOTS, t->v.kind2, t->v.tile2, t->v.child2, t->v.org2);
    BS_HIP(hipMemcpyAsync(t->block, host.data(), bytes, hipMemcpyHostToDevice, ctx->stream));
    BS_HIP(hipStreamSynchronize(ctx->stream));
    return t;
}

// ------------------------------------------------------------------ flood fill
// Scan-line sign propagation over the slots of one node (internal_node/
// flood_fill.rs:17-75), one block per node and a thread per z-row.  child_flags:
// bit 0 first, bit 1 last value negative, per child.  out_flags: the node's own
// (:94-108; the "last" sign of a branch in the last slot is that branch's first).
template <int LOG2>
__global__ __launch_bounds__(1 << (2 * LOG2)) void k_fill_nodes(const uint8_t* __restrict__ kind,
                                                                float* __restrict__ tile,
                                                                const int32_t* __restrict__ child,
                                                                const uint8_t* __restrict__ child_flags,
                                                                uint8_t* __restrict__ out_flags) {
    constexpr int D = 1 << LOG2, N = D * D * D;
    __shared__ uint8_t at0[D * D];  // slot (x, y, 0): 0 nothing there, 2 positive, 3 negative
    __shared__ uint32_t first_tile, first_branch, others;
    const uint64_t base = (uint64_t)blockIdx.x * N;
    const int row = threadIdx.x, x = row >> LOG2, y = row & (D - 1);
    if (row == 0) first_tile = first_branch = N, others = 0;
    __syncthreads();
    uint8_t state[D];
    uint32_t ft = N, fb = N, no = 0;
#pragma unroll
    for (int z = D - 1; z >= 0; --z) {
        const uint64_t s = base + (uint64_t)row * D + z;
        const uint8_t k = kind[s];
        state[z] = 0;
        if (k == SLOT_TILE) state[z] = 2 | (uint8_t)neg(tile[s]), ft = row * D + z;
        else no = 1;
        if (k == SLOT_BRANCH) state[z] = 2 | (child_flags[child[s]] >> 1 & 1), fb = row * D + z;
    }
    at0[row] = state[0];
    if (ft < (uint32_t)N) atomicMin(&first_tile, ft);
    if (fb < (uint32_t)N) atomicMin(&first_branch, fb);
    if (no) others = 1;
    __syncthreads();
    auto branch_first = [&](uint32_t o) { return (bool)(child_flags[child[base + o]] & 1); };
    if (others && (first_tile < (uint32_t)N || first_branch < (uint32_t)N)) {
        const bool seed = first_tile < first_branch ? neg(tile[base + first_tile]) : branch_first(first_branch);
        int k = seed;
        int at = x * D + y;  // the last (x, y', 0) at or before y, else the last (x', 0, 0) at or before x
        while (at > x * D && !at0[at]) --at;
        if (!at0[at])
            for (at = x * D; at > 0 && !at0[at];) at -= D;
        if (at0[at]) k = at0[at] & 1;
#pragma unroll
        for (int z = 0; z < D; ++z) {
            if (state[z]) k = state[z] & 1;
            else tile[base + (uint64_t)row * D + z] = k ? -FAR : FAR;
        }
    }
    __syncthreads();
    if (row == 0) {
        const bool first = kind[base] == SLOT_BRANCH ? branch_first(0) : neg(tile[base]);
        const bool last = kind[base + N - 1] == SLOT_BRANCH ? branch_first(N - 1) : neg(tile[base + N - 1]);
        out_flags[blockIdx.x] = (uint8_t)(first | last << 1);
    }
}

// ------------------------------------------------------------------ CSG
struct CsgCounts {
    uint32_t pairs, flips, n2, out, tiles, paired;
};
struct CsgWork {
    TreeView a, b;
    int op;
    int32_t n_a;             // leaves of a: a leaf of b is known as n_a + its index in nodes of a
    const uint8_t *fa, *fb;  // leaf flags
    int4* pairs;             // (slot of a's 32^3 nodes, 16^3 node of a, of b, 0)
    uint32_t *flips, *flipped;  // 16^3 nodes of b moved in and negated: their list, a word per node
    int32_t* partner;        // per leaf of a: the leaf of b it is combined with, -1
    uint32_t* negate;        // per leaf of b
    CsgCounts* counts;
};

template <class K>
__device__ inline bool inside(K k, float t) { return k != SLOT_BRANCH && neg(t); }
template <class K>
__device__ inline bool outside(K k, float t) { return k != SLOT_BRANCH && !neg(t); }

// What one slot of self (k, tile, child) becomes against other's slot
// (internal_node/csg.rs:68-152): CSG_PAIR both are branches, CSG_TAKEN other's
// branch moved in, CSG_TAKEN_FLIPPED and negated.
enum SlotResult : int { CSG_DONE, CSG_PAIR, CSG_TAKEN, CSG_TAKEN_FLIPPED };
__device__ inline SlotResult csg_slot(int op, uint8_t& k, float& tile, uint8_t ok, float otile) {
    if (op == CSG_UNION) {
        if (inside(k, tile)) return CSG_DONE;
        if (inside(ok, otile)) {
            k = SLOT_TILE;  // make_child_inside
            tile = -FAR;
            return CSG_DONE;
        }
        if (outside(k, tile)) return ok == SLOT_BRANCH ? CSG_TAKEN : CSG_DONE;
    } else if (op == CSG_SUBTRACT) {
        if (outside(k, tile) || outside(ok, otile)) return CSG_DONE;
        if (inside(ok, otile)) {
            k = SLOT_EMPTY;
            return CSG_DONE;
        }
        if (inside(k, tile)) return CSG_TAKEN_FLIPPED;
    } else {
        if (outside(k, tile) || inside(ok, otile)) return CSG_DONE;
        if (outside(ok, otile)) {
            k = SLOT_EMPTY;
            return CSG_DONE;
        }
        if (inside(k, tile)) return CSG_TAKEN;
    }
    return k == SLOT_BRANCH && ok == SLOT_BRANCH ? CSG_PAIR : CSG_DONE;
}

// The 32^3 nodes that both roots hold, n of them: pairs (node of a, node of b).
__global__ void k_csg_slots1(CsgWork w, uint32_t n, const int2* __restrict__ roots) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i / N1_SLOTS >= n) return;
    const int2 r = roots[i / N1_SLOTS];
    const uint64_t s = (uint64_t)r.x * N1_SLOTS + i % N1_SLOTS, o = (uint64_t)r.y * N1_SLOTS + i % N1_SLOTS;
    uint8_t k = w.a.kind1[s];
    float tile = w.a.tile1[s];
    const uint8_t k0 = k;
    const float tile0 = tile;
    const SlotResult res = csg_slot(w.op, k, tile, w.b.kind1[o], w.b.tile1[o]);
    if (res == CSG_PAIR) {
        w.pairs[atomicAdd(&w.counts->pairs, 1u)] = make_int4((int)s, w.a.child1[s], w.b.child1[o], 0);
    } else if (res == CSG_TAKEN || res == CSG_TAKEN_FLIPPED) {
        const int32_t node = w.b.child1[o];
        w.a.kind1[s] = SLOT_BRANCH;
        w.a.tile1[s] = w.b.tile1[o];
        w.a.child1[s] = (int32_t)w.a.n2 + node;  // a node of b
        if (res == CSG_TAKEN_FLIPPED) {
            w.flips[atomicAdd(&w.counts->flips, 1u)] = (uint32_t)node;
            w.flipped[node] = 1;
        }
    } else if (k != k0 || __float_as_uint(tile) != __float_as_uint(tile0)) {
        w.a.kind1[s] = k;
        w.a.tile1[s] = tile;
    }
}

// One block per listed pair of 16^3 nodes; union turns a node that it emptied
// into an inside tile.
__global__ __launch_bounds__(256) void k_csg_slots2(CsgWork w) {
    if (blockIdx.x >= w.counts->pairs) return;
    __shared__ uint32_t any;
    const int4 p = w.pairs[blockIdx.x];
    const uint64_t sa = (uint64_t)p.y * N2_SLOTS, sb = (uint64_t)p.z * N2_SLOTS;
    if (threadIdx.x == 0) any = 0;
    __syncthreads();
    bool mine = false;
    for (uint32_t q = threadIdx.x; q < N2_SLOTS; q += 256) {
        const uint64_t s = sa + q, o = sb + q;
        uint8_t k = w.a.kind2[s];
        float tile = w.a.tile2[s];
        int32_t child = w.a.child2[s];
        const SlotResult res = csg_slot(w.op, k, tile, w.b.kind2[o], w.b.tile2[o]);
        if (res == CSG_PAIR) {  // leaf_node/csg.rs:17-45: recorded, the assembly combines the leaves
            const int32_t lb = w.b.child2[o];
            w.partner[child] = lb;
            if (w.op == CSG_UNION && (w.fa[child] & w.fb[lb] & 4)) {
                k = SLOT_TILE;
                tile = -FAR;
            }
        } else if (res == CSG_TAKEN || res == CSG_TAKEN_FLIPPED) {
            const int32_t lb = w.b.child2[o];
            k = SLOT_BRANCH;
            tile = w.b.tile2[o];
            child = w.n_a + lb;
            if (res == CSG_TAKEN_FLIPPED) w.negate[lb] = 1;
        }
        w.a.kind2[s] = k;
        w.a.tile2[s] = tile;
        w.a.child2[s] = child;
        mine |= k != SLOT_EMPTY;
    }
    if (mine) any = 1;
    __syncthreads();
    if (threadIdx.x == 0 && !any && w.op == CSG_UNION) {
        w.a.kind1[p.x] = SLOT_TILE;
        w.a.tile1[p.x] = -FAR;
    }
}

// internal_node/csg.rs:154-162: the leaves here, the tiles where the result is
// written (b's own slots stay as they are)
__global__ __launch_bounds__(256) void k_csg_flip(CsgWork w) {
    if (blockIdx.x >= w.counts->flips) return;
    const uint64_t base = (uint64_t)w.flips[blockIdx.x] * N2_SLOTS;
    for (uint32_t q = threadIdx.x; q < N2_SLOTS; q += 256)
        if (w.b.kind2[base + q] == SLOT_BRANCH) w.negate[w.b.child2[base + q]] = 1;
}

// ------------------------------------------------------------------ result
// The result's 32^3 nodes in root order, each one of a tree's (node) or b's
// (-1 - node); item i is slot i % N1_SLOTS of result node i / N1_SLOTS.
struct Item {
    uint8_t kind;
    float tile;
    int32_t node2;  // of a, or a.n2 + that of b
    int4 org;
};
__device__ inline Item item_of(const TreeView& a, const TreeView& b, const int32_t* nodes, uint32_t i) {
    const int32_t r = nodes[i / N1_SLOTS];
    const bool of_b = r < 0;
    const uint64_t s = (uint64_t)(of_b ? -1 - r : r) * N1_SLOTS + i % N1_SLOTS;
    Item t;
    t.kind = of_b ? b.kind1[s] : a.kind1[s];
    t.tile = of_b ? b.tile1[s] : a.tile1[s];
    t.node2 = of_b ? b.child1[s] + (int32_t)a.n2 : a.child1[s];
    t.org = of_b ? b.org1[-1 - r] : a.org1[r];
    return t;
}

__global__ void k_item_branch(TreeView a, TreeView b, uint32_t n, const int32_t* __restrict__ nodes,
                              uint32_t* __restrict__ branch) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    branch[i] = i < n && item_of(a, b, nodes, i).kind == SLOT_BRANCH;  // entry n: 0, so that the scan ends in the total
}

// refs[k] = the k-th 16^3 node of the result
__global__ void k_item_refs(TreeView a, TreeView b, uint32_t n, const int32_t* __restrict__ nodes,
                            const uint32_t* __restrict__ branch, const uint32_t* __restrict__ at, int32_t* refs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !branch[i]) return;
    refs[at[i]] = item_of(a, b, nodes, i).node2;
}

// Leaves that the k-th result node keeps (leaf of a, or n_a + leaf of b), and its
// active tiles and its filled slots.
__global__ __launch_bounds__(256) void k_node_mark(TreeView a, TreeView b, int32_t n_a, const int32_t* __restrict__ refs,
                                                   const uint32_t* __restrict__ n, uint32_t* keep, uint32_t* tiles,
                                                   uint32_t* filled) {
    if (blockIdx.x >= *n) return;
    const int32_t r = refs[blockIdx.x];
    const bool of_b = r >= (int32_t)a.n2;
    const uint64_t base = (uint64_t)(of_b ? r - (int32_t)a.n2 : r) * N2_SLOTS;
    const uint8_t* kind = (of_b ? b.kind2 : a.kind2) + base;
    const int32_t* child = (of_b ? b.child2 : a.child2) + base;
    __shared__ uint32_t nt, nf;
    if (threadIdx.x == 0) nt = nf = 0;
    __syncthreads();
    uint32_t mt = 0, mf = 0;
    for (uint32_t q = threadIdx.x; q < N2_SLOTS; q += 256) {
        const uint8_t k = kind[q];
        if (k == SLOT_BRANCH && keep) keep[child[q] + (of_b ? n_a : 0)] = 1;
        mt += k == SLOT_TILE;
        mf += k != SLOT_EMPTY;
    }
    if (mt) atomicAdd(&nt, mt);
    if (mf) atomicAdd(&nf, mf);
    __syncthreads();
    if (threadIdx.x == 0) {
        tiles[blockIdx.x] = nt;
        if (filled) filled[blockIdx.x] = nf;
    }
}

// Active tiles (or, per_node = filled slots, units) of each item; entry n: 0.
__global__ void k_item_counts(TreeView a, TreeView b, uint32_t n, const int32_t* __restrict__ nodes,
                              const uint32_t* __restrict__ at, const uint32_t* __restrict__ per_node, uint32_t* count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    uint32_t c = 0;
    if (i < n) {
        const uint8_t k = item_of(a, b, nodes, i).kind;
        c = k == SLOT_TILE ? 1u : (k == SLOT_BRANCH ? per_node[at[i]] : 0u);
    }
    count[i] = c;
}

__device__ inline int4 slot1_origin(int4 org, uint32_t s) {
    return make_int4(org.x + (int)(s >> 10) * SPAN2, org.y + (int)(s >> 5 & 31) * SPAN2, org.z + (int)(s & 31) * SPAN2, SPAN2);
}
__device__ inline int4 slot2_origin(int4 org, uint32_t s) {
    return make_int4(org.x + (int)(s >> 8) * 8, org.y + (int)(s >> 4 & 15) * 8, org.z + (int)(s & 15) * 8, 8);
}

// Everything of the result in tree order, a wave per item: its active tiles to
// tile_org (x, y, z, size) and tile_val from tile_at[i] on; with units, its
// leaves (index) and tiles (-1 - tile) from unit_at[i] on.  flipped (or null): see CsgWork.
__global__ __launch_bounds__(256) void k_item_write(TreeView a, TreeView b, uint32_t n, const int32_t* __restrict__ nodes,
                                                    const uint32_t* __restrict__ flipped,
                                                    const uint32_t* __restrict__ tile_at, int4* tile_org, float* tile_val,
                                                    const uint32_t* __restrict__ unit_at, int64_t* units) {
    const uint32_t i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    uint32_t t0 = tile_at[i], u0 = units ? unit_at[i] : 0;
    if (tile_at[i + 1] == t0 && (!units || unit_at[i + 1] == u0)) return;
    const int lane = threadIdx.x & 63;
    const Item it = item_of(a, b, nodes, i);
    const int4 org = slot1_origin(it.org, i % N1_SLOTS);
    if (it.kind == SLOT_TILE) {
        if (lane == 0) {
            tile_org[t0] = org;
            tile_val[t0] = it.tile;
            if (units) units[u0] = -1 - (int64_t)t0;
        }
        return;
    }
    const bool of_b = it.node2 >= (int32_t)a.n2;
    const TreeView& t = of_b ? b : a;
    const int32_t node = of_b ? it.node2 - (int32_t)a.n2 : it.node2;
    const uint64_t base = (uint64_t)node * N2_SLOTS;
    const bool flip = of_b && flipped && flipped[node];
    const unsigned long long lt = (1ull << lane) - 1;
    for (uint32_t q = lane; q < N2_SLOTS; q += 64) {
        const uint8_t k = t.kind2[base + q];
        const unsigned long long bt = __ballot(k == SLOT_TILE), bu = __ballot(k != SLOT_EMPTY);
        const uint32_t ti = t0 + (uint32_t)__popcll(bt & lt);
        if (k == SLOT_TILE) {
            tile_org[ti] = slot2_origin(org, q);
            tile_val[ti] = flip ? -t.tile2[base + q] : t.tile2[base + q];
        }
        if (units && k != SLOT_EMPTY)
            units[u0 + (uint32_t)__popcll(bu & lt)] = k == SLOT_TILE ? -1 - (int64_t)ti : (int64_t)t.child2[base + q];
        t0 += (uint32_t)__popcll(bt);
        u0 += (uint32_t)__popcll(bu);
    }
}

__global__ void k_csg_totals(const uint32_t* n2, const uint32_t* kept, const uint32_t* tiles, CsgCounts* c) {
    if (threadIdx.x == 0) c->n2 = *n2, c->out = *kept, c->tiles = *tiles;
}

// Place of every kept leaf (of a, then of b) in origin order.  Each operand's
// leaves are in that order and a result leaf stands for one origin, so a leaf's
// place is its own rank plus the other operand's kept leaves below it (a binary
// search).  rank: exclusive sums of keep over the leaves of a, then of b.
__global__ void k_leaf_places(CsgWork w, uint32_t n_a, uint32_t n_b, const int4* __restrict__ oa,
                              const int4* __restrict__ ob, const uint32_t* __restrict__ keep,
                              const uint32_t* __restrict__ rank, int32_t* __restrict__ place, int4* __restrict__ refs,
                              int4* __restrict__ origins) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool paired = false;
    if (i < n_a + n_b && keep[i]) {
        const bool of_b = i >= n_a;
        const uint32_t l = of_b ? i - n_a : i;
        const int4 o = of_b ? ob[l] : oa[l];
        const uint64_t key = leaf_key(o.x >> 3, o.y >> 3, o.z >> 3);
        const int4* other = of_b ? oa : ob;
        uint32_t lo = 0, hi = of_b ? n_a : n_b;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            const int4 m = other[mid];
            if (leaf_key(m.x >> 3, m.y >> 3, m.z >> 3) < key) lo = mid + 1;
            else hi = mid;
        }
        const uint32_t at = rank[i] - rank[n_a] + (of_b ? rank[lo] : rank[n_a + lo]);  // unsigned: either order of the sums
        place[i] = (int32_t)at;
        const int32_t partner = of_b ? -1 : w.partner[l];
        paired = partner >= 0;
        const int op = of_b ? LEAF_COPY_B
                            : (partner < 0 ? LEAF_COPY_A
                                           : (w.op == CSG_UNION ? LEAF_UNION : (w.op == CSG_SUBTRACT ? LEAF_SUBTRACT : LEAF_INTERSECT)));
        refs[at] = make_int4(of_b ? 0 : (int)l, of_b ? (int)l : max(partner, 0), op | (of_b ? (int)w.negate[l] << 8 : 0), 0);
        origins[at] = make_int4(o.x, o.y, o.z, 0);
    }
    const unsigned long long b = __ballot(paired);
    if ((threadIdx.x & 63) == 0 && b) atomicAdd(&w.counts->paired, (uint32_t)__popcll(b));
}

// The result's nodes with renumbered children.
__global__ void k_copy_nodes1(TreeView a, TreeView b, uint32_t n, const int32_t* __restrict__ nodes,
                              const uint32_t* __restrict__ at, TreeView out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Item it = item_of(a, b, nodes, i);
    out.kind1[i] = it.kind;
    out.tile1[i] = it.tile;
    out.child1[i] = it.kind == SLOT_BRANCH ? (int32_t)at[i] : -1;
    if (i % N1_SLOTS == 0) out.org1[i / N1_SLOTS] = it.org;
}
__global__ __launch_bounds__(256) void k_copy_nodes2(TreeView a, TreeView b, int32_t n_a, const int32_t* __restrict__ refs,
                                                     const uint32_t* __restrict__ flipped,
                                                     const int32_t* __restrict__ place, TreeView out) {
    const int32_t r = refs[blockIdx.x];
    const bool of_b = r >= (int32_t)a.n2;
    const int32_t node = of_b ? r - (int32_t)a.n2 : r;
    const TreeView& t = of_b ? b : a;
    const bool flip = of_b && flipped[node];
    const uint64_t src = (uint64_t)node * N2_SLOTS, dst = (uint64_t)blockIdx.x * N2_SLOTS;
    for (uint32_t q = threadIdx.x; q < N2_SLOTS; q += 256) {
        const uint8_t k = t.kind2[src + q];
        out.kind2[dst + q] = k;
        out.tile2[dst + q] = flip && k == SLOT_TILE ? -t.tile2[src + q] : t.tile2[src + q];
        out.child2[dst + q] = k == SLOT_BRANCH ? place[t.child2[src + q] + (of_b ? n_a : 0)] : -1;
    }
    if (threadIdx.x == 0) out.org2[blockIdx.x] = t.org2[node];
}

// ------------------------------------------------------------------ offset
// Old 16^3 nodes that kept a leaf, and their 32^3 nodes.
__global__ void k_node_kept(uint64_t n, const int4* __restrict__ origins, const uint32_t* __restrict__ keep, TreeView old,
                            const int2* __restrict__ match, uint32_t n_match, uint32_t* kept1, uint32_t* kept2) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !keep[i]) return;
    const int4 o = origins[i];
    for (uint32_t m = 0; m < n_match; ++m) {
        const int4 r = old.org1[match[m].y];
        if ((o.x >> 12) != (r.x >> 12) || (o.y >> 12) != (r.y >> 12) || (o.z >> 12) != (r.z >> 12)) continue;
        kept1[match[m].y] = 1;
        kept2[old.child1[(uint64_t)match[m].y * N1_SLOTS + slot1(o.x, o.y, o.z)]] = 1;
        return;
    }
}
// match[m] = (32^3 node of the new tree, of the old one) at one origin: a block per
// slot of the new one takes the tile values of the old nodes that kept a leaf.
__global__ __launch_bounds__(256) void k_keep_tiles(TreeView old, const int2* __restrict__ match,
                                                    const uint32_t* __restrict__ kept1,
                                                    const uint32_t* __restrict__ kept2, TreeView t) {
    const int2 m = match[blockIdx.x / (N1_SLOTS / 256)];
    if (!kept1[m.y]) return;
    const uint32_t s0 = blockIdx.x % (N1_SLOTS / 256) * 256, s = s0 + threadIdx.x;
    const uint64_t a = (uint64_t)m.x * N1_SLOTS, b = (uint64_t)m.y * N1_SLOTS;
    t.tile1[a + s] = old.tile1[b + s];
    for (uint32_t k = s0; k < s0 + 256; ++k) {
        if (t.kind1[a + k] != SLOT_BRANCH || old.kind1[b + k] != SLOT_BRANCH || !kept2[old.child1[b + k]]) continue;
        const uint64_t d = (uint64_t)t.child1[a + k] * N2_SLOTS, e = (uint64_t)old.child1[b + k] * N2_SLOTS;
        for (uint32_t q = threadIdx.x; q < N2_SLOTS; q += 256) t.tile2[d + q] = old.tile2[e + q];
    }
}

// Device copies of small host lists, kept alive until the caller synchronises.
template <class T>
T* upload(bs_ctx* ctx, int slot, const std::vector<T>& h) {
    T* d = ctx->scratch.as<T>(slot, std::max<size_t>(h.size(), 1));
    if (!h.empty()) BS_HIP(hipMemcpyAsync(d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice, ctx->stream));
    return d;
}

std::vector<TileRec> read_tiles(bs_ctx* ctx, const int4* org, const float* val, uint32_t n) {
    std::vector<TileRec> tiles(n);
    if (!n) return tiles;
    std::vector<int4> o(n);
    std::vector<float> v(n);
    BS_HIP(hipMemcpyAsync(o.data(), org, sizeof(int4) * n, hipMemcpyDeviceToHost, ctx->stream));
    BS_HIP(hipMemcpyAsync(v.data(), val, sizeof(float) * n, hipMemcpyDeviceToHost, ctx->stream));
    BS_HIP(hipStreamSynchronize(ctx->stream));
    for (uint32_t i = 0; i < n; ++i) tiles[i] = {o[i].x, o[i].y, o[i].z, o[i].w, v[i]};
    return tiles;
}

}  // namespace

DeviceTree::~DeviceTree() {
    if (!block) return;
    const bool idle = !pending || hipStreamSynchronize(pending) == hipSuccess;
    free_block(block, !idle);
}

void require_tree(const bs_volume* v) {
    BS_REQUIRE(!v->tree_lost, BS_ERR_INTERNAL, "an earlier operation that failed left this volume without its upper levels");
}

bool known_root_gap(const bs_volume* v) {
    std::lock_guard<std::mutex> lk(v->forms);
    return v->tree ? has_root_gap(v->tree->root) : v->topo && has_root_gap(v->topo->root);
}

DeviceTree* ensure_tree(bs_ctx* ctx, bs_volume* v, bool no_gap) {
    require_tree(v);
    if (no_gap && known_root_gap(v)) return nullptr;
    std::lock_guard<std::mutex> lk(v->forms);
    if (v->tree) return v->tree.get();
    std::unique_ptr<DeviceTree> t;
    try {
        t = v->topo ? upload_tree(ctx, *v->topo)
                    : tree_from_leaves(ctx, reinterpret_cast<const int4*>(v->origins), v->n_leaves, v->tiles, no_gap);
    } catch (const Error& e) {
        if (!e.out_of_memory) throw;
        (void)hipStreamSynchronize(ctx->stream);
    }
    if (!t) return nullptr;
    t->pending = nullptr;  // both return with the stream's work done
    v->tree = std::move(t);
    return v->tree.get();
}

std::unique_ptr<DeviceTree> clone_tree(const DeviceTree& s) {
    auto t = new_tree(nullptr, s.v.n1, s.v.n2);
    t->root = s.root;
    BS_HIP(hipMemcpyAsync(t->block, s.block, tree_bytes(s), hipMemcpyDeviceToDevice));
    BS_HIP(hipStreamSynchronize(nullptr));
    return t;
}

std::unique_ptr<Topology> download_tree(bs_ctx* ctx, const bs_volume* v) {
    const DeviceTree& s = *v->tree;
    auto t = std::make_unique<Topology>();
    t->root = s.root;
    const uint64_t bytes = tree_bytes(s);
    std::vector<uint8_t> host(bytes);
    std::vector<int4> org(v->n_leaves);
    BS_HIP(hipMemcpyAsync(host.data(), s.block, bytes, hipMemcpyDeviceToHost, ctx->stream));
    if (v->n_leaves)
        BS_HIP(hipMemcpyAsync(org.data(), v->origins, sizeof(int4) * v->n_leaves, hipMemcpyDeviceToHost, ctx->stream));
    BS_HIP(hipStreamSynchronize(ctx->stream));
    auto at = [&](const void* p) { return host.data() + ((const uint8_t*)p - (const uint8_t*)s.block); };
    auto get = [&](auto& nodes, uint32_t n, uint64_t slots, const uint8_t* kind, const float* tile, const int32_t* child,
                   const int4* o4) {
        for (uint32_t i = 0; i < n; ++i) {
            int4 o;
            std::memcpy(&o, at(o4 + i), sizeof(o));
            nodes.emplace_back(o.x, o.y, o.z);
        }
        host_parallel_for(n, [&](size_t i) {
            std::memcpy(nodes[i].kind.data(), at(kind + i * slots), slots);
            std::memcpy(nodes[i].tile.data(), at(tile + i * slots), slots * sizeof(float));
            std::memcpy(nodes[i].child.data(), at(child + i * slots), slots * sizeof(int32_t));
        });
    };
    t->n1.reserve(s.v.n1);
    t->n2.reserve(s.v.n2);
    get(t->n1, s.v.n1, N1_SLOTS, s.v.kind1, s.v.tile1, s.v.child1, s.v.org1);
    get(t->n2, s.v.n2, N2_SLOTS, s.v.kind2, s.v.tile2, s.v.child2, s.v.org2);
    t->leaves.resize(v->n_leaves);
    LeafVec& recs = t->leaves.seg[0];
    for (uint64_t i = 0; i < v->n_leaves; ++i) recs[i] = leaf_ref(org[i].x, org[i].y, org[i].z, (int32_t)i);
    return t;
}

void tree_flood_fill(bs_ctx* ctx, const DeviceTree& t, const uint8_t* leaf_flags) {
    uint8_t* f2 = ctx->scratch.as<uint8_t>(S_TREE_FLAGS, (uint64_t)t.v.n2 + t.v.n1 + 2);
    if (t.v.n2) k_fill_nodes<4><<<t.v.n2, 256, 0, ctx->stream>>>(t.v.kind2, t.v.tile2, t.v.child2, leaf_flags, f2);
    if (t.v.n1) k_fill_nodes<5><<<t.v.n1, 1024, 0, ctx->stream>>>(t.v.kind1, t.v.tile1, t.v.child1, f2, f2 + t.v.n2);
    BS_HIP(hipGetLastError());
}

static void plan_csg(bs_ctx* ctx, const DeviceTree& a, const DeviceTree& b, const TreeOperand& la, const TreeOperand& lb,
                     CsgOp op, TreeCsg& r) {
    hipStream_t st = ctx->stream;
    Scratch& S = ctx->scratch;
    // the root's rules (root_node/csg.rs:9-54): nodes that both hold are combined, the others stay or move in
    std::vector<int2> roots;
    std::map<Topology::Key, int32_t> res;  // node of a, or -1 - node of b
    for (const auto& kv : a.root) {
        const auto it = b.root.find(kv.first);
        if (it != b.root.end()) roots.push_back(make_int2(kv.second, it->second));
        if (it != b.root.end() || op != CSG_INTERSECT) res[kv.first] = kv.second;
    }
    if (op == CSG_UNION)
        for (const auto& kv : b.root)
            if (!a.root.count(kv.first)) res[kv.first] = -1 - kv.second;
    std::vector<int32_t> nodes;
    for (const auto& kv : res) nodes.push_back(kv.second);
    if (nodes.size() > MAX_ROOTS) return;

    // 20 MB for 285 k leaves; working in place a subtraction of two such volumes takes 3.38 ms instead of 3.40, a
    // union of 1,400 leaves 0.53 either way.
    r.work = copy_slots(ctx, a);
    const TreeView av = r.work->v, bv = b.v;
    CsgWork w{};
    w.a = av;
    w.b = bv;
    w.op = op;
    w.n_a = (int32_t)la.n;
    w.fa = la.flags;
    w.fb = lb.flags;
    const uint64_t leaves = la.n + lb.n, n2 = (uint64_t)av.n2 + bv.n2;
    const uint32_t n_items = (uint32_t)(nodes.size() * N1_SLOTS);
    w.pairs = S.as<int4>(S_TREE_PAIRS, std::min(av.n2, bv.n2) + 1);
    w.flips = S.as<uint32_t>(S_TREE_FLIPS, bv.n2 + 1);
    w.partner = S.as<int32_t>(S_TREE_PARTNER, la.n);
    // cleared together: counts, negate, keep of a's leaves, then b's, and one entry more for the total, flipped
    const uint64_t zero_n = sizeof(CsgCounts) / 4 + lb.n + leaves + 1 + bv.n2;
    uint32_t* zero = S.as<uint32_t>(S_TREE_ZERO, zero_n);
    w.counts = reinterpret_cast<CsgCounts*>(zero);
    w.negate = zero + sizeof(CsgCounts) / 4;
    uint32_t* keep = w.negate + lb.n;
    w.flipped = keep + leaves + 1;
    uint32_t* rank = S.as<uint32_t>(S_TREE_RANK, leaves + 1);
    BS_HIP(hipMemsetAsync(zero, 0, sizeof(uint32_t) * zero_n, st));
    BS_HIP(hipMemsetAsync(w.partner, 0xFF, sizeof(int32_t) * la.n, st));
    const int2* d_roots = upload(ctx, S_TREE_ROOTS, roots);
    const int32_t* d_nodes = upload(ctx, S_TREE_NODES, nodes);
    if (!roots.empty()) {
        k_csg_slots1<<<blocks(roots.size() * N1_SLOTS), 256, 0, st>>>(w, (uint32_t)roots.size(), d_roots);
        BS_HIP(hipGetLastError());
        const uint32_t most = std::min(av.n2, bv.n2);
        if (most) k_csg_slots2<<<most, 256, 0, st>>>(w);
        if (op == CSG_SUBTRACT && bv.n2) k_csg_flip<<<bv.n2, 256, 0, st>>>(w);
        BS_HIP(hipGetLastError());
    }
    // the result's nodes, leaves and tiles
    uint32_t* branch = S.as<uint32_t>(S_TREE_ITEMS, 4 * ((uint64_t)n_items + 1));
    uint32_t *at = branch + n_items + 1, *tile_n = at + n_items + 1, *tile_at = tile_n + n_items + 1;
    int32_t* refs2 = S.as<int32_t>(S_TREE_REFS, n2 + 1);
    uint32_t* node_tiles = S.as<uint32_t>(S_TREE_NODE_N, n2 + 1);
    const unsigned ib = blocks((uint64_t)n_items + 1);
    k_item_branch<<<ib, 256, 0, st>>>(av, bv, n_items, d_nodes, branch);
    BS_HIP(hipGetLastError());
    scan_u32(ctx, branch, at, (uint64_t)n_items + 1);
    k_item_refs<<<ib, 256, 0, st>>>(av, bv, n_items, d_nodes, branch, at, refs2);
    if (n2) k_node_mark<<<(unsigned)n2, 256, 0, st>>>(av, bv, w.n_a, refs2, at + n_items, keep, node_tiles, nullptr);
    k_item_counts<<<ib, 256, 0, st>>>(av, bv, n_items, d_nodes, at, node_tiles, tile_n);
    BS_HIP(hipGetLastError());
    scan_u32(ctx, tile_n, tile_at, (uint64_t)n_items + 1);
    scan_u32(ctx, keep, rank, leaves + 1);
    k_csg_totals<<<1, 64, 0, st>>>(at + n_items, rank + leaves, tile_at + n_items, w.counts);
    int32_t* place = S.as<int32_t>(S_TREE_PLACE, leaves);
    int4* plan = S.as<int4>(S_CSG_PLAN, 2 * leaves);
    if (leaves)
        k_leaf_places<<<blocks(leaves), 256, 0, st>>>(w, (uint32_t)la.n, (uint32_t)lb.n, la.origins, lb.origins, keep, rank,
                                                      place, plan, plan + leaves);
    BS_HIP(hipGetLastError());
    CsgCounts* back = static_cast<CsgCounts*>(pinned_words(ctx, sizeof(CsgCounts) / 4));
    BS_HIP(hipMemcpyAsync(back, w.counts, sizeof(CsgCounts), hipMemcpyDeviceToHost, st));
    BS_HIP(hipStreamSynchronize(st));
    const CsgCounts c = *back;
    if (c.n2 > MAX_N2) return;
    r.n_out = c.out;
    r.n_paired = c.paired;
    r.refs = plan;
    r.origins = plan + leaves;
    auto tree = new_tree(ctx, (uint32_t)nodes.size(), c.n2);
    int32_t i1 = 0;
    for (const auto& kv : res) tree->root[kv.first] = i1++;
    if (n_items) k_copy_nodes1<<<blocks(n_items), 256, 0, st>>>(av, bv, n_items, d_nodes, at, tree->v);
    if (c.n2) k_copy_nodes2<<<c.n2, 256, 0, st>>>(av, bv, w.n_a, refs2, w.flipped, place, tree->v);
    BS_HIP(hipGetLastError());
    if (c.tiles) {
        int4* tile_org = S.as<int4>(S_TREE_TILES, c.tiles);
        float* tile_val = S.as<float>(S_TREE_TILE_VAL, c.tiles);
        k_item_write<<<blocks(n_items, 4), 256, 0, st>>>(av, bv, n_items, d_nodes, w.flipped, tile_at, tile_org, tile_val,
                                                         nullptr, nullptr);
        BS_HIP(hipGetLastError());
        r.tiles = read_tiles(ctx, tile_org, tile_val, c.tiles);
    }
    r.tree = std::move(tree);
}

TreeCsg tree_csg(bs_ctx* ctx, const DeviceTree& a, const DeviceTree& b, const TreeOperand& la, const TreeOperand& lb,
                 CsgOp op) {
    TreeCsg r;
    try {
        plan_csg(ctx, a, b, la, lb, op, r);
    } catch (const Error& e) {
        if (!e.out_of_memory) throw;
    }
    return r;
}

std::unique_ptr<DeviceTree> tree_after_offset(bs_ctx* ctx, const DeviceTree& old, const int4* old_origins,
                                              const uint32_t* keep, uint64_t n_old, const int4* origins, uint64_t n) {
    hipStream_t st = ctx->stream;
    std::unique_ptr<DeviceTree> t;
    try {
        t = tree_from_leaves(ctx, origins, n, {});
        if (!t) return nullptr;
        std::vector<int2> match;
        for (const auto& kv : t->root) {
            const auto it = old.root.find(kv.first);
            if (it != old.root.end()) match.push_back(make_int2(kv.second, it->second));
        }
        if (!match.empty() && n_old) {
            const int2* d_match = upload(ctx, S_TREE_ROOTS, match);
            uint32_t* kept = ctx->scratch.as<uint32_t>(S_TREE_ZERO, (uint64_t)old.v.n1 + old.v.n2);
            uint32_t* kept2 = kept + old.v.n1;
            BS_HIP(hipMemsetAsync(kept, 0, sizeof(uint32_t) * ((uint64_t)old.v.n1 + old.v.n2), st));
            k_node_kept<<<blocks(n_old), 256, 0, st>>>(n_old, old_origins, keep, old.v, d_match, (uint32_t)match.size(),
                                                       kept, kept2);
            k_keep_tiles<<<(unsigned)match.size() * (N1_SLOTS / 256), 256, 0, st>>>(old.v, d_match, kept, kept2, t->v);
            BS_HIP(hipGetLastError());
            BS_HIP(hipStreamSynchronize(st));
        }
    } catch (const Error& e) {
        if (!e.out_of_memory) throw;
        (void)hipStreamSynchronize(st);
        return nullptr;
    }
    t->pending = nullptr;
    return t;
}

uint64_t tree_units(bs_ctx* ctx, const DeviceTree& t, const int64_t** units, std::vector<TileRec>& tiles) {
    hipStream_t st = ctx->stream;
    Scratch& S = ctx->scratch;
    std::vector<int32_t> nodes;
    for (const auto& kv : t.root) nodes.push_back(kv.second);
    const uint32_t n_items = (uint32_t)(nodes.size() * N1_SLOTS);
    tiles.clear();
    *units = nullptr;
    if (!n_items) return 0;
    const TreeView none{};
    const int32_t* d_nodes = upload(ctx, S_TREE_NODES, nodes);
    uint32_t* branch = S.as<uint32_t>(S_TREE_ITEMS, 6 * ((uint64_t)n_items + 1));
    uint32_t *at = branch + n_items + 1, *tile_n = at + n_items + 1, *tile_at = tile_n + n_items + 1,
             *unit_n = tile_at + n_items + 1, *unit_at = unit_n + n_items + 1;
    int32_t* refs2 = S.as<int32_t>(S_TREE_REFS, (uint64_t)t.v.n2 + 1);
    uint32_t* node_tiles = S.as<uint32_t>(S_TREE_NODE_N, 2 * ((uint64_t)t.v.n2 + 1));
    uint32_t* node_units = node_tiles + t.v.n2 + 1;
    const unsigned ib = blocks((uint64_t)n_items + 1);
    k_item_branch<<<ib, 256, 0, st>>>(t.v, none, n_items, d_nodes, branch);
    BS_HIP(hipGetLastError());
    scan_u32(ctx, branch, at, (uint64_t)n_items + 1);
    k_item_refs<<<ib, 256, 0, st>>>(t.v, none, n_items, d_nodes, branch, at, refs2);
    if (t.v.n2) k_node_mark<<<t.v.n2, 256, 0, st>>>(t.v, none, 0, refs2, at + n_items, nullptr, node_tiles, node_units);
    k_item_counts<<<ib, 256, 0, st>>>(t.v, none, n_items, d_nodes, at, node_tiles, tile_n);
    k_item_counts<<<ib, 256, 0, st>>>(t.v, none, n_items, d_nodes, at, node_units, unit_n);
    BS_HIP(hipGetLastError());
    scan_u32(ctx, tile_n, tile_at, (uint64_t)n_items + 1);
    scan_u32(ctx, unit_n, unit_at, (uint64_t)n_items + 1);
    uint32_t* back = static_cast<uint32_t*>(pinned_words(ctx, 2));
    BS_HIP(hipMemcpyAsync(back, tile_at + n_items, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipMemcpyAsync(back + 1, unit_at + n_items, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    BS_HIP(hipStreamSynchronize(st));
    const uint32_t n_tiles = back[0], n_units = back[1];
    if (!n_units) return 0;
    int64_t* out = S.as<int64_t>(S_MC_UNITS, n_units);
    int4* tile_org = S.as<int4>(S_TREE_TILES, n_tiles);
    float* tile_val = S.as<float>(S_TREE_TILE_VAL, n_tiles);
    k_item_write<<<blocks(n_items, 4), 256, 0, st>>>(t.v, none, n_items, d_nodes, nullptr, tile_at, tile_org, tile_val,
                                                     unit_at, out);
    BS_HIP(hipGetLastError());
    tiles = read_tiles(ctx, tile_org, tile_val, n_tiles);
    *units = out;
    return n_units;
}

}  // namespace bs
