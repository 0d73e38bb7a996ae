// The upper levels of a volume's grid on the device: the same tree as Topology
// (topology.hpp), its 32^3-slot and 16^3-slot nodes as flat arrays in device
// memory and only the root map on the host.  CSG, offset and the visit order
// of marching cubes work on it; Topology is the host's form for the operations
// that walk the tree voxel by voxel, and for trees that do not fit here.
#pragma once
#include <hip/hip_runtime.h>

#include <array>
#include <cstdint>
#include <map>
#include <memory>
#include <vector>

#include "topology.hpp"

struct bs_ctx;
struct bs_volume;

namespace bs {

constexpr uint32_t N1_SLOTS = Node1::SIZE, N2_SLOTS = Node2::SIZE;

// Slot s of 32^3 node i is at [i * N1_SLOTS + s], of 16^3 node i at
// [i * N2_SLOTS + s]; origins are (x, y, z, 0).
struct TreeView {
    uint8_t *kind1, *kind2;
    float *tile1, *tile2;
    int32_t *child1, *child2;  // 16^3 node, leaf
    int4 *org1, *org2;
    uint32_t n1, n2;
};

struct DeviceTree {
    std::map<Topology::Key, int32_t> root;  // -> 32^3 node
    TreeView v{};
    void* block = nullptr;
    hipStream_t pending = nullptr;  // a stream that may still work on it, within a call
    DeviceTree() = default;
    DeviceTree(const DeviceTree&) = delete;
    DeviceTree& operator=(const DeviceTree&) = delete;
    ~DeviceTree();
};

// The volume's tree on the device, made from its leaves (and tiles) or from its
// Topology; nullptr when it does not fit: more than 2^24 128^3 blocks in the box
// of the leaves, 256 root blocks in it, 2^16 nodes, or device memory.  With `no_gap` nullptr also,
// and nothing is made, where the root's flood fill may close a gap on a z line
// between two root entries (root_node/flood_fill.rs:14-41), which is left to
// Topology.
DeviceTree* ensure_tree(bs_ctx* ctx, bs_volume* v, bool no_gap = false);
// A volume that has a form of its tree, with such a gap in its root.
bool known_root_gap(const bs_volume* v);
// Throws for a volume whose upper levels a failed call lost.
void require_tree(const bs_volume* v);
std::unique_ptr<DeviceTree> clone_tree(const DeviceTree& t);
// The host's form of a volume's device tree.
std::unique_ptr<Topology> download_tree(bs_ctx* ctx, const bs_volume* v);

// Flood fill of both internal levels (internal_node/flood_fill.rs:17-75);
// leaf_flags: bit 0 first value negative, bit 1 last value negative.
void tree_flood_fill(bs_ctx* ctx, const DeviceTree& t, const uint8_t* leaf_flags);

// CSG of two flood-filled trees (root_node/csg.rs:9-58, internal_node/csg.rs:
// 68-162) with `a` as self.  The slot rules work on a copy of a's, so that a call
// that fails leaves both operands' trees as they were.  The result's leaves in origin
// order: refs[i] = (leaf of a, leaf of b, LEAF_* | negate << 8, 0), origins[i].
// No tree when the result has more than 256 root blocks or 2^16 nodes, or when
// device memory runs out.
struct TreeOperand {
    const int4* origins;
    const uint8_t* flags;  // bit 2: mask empty
    uint64_t n;
};
struct TreeCsg {
    std::unique_ptr<DeviceTree> tree;
    std::unique_ptr<DeviceTree> work;  // the copy, read until the stream is done
    std::vector<TileRec> tiles;        // active tiles in tree order
    uint64_t n_out = 0, n_paired = 0;
    const int4 *refs = nullptr, *origins = nullptr;  // context scratch
};
TreeCsg tree_csg(bs_ctx* ctx, const DeviceTree& a, const DeviceTree& b, const TreeOperand& la, const TreeOperand& lb,
                 CsgOp op);

// The tree after Volume::offset (see Topology::after_offset) of a volume whose
// tree is `old`: the nodes of the result's leaves, with the tile values of the
// nodes that kept a leaf (keep: per leaf of the old volume); nullptr when it does
// not fit (see ensure_tree).
std::unique_ptr<DeviceTree> tree_after_offset(bs_ctx* ctx, const DeviceTree& old, const int4* old_origins,
                                              const uint32_t* keep, uint64_t n_old, const int4* origins, uint64_t n);

// The serial visit order (see Topology::visit_units): units (context scratch)
// and the active tiles they refer to.
uint64_t tree_units(bs_ctx* ctx, const DeviceTree& t, const int64_t** units, std::vector<TileRec>& tiles);

}  // namespace bs
