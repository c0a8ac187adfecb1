// tree_walk.h -- root-to-leaf descent of the N^3 tree (reference: query_single_from_root,
// svox/csrc/include/common.cuh:52-90).
//
// Two formulations that return the same leaf and the same leaf-local position:
//
//   descend_generic<T>   the reference's floating-point walk (multiply by N, floor, subtract) for
//                        any branching factor and scalar type.
//
//   OctreeCursor         (march_kernels.h) N == 2, fp32.  Multiplying by 2, taking the floor and subtracting it are
//                        exact in binary floating point, so the cell chosen at level l is bit
//                        (24 - l) of trunc(p * 2^24) and the leaf-local position at depth L is
//                        frac(p * 2^L).  The walk therefore runs on integers, and because a ray's
//                        next sample is close to the previous one, it restarts from the deepest
//                        node whose cell still contains the new point instead of from the root:
//                        the child rows of the previous path are kept in LDS, one column per lane
//                        (keeping only the deepest four levels in registers was measured slower:
//                        more restarts from the root and select chains on the critical path).
#pragma once

#include "fpmath.h"

namespace svox {

constexpr int kMaxWalkLevels = 64;   // a deeper (malformed) tree ends the walk with leaf -1
constexpr int kCoordBits = 24;       // integer cell coordinates hold 24 levels of an octree
constexpr int kPathLevels = 11;      // levels of the previous path remembered per lane

template <typename T>
struct TreeDev {
    T* data;
    const int32_t* child;
    const int32_t* parent_depth;
    const T* extra;
    const T* offset;   // may be null: zero
    const T* scaling;  // may be null: one
    T* weight_accum;
    const int32_t* walk;   // a walk table of the octree (kWalkNodeBits), or null
    bool walk_marked;      // ... made from marks
    int64_t capacity;
    int32_t N;
    int32_t K;
    int32_t extra_cols;
    int32_t weight_accum_max;
};

// The octree march kernels may be given, in place of the child table, the copy svox_mark_empty_leaves
// made of it, in which a negative entry is a leaf whose density is not > 0.  Their walk reads every
// negative entry so (the child table of a well-formed tree has none on a cell that can be reached)
// and sets this bit in the leaf id it returns for such a leaf (octree leaf ids stay below 2^30).
constexpr int32_t kEmptyLeafBit = 1 << 30;

// The point queries may be given a copy of an octree's child table in which an entry whose node has leaves only carries this
// bit: the row of such a node, where most searches end, need not be read.  (Entries of a well-formed table stay below 2^28.)
constexpr int32_t kLastNodeBit = 1 << 30;

// A walk table: the child table of an octree of fewer than 2^kWalkNodeBits nodes, or its copy with marks, made over for the march
// (walk_table_kernel).  The entry of a cell whose node has leaves only says so (kLastNodeBit), and in the bits from kWalkNodeBits on which of
// the eight are marked empty: the row of such a node, the one in eight of the table's that a ray finds in no cache, need not be read, and is
// not written.  A marked leaf is the sign bit and the same eight bits, all set.  So the sum of a node's number and an entry of its
// row is the child's number, kLastNodeBit and its marks: a word of the walk.
constexpr int kWalkNodeBits = 22;
constexpr uint32_t kWalkNodes = (1u << kWalkNodeBits) - 1u;
constexpr uint32_t kWalkEmptyLeaf = 0x80000000u | 0xffu << kWalkNodeBits;

template <typename T>
__device__ __forceinline__ void load_transform(const TreeDev<T>& tr, T* offset, T* scaling) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        offset[i] = tr.offset ? tr.offset[i] : T(0);
        scaling[i] = tr.scaling ? tr.scaling[i] : T(1);
    }
}

// transform_coord, common.cuh:43-50
template <typename T>
__device__ __forceinline__ void transform_coord(T* q, const T* offset, const T* scaling) {
#pragma unroll
    for (int i = 0; i < 3; ++i) q[i] = fma_(scaling[i], q[i], offset[i]);
}

// The reference's walk.  xyz: in = point in tree coordinates, out = position inside the leaf.
// Returns the packed leaf id node*N^3 + u*N^2 + v*N + w, or -1 for a malformed tree.
template <typename T>
__device__ __forceinline__ int64_t descend_generic(const int32_t* __restrict__ child,
                                                   int64_t capacity, int32_t Ni, T* xyz,
                                                   T* cube_sz, int* levels, bool marked = false) {
    const T N = (T)Ni;
    xyz[0] = clamp01(xyz[0]);
    xyz[1] = clamp01(xyz[1]);
    xyz[2] = clamp01(xyz[2]);
    int64_t node = 0;
    *cube_sz = N;
    for (int level = 1; level <= kMaxWalkLevels; ++level) {
        xyz[0] *= N;
        xyz[1] *= N;
        xyz[2] *= N;
        const int32_t u = (int32_t)floor_(xyz[0]);
        const int32_t v = (int32_t)floor_(xyz[1]);
        const int32_t w = (int32_t)floor_(xyz[2]);
        xyz[0] -= (T)u;
        xyz[1] -= (T)v;
        xyz[2] -= (T)w;
        const int64_t cell = ((node * Ni + u) * Ni + v) * Ni + w;
        const int32_t skip = child[cell];
        if (skip == 0 || (marked && skip < 0)) {
            *levels = level;
            return cell;
        }
        *cube_sz *= N;
        node += skip;
        if (node < 0 || node >= capacity) return -1;
    }
    return -1;
}

// Integer cell coordinates of a clamped point: trunc(p * 2^24), exact.
__device__ __forceinline__ uint32_t cell_coord(float pc) { return (uint32_t)(pc * 16777216.0f); }

__device__ __forceinline__ int cell_at(uint32_t ix, uint32_t iy, uint32_t iz, int level) {
    const unsigned s = (unsigned)(kCoordBits - level);
    const unsigned bx = __builtin_amdgcn_ubfe(ix, s, 1u), by = __builtin_amdgcn_ubfe(iy, s, 1u),
                   bz = __builtin_amdgcn_ubfe(iz, s, 1u);
    return (int)((((bx << 1) | by) << 1) | bz);
}

// One child entry for the point queries: from the rows staged in LDS for nodes below lds_nodes, else
// from memory.  Written as an LDS read that every lane makes (of entry 0 where the node is not
// staged) and a memory read under a condition: a choice between the two pointers would leave the
// compiler with one load through the generic address path, which is the slower way into LDS.
__device__ __forceinline__ int32_t child_entry(const int32_t* __restrict__ child, const int32_t* lds_child,
                                               int32_t lds_nodes, int32_t node, int32_t cell) {
    const bool staged = node < lds_nodes;
    int32_t skip = lds_child[staged ? cell : 0];
    asm volatile("" : "+v"(skip));   // (keeps the two reads apart)
    if (!staged) skip = child[cell];
    return skip;
}

// Octree walk over integer coordinates with no path memory (point queries).
// `lds_child` holds the child rows of nodes [0, lds_nodes); deeper nodes are read from memory (lds_nodes 0: all of them).
// `marked`: `child` is the copy with kLastNodeBit; in the table itself an entry that large leads past the end (malformed tree).
// Returns the leaf cell index node*8 + cell, or -1.
__device__ __forceinline__ int32_t descend_octree(const int32_t* __restrict__ child, const int32_t* lds_child,
                                                  int32_t lds_nodes, int64_t capacity, uint32_t ix, uint32_t iy,
                                                  uint32_t iz, bool marked) {
    int32_t node = 0, leaf = -1;
    bool live = true;
    for (int level = 1; level <= kCoordBits && live; ++level) {
        const int32_t cell = node * 8 + cell_at(ix, iy, iz, level);
        const int32_t skip = lds_child ? child_entry(child, lds_child, lds_nodes, node, cell) : child[cell];
        if (skip == 0) {
            leaf = cell;
            live = false;
        } else {
            const bool last = marked && skip >= kLastNodeBit;
            node = (int32_t)((uint32_t)node + (uint32_t)(last ? skip - kLastNodeBit : skip));
            if (node < 0 || node >= capacity) {
                live = false;
            } else if (last) {
                if (level < kCoordBits) leaf = node * 8 + cell_at(ix, iy, iz, level + 1);
                live = false;
            }
        }
    }
    return leaf;  // (-1 also where the tree is deeper than the integer coordinates resolve)
}

}  // namespace svox
