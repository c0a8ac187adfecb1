// query_kernels.h -- point queries on the N^3 tree (reference: svox/csrc/svox_kernel.cu:42-115).
//
// query / query-backward / assign run in two phases per wavefront:
//   1. one lane per point: world->tree transform, clamp, root-to-leaf walk.  For an fp32 octree the
//      walk runs on integer cell coordinates and reads the child rows of the first `lds_nodes`
//      nodes (the top of the tree: nodes are stored parents-before-children) from LDS;
//   2. the 64 lanes together move the 64 leaf records: the output (or grad_output / values) of a
//      wavefront is one contiguous run of 64*K scalars, so consecutive lanes touch consecutive
//      addresses on that side and K-long runs on the tree side, instead of one lane copying K
//      scalars in a serial loop.
// Blocks are persistent (grid-stride over tiles of 256 points) so the LDS copy of the child rows is
// filled once per block.
#pragma once

#include "tree_walk.h"

namespace svox {

constexpr int kQueryThreads = 256;
constexpr int kWave = 64;

enum QueryMode { kQueryGather = 0, kQueryScatterAdd = 1, kQueryAssign = 2 };
typedef unsigned int Piece16 __attribute__((ext_vector_type(4)));   // 16 bytes as the non-temporal builtins take them

// Leaf of a point (packed leaf id or -1).  lds_child: the child rows of the nodes below lds_nodes; walk: the child table or its
// copy with kLastNodeBit (octrees).
template <typename T, bool kOctree>
__device__ __forceinline__ int64_t query_leaf(const TreeDev<T>& tr, const int32_t* __restrict__ walk, const int32_t* lds_child, int32_t lds_nodes,
                                              const T* offset, const T* scaling, const T* __restrict__ points, int64_t q,
                                              bool valid) {
    T xyz[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) xyz[k] = valid ? points[q * 3 + k] : T(0);
    transform_coord(xyz, offset, scaling);
    int64_t leaf = -1;
    if constexpr (kOctree) {
        if (valid)
            leaf = descend_octree(walk, lds_child, lds_nodes, tr.capacity, cell_coord(clamp01(xyz[0])),
                                  cell_coord(clamp01(xyz[1])), cell_coord(clamp01(xyz[2])), walk != tr.child);
    }
    if (valid && leaf < 0) {   // deeper than the integer coordinates resolve: once more with the floating-point walk
        T cube;
        int levels;
        leaf = descend_generic<T>(tr.child, tr.capacity, tr.N, xyz, &cube, &levels);
    }
    return leaf;
}

// The rows of one run, scalar by scalar: flat index f = p * Kx + e of the run's contiguous side (`lin`) to lane f mod 64,
// row_leaf(p) the leaf of row p (called by every lane).  kBatch scalars per lane are read before the first is written:
// the compiler must assume that the two sides overlap, so it would wait for every read before the write behind it
// (1 000 points, 49 scalars: 32.4 -> 6.7 us, with query_few_kernel's smaller wavefronts).
template <typename T, int MODE, class RowLeaf>
__device__ __forceinline__ void move_rows(int lane, int n_rows, int32_t Kx, int64_t row, RowLeaf&& row_leaf, T* data, T* lin,
                                          T* target) {
    constexpr int kBatch = 4;
    const int total = n_rows * Kx;
    const int step_e = kWave % Kx, step_p = kWave / Kx;
    int p = lane / Kx, e = lane % Kx;
    for (int f0 = 0; f0 < total; f0 += kWave * kBatch) {
        T buf[kBatch];
        int64_t at[kBatch];   // on the tree's side; -1: no leaf (malformed tree) or past the end
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const int f = f0 + b * kWave + lane;
            const int64_t leaf = row_leaf(f < total ? p : 0);
            at[b] = f < total && leaf >= 0 ? leaf * row + e : -1;
            buf[b] = T(0);
            if (MODE == kQueryGather) {
                if (at[b] >= 0) buf[b] = data[at[b]];
            } else {
                if (at[b] >= 0) buf[b] = __builtin_nontemporal_load(&lin[f]);
            }
            e += step_e;
            p += step_p;
            if (e >= Kx) {
                e -= Kx;
                p += 1;
            }
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const int f = f0 + b * kWave + lane;
            if (MODE == kQueryGather) {
                if (f < total) __builtin_nontemporal_store(buf[b], &lin[f]);
            } else if (MODE == kQueryScatterAdd) {
                if (at[b] >= 0) atomicAdd(target + at[b], buf[b]);
            } else {
                if (at[b] >= 0) data[at[b]] = buf[b];
            }
        }
    }
}

// MODE gather:      values[q][0..Kx) = data[leaf_q][0..Kx), ids[q] = leaf_q        (Kx = K)
// MODE scatter-add: target[leaf_q][0..Kx) += values[q][0..Kx)   (target row stride Kx); with ids given, leaf_q = ids[q], and the
//                   points are not looked up
// MODE assign:      data[leaf_q][0..Kx) = values[q][0..Kx)      (tree row stride K)
// The leaf the scatter was told of, -1 if it is none of the tree's.
template <typename T>
__device__ __forceinline__ int64_t known_leaf(const TreeDev<T>& tr, const int64_t* __restrict__ ids, int64_t q, bool valid) {
    const int64_t leaf = valid ? ids[q] : -1;
    return leaf < tr.capacity * tr.N * tr.N * tr.N ? leaf : -1;
}

template <typename T, int MODE, bool kOctree>
__global__ __launch_bounds__(kQueryThreads) void query_kernel(TreeDev<T> tr, const T* __restrict__ points,
                                                              int64_t n_points, T* values, T* target,
                                                              int64_t* __restrict__ ids, int32_t Kx,
                                                              const int32_t* __restrict__ walk, int32_t lds_nodes) {
    extern __shared__ int32_t lds_child[];
    if constexpr (kOctree) {
        for (int i = threadIdx.x; i < lds_nodes * 8; i += kQueryThreads) lds_child[i] = walk[i];
        __syncthreads();
    }
    T offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t n_tiles = (n_points + kQueryThreads - 1) / kQueryThreads;
    const int64_t row = (MODE == kQueryAssign) ? (int64_t)tr.K : (int64_t)Kx;
    // records and output rows start on 16-byte boundaries: move 16-byte pieces
    const bool vec16 = (Kx * (int)sizeof(T)) % 16 == 0 && (((uintptr_t)tr.data | (uintptr_t)values) & 15u) == 0;

    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        // a wavefront owns 64 consecutive points; lane l walks point l
        const int64_t wave_base = tile * kQueryThreads + (int64_t)(threadIdx.x / kWave) * kWave;
        const int64_t q = wave_base + lane;
        const int64_t leaf = MODE == kQueryScatterAdd && ids ? known_leaf(tr, ids, q, q < n_points)
                                                             : query_leaf<T, kOctree>(tr, walk, lds_child, lds_nodes, offset, scaling, points, q, q < n_points);
        if (MODE == kQueryGather && ids && q < n_points) ids[q] = leaf;
        // phase 2: the 64 rows of the run, flat index f = p * Kx + e
        const int64_t remaining = n_points - wave_base;
        const int n_rows = remaining < kWave ? (int)(remaining > 0 ? remaining : 0) : kWave;
        T* lin = values + wave_base * Kx;
        const int leaf_lo = (int)(leaf & 0xffffffff), leaf_hi = (int)(leaf >> 32);
        if (MODE == kQueryGather && vec16) {
            // 16-byte pieces: a record is `pieces` of them, and kBatch loads per lane are in flight
            // before the first store (the compiler must assume that the output aliases the tree)
            constexpr int kPer = 16 / (int)sizeof(T);
            constexpr int kBatch = 4;
            const int pieces = Kx / kPer;
            const int total = n_rows * pieces;
            const int step_e = kWave % pieces, step_p = kWave / pieces;
            int p = lane / pieces, e = lane % pieces;
            uint4* lin16 = (uint4*)lin;
            for (int f0 = 0; f0 < total; f0 += kWave * kBatch) {
                uint4 buf[kBatch];
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    const int f = f0 + b * kWave + lane;
                    // every lane takes part in the shuffle; rows past the end read lane 0's leaf
                    const int src_lane = f < total ? p : 0;
                    const int lo = __shfl(leaf_lo, src_lane);
                    const int hi = __shfl(leaf_hi, src_lane);
                    const int64_t lf = ((int64_t)hi << 32) | (uint32_t)lo;
                    buf[b] = make_uint4(0u, 0u, 0u, 0u);
                    if (f < total && lf >= 0) buf[b] = ((const uint4*)(tr.data + lf * row))[e];
                    e += step_e;
                    p += step_p;
                    if (e >= pieces) {
                        e -= pieces;
                        p += 1;
                    }
                }
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    const int f = f0 + b * kWave + lane;
                    // (stored past the caches' keep-list: the output is written once, and the tree it is gathered
                    // from should stay in the last-level cache: 4 Mi points of a 268 MB tree 0.346 -> 0.332 ms)
                    if (f < total) __builtin_nontemporal_store((Piece16){buf[b].x, buf[b].y, buf[b].z, buf[b].w}, (Piece16*)lin16 + f);
                }
            }
        } else {
            move_rows<T, MODE>(lane, n_rows, Kx, row, [&](int p) {
                const int lo = __shfl(leaf_lo, p), hi = __shfl(leaf_hi, p);
                return ((int64_t)hi << 32) | (uint32_t)lo;
            }, tr.data, lin, target);
        }
    }
}

// Few points: 16 to a wavefront, four lanes walking each, nothing staged in LDS -- a call this small is one chain of
// dependent reads, and the shorter its pieces the sooner it is over.  (Before, as two runs of 64 points per wavefront:
// 1 000 points of a 32^3 SH4 tree 13.7 -> 4.7 us.)
constexpr int kFewPoints = 16;
template <typename T, int MODE, bool kOctree>
__global__ __launch_bounds__(kWave) void query_few_kernel(TreeDev<T> tr, const T* __restrict__ points, int64_t n_points,
                                                          T* values, T* target, int64_t* __restrict__ ids, int32_t Kx) {
    const int lane = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * kFewPoints, q = base + lane / (kWave / kFewPoints);
    const bool valid = q < n_points;
    T offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const int64_t leaf = MODE == kQueryScatterAdd && ids ? known_leaf(tr, ids, q, valid)
                                                         : query_leaf<T, kOctree>(tr, tr.child, nullptr, 0, offset, scaling, points, q, valid);
    if (MODE == kQueryGather && ids && valid && lane % (kWave / kFewPoints) == 0) ids[q] = leaf;
    const int64_t remaining = n_points - base;
    const int n_rows = remaining < kFewPoints ? (int)remaining : kFewPoints;
    const int leaf_lo = (int)(leaf & 0xffffffff), leaf_hi = (int)(leaf >> 32);
    move_rows<T, MODE>(lane, n_rows, Kx, MODE == kQueryAssign ? (int64_t)tr.K : (int64_t)Kx, [&](int p) {
        const int from = p * (kWave / kFewPoints);
        const int lo = __shfl(leaf_lo, from), hi = __shfl(leaf_hi, from);
        return ((int64_t)hi << 32) | (uint32_t)lo;
    }, tr.data, values + base * Kx, target);
}

// The octree's child table with kLastNodeBit (tree_walk.h).  One thread per cell.
static __global__ __launch_bounds__(256) void last_nodes_kernel(const int32_t* __restrict__ child, int32_t capacity,
                                                                int32_t* __restrict__ walk) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    if (i >= capacity * 8ll) return;
    int32_t c = child[i];
    const int64_t node = (i >> 3) + c;
    if (c >= kLastNodeBit) {
        c = kLastNodeBit - 1;   // (a malformed tree's: still past the end)
    } else if (c > 0 && node < capacity) {
        const int4 lo = ((const int4*)child)[node * 2], hi = ((const int4*)child)[node * 2 + 1];
        if ((lo.x | lo.y | lo.z | lo.w | hi.x | hi.y | hi.z | hi.w) == 0) c |= kLastNodeBit;
    }
    walk[i] = c;
}

// The walk table (kWalkNodeBits) of an octree from its child table or a copy with marks, which begins at a multiple of 16 bytes.  One thread per cell.
static __global__ __launch_bounds__(256) void walk_table_kernel(const int32_t* __restrict__ child, int32_t capacity,
                                                                uint32_t* __restrict__ walk) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    const int32_t c = i < capacity * 8ll ? child[i] : 0;
    // the rows of nodes that have leaves only are read by nobody (but the root's)
    const unsigned long long inner = __ballot(c > 0);
    const bool last = (inner >> (threadIdx.x & 56u) & 0xffull) == 0;
    if (i >= capacity * 8ll || (last && i >= 8)) return;
    uint32_t word = c < 0 ? kWalkEmptyLeaf : 0u;
    if (c > 0) {
        const int64_t node = (i >> 3) + c;
        word = kWalkNodes;   // (a malformed tree's: past the end of every table)
        if (node < capacity) {
            const int4 lo = ((const int4*)child)[node * 2], hi = ((const int4*)child)[node * 2 + 1];
            word = (uint32_t)c;
            if (max(max(max(lo.x, lo.y), max(lo.z, lo.w)), max(max(hi.x, hi.y), max(hi.z, hi.w))) <= 0) {
                const uint32_t marks = (lo.x < 0 ? 1u : 0u) | (lo.y < 0 ? 2u : 0u) | (lo.z < 0 ? 4u : 0u) | (lo.w < 0 ? 8u : 0u) |
                                       (hi.x < 0 ? 16u : 0u) | (hi.y < 0 ? 32u : 0u) | (hi.z < 0 ? 64u : 0u) | (hi.w < 0 ? 128u : 0u);
                word |= (uint32_t)kLastNodeBit | marks << kWalkNodeBits;
            }
        }
    }
    walk[i] = word;
}

// calc_corner_kernel, svox_kernel.cu:91-115: climb parent links from the leaf's node to the
// root; per level result = (result + cell index) / N.
template <typename T>
__global__ __launch_bounds__(kQueryThreads) void corners_kernel(const int32_t* __restrict__ parent_depth,
                                                                int32_t N, int64_t capacity,
                                                                const int64_t* __restrict__ indexer,
                                                                int64_t n_leaves, T* __restrict__ out) {
    const int64_t q = blockIdx.x * (int64_t)kQueryThreads + threadIdx.x;
    if (q >= n_leaves) return;
    int32_t node = (int32_t)indexer[q * 4];
    int32_t c[3] = {(int32_t)indexer[q * 4 + 1], (int32_t)indexer[q * 4 + 2],
                    (int32_t)indexer[q * 4 + 3]};
    T res[3] = {T(0), T(0), T(0)};
    const T Nf = (T)N;
    for (int guard = 0; guard < kMaxWalkLevels; ++guard) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            res[i] += (T)c[i];
            res[i] /= Nf;
        }
        if (node <= 0 || node >= capacity) break;
        int32_t packed = parent_depth[(int64_t)node * 2];
        c[2] = packed % N;
        packed /= N;
        c[1] = packed % N;
        packed /= N;
        c[0] = packed % N;
        node = packed / N;
    }
    out[q * 3] = res[0];
    out[q * 3 + 1] = res[1];
    out[q * 3 + 2] = res[2];
}

// The child table with the leaves a render skips marked: a leaf cell (child == 0) whose density -- after the shifted
// softplus of rt_kernel.cu:276-277 where `softplus` says so -- is not > thresh receives SVOX_EMPTY_LEAF, every other
// cell its child entry.  One thread per cell.
template <typename T>
__global__ __launch_bounds__(256) void mark_leaves_kernel(const T* __restrict__ data, const int32_t* __restrict__ child,
                                                          int64_t cells, int K, T thresh, bool softplus,
                                                          int32_t* __restrict__ marks) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    if (i >= cells) return;
    const int32_t c = child[i];
    int32_t m = c;
    if (c == 0) {
        // read past the caches' keep-list: a density is 4 bytes of a line nobody asks for again soon, and 0.7 GB of
        // such lines would push the child table and the marks out of L2 ahead of the render that follows
        // (8 poses of 800x800: marking 0.141 -> 0.129 ms, the render call as a whole 0.811 -> 0.790 ms)
        T sigma = __builtin_nontemporal_load(&data[i * K + (K - 1)]);
        if (softplus) sigma = softplus_m1(sigma);
        m = sigma > thresh ? 0 : SVOX_EMPTY_LEAF;
    }
    marks[i] = m;
}

// Zero-fill used in place of a memset so that a caller may capture the call in a graph.  16 bytes a thread and no loop: the
// blocks finish in the order they start, so what is written at any time lies close together (1.21 GB: 178 us, 6.8 TB/s;
// 8192 blocks that stride through all of it 210 to 272 us, 16 pieces a thread 215 us, non-temporal stores 199 us and more;
// 268 MB: 34 us instead of 37).
__global__ __launch_bounds__(256) void zero_kernel(uint4* __restrict__ p16, int64_t n16,
                                                   uint32_t* __restrict__ tail, int n_tail) {
    const int64_t i = blockIdx.x * 256ll + threadIdx.x;
    if (i < n16) p16[i] = make_uint4(0u, 0u, 0u, 0u);
    if (blockIdx.x == 0 && (int)threadIdx.x < n_tail) tail[threadIdx.x] = 0u;
}

}  // namespace svox
