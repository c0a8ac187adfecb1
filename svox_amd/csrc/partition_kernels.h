// partition_kernels.h -- the gradient of a point query by rows of the tree instead of by points.
//
// Adding a point's gradient row to its leaf with atomics (query_kernel) costs the memory system a request per 64 bytes,
// about 16 a nanosecond, after the gradient has been cleared.  Where the points are many beside the tree, it is cheaper to
// bring the points of neighbouring leaves together and write every row of the gradient once:
//   count    every block of points counts how many fall into each bin of rows (a bin: a few thousand rows), from the leaves
//            the query found where the caller kept them (28 -> 9 us for the points below);
//   offsets  prefix sums of the counts over the blocks, bin by bin;
//   place    (row, point) pairs, bin after bin;
//   collect  a block per tile of rows (up to 256) picks its pairs out of the bin, puts them in order and
//            writes the sums.
// 1 000 003 points, 128^3 SH9 tree: cleared in 38 us and added to in 168 us -> counted in 28, placed in 20, collected in 89 us.
#pragma once

#include "query_kernels.h"

namespace svox {

constexpr int kPartThreads = 256;
constexpr int kPointThreads = 1024;   // of the passes over points, which wait for memory
constexpr int kPartBins = 2048;       // at most
constexpr int kPartBlocks = 512;      // blocks of points at most

struct Partition {
    int64_t n_points, n_rows;
    int32_t per_block;      // points of a block
    int32_t n_blocks, n_bins;
    int32_t bin_shift;      // rows of a bin, log2
    int32_t tile_shift;     // rows of a tile, log2
    const int64_t* ids;     // [n_points]: leaves of the points, where the caller knows them, or null
    int32_t* leaf;          // [n_points]
    int32_t* counts;        // [n_bins][n_blocks]
    int32_t* totals;        // [n_bins]
    int32_t* starts;        // [n_bins + 1]
    uint2* pairs;           // [n_points]: row, point
};

template <bool kOctree>
static __global__ __launch_bounds__(kPointThreads) void partition_count_kernel(TreeDev<float> tr, const float* __restrict__ points,
                                                                              Partition part, int32_t lds_nodes) {
    extern __shared__ int32_t lds_child[];   // the child rows of the first lds_nodes nodes, as in query_kernel
    __shared__ int32_t hist[kPartBins];
    for (int i = threadIdx.x; i < part.n_bins; i += kPointThreads) hist[i] = 0;
    if constexpr (kOctree) {
        for (int i = threadIdx.x; i < lds_nodes * 8; i += kPointThreads) lds_child[i] = tr.child[i];
    }
    __syncthreads();
    float offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const int64_t first = (int64_t)blockIdx.x * part.per_block;
    for (int i = threadIdx.x; i < part.per_block; i += kPointThreads) {
        const int64_t q = first + i;
        if (q >= part.n_points) break;
        const int64_t leaf = part.ids ? part.ids[q] : query_leaf<float, kOctree>(tr, tr.child, lds_child, lds_nodes, offset, scaling, points, q, true);
        // (no leaf: a malformed tree; and what is no row of this tree is left out)
        const bool ok = leaf >= 0 && leaf < part.n_rows;
        part.leaf[q] = ok ? (int32_t)leaf : -1;
        if (ok) atomicAdd(&hist[leaf >> part.bin_shift], 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < part.n_bins; i += kPointThreads) part.counts[(int64_t)i * part.n_blocks + blockIdx.x] = hist[i];
}

// exclusive prefix sum of v over the block's threads; `total`: the sum of all
template <int kThreads>
__device__ __forceinline__ int32_t block_prefix(int32_t v, int32_t* wave_sums, int32_t& total) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int32_t sum = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t other = __shfl_up(sum, off);
        if (lane >= off) sum += other;
    }
    if (lane == kWave - 1) wave_sums[wave] = sum;
    __syncthreads();
    int32_t before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; ++w) {
        if (w < wave) before += wave_sums[w];
        total += wave_sums[w];
    }
    __syncthreads();
    return before + sum - v;
}

static __global__ __launch_bounds__(kPartThreads) void partition_offsets_kernel(Partition part) {
    __shared__ int32_t wave_sums[kPartThreads / kWave];
    int32_t* const row = part.counts + (int64_t)blockIdx.x * part.n_blocks;
    int32_t run = 0;
    for (int b = 0; b < part.n_blocks; b += kPartThreads) {
        const int i = b + threadIdx.x;
        int32_t total;
        const int32_t before = block_prefix<kPartThreads>(i < part.n_blocks ? row[i] : 0, wave_sums, total);
        if (i < part.n_blocks) row[i] = run + before;
        run += total;
    }
    if (threadIdx.x == 0) part.totals[blockIdx.x] = run;
}

static __global__ __launch_bounds__(kPointThreads) void partition_place_kernel(Partition part) {
    __shared__ int32_t cursor[kPartBins];
    __shared__ int32_t wave_sums[kPointThreads / kWave];
    int32_t run = 0;
    for (int b = 0; b < part.n_bins; b += kPointThreads) {
        const int i = b + threadIdx.x;
        int32_t total;
        const int32_t before = block_prefix<kPointThreads>(i < part.n_bins ? part.totals[i] : 0, wave_sums, total);
        if (i < part.n_bins) {
            cursor[i] = run + before + part.counts[(int64_t)i * part.n_blocks + blockIdx.x];
            if (blockIdx.x == 0) part.starts[i] = run + before;
        }
        run += total;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) part.starts[part.n_bins] = run;
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * part.per_block;
    for (int i = threadIdx.x; i < part.per_block; i += kPointThreads) {
        const int64_t q = first + i;
        if (q >= part.n_points) break;
        const int32_t leaf = part.leaf[q];
        if (leaf >= 0) part.pairs[atomicAdd(&cursor[leaf >> part.bin_shift], 1)] = make_uint2((uint32_t)leaf, (uint32_t)q);
    }
}

// One tile of rows: grad[row][0..K) = sum of values[point][0..K) over the row's points (0 where there are none).
// The tile's pairs are picked out of the bin and put in order of their rows in LDS; then every thread sums pieces of rows,
// one piece of the tile after the other, so that the writes are one run.  What bounds it is that writing and the reading
// of the points' rows, which lie anywhere: every thread asks for the first points of kBatch pieces before it adds.
// (Adding the points' rows into the tile in LDS, with LDS atomics: 193 us instead of 89.)
// kVec: K is a multiple of 4 and both arrays start on 16-byte boundaries.
constexpr int kTileRows = 256;    // at most
constexpr int kTilePairs = 1024;  // pairs in LDS; a tile with more is summed in several rounds
template <bool kVec>
static __global__ __launch_bounds__(kPartThreads) void partition_collect_kernel(Partition part, const float* __restrict__ values,
                                                                                int32_t K, float* __restrict__ grad) {
    __shared__ uint2 pairs[kTilePairs];        // row of the tile | place among the row's << 16, point
    __shared__ uint32_t order[kTilePairs];     // points by row
    __shared__ int32_t start[kTileRows + 1];   // of a row's in `order`
    __shared__ int32_t wave_sums[kPartThreads / kWave];
    __shared__ int32_t n_pairs;
    static_assert(kTileRows == kPartThreads, "one thread per row of a tile");
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t first_row = (int64_t)blockIdx.x << part.tile_shift;
    const int64_t rows_left = part.n_rows - first_row;
    const int n_rows = rows_left < (1 << part.tile_shift) ? (int)rows_left : 1 << part.tile_shift;
    float* const out = grad + first_row * K;
    constexpr int kPer = kVec ? 4 : 1, kBatch = 4;
    const int pieces = K / kPer, n_pieces = n_rows * pieces;
    bool again = false;   // an earlier round has written the tile
    auto round = [&]() {
        __syncthreads();
        const int n = n_pairs;
        start[threadIdx.x] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kPartThreads) {
            const uint32_t row = pairs[i].x;
            pairs[i].x = row | (uint32_t)atomicAdd(&start[row], 1) << 16;
        }
        __syncthreads();
        int32_t total;
        const int32_t before = block_prefix<kPartThreads>(start[threadIdx.x], wave_sums, total);
        start[threadIdx.x] = before;
        if (threadIdx.x == 0) {
            start[kTileRows] = total;
            n_pairs = 0;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kPartThreads) order[start[pairs[i].x & 0xffffu] + (pairs[i].x >> 16)] = pairs[i].y;
        __syncthreads();
        for (int f0 = 0; f0 < n_pieces; f0 += kPartThreads * kBatch) {
            float4 sum[kBatch];
            int at[kBatch], to[kBatch], e[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int f = f0 + b * kPartThreads + (int)threadIdx.x;
                const int row = f < n_pieces ? f / pieces : kTileRows - 1;
                e[b] = (f - row * pieces) * kPer;
                at[b] = start[row];
                to[b] = f < n_pieces ? start[row + 1] : at[b];
                sum[b] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (at[b] < to[b]) {
                    const float* const from = values + (int64_t)order[at[b]] * K + e[b];
                    if constexpr (kVec)
                        sum[b] = *(const float4*)from;
                    else
                        sum[b].x = *from;
                }
            }
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int f = f0 + b * kPartThreads + (int)threadIdx.x;
                for (int i = at[b] + 1; i < to[b]; ++i) {
                    const float* const from = values + (int64_t)order[i] * K + e[b];
                    if constexpr (kVec) {
                        const float4 v = *(const float4*)from;
                        sum[b].x += v.x;
                        sum[b].y += v.y;
                        sum[b].z += v.z;
                        sum[b].w += v.w;
                    } else {
                        sum[b].x += *from;
                    }
                }
                if (f < n_pieces) {
                    if constexpr (kVec) {
                        float4* const to4 = (float4*)out + f;
                        if (again) {
                            const float4 v = *to4;
                            sum[b].x += v.x;
                            sum[b].y += v.y;
                            sum[b].z += v.z;
                            sum[b].w += v.w;
                        }
                        *to4 = sum[b];
                    } else {
                        out[f] = again ? out[f] + sum[b].x : sum[b].x;
                    }
                }
            }
        }
        again = true;
    };
    if (threadIdx.x == 0) n_pairs = 0;
    const int bin = (int)(first_row >> part.bin_shift);
    const int begin = part.starts[bin], end = part.starts[bin + 1];
    for (int base = begin; base < end; base += kPartThreads) {
        __syncthreads();
        if (n_pairs + kPartThreads > kTilePairs) round();
        __syncthreads();
        const int i = base + (int)threadIdx.x;
        const uint2 pair = i < end ? part.pairs[i] : make_uint2(0xffffffffu, 0u);
        const bool take = i < end && (int64_t)pair.x >= first_row && (int64_t)pair.x < first_row + n_rows;
        const unsigned long long m = __ballot(take);
        int to = 0;
        if (lane == 0 && m) to = atomicAdd(&n_pairs, __popcll(m));
        to = __builtin_amdgcn_readfirstlane(to);
        if (take) pairs[to + __popcll(m & ((1ull << lane) - 1ull))] = make_uint2(pair.x - (uint32_t)first_row, pair.y);
    }
    round();
}

}  // namespace svox
