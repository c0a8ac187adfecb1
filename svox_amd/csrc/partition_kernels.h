// partition_kernels.h -- the gradient of a point query by rows of the tree instead of by points.
//
// Adding a point's gradient row to its leaf with atomics (query_kernel) costs the memory system a request per 64 bytes,
// about 16 a nanosecond, after the gradient has been cleared.  Where the points are many beside the tree, it is cheaper to
// bring the points of neighbouring leaves together and write every row of the gradient once:
//   count    every block of points counts how many fall into each bin of rows (a bin: a few thousand rows), from the leaves
//            the query found where the caller kept them (28 -> 9 us for the points below);
//   offsets  prefix sums of the counts over the blocks, bin by bin; the rows of a crowded bin are cleared;
//   place    (row, point) pairs, bin after bin;
//   collect  a block per tile of rows (up to 256) of a bin that is not crowded picks its pairs out of the bin, puts them in
//            order and writes the sums;
//   crowded  the pairs of the crowded bins, cut into runs of equal length whatever rows they fall into: a block adds up what
//            a run has for a row and adds the sum to the gradient with atomics.
// A bin is crowded if it has more than Partition::crowded pairs, twice what a bin would have if the points were spread evenly
// over the rows.  On a dense tree under points from all of space none is; on a sparse tree a few large leaves hold most of
// space, they lie side by side in memory (a level after the other), and a block that did such rows alone would do most of the
// call's work: 1 Mi points from all of space in a 256^3 SH9 shell took 17.7 ms without the runs, 131 us with them (atomics 465 us).
// 1 000 003 points, 128^3 SH9 tree, atomics: cleared in 34 us, added to in 142; by rows: counted in 10 (28 where the leaves are
// looked up), offsets 4, placed in 14, collected in 97, no runs 4 us.
#pragma once

#include <type_traits>

#include "query_kernels.h"

namespace svox {

constexpr int kPartThreads = 256;
constexpr int kPointThreads = 1024;   // of the passes over points, which wait for memory
constexpr int kPartBins = 8192;       // at most
constexpr int kMaxBinShift = 13;      // rows of a bin at most, log2: crowded_kernel counts the pairs of each in LDS
// Blocks of points, at most: each writes and reads a count for every bin (1 000 003 points, 128^3 SH9: 256 blocks 130 us, 512 134).
constexpr int kPartBlocks = 256;

struct Partition {
    int64_t n_points, n_rows;
    int32_t per_block;      // points of a block
    int32_t n_blocks, n_bins;
    int32_t bin_shift;      // rows of a bin, log2
    int32_t tile_shift;     // rows of a tile, log2
    int32_t crowded;        // a bin with more pairs than this is crowded
    int32_t run_pairs;      // pairs of a run
    int32_t max_runs;       // room in `runs`: what every crowded bin can have together
    const int64_t* ids;     // [n_points]: leaves of the points, where the caller knows them, or null
    int32_t* leaf;          // [n_points]
    int32_t* counts;        // [n_bins][n_blocks]
    int32_t* totals;        // [n_bins]
    int32_t* starts;        // [n_bins + 1]
    uint2* pairs;           // [n_points]: row, point
    int2* runs;             // [max_runs]: bin, and which of its runs
    int32_t* n_runs;
};
constexpr int kRunPairs = 4096;   // of a crowded bin, one block's, at most

template <bool kOctree>
static __global__ __launch_bounds__(kPointThreads) void partition_count_kernel(TreeDev<float> tr, const float* __restrict__ points,
                                                                              Partition part, int32_t lds_nodes) {
    extern __shared__ int32_t lds_child[];   // the child rows of the first lds_nodes nodes, as in query_kernel
    int32_t* const hist = lds_child + lds_nodes * 8;   // [n_bins]
    for (int i = threadIdx.x; i < part.n_bins; i += kPointThreads) hist[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *part.n_runs = 0;
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

static __global__ __launch_bounds__(kPartThreads) void partition_offsets_kernel(Partition part, int32_t K, float* __restrict__ grad) {
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
    if (run > part.crowded) {
        __shared__ int32_t at;
        const int32_t n_runs = (run + part.run_pairs - 1) / part.run_pairs;
        if (threadIdx.x == 0) at = atomicAdd(part.n_runs, n_runs);
        __syncthreads();
        for (int r = threadIdx.x; r < n_runs; r += kPartThreads) part.runs[at + r] = make_int2(blockIdx.x, r);
        const int64_t first = (int64_t)blockIdx.x << part.bin_shift, left = part.n_rows - first;
        const int64_t n = (left < ((int64_t)1 << part.bin_shift) ? left : (int64_t)1 << part.bin_shift) * K;
        float* const out = grad + first * K;
        // (a bin is a whole number of 16-byte pieces, but for the last one's end)
        const int64_t n16 = ((uintptr_t)out & 15u) == 0 ? n / 4 : 0;
        for (int64_t i = threadIdx.x; i < n16; i += kPartThreads) ((uint4*)out)[i] = make_uint4(0u, 0u, 0u, 0u);
        for (int64_t i = n16 * 4 + threadIdx.x; i < n; i += kPartThreads) out[i] = 0.0f;
    }
}

static __global__ __launch_bounds__(kPointThreads) void partition_place_kernel(Partition part) {
    extern __shared__ int32_t cursor[];   // [n_bins]
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

// The points' rows of `count` pairs of one row, from `order`, added up by a wavefront: kCols scalars of the row, the first of
// them `col0`, of 64 / kCols points at a time.  Every lane of the first kCols is left with the sum of its scalar.
template <int kCols>
__device__ __forceinline__ float add_long_row(const uint32_t* order, int count, const float* __restrict__ values, int32_t K, int col0) {
    constexpr int kPoints = kWave / kCols, kBatch = 8;
    int lane = threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));   // (what follows is not to take registers outside)
    const int col = col0 + (lane & (kCols - 1));
    float sum = 0.0f;
    for (int i0 = lane / kCols; i0 < count; i0 += kPoints * kBatch) {
        float v[kBatch];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const int i = i0 + b * kPoints;
            v[b] = i < count && col < K ? values[(int64_t)order[i] * K + col] : 0.0f;
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b) sum += v[b];
    }
#pragma unroll
    for (int off = kCols; off < kWave; off <<= 1) sum += __shfl_xor(sum, off);
    return sum;
}

// One tile of rows: grad[row][0..K) = sum of values[point][0..K) over the row's points (0 where there are none).
// The tile's pairs are picked out of the bin and put in order of their rows in LDS; then every thread sums pieces of rows,
// one piece of the tile after the other, so that the writes are one run.  What bounds it is that writing and the reading
// of the points' rows, which lie anywhere: every thread asks for the first points of kBatch pieces before it adds.
// (Adding the points' rows into the tile in LDS, with LDS atomics: 193 us instead of 89.)
// A row with more than kLongRow points is left to a wavefront of its own, which has 32 of them under way at once: added by one
// thread per piece they would wait for one another, 0.3 us each.
// kVec: K is a multiple of 4 and both arrays start on 16-byte boundaries.
typedef float Float4 __attribute__((ext_vector_type(4)));
constexpr int kTileRows = 256;    // at most
constexpr int kTilePairs = 1024;  // pairs in LDS; a tile with more is summed in several rounds
constexpr int kLongRow = 32;
template <bool kVec>
static __global__ __launch_bounds__(kPartThreads, 7) void partition_collect_kernel(Partition part, const float* __restrict__ values,
                                                                                   int32_t K, float* __restrict__ grad) {
    __shared__ uint2 pairs[kTilePairs];        // row of the tile | place among the row's << 16, point
    __shared__ uint32_t order[kTilePairs];     // points by row
    __shared__ int32_t start[kTileRows + 1];   // of a row's in `order`
    __shared__ int32_t wave_sums[kPartThreads / kWave];
    __shared__ int32_t long_rows[kTilePairs / kLongRow];
    __shared__ int32_t n_pairs, n_long;
    static_assert(kTileRows == kPartThreads, "one thread per row of a tile");
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t first_row = (int64_t)blockIdx.x << part.tile_shift;
    const int bin = (int)(first_row >> part.bin_shift);
    const int begin = part.starts[bin], end = part.starts[bin + 1];
    if (end - begin > part.crowded) return;
    const int64_t rows_left = part.n_rows - first_row;
    const int n_rows = rows_left < (1 << part.tile_shift) ? (int)rows_left : 1 << part.tile_shift;
    float* const out = grad + first_row * K;
    constexpr int kPer = kVec ? 4 : 1, kBatch = 4;
    using Piece = std::conditional_t<kVec, Float4, float>;
    const int pieces = K / kPer, n_pieces = n_rows * pieces;
    bool again = false;   // an earlier round has written the tile
    if (threadIdx.x == 0) n_pairs = 0;
    for (int base = begin;;) {
        for (; base < end; base += kPartThreads) {
            __syncthreads();
            const bool full = n_pairs + kPartThreads > kTilePairs;
            __syncthreads();
            if (full) break;
            const int i = base + (int)threadIdx.x;
            const uint2 pair = i < end ? part.pairs[i] : make_uint2(0xffffffffu, 0u);
            const bool take = i < end && (int64_t)pair.x >= first_row && (int64_t)pair.x < first_row + n_rows;
            const unsigned long long m = __ballot(take);
            int to = 0;
            if (lane == 0 && m) to = atomicAdd(&n_pairs, __popcll(m));
            to = __builtin_amdgcn_readfirstlane(to);
            if (take) pairs[to + __popcll(m & ((1ull << lane) - 1ull))] = make_uint2(pair.x - (uint32_t)first_row, pair.y);
        }
        __syncthreads();
        const int n = n_pairs;
        start[threadIdx.x] = 0;
        if (threadIdx.x == 0) n_long = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kPartThreads) {
            const uint32_t row = pairs[i].x;
            pairs[i].x = row | (uint32_t)atomicAdd(&start[row], 1) << 16;
        }
        __syncthreads();
        const int32_t mine = start[threadIdx.x];
        int32_t total;
        const int32_t before = block_prefix<kPartThreads>(mine, wave_sums, total);
        start[threadIdx.x] = before;
        if (mine > kLongRow) long_rows[atomicAdd(&n_long, 1)] = threadIdx.x;
        if (threadIdx.x == 0) {
            start[kTileRows] = total;
            n_pairs = 0;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kPartThreads) order[start[pairs[i].x & 0xffffu] + (pairs[i].x >> 16)] = pairs[i].y;
        __syncthreads();
        for (int f0 = 0; f0 < n_pieces; f0 += kPartThreads * kBatch) {
            Piece sum[kBatch];
            int rows[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int f = f0 + b * kPartThreads + (int)threadIdx.x;
                const int row = f < n_pieces ? f / pieces : kTileRows - 1;
                const int at = start[row], count = start[row + 1] - at;
                rows[b] = row;
                sum[b] = Piece{};
                if (f < n_pieces && count > 0 && count <= kLongRow)
                    sum[b] = *(const Piece*)(values + (int64_t)order[at] * K + (f - row * pieces) * kPer);
            }
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int f = f0 + b * kPartThreads + (int)threadIdx.x, row = rows[b];
                const int at = start[row], count = start[row + 1] - at;
                // (a long row is left to a wavefront, and a round after the first has nothing for a row without pairs)
                if (f >= n_pieces || count > kLongRow || (again && count == 0)) continue;
                const float* const from = values + (f - row * pieces) * kPer;
                int i = 1;
                for (; i + 1 < count; i += 2) {
                    const Piece v = *(const Piece*)(from + (int64_t)order[at + i] * K);
                    const Piece w = *(const Piece*)(from + (int64_t)order[at + i + 1] * K);
                    sum[b] += v;
                    sum[b] += w;
                }
                if (i < count) sum[b] += *(const Piece*)(from + (int64_t)order[at + i] * K);
                Piece* const to = (Piece*)out + f;
                *to = again ? *to + sum[b] : sum[b];
            }
        }
        constexpr int kCols = 16;
        const int groups = (K + kCols - 1) / kCols, units = n_long * groups;
        for (int u = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); u < units; u += kPartThreads / kWave) {
            const int row = long_rows[u / groups], col0 = u % groups * kCols;
            const float sum = add_long_row<kCols>(order + start[row], start[row + 1] - start[row], values, K, col0);
            float* const to = out + (int64_t)row * K + col0 + lane;
            if (lane < kCols && col0 + lane < K) *to = again ? *to + sum : sum;
        }
        if (base >= end) break;
        again = true;
    }
}

// The crowded bins, run by run: a run's pairs are put in order of their rows in LDS.  A row with up to kLongRow of them is added
// scalar by scalar, kSlot consecutive pairs of the run to a thread, and goes to the gradient at every change of the row; a
// longer one is added by a wavefront, kLongPart pairs at a time, before anything goes out -- atomics on one address follow one
// another at 22 ns (1 Mi points in one leaf of a 128^3 SH9 tree, all by atomics: 23 ms).
constexpr int kSlot = 16, kLongPart = 512;
static __global__ __launch_bounds__(kPointThreads, 8) void partition_crowded_kernel(Partition part, const float* __restrict__ values,
                                                                                    int32_t K, float* __restrict__ grad) {
    extern __shared__ int32_t start[];         // [rows of a bin + 1]
    __shared__ uint32_t order[kRunPairs];      // points by row
    __shared__ uint16_t row_of[kRunPairs];     // ... and their rows
    constexpr int kLongMax = kRunPairs / (kLongRow + 1) + kRunPairs / kLongPart + 1;
    __shared__ int32_t long_parts[kLongMax];   // row | number of the part << 16
    __shared__ int32_t wave_sums[kPointThreads / kWave];
    __shared__ int32_t n_long;
    const int rows = 1 << part.bin_shift, lane = threadIdx.x & (kWave - 1);
    const int n_runs = *part.n_runs;
    for (int r = blockIdx.x; r < n_runs; r += gridDim.x) {
        const int2 run = part.runs[r];
        const int begin = part.starts[run.x] + run.y * part.run_pairs, left = part.starts[run.x + 1] - begin;
        const int n = left < part.run_pairs ? left : part.run_pairs;
        const int64_t first_row = (int64_t)run.x << part.bin_shift;
        __syncthreads();
        for (int i = threadIdx.x; i < rows; i += kPointThreads) start[i] = 0;
        if (threadIdx.x == 0) n_long = 0;
        __syncthreads();
        uint2 pair[kRunPairs / kPointThreads];
        int place[kRunPairs / kPointThreads];
#pragma unroll
        for (int j = 0; j < kRunPairs / kPointThreads; ++j) {
            const int i = j * kPointThreads + (int)threadIdx.x;
            place[j] = -1;
            if (i < n) {
                pair[j] = part.pairs[begin + i];
                pair[j].x -= (uint32_t)first_row;
                place[j] = atomicAdd(&start[pair[j].x], 1);
            }
        }
        __syncthreads();
        int32_t before_all = 0;
        for (int r0 = 0; r0 < rows; r0 += kPointThreads) {
            const int row = r0 + (int)threadIdx.x;
            const int32_t mine = row < rows ? start[row] : 0;
            int32_t total;
            const int32_t before = block_prefix<kPointThreads>(mine, wave_sums, total);
            if (row < rows) start[row] = before_all + before;
            if (mine > kLongRow) {
                const int parts = (mine + kLongPart - 1) / kLongPart, at = atomicAdd(&n_long, parts);
                for (int k = 0; k < parts; ++k) long_parts[at + k] = row | k << 16;
            }
            before_all += total;
        }
        if (threadIdx.x == 0) start[rows] = n;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kRunPairs / kPointThreads; ++j) {
            if (place[j] >= 0) {
                const int at = start[pair[j].x] + place[j];
                order[at] = pair[j].y;
                row_of[at] = (uint16_t)pair[j].x;
            }
        }
        __syncthreads();
        float* const out = grad + first_row * K;
        const uint32_t units = (uint32_t)((n + kSlot - 1) / kSlot) * (uint32_t)K;
        for (uint32_t u = threadIdx.x; u < units; u += kPointThreads) {
            const uint32_t slot = u / (uint32_t)K, e = u - slot * (uint32_t)K;
            constexpr int kBatch = 8;
            float sum = 0.0f;
            int current = -1;
            for (int p0 = 0; p0 < kSlot; p0 += kBatch) {
                float v[kBatch];
                int row[kBatch];
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    const int at = (int)slot * kSlot + p0 + b;
                    row[b] = -1;
                    v[b] = 0.0f;
                    if (at < n) {
                        const int here = row_of[at];
                        if (start[here + 1] - start[here] <= kLongRow) {
                            row[b] = here;
                            v[b] = values[(int64_t)order[at] * K + e];
                        }
                    }
                }
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    if (row[b] != current) {
                        if (current >= 0) atomicAdd(out + (int64_t)current * K + e, sum);
                        sum = 0.0f;
                        current = row[b];
                    }
                    sum += v[b];
                }
            }
            if (current >= 0) atomicAdd(out + (int64_t)current * K + e, sum);
        }
        constexpr int kCols = 16;
        const int groups = (K + kCols - 1) / kCols, n_units = n_long * groups;
        for (int u = threadIdx.x / kWave; u < n_units; u += kPointThreads / kWave) {
            const int row = long_parts[u / groups] & 0xffff, from = start[row] + (long_parts[u / groups] >> 16) * kLongPart;
            const int col0 = u % groups * kCols, count = start[row + 1] - from;
            const float sum = add_long_row<kCols>(order + from, count < kLongPart ? count : kLongPart, values, K, col0);
            if (lane < kCols && col0 + lane < K) atomicAdd(out + (int64_t)row * K + col0 + lane, sum);
        }
    }
}

}  // namespace svox
