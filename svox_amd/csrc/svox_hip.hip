// svox_hip.hip -- the extern "C" entry points of libsvox_hip.so (declared in include/svox_hip.h):
// argument validation, kernel selection and launches.  Each entry point stands where one function
// of the reference's extension module stood (svox/csrc/svox.cpp:106-121; host launchers
// svox/csrc/svox_kernel.cu:120-203 and svox/csrc/rt_kernel.cu:1009-1109).
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../include/svox_hip.h"
#include "group_kernels.h"
#include "march_launch.h"
#include "partition_kernels.h"

#include <mutex>
#include <numeric>

// Workspace of svox_volume_render_backward_static: one array per GPU, inside the library's code object.
// In host code the name `scratch` is only a handle for hipGetSymbolAddress (static_workspace below); it
// is never passed to a kernel or a runtime call as an address.
static_assert(SVOX_STATIC_WORKSPACE_BYTES % 256 == 0, "whole 256-byte units");
static __device__ __align__(256) unsigned char scratch[SVOX_STATIC_WORKSPACE_BYTES];
// Wavefronts of render_forward_split_kernel that gave up waiting since the library was loaded (svox_give_up_count);
// the kernels get its address in ReplaySpace::give_ups.
static __device__ unsigned int split_give_ups = 0;

namespace {

using namespace svox;

thread_local char g_error[512] = "";
// Debug flags of the calling thread (svox_set_debug_flags): bit 0: always take the generic kernels; bit 1: small
// batches run like large ones; bit 2: forward launches never take the two-wavefront kernel; bit 3: they always
// do (where it applies); bit 4: the bounded waits of that kernel give up at once; bit 5: forward launches cut their rays, as bits 8 and
// up say (pick_cut, group_cut); bit 6: noting passes list their rays (list_shapes).  Per thread, so that one thread's tests cannot change the kernels of another's calls.
thread_local int g_debug_flags = 0;

// Launch-shape overrides for experiments, read from the environment once, when the first launch of the process
// picks a shape; the library has no other mutable state besides g_error / g_debug_flags (per thread) and the
// per-device address of `scratch`.  Every field is 0 / -1 ("not set") in normal use:
//   SVOX_PER_WAVE      rays a persistent wavefront of a batch launch owns (64, 128, 256, 512 or 1024)
//   SVOX_REFILL        idle lanes at which such a wavefront takes new rays (1..64)
//   SVOX_XCD_GROUP     consecutive image tiles handed to one XCD (1..4096)
//   SVOX_TILE_ORDER    0: 16x16 blocks of an image row by row, 1: ring by ring from the middle
//   SVOX_IMAGE_RUN     16x16 blocks of one image in a row before the next image's, in multi-image launches
//   SVOX_SPLIT_FORWARD 0 / 1: forward launches never / always on two wavefronts per tile
//   SVOX_SPLIT_BLOCKS  largest forward launch (in tiles) that takes two wavefronts per tile
//   SVOX_REPLAY_SHIFT  4, 5 or 6: log2 of the rays a block of the replay kernels takes
//   SVOX_CUT           single precision, 0: forward passes never cut their rays into pieces, 1 to 8: always, so many rays to a
//                      wavefront, + 10 x: into 2^x pieces at most (62: two rays, 32 pieces of each, or 64 of one if the other misses)
struct Tuning {
    int per_wave = 0, refill = 0, xcd_group = 0, tile_order = -1, image_run = -1, split_forward = -1, replay_shift = -1;
    long split_blocks = -1;
    int cut = -1;
};
const Tuning& tuning() {
    static const Tuning t = [] {
        Tuning v;
        auto num = [](const char* name, long unset) {
            const char* e = getenv(name);
            return e ? atol(e) : unset;
        };
        v.per_wave = (int)num("SVOX_PER_WAVE", 0);
        v.refill = (int)num("SVOX_REFILL", 0);
        v.xcd_group = (int)num("SVOX_XCD_GROUP", 0);
        v.tile_order = (int)num("SVOX_TILE_ORDER", -1);
        v.image_run = (int)num("SVOX_IMAGE_RUN", -1);
        v.split_forward = (int)num("SVOX_SPLIT_FORWARD", -1);
        v.split_blocks = num("SVOX_SPLIT_BLOCKS", -1);
        v.replay_shift = (int)num("SVOX_REPLAY_SHIFT", -1);
        v.cut = (int)num("SVOX_CUT", -1);
        return v;
    }();
    return t;
}

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
    return code;
}

int check_launch(const char* what) {
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return fail(SVOX_ERR_LAUNCH, "svox.%s: %s", what, hipGetErrorString(err));
    return SVOX_OK;
}

// The device address of a __device__ variable of this library on the current device, looked up once per device (every
// GPU holds its own copy at its own address); nullptr where there is no usable device.
constexpr int kStaticDevicesMax = 64;
struct DeviceAddress {
    std::mutex guard;
    void* address[kStaticDevicesMax] = {nullptr};
    template <typename Symbol>
    void* get(const Symbol& symbol) {
        int device = -1;
        if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kStaticDevicesMax) return nullptr;
        std::lock_guard<std::mutex> lock(guard);
        if (!address[device]) {
            void* ptr = nullptr;
            if (hipGetSymbolAddress(&ptr, symbol) != hipSuccess) return nullptr;
            address[device] = ptr;
        }
        return address[device];
    }
};
unsigned int* give_up_counter() {
    static DeviceAddress at;
    return (unsigned int*)at.get(HIP_SYMBOL(split_give_ups));
}

int check_tree(const SvoxTreeSpec* t, bool need_data) {
    if (!t) return fail(SVOX_ERR_NULL_POINTER, "tree spec is NULL");
    if (need_data && !t->data) return fail(SVOX_ERR_NULL_POINTER, "tree.data is NULL");
    if (!t->child) return fail(SVOX_ERR_NULL_POINTER, "tree.child is NULL");
    if (!t->parent_depth) return fail(SVOX_ERR_NULL_POINTER, "tree.parent_depth is NULL");
    if (t->dtype != SVOX_F32 && t->dtype != SVOX_F64)
        return fail(SVOX_ERR_BAD_DTYPE, "tree.dtype must be SVOX_F32 or SVOX_F64, got %d", t->dtype);
    if (t->capacity < 1) return fail(SVOX_ERR_BAD_SHAPE, "tree.capacity must be >= 1, got %lld", (long long)t->capacity);
    if (t->N < 2) return fail(SVOX_ERR_BAD_SHAPE, "tree.N must be >= 2, got %d", t->N);
    if (t->data_dim < 1) return fail(SVOX_ERR_BAD_SHAPE, "tree.data_dim must be >= 1, got %d", t->data_dim);
    const double cells = (double)t->capacity * t->N * t->N * t->N;
    if (cells >= 9.0e18 / (double)(t->data_dim > 0 ? t->data_dim : 1))
        return fail(SVOX_ERR_BAD_SHAPE, "tree is too large to index");
    if (t->capacity > 0x7fffffffll)
        return fail(SVOX_ERR_BAD_SHAPE, "tree.capacity exceeds the int32 node ids of the child table");
    return SVOX_OK;
}

template <typename T>
TreeDev<T> make_tree(const SvoxTreeSpec* t) {
    TreeDev<T> d;
    d.data = (T*)t->data;
    d.child = t->child;
    d.parent_depth = t->parent_depth;
    d.extra = (const T*)t->extra_data;
    d.offset = (const T*)t->offset;
    d.scaling = (const T*)t->scaling;
    d.weight_accum = (T*)t->weight_accum;
    d.walk = nullptr;
    d.walk_marked = false;
    d.capacity = t->capacity;
    d.N = t->N;
    d.K = t->data_dim;
    d.extra_cols = t->extra_cols;
    d.weight_accum_max = t->weight_accum_max;
    return d;
}

// an fp32 tree whose cells number less than 2^30 (int32 cell indices with two spare bits; for an octree that is
// fewer than 2^27 nodes and a child table below 4 GiB, which its walk addresses with 32-bit byte offsets).  Octrees
// walk on integer coordinates from the previous path; other branching factors take the reference's floating-point
// walk inside the same kernels and share the rounds, the shade list, the record lists and the notes.
bool march_fast_ok(const SvoxTreeSpec* t) {
    return !(g_debug_flags & 1) && t->dtype == SVOX_F32 && (double)t->capacity * t->N * t->N * t->N < 1073741824.0;
}
// ... and an octree among them: the point queries' integer walk
bool octree_fast_ok(const SvoxTreeSpec* t) { return march_fast_ok(t) && t->N == 2; }

int zero_fill(void* ptr, int64_t bytes, hipStream_t stream) {
    if (bytes <= 0) return SVOX_OK;
    if (((uintptr_t)ptr & 15u) != 0 || (bytes & 3) != 0)
        return fail(SVOX_ERR_BAD_SHAPE, "gradient buffer must be 16-byte aligned and a multiple of 4 bytes");
    // (a launch has fewer than 2^32 threads, and each of these clears 16 bytes)
    constexpr int64_t kMost = (int64_t)0xffffff * 256;
    int64_t left = bytes / 16;
    uint4* at = (uint4*)ptr;
    for (; left > kMost; left -= kMost, at += kMost)
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)(kMost / 256)), dim3(256), 0, stream, at, kMost, (uint32_t*)nullptr, 0);
    const int64_t blocks = left < 1 ? 1 : (left + 255) / 256;
    hipLaunchKernelGGL(zero_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, at, left, (uint32_t*)(at + left),
                       (int)(bytes % 16 / 4));
    return check_launch("zero_fill");
}

// ---------------------------------------------------------------------------------------------
// queries
// ---------------------------------------------------------------------------------------------
// Calls of up to kFewPointsMax points take query_few_kernel: its wavefronts have 16 points instead of 64, so that small
// calls spread further and end sooner, but each walks from the root through memory and moves scalars.  Gather, us, 64 /
// 16 points: 262 144 points, SH9 25.7 / 25.2, SH4 11.7 / 11.5, SH16 36.9 / 30.2; 524 288 points 44.7 / 44.6, 16.3 / 19.3,
// 52.7 / 54.8.  (Larger wavefronts of 128 points, two to a lane, for the rest: SH16, 1 Mi points 92 / 92, 262 144 points
// 37 / 47.)
constexpr int64_t kFewPointsMax = 262144;
// Whether a tree's nodes number as many as a complete octree's, or up to an eighth more: a grid that is as fine everywhere, perhaps
// refined here and there.  (A tree of another shape with such a number only takes a rule that is not made for it.)
bool like_complete_octree(const SvoxTreeSpec* tree) {
    int64_t nodes = 1;
    while (nodes * 8 + 1 <= tree->capacity) nodes = nodes * 8 + 1;
    return tree->N == 2 && tree->capacity - nodes <= nodes / 8;
}
// Whether a query of n points is worth a copy of the child table in which the nodes of leaves only are marked
// (last_nodes_kernel).  It takes 5 us and 14 ps a node, and what it saves -- a request for a line of the table, which the
// memory system serves 55 of a nanosecond once the table is larger than an L2 cache -- goes to the points that end in such a
// node: all of a grid's, few of those thrown at random on a sparse tree.  So for a grid by that cost, with 17 ps saved a point and
// a quarter in hand (a table that L2 holds: from 12 points a node on, even at 27); for others from 24 points a node on, where it is
// even, and not where L2 holds the table.
// (us, plain / with the copy, its making included.  Grids: 128^3 SH9, 600 000 points 52 / 48, 1 000 003 78 / 69, 4 M 274 / 249; RGBA
// 36 / 33, 52 / 43, 167 / 109; 64^3 SH4, 450 000 points 26 / 28, 1.0 M 44 / 43, 4 M 131 / 120, SH16 45 / 48, 83 / 85, 285 / 274; 256^3
// SH1, 2 M points 134 / 133, 4 M 257 / 214; 32^3 SH4, 4 M 77 / 77.  Shells, 13 / 24 / 48 points a node: 256^3 RGBA 40 / 43, 62 / 64,
// 114 / 113, SH9 79 / 81, 136 / 134, 417 / 415; 512^3 SH4 338 / 349, 622 / 623, 1238 / 1224; 128^3 RGBA 18 / 21, 24 / 31, 35 / 37.)
bool walk_copy_pays(const SvoxTreeSpec* tree, int64_t n) {
    if (!octree_fast_ok(tree) || tree->capacity < 30000 || n <= kFewPointsMax) return false;
    const bool beyond_l2 = tree->capacity >= 131072;   // (32 bytes a node, 4 MB)
    if (!like_complete_octree(tree)) return beyond_l2 && n >= 24 * tree->capacity;
    return beyond_l2 ? (double)n * 17.0 >= 1.25 * (5e6 + 14.0 * (double)tree->capacity) : n >= 12 * tree->capacity;
}
constexpr int kLdsNodesMax = 584;  // child rows kept in LDS per block: 584 * 32 B = 18.25 KiB

template <typename T, int MODE>
int launch_query(const SvoxTreeSpec* tree, const void* points, int64_t n, void* values, void* target,
                 int64_t* ids, int32_t Kx, hipStream_t stream, const char* what, int32_t* walk_space = nullptr) {
    if (n == 0) return SVOX_OK;
    const TreeDev<T> tr = make_tree<T>(tree);
    if (n <= kFewPointsMax) {
        const dim3 blocks((unsigned)((n + kFewPoints - 1) / kFewPoints));
        if (sizeof(T) == 4 && octree_fast_ok(tree))
            hipLaunchKernelGGL((query_few_kernel<T, MODE, sizeof(T) == 4>), blocks, dim3(kWave), 0, stream, tr, (const T*)points, n,
                               (T*)values, (T*)target, ids, Kx);
        else
            hipLaunchKernelGGL((query_few_kernel<T, MODE, false>), blocks, dim3(kWave), 0, stream, tr, (const T*)points, n,
                               (T*)values, (T*)target, ids, Kx);
        return check_launch(what);
    }
    const int64_t tiles = (n + kQueryThreads - 1) / kQueryThreads;
    const int64_t blocks = tiles < 256 * 8 ? tiles : 256 * 8;
    if constexpr (sizeof(T) == 4) {
        if (octree_fast_ok(tree)) {
            // (a scatter with the leaves at hand walks nothing)
            const bool walks = MODE != kQueryScatterAdd || !ids;
            const int32_t lds_nodes = !walks ? 0 : tree->capacity < kLdsNodesMax ? (int32_t)tree->capacity : kLdsNodesMax;
            const int32_t* walk = tr.child;
            if (walk_space) {
                hipLaunchKernelGGL(last_nodes_kernel, dim3((unsigned)((tree->capacity * 8 + 255) / 256)), dim3(256), 0, stream, tr.child,
                                   (int32_t)tree->capacity, walk_space);
                walk = walk_space;
            }
            hipLaunchKernelGGL((query_kernel<T, MODE, true>), dim3((unsigned)blocks), dim3(kQueryThreads),
                               (size_t)lds_nodes * 32, stream, tr, (const T*)points, n, (T*)values,
                               (T*)target, ids, Kx, walk, lds_nodes);
            return check_launch(what);
        }
    }
    hipLaunchKernelGGL((query_kernel<T, MODE, false>), dim3((unsigned)blocks), dim3(kQueryThreads), 0, stream,
                       tr, (const T*)points, n, (T*)values, (T*)target, ids, Kx, tr.child, 0);
    return check_launch(what);
}

// log2 of the rows of a bin, from that of a tile on: 2 048 bins at most while that leaves them small (2 048 rows: 8 tiles, each of
// which looks through the bin's pairs), because every block of points writes a count for every bin; more in larger trees.
int bin_shift_of(int64_t n_rows, int shift) {
    auto bins = [&] { return ((n_rows - 1) >> shift) + 1; };
    while (bins() > kPartBins || (bins() > 2048 && shift < 11)) ++shift;
    return shift;
}

// How the gradient of n points is collected row by row (partition_kernels.h): fills `part` and returns the bytes of
// workspace it needs, or returns 0 where the points are added with atomics, whichever is estimated to take less where the
// points are spread evenly over the rows.  With atomics: the gradient cleared at 6.8 bytes a picosecond, then 16.5 requests a
// nanosecond, a request for every 64 bytes a row touches.  By rows: the launches, 45 ps a point to count and place it, rows and
// points' rows at 4.4 bytes a picosecond, and the pairs of a bin once for each of its tiles at 8.
// Where the points crowd, atomics on one address wait for one another and rows gain by more; the cost of the runs can eat that up
// again where a run has one or two points to a row (the slab and the blob below).
// (us, atomics / rows, leaves known.  Even: 1 000 003 points, 128^3 SH9 178 / 131, 64^3 SH16 253 / 101, 32^3 SH4 106 / 61, 128^3
// RGBA 62 / 76; 4 Mi points, 128^3 SH9 612 / 319, RGBA 216 / 198; 262 144 points, 32^3 SH4 34 / 40, 64^3 SH16 78 / 60; 131 072 of
// the latter 47 / 52; 16 Mi points, 256^3 SH1 869 / 1120.  All of space, in shells: 1 Mi points, 64^3 SH16 559 / 152, 256^3 SH9
// 465 / 131, 512^3 SH16 887 / 554; 262 144 points, 64^3 SH16 148 / 86; 16 Mi points, 48 M rows of SH25 8030 / 6740.  1 Mi points of
// the 128^3 SH9 tree: in 1 % of the volume 200 / 173, in 0.1 % 291 / 148, in a slab of 2 % 190 / 194, around the middle with a
// deviation of 0.12 184 / 188, in one leaf 23 300 / 160; around the middle of the 64^3 SH16 tree 272 / 181, in 1 % of it 318 / 134.)
int64_t plan_partition(const SvoxTreeSpec* tree, int64_t n, int32_t K, Partition* part) {
    const double rows = (double)tree->capacity * tree->N * tree->N * tree->N;
    const double most_rows = (double)((int64_t)kPartBins << kMaxBinShift);
    if (tree->dtype != SVOX_F32 || (g_debug_flags & 1) || rows > most_rows || n > (1 << 30) || K > (1 << 20)) return 0;
    *part = Partition{};
    part->n_points = n;
    part->n_rows = (int64_t)rows;
    // tiles of about 256 points, and not more than 256 rows
    int tile = 8;
    while (tile > 2 && (double)n * (1 << tile) > 512.0 * rows) --tile;
    part->tile_shift = tile;
    part->bin_shift = bin_shift_of(part->n_rows, tile);
    part->n_bins = (int32_t)(((part->n_rows - 1) >> part->bin_shift) + 1);
    const double row_bytes = 4.0 * K;
    const int align = K % 16 == 0 ? 64 : K % 8 == 0 ? 32 : K % 4 == 0 ? 16 : K % 2 == 0 ? 8 : 4;   // where rows may start
    const double atomics_us = rows * row_bytes / 6.8e6 + (double)n * (row_bytes + 64.0 - align) / 64.0 / 16500.0;
    const double looks = (double)n * 8.0 * (1 << (part->bin_shift - tile));   // bytes
    const double rows_us = 30.0 + (double)n * 45e-6 + (rows * row_bytes + (double)n * (row_bytes + 32.0)) / 4.4e6 + looks / 8e6;
    if (atomics_us <= rows_us) return 0;
    int64_t per = (n + kPartBlocks - 1) / kPartBlocks;
    if (per < 2048) per = 2048;
    part->per_block = (int32_t)((per + kPointThreads - 1) / kPointThreads * kPointThreads);
    part->n_blocks = (int32_t)((n + part->per_block - 1) / part->per_block);
    // Crowded: beyond twice the even share, and 1 024 pairs, which a tile sorts at once.  (us, twice and 1 024 / three times and 1 024 /
    // four times and 2 048; 1 Mi points: deviation of 0.12 in the 64^3 SH16 tree 189 / 255 / 262, 64^3 SH16 shell 157 / 207 / 215, slab
    // 200 / 190 / 190; 262 144 points in the shell 87 / 87 / 166; even points, half of the capacity unused, 216 / 192 / 192, atomics 253.)
    // Runs: two for every CU, 512 to 4 096 pairs.  (262 144 points in the shell: the crowded kernel 96 us at 4 096, 23 at 512.)
    // And not beyond 2 048 pairs a tile, however few the rows are.  (40 000 points in one node of 300 numbers: 2 280 us as two tiles,
    // 195 with atomics.)
    const int64_t even = (n + part->n_bins - 1) / part->n_bins, most = 2048ll << (part->bin_shift - tile);
    part->crowded = (int32_t)(even * 2 < 1024 ? 1024 : even * 2 < most ? even * 2 : most);
    part->run_pairs = n < 512 * 512 ? 512 : n > 512 * kRunPairs ? kRunPairs : (int32_t)(n / 512);
    part->max_runs = (int32_t)(n / part->run_pairs + n / part->crowded + 1);
    return n * 12 + part->max_runs * 8ll + ((int64_t)part->n_bins * part->n_blocks + 2 * part->n_bins + 16) * 4;
}
int launch_partition(const SvoxTreeSpec* tree, Partition part, const float* points, const int64_t* ids, const float* values, int32_t K,
                     float* grad, void* workspace, hipStream_t stream) {
    part.ids = ids;
    part.pairs = (uint2*)workspace;
    part.runs = (int2*)(part.pairs + part.n_points);
    part.leaf = (int32_t*)(part.runs + part.max_runs);
    part.counts = part.leaf + part.n_points;
    part.totals = part.counts + (int64_t)part.n_bins * part.n_blocks;
    part.starts = part.totals + part.n_bins;
    part.n_runs = part.starts + part.n_bins + 1;
    const TreeDev<float> tr = make_tree<float>(tree);
    const dim3 threads(kPartThreads);
    const size_t bin_words = (size_t)part.n_bins * 4;
    if (octree_fast_ok(tree)) {
        const int32_t lds_nodes = ids ? 0 : tree->capacity < kLdsNodesMax ? (int32_t)tree->capacity : kLdsNodesMax;
        hipLaunchKernelGGL((partition_count_kernel<true>), dim3(part.n_blocks), dim3(kPointThreads), (size_t)lds_nodes * 32 + bin_words,
                           stream, tr, points, part, lds_nodes);
    } else {
        hipLaunchKernelGGL((partition_count_kernel<false>), dim3(part.n_blocks), dim3(kPointThreads), bin_words, stream, tr, points, part, 0);
    }
    hipLaunchKernelGGL(partition_offsets_kernel, dim3(part.n_bins), threads, 0, stream, part, K, grad);
    hipLaunchKernelGGL(partition_place_kernel, dim3(part.n_blocks), dim3(kPointThreads), bin_words, stream, part);
    const unsigned tiles = (unsigned)(((part.n_rows - 1) >> part.tile_shift) + 1);
    if (K % 4 == 0 && (((uintptr_t)values | (uintptr_t)grad) & 15u) == 0)
        hipLaunchKernelGGL((partition_collect_kernel<true>), dim3(tiles), threads, 0, stream, part, values, K, grad);
    else
        hipLaunchKernelGGL((partition_collect_kernel<false>), dim3(tiles), threads, 0, stream, part, values, K, grad);
    const unsigned run_blocks = (unsigned)(part.max_runs < 512 ? part.max_runs : 512);
    hipLaunchKernelGGL(partition_crowded_kernel, dim3(run_blocks), dim3(kPointThreads), ((size_t)4 << part.bin_shift) + 4, stream, part,
                       values, K, grad);
    return check_launch("query_vertical_backward");
}

// ---------------------------------------------------------------------------------------------
// rendering
// ---------------------------------------------------------------------------------------------
int check_render(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int* out_dim) {
    int rc = check_tree(tree, true);
    if (rc) return rc;
    if (!opt) return fail(SVOX_ERR_NULL_POINTER, "render options are NULL");
    if (opt->format < SVOX_FORMAT_RGBA || opt->format > SVOX_FORMAT_ASG)
        return fail(SVOX_ERR_BAD_SHAPE, "unknown data format %d", opt->format);
    const int od = svox_out_data_dim(opt->format, opt->basis_dim, tree->data_dim);
    if (od < 0)
        return fail(SVOX_ERR_BAD_SHAPE, "basis_dim %d is invalid for format %d", opt->basis_dim, opt->format);
    if (od > SVOX_MAX_OUT_DIM)
        return fail(SVOX_ERR_UNSUPPORTED, "rendered colour dimension %d exceeds %d", od, SVOX_MAX_OUT_DIM);
    if (opt->format != SVOX_FORMAT_RGBA) {
        if (opt->basis_dim > SVOX_MAX_BASIS_DIM)
            return fail(SVOX_ERR_UNSUPPORTED, "basis_dim %d exceeds %d", opt->basis_dim, SVOX_MAX_BASIS_DIM);
        if (opt->min_comp < 0 || opt->max_comp >= opt->basis_dim)
            return fail(SVOX_ERR_BAD_SHAPE, "component range [%d, %d] outside [0, %d)", opt->min_comp,
                        opt->max_comp, opt->basis_dim);
        if (opt->format == SVOX_FORMAT_SG || opt->format == SVOX_FORMAT_ASG) {
            const int need = opt->format == SVOX_FORMAT_SG ? 4 : 11;
            if (!tree->extra_data || tree->extra_rows < opt->basis_dim || tree->extra_cols < need)
                return fail(SVOX_ERR_BAD_SHAPE, "extra_data must be (%d, >=%d) for this format", opt->basis_dim, need);
        }
    }
    *out_dim = od;
    return SVOX_OK;
}

int check_camera(const SvoxCameraSpec* cam, int n_images = 1, int64_t pose_stride = 12) {
    if (!cam) return fail(SVOX_ERR_NULL_POINTER, "camera spec is NULL");
    if (!cam->c2w) return fail(SVOX_ERR_NULL_POINTER, "cam.c2w is NULL");
    if (cam->width < 0 || cam->height < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative image size");
    if (n_images < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative image count");
    if (n_images > 1 && pose_stride < 12) return fail(SVOX_ERR_BAD_SHAPE, "pose_stride must be >= 12 scalars");
    // (+ 64: multi-image launches pad every image to a whole number of block runs)
    const double tiles = 4.0 * ((double)blocks16_of(cam->width) * blocks16_of(cam->height) + 64.0) * (n_images > 0 ? n_images : 1);
    if (tiles >= 2147483647.0) return fail(SVOX_ERR_BAD_SHAPE, "too many pixels for one launch");
    return SVOX_OK;
}

int check_rays(const SvoxRaysSpec* rays) {
    if (!rays) return fail(SVOX_ERR_NULL_POINTER, "rays spec is NULL");
    if (rays->n_rays < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative ray count");
    if (rays->n_rays >= (1ll << 36)) return fail(SVOX_ERR_BAD_SHAPE, "too many rays for one launch");
    if (rays->n_rays > 0 && (!rays->origins || !rays->dirs || !rays->vdirs))
        return fail(SVOX_ERR_NULL_POINTER, "rays.origins / dirs / vdirs is NULL");
    return SVOX_OK;
}

// default options on an fp32 octree whose record matches the format: the specialised kernels (with or without
// density_softplus, which they apply to the densities they fetch).  Returns what SVOX_DISPATCH_OCTREE
// switches on: 0 for RGBA, basis_dim for spherical harmonics, kLobeKernels + basis_dim for lobes (spherical
// gaussians and anisotropic ones), -1 for everything the generic kernels serve.
constexpr int kLobeKernels = 100;
int fast_basis(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt) {
    if (!march_fast_ok(tree)) return -1;
    if (opt->format == SVOX_FORMAT_RGBA) return tree->data_dim == 4 ? 0 : -1;
    if (opt->format != SVOX_FORMAT_SH && opt->format != SVOX_FORMAT_SG && opt->format != SVOX_FORMAT_ASG) return -1;
    const int D = opt->basis_dim;
    if (D != 1 && D != 4 && D != 9 && D != 16 && D != 25) return -1;
    if (tree->data_dim != 3 * D + 1 || opt->min_comp < 0 || opt->max_comp > D - 1) return -1;
    // A range of components narrower than the basis runs on the kernels that keep a ray's basis as a row in LDS (the
    // lobe policy: its rows come from precalc_basis, for spherical harmonics too), the row zero outside the range;
    // min_comp > max_comp is the reference's empty range, mid grey.
    const bool partial = opt->min_comp > 0 || opt->max_comp < D - 1;
    if (opt->format == SVOX_FORMAT_SH && partial) return kLobeKernels + D;
    if (opt->format != SVOX_FORMAT_SH) {
        // lobes: the table must be there, [lambda, mu] per spherical gaussian (rt_kernel.cu:133-139),
        // [lambda_x, lambda_y, three axes] per anisotropic one (rt_kernel.cu:120-131)
        const int need = opt->format == SVOX_FORMAT_SG ? 4 : 11;
        if (!tree->extra_data || tree->extra_rows < D || tree->extra_cols < need) return -1;
        return kLobeKernels + D;
    }
    return D;
}

// The basis size a double-precision octree is rendered with by the kernels that give four lanes to a ray
// (group_kernels.h; 0 for RGBA), or -1: three colour channels of a basis size they are built for, cells that 32-bit
// indices reach, no weight accumulator, and not more rays than kGroupMaxRays.
//
// kGroupMaxRays: with more rays than fill the chip four lanes to a ray, or pieces of it, are work done several times over.
constexpr int64_t kGroupMaxRays = 1 << 17;

int group_basis(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int64_t n_rays) {
    if ((g_debug_flags & 1) || tree->dtype != SVOX_F64 || tree->N != 2 || tree->weight_accum || n_rays > kGroupMaxRays ||
        (double)tree->capacity * 8.0 >= 1073741824.0)
        return -1;
    if (opt->format == SVOX_FORMAT_RGBA) return tree->data_dim == 4 ? 0 : -1;
    const int D = opt->basis_dim;
    if (D != 1 && D != 4 && D != 9 && D != 16 && D != 25) return -1;
    return tree->data_dim == 3 * D + 1 ? D : -1;
}

// Rays that a wavefront of those kernels is dealt, and log2 of the pieces a ray is walked in at most (at least 2); none dealt: four
// lanes walk a ray together.
struct Cut {
    int per_wave = 0, most = 6;
};
Cut group_cut(const SvoxTreeSpec* tree, int64_t n_rays, bool gradient, bool image) {
    Cut c;
    if (g_debug_flags != 0) {
        const int forced = (g_debug_flags & 32) ? g_debug_flags >> 8 : 0;
        c.per_wave = std::min(forced % 100, kGroupRays);
        c.most = std::min(std::max(forced / 100, 2), 6);
        return c;
    }
    // As many pieces as still are some leaves long, while the wavefronts have room on the GPU, fewer with more rays, and as few rays to a
    // wavefront as leaves the lists room for all they find: the launcher cannot know how many leaves have density, so the lines are
    // drawn where trees all of whose leaves do lose nothing or little.  What was measured (us; lanes that walk a ray together / pieces, in
    // parentheses where they are not taken; half of the leaves with density, all of them):
    //   forward           20 000 rays               26 000                    40 960
    //   16^3 SH4          66, 67 / 46, 52           68, 70 / (72, 78)         78, 81 / (88, 100)
    //   32^3 SH9          158, 163 / 95, 139        160, 167 / 104, 151       177, 182 / (136, 207)
    //   64^3 SH4          278, 285 / 144, 220       285, 294 / 165, 254       318, 328 / (242, 365)
    //   64^3 SH16         404, 427 / 174, 280       439, 463 / 219, 338       478, 496 / (312, 487)
    //   128^3 SH4         550, 565 / 296, 430       576, 590 / 358, 531       622, 646 / (528, 797)
    //   shell 128^3 SH9   290, 315 / 195, 247       320, 354 / 238, 291       330, 351 / (329, 421)
    //   shell 256^3 SH16  507, 599 / 253, 349       526, 620 / 303, 432       575, 677 / (434, 618)
    //   gradient          20 000 rays               26 000                    40 960                    65 536                    131 072
    //   16^3 SH4          120, 157 / 95, 158        129, 180 / 115, 147       162, 228 / 155, 209       224, 332 / 201, 276       341, 502 / (355, 486)
    //   32^3 SH9          308, 435 / 204, 327       343, 480 / 242, 398       418, 627 / 350, 542       610, 959 / 521, 771       917, 1502 / (974, 1451)
    //   64^3 SH4          553, 686 / 245, 518       597, 745 / 279, 601       696, 904 / 402, 867       1036, 1404 / 596, 1308    1574, 2196 / (1106, 2469)
    //   64^3 SH16         935, 1268 / 473, 965      1041, 1400 / 578, 1149    1271, 1850 / 815, 1625    1926, 2878 / 1201, 2454   3110, 4904 / (2221, 4617)
    //   128^3 SH4         1312, 1515 / 500, 1020    1355, 1599 / 597, 1261    1534, 1854 / 876, 1877    2385, 2987 / 1329, 2858   3678, 4680 / (2535, 5498)
    //   shell 128^3 SH9   611, 812 / 292, 563       644, 911 / 360, 654       688, 1071 / 487, 911      869, 1554 / 754, 1396     1362, 2308 / (1359, 2464)
    //   shell 256^3 SH16  1182, 1617 / 503, 1019    1147, 1732 / 587, 1223    1336, 1993 / 777, 1649    1600, 2816 / 1161, 2553   2532, 4447 / (2011, 4364)
    // (1 000 and 5 000 rays, pieces: 64^3 SH4 51, 54 and 68, 96, gradient step 123, 178 and 166, 329.  25 functions: 64^3, forward pass and gradient of 20 000 rays 203, 335 and 683,
    // 1432, gradient of 40 960 1136, 2449, shell 256^3 of 65 536 1675.)  Full 128^3 grids lose 1 % of a gradient of
    // 40 960 rays; of 131 072 rays they would lose 17 % (half-empty trees would gain up to a third).
    // The rays that meet the cube lie together in a picture, and fill the lists of a few wavefronts, while a batch deals them out: with more than kFill pixels small trees have
    // no gradient in pieces, and those of up to 32^3 leaves with fewer than nine functions no picture.  (Gradient of a picture from radius 1.5, 2.5 and 4, 150x150: 16^3 RGBA
    // 59 / 68, 52 / 72, 46 / 60, SH9 133 / 122, 90 / 94, 79 / 75, 250x250: 94 / 142, 58 / 135, 51 / 105, 261 / 267, 124 / 191, 86 / 137; picture, 150x150: 32^3 RGBA 65 / 69,
    // 60 / 77, 57 / 55, SH9 98 / 80, 86 / 83, 77 / 62.)  Larger trees lose at some distances and gain at others: 64^3 SH4, gradient, 200x200 459 / 353,
    // 330 / 267, 307 / 189, 250x250 593 / 518, 349 / 414, 300 / 249, 128^3 1129 / 1139, 876 / 798, 769 / 403.
    const double cells = (double)tree->capacity * 8.0;
    const bool tiny = cells < 2048.0, small = cells < 16384.0, medium = cells < 131072.0, large = cells >= 1048576.0;
    const bool grid = like_complete_octree(tree);
    constexpr int64_t kFill = 20480;
    if (tiny && !(gradient && n_rays <= 2560)) return c;
    const bool few = image && (gradient ? small : medium && tree->data_dim < 28);
    const int64_t most_rays = few ? kFill : gradient ? 65536 : small ? kFill : 26624;
    if (n_rays > most_rays) return c;
    if (small) {
        const bool eight = n_rays <= 14336 || n_rays > kFill;
        c.per_wave = eight ? 8 : 12;     // (8 rays to each of as many wavefronts as run at once)
        c.most = eight ? 3 : 2;
    } else if (medium) {
        const bool short_lists = n_rays <= 8192 || (gradient && n_rays > 14336);
        c.per_wave = short_lists ? 4 : 8;
        c.most = short_lists ? 4 : 3;
    } else {
        // (of a 128^3 grid the lists hold the leaves of two rays, four in a pinch: SH4, 4 x 16 / 2 x 32, gradient 12 000 rays 465, 910 / 342, 705, 20 000 650, 1302 / 503,
        // 1056, forward pass 12 000 rays 207, 361 / 189, 292, 20 000 286, 523 / 290, 450: from fewer rays on than here)
        const bool two = grid && large && (gradient || n_rays > 16384);
        c.per_wave = large && n_rays <= 1280 ? 1 : n_rays <= 2560 || two ? 2 : 4;
        c.most = large ? 6 : 5;
    }
    return c;
}

Lobes lobes_of(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt) {
    return Lobes{(const float*)tree->extra_data, tree->extra_cols, opt->format};
}

// Whether child_marks is a walk table, as svox_walk_table leaves it: one of its numbers in child_marks_softplus, and a child_marks_thresh below
// zero (or no number), which marks that apply to any call do not have.  Marks by themselves may say by any number but 0 that they were made with
// density_softplus.
bool has_walk_table(const SvoxTreeSpec* tree) {
    uint32_t bits;
    memcpy(&bits, &tree->child_marks_thresh, 4);
    const int32_t is = tree->child_marks_softplus;
    return tree->child_marks && bits > 0x80000000u &&
           (is == SVOX_MARKS_WALK || is == (SVOX_MARKS_WALK | 1) || is == (SVOX_MARKS_WALK | SVOX_MARKS_NONE));
}
// The threshold of the marks a walk table was made from, as it carries it: the next number of the other sign.
float walk_thresh(float thresh) {
    uint32_t bits;
    thresh += 0.0f;   // (-0 is 0)
    memcpy(&bits, &thresh, 4);
    bits = (bits + 1u) | 0x80000000u;
    memcpy(&thresh, &bits, 4);
    return thresh;
}
float marks_thresh(const SvoxTreeSpec* tree) {
    float thresh = tree->child_marks_thresh;
    if (!has_walk_table(tree)) return thresh;
    uint32_t bits;
    memcpy(&bits, &thresh, 4);
    bits = (bits & 0x7fffffffu) - 1u;
    memcpy(&thresh, &bits, 4);
    return thresh;
}
// Whether they are a walk table made without marks, which hides no leaf.
bool marks_none(const SvoxTreeSpec* tree) { return has_walk_table(tree) && (tree->child_marks_softplus & SVOX_MARKS_NONE); }

// Whether a launch that works on every leaf with density > need_thresh (the forward pass: opt->sigma_thresh; the
// backward passes, se_grad and the noting passes: 0) may read the caller's marks in place of the child table: the
// marks hide the leaves whose density is not > the threshold they were made with, which must all be leaves the launch skips.
bool marks_apply(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, float need_thresh) {
    if (marks_none(tree)) return true;
    const bool softplus = has_walk_table(tree) ? (tree->child_marks_softplus & 1) != 0 : tree->child_marks_softplus != 0;
    const float thresh = marks_thresh(tree);
    return tree->child_marks && thresh >= 0.0f && need_thresh >= thresh && softplus == (opt->density_softplus != 0);
}
// ... and whether the marks hide exactly the leaves the launch skips: every leaf they let through is shaded.
bool marks_decide(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, float need_thresh) {
    return marks_apply(tree, opt, need_thresh) && !marks_none(tree) && need_thresh == marks_thresh(tree);
}

// The tree as the octree march kernels see it: with the caller's marks in place of the child table where they apply.
TreeDev<float> march_tree(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, float need_thresh = 0.0f) {
    TreeDev<float> d = make_tree<float>(tree);
    if (marks_apply(tree, opt, need_thresh)) (has_walk_table(tree) ? d.walk : d.child) = tree->child_marks;
    d.walk_marked = d.walk && !marks_none(tree);
    return d;
}

// ... and of rays in pieces, who walk on the child table alone (calls of so few rays make no walk table)
TreeDev<float> on_child_table(TreeDev<float> tr) {
    tr.walk = nullptr;
    return tr;
}

// The table a walk table is made from.  Its rows are read 16 bytes at a time (walk_table_kernel): one that begins elsewhere, which the march itself
// reads entry by entry, serves no walk table.
const int32_t* walk_source(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, bool every_positive_leaf) {
    const int32_t* from = marks_apply(tree, opt, every_positive_leaf ? 0.0f : opt->sigma_thresh) ? tree->child_marks : tree->child;
    return ((uintptr_t)from & 15u) == 0 ? from : nullptr;
}

// Whether a call makes a walk table (svox_walk_table) for its march.  Making it costs 4 us and 11 ps a node, and a march that starts on a
// table no cache holds; a turn of the walk then waits for one read instead of two, or for none, though in three turns of ten it only descends.  So it pays
// where rays are many and apart.  us, whole calls without and with it, forward and with notes (SH9, SH4 on 128^3 and 512^3):
//   batches that all hit        13 000 rays                   40 000              100 000             300 000
//     64^3                      178, 196 / 153, 186           184, 240 / 163, 209 264, 351 / 232, 313 662, 983 / 527, 843
//     128^3                     351, 377 / 279, 334           363, 410 / 302, 384 568, 743 / 467, 610 2106, 2611 / 1495, 1992
//     shell 256^3               126, 241 / 107, 206           142, 307 / 120, 240 183, 341 / 162, 334 515, 1052 / 441, 910
//     shell 512^3               188, 308 / 166, 265           224, 334 / 198, 285 254, 439 / 224, 385 759, 1210 / 648, 1110
//   ... 18 % of which do: shell 128^3  53, 92 / 58, 96        53, 147 / 55, 136   69, 151 / 67, 141   132, 206 / 131, 169
//     shell 256^3               68, 130 / 82, 140             86, 205 / 89, 165   110, 224 / 105, 189 172, 265 / 181, 213
//     shell 512^3               96, 163 / 126, 189            128, 270 / 132, 228 161, 252 / 147, 231 240, 306 / 252, 259
//   pictures, 128, 200, 400, 800 pixels a side: shell 128^3  78, 71, 73, 79 / 70, 71, 70, 75;  256^3  132, 138, 136, 137 / 109, 119, 121, 122;
//     512^3  187, 193, 204, 205 / 166, 167, 175, 188, eight poses 764 / 687;  64^3  166, 157, 148, 158 / 166, 155, 150, 179;  128^3  332, 317, 290, 294 / 304, 300,
//     271, 319;  NDC 512^3, 128x96, 256x192, 504x378, 1008x756  123, 136, 171, 350 / 120, 120, 187, 366 (rays that share their nodes find them in L1)
//   ... with notes, 128, 200, 400, 800, which wait for the colours as much as for the walk: shell 128^3  172, 203, 218, 259 / 157, 203, 219, 256;  256^3  258, 287,
//     299, 347 / 212, 259, 295, 350;  512^3 SH16  341, 377, 400, 543 / 289, 329, 383, 530;  128^3 SH4  317, 317, 306, 429 / 320, 326, 311, 440
//   32^3 and smaller (batches of 13 000 and 300 000, picture of 800): 68, 253, 81 / 63, 232, 99
// Forward batches through shells most of whose rays miss lose by it from some 200 000 rays on, where making the table costs more than the few rays that hit
// gain: 18 % of 200 000, 300 000, 500 000 and 1 Mi rays, with thresholds, without and with it 256^3 SH9 150, 163, 240, 214 / 152, 174, 248, 226, 512^3 SH9 215, 231, 342,
// 321 / 220, 246, 362, 330, 256^3 RGBA 128, 153, 223, 194 / 142, 161, 234, 213.  They make one all the same, for those that all hit: 239, 373, 490, 881 / 218, 332, 442,
// 753, 366, 625, 787, 1400 / 355, 578, 717, 1238, 203, 297, 388, 621 / 196, 273, 370, 589.  How many hit the launcher does not know.
bool walk_table_pays(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int64_t n_rays, bool image, bool every_positive_leaf) {
    if (tree->N != 2 || tree->capacity > (int64_t)kWalkNodes || fast_basis(tree, opt) < 0) return false;
    if (has_walk_table(tree) || !walk_source(tree, opt, every_positive_leaf)) return false;
    if (g_debug_flags & 128) return true;
    if (tree->capacity < 32768 || n_rays <= 12288) return false;
    const bool grid = like_complete_octree(tree);
    // (with the shifted softplus rays end behind the first leaves they meet.  us, without and with: batches that all hit, 13 000, 66 000, 200 000 rays: 64^3
    // SH9 228, 265, 690 / 222, 263, 617, 128^3 SH4 423, 509, 1473 / 399, 476, 1143; shells, 66 000, 200 000 rays that all hit, 66 000 and 200 000 of which 18 % do: 128^3 SH9
    // 88, 156, 47, 100 / 85, 169, 51, 106, 256^3 134, 204, 63, 129 / 124, 215, 71, 143, 512^3 162, 306, 77, 146 / 159, 326, 90, 172; pictures, 128, 200, 400, 800: 128^3
    // shell 67, 67, 78, 91 / 70, 70, 85, 102, 512^3 SH1 83, 96, 112, 140 / 108, 118, 128, 148, 128^3 SH4 481, -, 415, 426 / 492, -, 428, 425)
    if (opt->density_softplus && (every_positive_leaf || image || !grid)) return false;
    if (image && opt->ndc_width > 0) return !grid && n_rays <= 65536;
    if (image && every_positive_leaf) return !grid && tree->capacity >= 131072;
    if (image) return !grid || (tree->capacity >= 262144 && n_rays <= 262144);
    return grid || n_rays >= (every_positive_leaf ? 40000 : 65536);
}

// the workspace argument of a forward launch that takes no notes
ReplaySpace no_notes() {
    ReplaySpace ws{};
    ws.spin_limit = (g_debug_flags & 16) ? 1 : 0;
    ws.give_ups = give_up_counter();
    return ws;
}

// Items (rays) a persistent wavefront owns.  With few rays every wavefront gets one 64-item chunk so
// that the launch spreads over as many SIMDs as possible; with many, several chunks, which lets lanes
// whose rays end early pick up new ones (measured on 1M random rays: forward best at 256 rays per
// wavefront, backward -- two marches per ray, longer-lived lanes -- at 512).
constexpr int64_t kRefillRays = 64 * 1024 * 8;
int pick_per_wave(int64_t total_items, bool backward) {
    const int forced = tuning().per_wave;
    if (forced == 64 || forced == 128 || forced == 256 || forced == 512 || forced == 1024) return forced;
    if (total_items < kRefillRays && !(g_debug_flags & 2)) return 64;
    return backward ? 512 : 256;
}

int pick_refill() {
    const int forced = tuning().refill;
    return forced >= 1 && forced <= 64 ? forced : 16;
}

// Image tiles handed to one XCD in a row (chunk_of_block): 16 tiles are four 16x16 pixel blocks.
// Measured on 8 poses of 800x800: 1 -> 16 shortens the launch by 2-3 %, larger runs gain no more and
// start to unbalance the XCDs.
int pick_xcd_group() {
    const int forced = tuning().xcd_group;
    return forced >= 1 && forced <= 4096 ? forced : 16;
}

template <typename T>
BatchSource<T> batch_source(const SvoxRaysSpec* rays, bool backward = false) {
    BatchSource<T> s;
    s.rays.origins = (const T*)rays->origins;
    s.rays.dirs = (const T*)rays->dirs;
    s.rays.vdirs = (const T*)rays->vdirs;
    s.rays.n_rays = rays->n_rays;
    s.per_wave = pick_per_wave(rays->n_rays, backward);
    s.refill_at = pick_refill();
    s.xcd_group = 1;
    s.n_waves = 0;
    return s;
}

// The persistent kernels deal the rays of a batch out over their wavefronts (BatchSource::n_waves).
template <typename T>
BatchSource<T> dealt_out(BatchSource<T> s, unsigned n_waves) {
    if (s.per_wave > kMarchThreads && (s.per_wave & (s.per_wave - 1)) == 0) s.n_waves = n_waves;
    return s;
}
template <typename T>
ImageSource<T> dealt_out(const ImageSource<T>& s, unsigned) { return s; }

// bytes after the chunks and the bitmap of a workspace: the stamp of the notes
constexpr int64_t kTailBytes = 256;

template <typename T>
ImageSource<T> image_source(const SvoxCameraSpec* cam, int n_images, int64_t pose_stride,
                            const SvoxRenderOptions* opt) {
    ImageSource<T> s;
    s.cam.c2w = (const T*)cam->c2w;
    s.cam.fx = cam->fx;
    s.cam.fy = cam->fy;
    s.cam.width = cam->width;
    s.cam.height = cam->height;
    s.n_images = n_images;
    s.pose_stride = pose_stride;
    // image tiles are coherent (rays of a tile end together) and only part of an image hits the
    // tree: one tile per wavefront keeps the busy tiles spread over the whole GPU
    s.per_wave = 64;
    s.refill_at = pick_refill();
    s.xcd_group = pick_xcd_group();
    s.run = 0;
    // Blocks from the middle of the image outwards, unless the camera is an NDC one: there every
    // ray crosses the whole tree, no part of the picture is longer than another, and rows of
    // blocks (slabs of the tree) share more leaves in L2 than rings do.  Measured (us, rows / rings):
    // one 800x800 pose of the sparse SH16 tree 317 / 304, 2 poses 344 / 314, 8 poses 695 / 670,
    // 16 poses 1159 / 1174; one pose of the dense 128^3 tree 385 / 340; 4 NDC poses 3538 / 3957.
    {
        const int forced = tuning().tile_order;
        s.inside_out = forced == 0 || forced == 1 ? forced : (opt->ndc_width > 0 ? 0 : 1);
    }
    if (n_images > 1) {
        const int forced = tuning().image_run;
        s.run = forced >= 0 ? forced : 4;
    }
    return s;
}

template <typename T>
int64_t total_items_of(const BatchSource<T>& s) { return s.rays.n_rays; }
template <typename T>
int64_t total_items_of(const ImageSource<T>& s) {
    const int64_t per_image = (int64_t)blocks16_of(s.cam.width) * blocks16_of(s.cam.height);
    const int64_t padded = s.run > 0 ? (per_image + s.run - 1) / s.run * s.run : per_image;
    return (int64_t)s.n_images * padded * 256;
}

unsigned blocks_for(int64_t items, int per_block) { return (unsigned)((items + per_block - 1) / per_block); }

#define SVOX_DISPATCH_OCTREE(D, ...)                                         \
    switch (D) {                                                             \
        case 0: { using P = OctreePolicy<SVOX_FORMAT_RGBA, 0>; __VA_ARGS__; } break; \
        case 1: { using P = OctreePolicy<SVOX_FORMAT_SH, 1>; __VA_ARGS__; } break;   \
        case 4: { using P = OctreePolicy<SVOX_FORMAT_SH, 4>; __VA_ARGS__; } break;   \
        case 9: { using P = OctreePolicy<SVOX_FORMAT_SH, 9>; __VA_ARGS__; } break;   \
        case 16: { using P = OctreePolicy<SVOX_FORMAT_SH, 16>; __VA_ARGS__; } break; \
        case 25: { using P = OctreePolicy<SVOX_FORMAT_SH, 25>; __VA_ARGS__; } break; \
        case kLobeKernels + 1: { using P = OctreePolicy<SVOX_FORMAT_SG, 1>; __VA_ARGS__; } break;   \
        case kLobeKernels + 4: { using P = OctreePolicy<SVOX_FORMAT_SG, 4>; __VA_ARGS__; } break;   \
        case kLobeKernels + 9: { using P = OctreePolicy<SVOX_FORMAT_SG, 9>; __VA_ARGS__; } break;   \
        case kLobeKernels + 16: { using P = OctreePolicy<SVOX_FORMAT_SG, 16>; __VA_ARGS__; } break; \
        default: { using P = OctreePolicy<SVOX_FORMAT_SG, 25>; __VA_ARGS__; } break; \
    }

// Whether a forward launch of `blocks` 64-ray wavefronts takes render_forward_split_kernel (two wavefronts per 64
// rays: one walks, one shades).  It shortens the chain of a tile's longest ray, which is what a launch that does not
// fill the GPU with heavy tiles waits for; where every tile is heavy and the GPU full, the second wavefront only
// takes a place another tile could have.  Measured on 800x800 poses of the sparse 512^3 SH16 tree (ms, one / two
// wavefronts per tile), orbit of radius 4 (18 % of the rays hit the tree): 1 pose 0.41 / 0.34, 2 poses 0.45 / 0.37,
// 4 poses 0.62 / 0.56, 8 poses 0.90 / 0.85, 16 poses 1.55 / 1.60; radius 2.5 (49 % hit): 0.43 / 0.38, 0.57 / 0.54,
// 0.97 / 0.95, 1.61 / 1.64, 2.91 / 3.14; radius 1.5 (every ray hits): 0.54 / 0.52, 0.88 / 0.90, 1.71 / 1.82,
// 3.14 / 3.40, 5.92 / 6.49.  With marks that decide the shading (`decided`: the one-wavefront kernel then reads a
// leaf's density with its coefficients, the two-wavefront kernel gains nothing from them) the balance tips earlier,
// launches alone: radius 4, 4 poses 0.48 / 0.47, 8 poses 0.69 / 0.72, 16 poses 1.13 / 1.30; radius 2.5, 8 poses
// 1.22 / 1.33.  The launcher cannot know how many rays hit, so the rule goes by tiles: images of up to 65 536 tiles
// (six 800x800 poses) -- 49 152 with deciding marks, 6 144 under NDC, where every ray passes through the tree (us, one /
// two, SH16 trees of 128^3 and 512^3: 3 024 tiles 117 / 115 and 310 / 279, 6 745 tiles 155 / 190 and 423 / 420, 11 970
// tiles 201 / 243 and 482 / 506) --, ray batches as
// long as all their blocks run at once (`at_once`; 3 072 tiles with up to 80 registers, fewer with more of them), beyond which the
// longest chain waits for a place: us, one / two wavefronts, unrelated rays that all hit, forward, training step, squared error:
//   SH9, at once 3 072 / 3 072: 256^3 shell, 196 001 rays 481 / 438, 1150 / 1074, 1543 / 1469; 200 003 rays 486 / 543, 1171 / 1194,
//   1563 / 1579; SH4 in a 512^3 shell 621 / 556, 1185 / 1086, 1494 / 1390 and 581 / 680, 1146 / 1208, 1466 / 1525;
//   SH16, 3 072 / 2 560: 256^3 shell, 160 001 rays 473 / 417, 1282 / 1195, 1818 / 1731; 170 001 rays 490 / 429, 1313 / 1378, 1904 / 1957;
//   SH25, 2 560 / 2 048: 256^3 shell, 130 001 rays 500 / 422, 1473 / 1366, 2174 / 2066; 150 001 rays 505 / 460, 1582 / 1628, 2381 / 2416;
//   170 001 rays 540 / 637, 1689 / 1752, 2591 / 2624;
//   the gradient by itself (2 560 to SH9, 2 048 beyond): SH9, 163 001 rays 1060 / 957, 170 001 rays 1081 / 1109.
// (Where most rays miss, as in pictures of a shell, noting passes gain a little beyond: SH9, 200 003 rays 572 / 533, 230 401 598 / 597;
// SH16 loses there too.)  On grids of 64^3 leaves and more not beyond 2 048: no ray is short there, a leaf to every layer
// of the grid, and the second wavefront has paid for itself sooner:
//   131 001 rays: 64^3 SH16 443 / 412, 1841 / 1971, 2866 / 2852; 128^3 SH9 895 / 866, 2888 / 2897, 4046 / 4069;
//   150 001 rays: 64^3 SH4 367 / 319, 1234 / 1191, 1794 / 1740, SH16 491 / 531, 2064 / 2087, 3284 / 3296; 128^3 SH9 1036 / 1062, 3076 /
//   3175, 4522 / 4633; 180 001 rays: 64^3 SH4 387 / 346, 1364 / 1343, 2052 / 2019, SH16 555 / 615, 2432 / 2557, 3828 / 3951; 128^3 SH9
//   1215 / 1316, 3546 / 3686, 5242 / 5389; 32^3 SH4 167 / 151, 739 / 721.  (N = 3, 81^3 SH9, walks longer: 736 / 665, 2517 / 2470,
//   3597 / 3617.)
bool use_split_forward(const SvoxTreeSpec* tree, unsigned blocks, bool image, const SvoxRenderOptions* opt, bool decided,
                       unsigned at_once) {
    const int forced = tuning().split_forward;
    const long limit = tuning().split_blocks;
    if (g_debug_flags & 12) return (g_debug_flags & 8) != 0;
    if (forced >= 0) return forced > 0;
    if (limit >= 0) return (long)blocks <= limit;
    if (!image) return blocks <= at_once && (blocks <= 2048u || tree->capacity < 37449 || !like_complete_octree(tree));
    if (opt->ndc_width > 0) return blocks <= 6144u;
    return blocks <= (decided ? 49152u : 65536u);
}
template <typename T>
constexpr bool is_image_source(const ImageSource<T>&) { return true; }
template <typename T>
constexpr bool is_image_source(const BatchSource<T>&) { return false; }

// How a forward pass cuts its rays into pieces (cut_kernel.h); no rays dealt to a wavefront: it does not.
// The pieces pay as long as they find the GPU idle: what each of them walks in vain -- the leaves until two walks agree -- is
// as much as a fair part of it, and the more of them the shorter; and as long as the lists hold what they find, which the more rays of a wavefront and
// the more leaves with density fills them the sooner.  The launcher knows neither how many rays meet the cube nor how many leaves have
// density, so the lines are drawn where launches of rays that all do gain nothing more and, within some per cent, trees all of whose
// leaves do lose nothing.  Trees are grids (like_complete_octree) or sparse ones, small (up to 32^3 leaves), fine (from 64^3, or the
// surface of 128^3, on) or large (128^3, the surface of 256^3).  us, march without notes and with, from end to end / in pieces, rays that all hit, half of
// a grid's leaves empty and a shell's all but the surface | no leaf empty:
//                1 000 rays                              4 096                                   8 192 (with notes, shells: 7 168)
//   8^3 SH1      not taken                               | 20, 26 / 34, 36 if it were
//   32^3 SH9     80, 80 / 27, 34    | 83, 92 / 40, 44    77, 77 / 41, 52     | 80, 91 / 53, 61    79, 82 / 53, 54      | 83, 107 / 76, 82
//   64^3 SH9     153, 153 / 37, 45  | 171, 194 / 65, 62  194, 192 / 62, 62   | 216, 234 / 143, 115   197, 196 / 110, 115 | 218, 237 / 154, 169
//   128^3 SH4    377, 377 / 62, 74  | 395, 423 / 86, 99  390, 387 / 112, 141 | 406, 432 / 245, 224   403, 400 / 192, 259 | 416, 437 / 361, 372
//   shell 128^3 SH9   128, 126 / 54, 60   | 131, 135 / 92, 76   170, 169 / 87, 99    | 185, 194 / 110, 127   180, 180 / 116, 149 | 187, 195 / 163, 206
//   shell 256^3 SH9   178, 173 / 48, 57   | 181, 188 / 83, 86   260, 257 / 114, 167  | 273, 273 / 150, 222   272, 242 / 185, 198 | 276, 254 / 249, 333
// (10 000 rays: 64^3 SH9 204, 204 / 132, 147 | 227, 247 / 183, 210, 128^3 417, 414 / 204, 304 | 435, 459 / 419, 447; 12 288 rays: 64^3 SH9 198, 200 /
// 158, 165 | 220, 243 / 222, 248, SH4 188, 195 / 161, 158 | 205, 228 / 214, 242, RGBA, not taken, 165, 176 / 144, 147 | 166, 187 / 200, 226.  Of views from afar, 18 % of whose
// rays hit a shell, 7 000 with notes take 169 / 89 at 256^3: for those the line of a full shell, 6 000 rays, is passed over.)
// With the shifted softplus every leaf is listed and rays end behind what they met (opaque_light), from end to end as in pieces.  A shell of 256^3,
// without notes and with: 1 000 rays 74, 80 / 45, 61, 4 096 84, 95 / (116, 186).
// Square pictures, 64, 90 pixels a side, from close up (every pixel hits) and from afar, half empty | full:
//   64^3 SH9          121, 145 / 63, 60, 100, 105 / 32, 40 | 165, 210 / 93, 97     121, 140 / 86, 140 | 157, 191 / 136, 198
//   128^3 SH4         299, 302 / 115, 129, 209, 222 / 43, 57 | 351, 389 / 167, 218 273, 274 / 182, 279 | 321, 353 / 296, 403
//   shell 128^3 SH9   142, 149 / 69, 80 | 193, 218 / 91, 116                       149, 159 / 117, 150 | 198, 224 / 158, 210
//   shell 256^3 SH9   225, 225 / 111, 123 | 257, 285 / 143, 175                    223, 222 / 203, 224 | 266, 295 / 267, 316
//   NDC, every ray in the tree, half empty, 256^3 and 512^3  133, 86 / 108, 49  151, 114 / 172, 79;  227, 129 / 225, 83  245, 158 / 335, 116 (with notes, without)
Cut pick_cut(const SvoxTreeSpec* tree, int64_t items, bool image, const SvoxRenderOptions* opt, bool noted) {
    const int forced = (g_debug_flags & 32) ? g_debug_flags >> 8 : g_debug_flags == 0 ? tuning().cut : 0;
    Cut c;
    if (forced >= 0) {
        c.per_wave = std::min(forced % 10, kCutMostRays);
        c.most = std::min(forced / 10, 6);
        return c;
    }
    const double cells = (double)tree->capacity * tree->N * tree->N * tree->N;
    const bool tiny = cells < 2048.0, small = cells < 65536.0, large = cells >= 1048576.0;
    const bool grid = like_complete_octree(tree), sparse = !grid && !small, fine = cells >= 262144.0;
    const bool softplus = opt->density_softplus;
    if (tiny) return c;
    if (image && opt->ndc_width > 0) {
        if (items <= (noted ? 4096 : 8192)) c.per_wave = small ? 8 : 4;
        return c;
    }
    int64_t limit = 8192;
    if (image && !small) limit = grid && !noted ? 12288 : 9216;   // (in blocks of 16 x 16)
    if (!image && !small) limit = grid ? (large || tree->data_dim < 13 ? 10240 : 12288) : noted ? 7168 : 8192;
    if (softplus) limit = small ? 4096 : grid ? (noted ? 4096 : 8192) : noted ? (image ? 1024 : 2048) : image ? 4096 : 3072;
    if (items > limit) return c;
    if (image) {
        // (most pixels of a picture miss: a wavefront finds one ray or two among its few)
        if (small || (grid && !large && items > 9216))
            c.per_wave = 8, c.most = 4;
        else if (!large && (grid || !fine))
            c.per_wave = 4, c.most = 4;
        else if (sparse && large && !noted && !softplus)
            c.per_wave = 1;
        else if (sparse && !large && noted && items > 8192)
            c.per_wave = 4;
        else
            c.per_wave = 2, c.most = 5;
    } else if (small) {
        c.per_wave = items <= 4096 || (cells >= 16384.0 && !noted) ? 4 : 8;
    } else if (!large) {
        if (noted)
            c.per_wave = items <= 2048 || (sparse && fine && (tree->N == 2 || items <= 4096)) ? 2 : 4;
        else
            c.per_wave = items > (grid ? 3072 : 4096) && items <= 6144 && (grid || !fine) ? 4 : 2;
    } else if (grid) {
        c.per_wave = items <= 1536 ? 1 : 2;
    } else {
        c.per_wave = items <= (softplus ? 1024 : noted ? 4096 : 8192) ? 1 : 2;
    }
    return c;
}

template <class Source, typename T>
void launch_forward(const SvoxTreeSpec* tree, const Source& src, const SvoxRenderOptions* opt, int out_dim,
                    void* out, hipStream_t stream) {
    const int64_t items = total_items_of(src);
    if constexpr (sizeof(T) == 4) {
        const int D = fast_basis(tree, opt);
        if (D >= 0) {
            const TreeDev<float> tr = march_tree(tree, opt, opt->sigma_thresh);
            const ReplaySpace none = no_notes();
            const Cut cut = tree->weight_accum ? Cut() : pick_cut(tree, items, is_image_source(src), opt, false);
            if (cut.per_wave > 0) {
                SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::cut(dim3(blocks_for(items, cut.per_wave)), stream, on_child_table(tr), src, *opt, (float*)out,
                                                                    none, false, nullptr, nullptr, cut.per_wave, cut.most));
                return;
            }
            const unsigned blocks = blocks_for(items, src.per_wave);
            const Source dealt = dealt_out(src, blocks);
            // Marks made with this launch's own threshold: every leaf they let through is shaded, and the kernel with
            // one wavefront per tile or chunk then reads a leaf's density with its coefficients (one round trip per
            // round instead of two that wait for one another: 4 NDC poses 3.10 -> 2.93 ms).  The two-wavefront kernel
            // keeps its density phase: there the walk is the critical path, the density read of a leaf brings the
            // last line of its record into L2 ahead of the coefficient reads, and without it the kernel needs more
            // registers (5 instead of 6 wavefronts per SIMD): measured 0.70 -> 0.73 ms on 8 poses of 800x800,
            // although the launch sends 17 % fewer requests to L2.
            const bool all_shaded = !tree->weight_accum && marks_decide(tree, opt, opt->sigma_thresh);
            const bool refill = src.per_wave > kMarchThreads;
            unsigned at_once = 0;
            SVOX_DISPATCH_OCTREE(D, at_once = MarchLaunch<P, Source>::split_tiles_at_once(false, false));
            const bool split = !refill && !tree->weight_accum &&
                               use_split_forward(tree, blocks, is_image_source(src), opt, all_shaded, at_once);
            SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::forward(dim3(blocks), stream, tr, dealt, *opt, (float*)out, none,
                                                                    split, tree->weight_accum != nullptr, refill, all_shaded));
            return;
        }
    }
    if constexpr (sizeof(T) == 8) {
        const int D = group_basis(tree, opt, items);
        if (D >= 0) {
            const Cut cut = group_cut(tree, items, false, is_image_source(src));
            if (cut.per_wave > 0)
                launch_group_forward(D, dim3(blocks_for(items, cut.per_wave)), stream, make_tree<double>(tree), src, *opt, (double*)out,
                                     cut.per_wave, cut.most);
            else
                launch_shared_forward(D, dim3(blocks_for(items, kSharedRays)), stream, make_tree<double>(tree), src, *opt, (double*)out);
            return;
        }
    }
    const int basis_rows = opt->format == SVOX_FORMAT_RGBA ? 1 : opt->basis_dim;
    hipLaunchKernelGGL((render_forward_generic_kernel<T, Source>), dim3(blocks_for(items, kMarchThreads)),
                       dim3(kMarchThreads), generic_forward_lds_bytes<T>(basis_rows, out_dim), stream,
                       make_tree<T>(tree), src, *opt, out_dim, (T*)out);
}

constexpr int64_t kChunkBytes = (int64_t)kChunkFloat2 * 8;   // 384: 15 records and a link

// What the notes in a workspace belong to (ReplaySpace::stamp).
struct NoteStamp {
    unsigned long long word[kStampWords];
};
NoteStamp stamp_of(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt) {
    NoteStamp st;
    uint32_t step_bits, thresh_bits;
    memcpy(&step_bits, &opt->step_size, 4);
    memcpy(&thresh_bits, &opt->sigma_thresh, 4);
    st.word[0] = 0x73766f786e6f7465ull ^ (unsigned long long)rays->n_rays ^ (opt->density_softplus ? 1ull << 62 : 0ull);
    st.word[1] = (unsigned long long)(uintptr_t)tree->data;
    st.word[2] = (unsigned long long)(uintptr_t)rays->origins;
    st.word[3] = ((unsigned long long)thresh_bits << 32) | step_bits;
    st.word[4] = (unsigned long long)(uintptr_t)tree->child;
    st.word[5] = (unsigned long long)(uintptr_t)rays->dirs;
    return st;
}

// Whether a noting pass over pictures lists the pixels that meet the cube first, and deals them out so that every tile has some from all over the
// picture (PicturesSpread).  A tile of 8 x 8 pixels has long rays or short ones, and leaves to shade in the same rounds or none, and the pass takes as long as
// the worst of them; dealt out they are alike: 800x800 picture of a 512^3 SH16 shell 538 -> 417 us, of a 256^3 SH16 shell 453 -> 332, of 400x400 322 -> 251.
// Not for grids that are as fine everywhere, whose rays are alike and read the same lines (64^3 SH9 400x400 175 / 178, 800x800 218 / 239; 128^3 SH4 435 / 507), trees
// of fewer than 65 536 cells (16^3 RGBA 132 / 245), trees of other branching factors, whose rays walk longer and are no longer alike (gradient of an 800x800 picture,
// us, as it is / listed: 81^3 SH9 full 1047 / 1100, one leaf in twenty 363 / 435, 64^3 (N = 4) SH1 400x400 208 / 221), pictures in normalised device coordinates, all of
// whose rays meet the cube, and where what is to be gone through is small beside the launches or large beside the hits: under 16 384 pixels, over 2 Mi (1700x1700, 16 000 hits: 412 / 428).
bool lists_pixels(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int64_t n_pixels) {
    if (g_debug_flags & 64) return true;
    const Tuning& t = tuning();
    return g_debug_flags == 0 && t.per_wave <= 0 && t.split_forward < 0 && t.split_blocks < 0 && opt->ndc_width <= 0 && n_pixels >= 1 << 14 &&
           n_pixels <= 1 << 21 && tree->N == 2 && tree->capacity * 8 >= 65536 && !like_complete_octree(tree);
}
// Up to how many: tiles that are alike must all find a place at once, or the last of them take as long again when the first have ended (800x800, 256^3 SH9 shell:
// 2 530 tiles 262 -> 225 us, 2 712 tiles 256 -> 402, of 2 816 places; SH16, of 2 560: 2 290 tiles 439 -> 343, 2 446 445 -> 490).  Few functions leave little to
// level, while rays from all over read more lines: half as many then (512^3 SH1 shell 125 000 hits 318 / 332; 74 000 hits, 512^3 SH4 392 -> 334, 256^3 SH1 252 -> 241).
// Pictures with more hits pay for the sample and a launch without tiles: 5 to 10 us (800x800 close up, 512^3 SH16 868 / 876, 128^3 SH4 328 / 334).
int64_t most_listed_pixels(const SvoxRenderOptions* opt, int64_t n_pixels, unsigned at_once) {
    if (g_debug_flags & 64) return std::min((int64_t)(g_debug_flags >> 8 & 255) * kMarchThreads, n_pixels);
    const bool light = opt->format == SVOX_FORMAT_RGBA || opt->basis_dim < 9;
    const int64_t tiles = (int64_t)std::min(at_once, 2816u) * 9 / 10;
    return std::min((light ? tiles / 2 : tiles) * kMarchThreads, n_pixels);
}
constexpr int64_t kListRays = 1 << 17;
bool list_at_end(int64_t n_slots) { return n_slots >= kListRays || (g_debug_flags & 64); }
template <class Source>
bool keeps_list(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, const Source& src, int64_t n_slots) {
    return is_image_source(src) ? lists_pixels(tree, opt, n_slots) : list_at_end(n_slots);
}

// The workspace of the replaying kernels: chunks of notes, then one bit per ray (rays left undone by
// replay_backward_kernel), then 256 bytes that hold the stamp of the notes and, from byte 128 on, four
// words (cleared before every launch that takes notes): the chunk stocks handed out, the chunks that rays in
// pieces took one by one (take_chunks, which keeps the first in step), and the rays listed (list_hits_kernel); and whether any ray was left undone.
constexpr int64_t kStampOffset = 0;
constexpr int64_t kStockCounterOffset = 128;
int64_t bitmap_bytes(int64_t n_slots) { return ((n_slots + 63) / 64 * 8 + 15) / 16 * 16; }
// (and, of a batch or pictures whose rays may be listed, where the rays' shared chunks are many beside it, in the place of the last of them: a number per
// ray.  Every pass over the notes says so alike (keeps_list), or the room they are in would not be the same.  Of pictures with fewer pixels than
// kListRays the list lies in the first stocks instead, which a launch that lists takes like any others: svox_notes_pool_info, which knows of
// a workspace neither the tree nor whether its rays are a batch, has to know how many stocks it had.)
bool carve_workspace(void* workspace, int64_t workspace_bytes, int64_t n_slots, bool list, ReplaySpace* ws) {
    *ws = ReplaySpace{};
    int64_t chunks = workspace && n_slots > 0
                         ? (workspace_bytes - kTailBytes - bitmap_bytes(n_slots)) / kChunkBytes : 0;
    if (n_slots <= 0 || chunks < n_slots || chunks >= 0x7fffffffll || ((uintptr_t)workspace & 15u) != 0) return false;
    ws->base = (float2*)workspace;
    ws->undone = (unsigned long long*)((char*)workspace + chunks * kChunkBytes);
    const int64_t list_chunks = (n_slots * 4 + kChunkBytes - 1) / kChunkBytes;
    if (list && chunks - n_slots >= 16 * list_chunks) {
        if (list_at_end(n_slots))
            chunks -= list_chunks;
        else
            ws->list_stocks = (uint32_t)((list_chunks + kChunkStock - 1) / kChunkStock);
        ws->list = (int32_t*)((char*)workspace + (ws->list_stocks ? n_slots : chunks) * kChunkBytes);
    }
    ws->first_shared = n_slots;
    ws->n_chunks = chunks;
    ws->n_stocks = (uint32_t)((chunks - n_slots + kChunkStock - 1) / kChunkStock);
    ws->stamp_at = (unsigned long long*)((char*)ws->undone + bitmap_bytes(n_slots) + kStampOffset);
    ws->stocks_taken = (unsigned long long*)((char*)ws->undone + bitmap_bytes(n_slots) + kStockCounterOffset);
    ws->any_undone = ws->stocks_taken + 3;
    return true;
}

// The backward pass by two marches per ray (no workspace, or one that cannot serve: see backward_by_noting).
template <class Source, typename T>
void launch_backward(const SvoxTreeSpec* tree, const Source& src, const SvoxRenderOptions* opt, int out_dim,
                     const void* grad_out, void* grad_data, hipStream_t stream) {
    const int64_t items = total_items_of(src);
    if constexpr (sizeof(T) == 4) {
        const int D = fast_basis(tree, opt);
        if (D >= 0) {
            const unsigned blocks = blocks_for(items, src.per_wave);
            const Source dealt = dealt_out(src, blocks);
            const ReplaySpace none{};
            SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::backward(dim3(blocks), stream, march_tree(tree, opt), dealt, *opt,
                                                                     (const float*)grad_out, (float*)grad_data, none,
                                                                     src.per_wave > kMarchThreads, false));
            return;
        }
    }
    if constexpr (sizeof(T) == 8) {
        const int D = group_basis(tree, opt, items);
        if (D >= 0) {
            const Cut cut = group_cut(tree, items, true, is_image_source(src));
            if (cut.per_wave > 0)
                launch_group_backward(D, dim3(blocks_for(items, cut.per_wave)), stream, make_tree<double>(tree), src, *opt,
                                      (const double*)grad_out, (double*)grad_data, cut.per_wave, cut.most);
            else
                launch_shared_backward(D, dim3(blocks_for(items, kSharedRays)), stream, make_tree<double>(tree), src, *opt,
                                       (const double*)grad_out, (double*)grad_data);
            return;
        }
    }
    const int basis_rows = opt->format == SVOX_FORMAT_RGBA ? 1 : opt->basis_dim;
    hipLaunchKernelGGL((render_backward_generic_kernel<T, Source>), dim3(blocks_for(items, kMarchThreads)),
                       dim3(kMarchThreads), generic_backward_lds_bytes<T>(basis_rows, out_dim), stream,
                       make_tree<T>(tree), src, *opt, out_dim, (const T*)grad_out, (T*)grad_data);
}

// The launch shape of the noting forward pass for the rays of `s`: that of a forward pass (a batch
// source made for a backward pass gives its wavefronts more rays than the forward kernels like).
template <typename T>
BatchSource<T> noting_shape(BatchSource<T> s) {
    s.per_wave = pick_per_wave(s.rays.n_rays, false);
    return s;
}
template <typename T>
ImageSource<T> noting_shape(const ImageSource<T>& s) { return s; }

// The rays of a batch or of pictures that meet the cube, in the order they come in block by block (the blocks as they get there); the others are
// answered as a noting pass answers them.  200 003 rays 9 us, 1 Mi rays 30: 24 bytes
// read of each, and a line written for every one that misses, the head of its notes.  Where a sample of the rays says that more than
// `most` hit, nothing is listed (4.5 us), and the number stands for the batch as it is.  Pixels of an 800x800 picture 20 us.
constexpr int kListThreads = 1024;
// The rays as a listing launch goes through them, place by place.
struct BatchInOrder {
    static constexpr int kSample = 256;
    BatchSource<float> rays;
    __device__ __forceinline__ int64_t n_rays() const { return rays.rays.n_rays; }
    __device__ __forceinline__ int64_t sample(int i) const { return (int64_t)i * n_rays() / kSample; }
    __device__ __forceinline__ int64_t fetch(int64_t place, const SvoxRenderOptions& opt, const float* offset, const float* scaling,
                                             float* origin, float* dir, float* vdir) const {
        return rays.fetch_item(place, opt, offset, scaling, origin, dir, vdir);
    }
};
// Pieces of a row of 16 pixels, from all over the pictures in turn: the next piece lies `step` pieces on, about 0.618 of all there are and without a common
// factor with their number, so that any run of places is spread evenly.
constexpr int kListPiece = 16;
struct PicturesSpread {
    static constexpr int kSample = 256;
    ImageSource<float> pictures;
    int64_t n_pieces, step;
    __device__ __forceinline__ int64_t n_rays() const { return pictures.n_slots(); }
    __device__ __forceinline__ int64_t sample(int i) const { return (int64_t)i * kListPiece + i % kListPiece; }
    __device__ __forceinline__ int64_t fetch(int64_t place, const SvoxRenderOptions& opt, const float* offset, const float* scaling,
                                             float* origin, float* dir, float* vdir) const {
        const int64_t piece = place / kListPiece;
        const int64_t slot = piece * step % n_pieces * kListPiece + place % kListPiece;
        if (piece >= n_pieces || slot >= n_rays()) return -1;
        return pictures.fetch_slot(slot, opt, offset, scaling, origin, dir, vdir);
    }
};
int64_t spread_step(int64_t n_pieces) {
    int64_t step = std::max((int64_t)((double)n_pieces * 0.6180339887), (int64_t)1);
    while (std::gcd(step, n_pieces) != 1) ++step;
    return step;
}
template <class Places>
__global__ __launch_bounds__(kListThreads) void list_hits_kernel(TreeDev<float> tr, Places src, SvoxRenderOptions opt,
                                                                 float* __restrict__ out, ReplaySpace ws,
                                                                 unsigned long long* __restrict__ n_listed, int64_t most) {
    __shared__ int32_t hits[kListThreads / kMarchThreads];
    __shared__ unsigned long long first;
    float offset[3], scaling[3], origin[3], dir[3], vdir[3];
    load_transform(tr, offset, scaling);
    const int wave = threadIdx.x / kMarchThreads, lane = threadIdx.x & (kMarchThreads - 1);
    RayState<float> r;
    // (the same rays for every block, which all come to the same answer)
    if (threadIdx.x < Places::kSample) {
        const int64_t some = src.fetch(src.sample(threadIdx.x), opt, offset, scaling, origin, dir, vdir);
        const unsigned long long m = __ballot(some >= 0 && setup_ray(r, origin, dir, scaling));
        if (lane == 0) hits[wave] = __popcll(m);
    }
    __syncthreads();
    int sampled = 0;
#pragma unroll
    for (int i = 0; i < Places::kSample / kMarchThreads; ++i) sampled += hits[i];
    if (sampled * src.n_rays() > Places::kSample * most) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *n_listed = (unsigned long long)src.n_rays();
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && ws.list_stocks) *ws.stocks_taken = ws.list_stocks;
    __syncthreads();
    const int64_t slot = src.fetch(blockIdx.x * (int64_t)kListThreads + threadIdx.x, opt, offset, scaling, origin, dir, vdir);
    const bool hit = slot >= 0 && setup_ray(r, origin, dir, scaling);
    if (slot >= 0 && !hit) {
        if (out) {
            out[slot * 3] = opt.background_brightness;
            out[slot * 3 + 1] = opt.background_brightness;
            out[slot * 3 + 2] = opt.background_brightness;
        }
        NoteTaker::missed(ws, slot);
    }
    const unsigned long long m = __ballot(hit);
    if (lane == 0) hits[wave] = __popcll(m);
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int i = 0; i < kListThreads / kMarchThreads; ++i) {
        before += i < wave ? hits[i] : 0;
        all += hits[i];
    }
    if (threadIdx.x == 0) first = all > 0 ? atomicAdd(n_listed, (unsigned long long)all) : 0ull;
    __syncthreads();
    if (hit) ws.list[first + before + rank_in(m)] = (int32_t)slot;
}

// The shapes of a noting pass whose rays are listed first (ListedSource): up to `two` rays that meet the cube two wavefronts per tile,
// up to `one` one; beyond -- most of the batch does -- the batch as it is.  Only where the batch, if all of it met the cube, would not
// take two wavefronts anyway (the same rays listed or not: 256^3 shell, 100 000 rays 254 / 255 us, 200 000 rays 283 / 292), and not on
// trees to 32^3, whose marches are short beside the listing (16^3 RGBA, 300 000 rays that all hit 181 / 192).  us, batch as it is / listed,
// the noting march, the gradient by itself, the squared error; 18 % of the rays of a shell hit:
//   256^3 shell SH9   200 003 rays 339, 483, 577 / 290, 413, 524   300 000 rays 405, 573, 665 / 317, 450, 568   500 000 rays 566, 794, 921 / 332, 518, 680
//   512^3 shell SH16  170 000 rays 452, 820 / 383, 723   500 000 rays 775, 1208 / 457, 870   1 048 576 rays 749, 1332 / 708, 1313
//   512^3 shell SH25  400 000 rays 727, 1389 / 453, 1025    256^3 shell SH4 700 000 rays 458, 632, 741 / 344, 505, 632
// Where all of them hit, what the sample, the launches without rays and the look at which launch has them cost (the noting march, the gradient,
// the squared error; not listed / listed): 256^3 shell SH9 200 003 rays 540, 1044, 1463 / 548, 1039, 1457, 500 000 rays 1096, 2190, 3129 / 1105,
// 2189, 3124, 1 000 000 rays 1938, 3949, 5804 / 1951, 3967, 5800; 64^3 SH9 200 003 rays 663, 1877, 2854 / 673, 1893, 2863.
struct ListShapes {
    bool any = false;
    int64_t two = 0, one = 0;
};
ListShapes list_shapes(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int64_t n_rays, unsigned at_once) {
    ListShapes s;
    if (g_debug_flags & 64) {
        s.any = true;
        s.two = (g_debug_flags >> 8 & 255) * kMarchThreads;
        s.one = (g_debug_flags >> 16) * kMarchThreads;
        return s;
    }
    const Tuning& t = tuning();
    if (g_debug_flags != 0 || t.per_wave > 0 || t.split_forward >= 0 || t.split_blocks >= 0) return s;
    s.two = (int64_t)(use_split_forward(tree, at_once, false, opt, false, at_once) ? at_once : std::min(at_once, 2048u)) * kMarchThreads;
    s.one = std::max(std::min(kRefillRays - 1, n_rays - n_rays / 4), s.two);
    s.any = n_rays > s.two && (double)tree->capacity * tree->N * tree->N * tree->N >= 131072.0;
    return s;
}

// What a noting launch clears on the way (clear_share): up to two arrays of so many bytes.
struct ClearWork {
    void* at[2] = {nullptr, nullptr};
    int64_t bytes = 0;
};
constexpr int64_t kMostCleared = kClearWords * 4 * (1 << 24);   // (a launch has fewer than 2^32 threads)

// The forward pass of a training step: the picture into `out` and, in the workspace, the notes of
// every ray under `stamp`.  Needs a usable workspace and the octree kernels, which noted_ok() tells
// beforehand.  A launch that does not fill the GPU runs on two wavefronts per 64 rays.  out may be
// nullptr (notes only); grad_out, if given, is the gradient of the picture the backward pass will be
// called with: the notes' heads then also carry the sum of that pass's first march.
template <class Source>
int launch_noted(const SvoxTreeSpec* tree, const Source& src, const SvoxRenderOptions* opt, void* out,
                 void* workspace, int64_t workspace_bytes, int64_t n_slots, const NoteStamp& stamp,
                 hipStream_t stream, const void* grad_out = nullptr, const void* color_ref = nullptr,
                 const ClearWork& clear = ClearWork()) {
    const int D = fast_basis(tree, opt);
    const unsigned blocks = blocks_for(total_items_of(src), src.per_wave);
    const Source dealt = dealt_out(src, blocks);
    ReplaySpace ws;
    if (D < 0 || !carve_workspace(workspace, workspace_bytes, n_slots, keeps_list(tree, opt, src, n_slots), &ws))
        return fail(SVOX_ERR_BAD_SHAPE, "notes asked for where they cannot be taken");
    const int rc = zero_fill(ws.stocks_taken, 32, stream);
    if (rc) return rc;
    memcpy(ws.stamp, stamp.word, sizeof(ws.stamp));
    ws.spin_limit = (g_debug_flags & 16) ? 1 : 0;
    ws.give_ups = give_up_counter();
    // (the launch that has the rays clears what is to be cleared)
    ws.clear_at[0] = (uint32_t*)clear.at[0];
    ws.clear_at[1] = (uint32_t*)clear.at[1];
    ws.clear_words = clear.bytes / 4;
    auto with_clearing = [&](unsigned march) {
        ws.march_blocks = march;
        return dim3(march + (unsigned)((ws.clear_words + kClearWords - 1) / kClearWords));
    };
    const Cut cut = pick_cut(tree, total_items_of(src), is_image_source(src), opt, true);
    if (cut.per_wave > 0) {
        const dim3 grid = with_clearing(blocks_for(total_items_of(src), cut.per_wave));
        SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::cut(grid, stream,
                                                            on_child_table(march_tree(tree, opt)), src, *opt, (float*)out, ws, true,
                                                            (const float*)grad_out, (const float*)color_ref, cut.per_wave, cut.most));
        return SVOX_OK;
    }
    const bool refill = src.per_wave > kMarchThreads;
    unsigned at_once = 0;
    SVOX_DISPATCH_OCTREE(D, at_once = MarchLaunch<P, Source>::split_tiles_at_once(true, grad_out != nullptr));
    if constexpr (!is_image_source(Source())) {
        // (most of a batch often misses the cube, and the lanes of the rays that do idle; which shape suits those that meet it, the
        // device decides: every launch but one has no rays)
        const ListShapes shapes = list_shapes(tree, opt, src.rays.n_rays, at_once);
        if (ws.list && shapes.any) {
            unsigned long long* const n_listed = ws.stocks_taken + 2;
            const int64_t listed = std::max(shapes.one, shapes.two);
            BatchInOrder places{src};
            places.rays.n_waves = 0;
            hipLaunchKernelGGL(list_hits_kernel<BatchInOrder>, dim3(blocks_for(src.rays.n_rays, kListThreads)), dim3(kListThreads), 0, stream,
                               march_tree(tree, opt), places, *opt, (float*)out, ws, n_listed, listed);
            ws.n_listed = n_listed;
            auto launch_listed = [&](int64_t least, int64_t most, bool two) {
                ListedSource tiles;
                (Source&)tiles = src;
                tiles.per_wave = kMarchThreads;
                tiles.list = ws.list;
                tiles.n_listed = n_listed;
                ws.least = least;
                ws.most = most;
                const dim3 grid = with_clearing(blocks_for(std::min(most, src.rays.n_rays), kMarchThreads));
                SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, ListedSource>::noting(grid, stream, march_tree(tree, opt), tiles, *opt, (float*)out,
                                                                             ws, (const float*)grad_out, (const float*)color_ref, two, false));
            };
            if (shapes.two > 0) launch_listed(0, shapes.two, true);
            if (shapes.one > shapes.two) launch_listed(shapes.two > 0 ? shapes.two + 1 : 0, shapes.one, false);
            if (src.rays.n_rays > listed) {
                ws.least = listed > 0 ? listed + 1 : 0;
                ws.most = INT64_MAX;
                WholeSource whole;
                (Source&)whole = dealt;
                const dim3 grid = with_clearing(blocks);
                SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, WholeSource>::noting(grid, stream, march_tree(tree, opt), whole, *opt, (float*)out, ws,
                                                                            (const float*)grad_out, (const float*)color_ref, false, refill));
            }
            return SVOX_OK;
        }
    }
    const bool split = !refill && use_split_forward(tree, blocks, is_image_source(src), opt, false, at_once);
    if constexpr (is_image_source(Source())) {
        const int64_t most = split && ws.list ? most_listed_pixels(opt, n_slots, at_once) : 0;
        if (most > 0) {
            unsigned long long* const n_listed = ws.stocks_taken + 2;
            const int64_t n_pieces = (n_slots + kListPiece - 1) / kListPiece;
            const PicturesSpread places{src, n_pieces, spread_step(n_pieces)};
            // (nothing is listed only where the number that then stands for all of them, n_slots, is more than the listed shape takes; a sample is
            // some per cent off)
            const int64_t sampled_most = n_slots > most ? most - most / 32 : n_slots;
            hipLaunchKernelGGL(list_hits_kernel<PicturesSpread>, dim3(blocks_for(n_pieces * kListPiece, kListThreads)), dim3(kListThreads), 0,
                               stream, march_tree(tree, opt), places, *opt, (float*)out, ws, n_listed, sampled_most);
            ws.n_listed = n_listed;
            auto launch_pixels = [&](auto pixels, int64_t tiles, int64_t least, int64_t most_here) {
                ws.least = least;
                ws.most = most_here;
                const dim3 grid = with_clearing((unsigned)tiles);
                SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, decltype(pixels)>::noting(grid, stream, march_tree(tree, opt), pixels, *opt, (float*)out,
                                                                                 ws, (const float*)grad_out, (const float*)color_ref, true, false));
            };
            ListedImageSource listed;
            (Source&)listed = src;
            listed.xcd_group = 1;
            listed.list = ws.list;
            listed.n_listed = n_listed;
            launch_pixels(listed, blocks_for(most, kMarchThreads), 0, most);
            if (n_slots > most) {
                WholeImageSource whole;
                (Source&)whole = src;
                launch_pixels(whole, blocks, most + 1, INT64_MAX);
            }
            return SVOX_OK;
        }
    }
    const dim3 grid = with_clearing(blocks);
    SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::noting(grid, stream, march_tree(tree, opt), dealt, *opt,
                                                           (float*)out, ws, (const float*)grad_out,
                                                           (const float*)color_ref, split, refill));
    return SVOX_OK;
}

int64_t data_bytes(const SvoxTreeSpec* t) {
    const int64_t esz = t->dtype == SVOX_F32 ? 4 : 8;
    return t->capacity * t->N * t->N * t->N * t->data_dim * esz;
}

// `only`: a bitmap of the rays to do (octree kernels only; the batch rays are then not dealt out)
template <class Source, typename T>
void launch_se_grad(const SvoxTreeSpec* tree, const Source& src, const SvoxRenderOptions* opt, int out_dim,
                    const void* color_ref, void* color_out, void* grad, void* hess, hipStream_t stream,
                    const unsigned long long* only = nullptr, const unsigned long long* any_undone = nullptr) {
    const int64_t items = total_items_of(src);
    if constexpr (sizeof(T) == 4) {
        const int D = fast_basis(tree, opt);
        if (D >= 0) {
            const unsigned blocks = blocks_for(items, src.per_wave);
            const Source dealt = only ? src : dealt_out(src, blocks);
            SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::se_grad(dim3(blocks), stream, march_tree(tree, opt), dealt, *opt,
                                                                    (const float*)color_ref, (float*)color_out,
                                                                    (float*)grad, (float*)hess, only, any_undone,
                                                                    src.per_wave > kMarchThreads));
            return;
        }
    }
    const int basis_rows = opt->format == SVOX_FORMAT_RGBA ? 1 : opt->basis_dim;
    hipLaunchKernelGGL((se_grad_generic_kernel<T, Source>), dim3(blocks_for(items, kMarchThreads)),
                       dim3(kMarchThreads), generic_backward_lds_bytes<T>(basis_rows, out_dim), stream,
                       make_tree<T>(tree), src, *opt, out_dim, (const T*)color_ref, (T*)color_out, (T*)grad, (T*)hess);
}

// shared argument checks and zero-fills of the two squared-error entry points
int se_grad_prepare(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, void* grad, void* hess, int* od,
                    hipStream_t stream, bool fill = true) {
    int rc = check_render(tree, opt, od);
    if (rc) return rc;
    if (*od > 4) return fail(SVOX_ERR_BAD_SHAPE, "Tree's output dim cannot be > 4 for se_grad");
    if (!grad || !hess) return fail(SVOX_ERR_NULL_POINTER, "grad_out / hessdiag_out is NULL");
    if (!fill) return SVOX_OK;
    rc = zero_fill(grad, data_bytes(tree), stream);
    if (rc) return rc;
    return zero_fill(hess, data_bytes(tree), stream);
}

// Can notes be taken (launch_noted) and used (replay_backward_kernel)?  The octree kernels, a forward
// pass whose threshold does not admit leaves the backward pass ignores, no weight accumulator, and a
// workspace with a chunk for every ray.
bool notes_possible(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt) {
    return tree->dtype == SVOX_F32 && fast_basis(tree, opt) >= 0 && !tree->weight_accum && opt->sigma_thresh >= 0.0f;
}
bool noted_ok(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int64_t n_slots, void* workspace,
                     int64_t workspace_bytes) {
    if (!notes_possible(tree, opt)) return false;
    ReplaySpace ws;
    return carve_workspace(workspace, workspace_bytes, n_slots, false, &ws);   // (whether there is room for a list does not matter)
}

NoteStamp stamp_of_image(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                                const SvoxRenderOptions* opt) {
    SvoxRaysSpec as_rays;
    as_rays.origins = cam->c2w;
    as_rays.dirs = nullptr;
    as_rays.n_rays = ((int64_t)n_images * cam->height * cam->width) ^ ((int64_t)cam->width << 40);
    return stamp_of(tree, &as_rays, opt);
}

// log2 of the rays a block of the replay kernels takes: as many as leave 1024 blocks (four wavefronts for every SIMD),
// between 16 and 64.  Fewer cost the blocks' own time (start, heads of the notes), more leave the last blocks running
// alone: 50 001 rays 99 / 91 / 96 us with 16 / 32 / 64, an 800x800 picture 337 / 300 / 310 / 333 us with
// 32 / 64 / 128 / 256, 1 Mi rays 376 / 376 / 381 / 398 us.
int replay_shift(int64_t n_rays) {
    const int forced = tuning().replay_shift;
    if (forced >= 4 && forced <= kReplayMaxShift) return forced;
    int shift = 4;
    while (shift < kReplayMaxShift && n_rays >= ((int64_t)1024 << (shift + 1))) ++shift;
    return shift;
}

// The backward pass of `all` from the notes in the workspace: the rays with complete notes by
// replay_backward_kernel, the others, which it marks in the bitmap, by marching (`rest`: the launch
// shape for those): twice, or -- march1_known: the noting pass had grad_output and left the sum of
// the first march in the heads of the notes -- once.
template <class Source>
int backward_from_notes(const SvoxTreeSpec* tree, const Source& all, Source rest, const SvoxRenderOptions* opt,
                               const void* grad_output, void* grad_data_out, void* workspace, int64_t workspace_bytes,
                               int64_t n_slots, const NoteStamp& stamp, hipStream_t stream, bool march1_known = false,
                               int64_t* report = nullptr) {
    const int D = fast_basis(tree, opt);
    const int ray_shift = replay_shift(n_slots);
    const unsigned replay_blocks = blocks_for(n_slots, 1 << ray_shift);
    ReplaySpace ws;
    carve_workspace(workspace, workspace_bytes, n_slots, keeps_list(tree, opt, all, n_slots), &ws);
    memcpy(ws.stamp, stamp.word, sizeof(ws.stamp));
    ws.report = (unsigned long long*)report;
    SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::replay_backward(dim3(replay_blocks), stream, all, *opt, (const float*)grad_output,
                                                                    (float*)grad_data_out, ws, ray_shift,
                                                                    lobes_of(tree, opt)));
    int rc = check_launch("volume_render_backward_noted");
    if (rc) return rc;
    ReplaySpace only{};
    only.base = ws.base;
    only.only = ws.undone;
    only.any_undone = ws.any_undone;
    const unsigned blocks = blocks_for(total_items_of(rest), rest.per_wave);
    SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::backward(dim3(blocks), stream, march_tree(tree, opt), rest, *opt,
                                                             (const float*)grad_output, (float*)grad_data_out, only,
                                                             rest.per_wave > kMarchThreads, march1_known));
    return check_launch("volume_render_backward_noted");
}

// the options under which notes are taken where no picture hangs on them (se_grad, the backward pass alone): every leaf with sigma > 0, no early stop
SvoxRenderOptions without_thresholds(const SvoxRenderOptions* opt) {
    SvoxRenderOptions o = *opt;
    o.sigma_thresh = 0.0f;
    o.stop_thresh = 0.0f;
    return o;
}

// Whether the arrays of a gradient are cleared by the launch that takes its notes: aligned as clear_share stores, not more than a
// launch has blocks for, and beside a march that leaves the memory room: the more there is to clear the fewer rays that all hit do, and the march is
// slowed.  us, apart / on the way:
//   squared error, 256^3 SH9 shell (345 MB), 18 % hit  5 000 rays 190 / 147  20 000 350 / 299  100 000 422 / 363  200 003 543 / 425  500 000 680 / 655
//                                            all hit   9 000 421 / 381  50 000 629 / 597  100 000 882 / 853  160 000 1173 / 1153  200 003 1463 / 1457
//   256^3 SH16 shell (310 MB a gradient), all hit      gradient 20 000 476 / 429  160 000 1193 / 1177;  squared error 605 / 549  1625 / 1578
//   512^3 SH16 shell (1.2 GB), all hit                 gradient 9 000 653 / 549  50 000 871 / 877  100 000 1072 / 1079  200 003 1616 / 1664
//                                                      squared error 858 / 742  980 / 909  1184 / 1231  2331 / 2453
//                              18 % hit                gradient 50 000 549 / 455  100 000 593 / 472  500 000 870 / 877;  squared error 50 000 744 / 640
bool clears_on_the_way(const SvoxTreeSpec* tree, int64_t n_rays, const void* a, const void* b = nullptr) {
    if (((uintptr_t)a & 15u) != 0 || ((uintptr_t)b & 15u) != 0 || data_bytes(tree) > kMostCleared) return false;
    const int64_t bytes = data_bytes(tree) * (b ? 2 : 1);
    return bytes <= 512ll << 20 || n_rays <= (bytes <= 1ll << 30 ? 1 << 18 : bytes <= 2ll << 30 ? 1 << 17 : 1 << 15);
}

// The backward pass of a call that brings a workspace but no notes: one noting march without a picture
// (thresholds play no part in the backward pass, rt_kernel.cu:377, 441), then backward_from_notes.  The
// reference's two marches per ray become one walk of the tree and one pass over 24 bytes per leaf with
// density.  `all`, `rest` as in backward_from_notes; returns 1 if notes cannot be taken here (the
// caller then marches twice), else a status.
template <class Source>
int backward_by_noting(const SvoxTreeSpec* tree, const Source& all, const Source& rest, const SvoxRenderOptions* opt,
                       const void* grad_output, void* grad_data_out, void* workspace, int64_t workspace_bytes,
                       int64_t n_slots, NoteStamp stamp, bool accumulate, hipStream_t stream) {
    SvoxTreeSpec quiet = *tree;
    quiet.weight_accum = nullptr;   // (the backward pass accumulates no weights)
    const SvoxRenderOptions plain = without_thresholds(opt);
    if (!noted_ok(&quiet, &plain, n_slots, workspace, workspace_bytes)) return 1;
    // (the notes belong to this call alone: the stamp carries its gradient buffer too)
    stamp.word[0] ^= (unsigned long long)(uintptr_t)grad_output;
    ClearWork clear;
    int rc = SVOX_OK;
    if (!accumulate) {
        if (clears_on_the_way(tree, n_slots, grad_data_out)) {
            clear.at[0] = grad_data_out;
            clear.bytes = data_bytes(tree);
        } else {
            rc = zero_fill(grad_data_out, data_bytes(tree), stream);
        }
    }
    if (rc) return rc;
    rc = launch_noted(&quiet, noting_shape(all), &plain, nullptr, workspace, workspace_bytes, n_slots, stamp, stream,
                      grad_output, nullptr, clear);
    if (rc) return rc;
    rc = check_launch("volume_render_backward");
    if (rc) return rc;
    return backward_from_notes(&quiet, all, rest, &plain, grad_output, grad_data_out, workspace, workspace_bytes,
                               n_slots, stamp, stream, true);
}

// se_grad of the rays of `all` with their notes kept in the workspace between its two halves: one
// march that takes the notes (thresholds play no part in se_grad, rt_kernel.cu:479-715), then
// replay_se_grad_kernel; rays it marks in the bitmap are done by se_grad_kernel (`rest`: the launch
// shape for those).  The caller has checked noted_ok() with the same options.
template <class Source>
int se_grad_from_notes(const SvoxTreeSpec* tree, const Source& all, const Source& rest, const SvoxRenderOptions* opt,
                       const void* color_ref, void* color_out, void* grad, void* hess, void* workspace,
                       int64_t workspace_bytes, int64_t n_slots, const NoteStamp& stamp, hipStream_t stream) {
    const int D = fast_basis(tree, opt);
    ClearWork clear;
    if (clears_on_the_way(tree, n_slots, grad, hess)) {
        clear.at[0] = grad;
        clear.at[1] = hess;
        clear.bytes = data_bytes(tree);
    }
    int rc = launch_noted(tree, noting_shape(all), opt, color_out, workspace, workspace_bytes, n_slots, stamp, stream, nullptr,
                          color_ref, clear);
    if (rc) return rc;
    rc = check_launch("se_grad");
    if (rc) return rc;
    ReplaySpace ws;
    carve_workspace(workspace, workspace_bytes, n_slots, keeps_list(tree, opt, all, n_slots), &ws);
    memcpy(ws.stamp, stamp.word, sizeof(ws.stamp));
    const int ray_shift = replay_shift(n_slots);
    SVOX_DISPATCH_OCTREE(D, MarchLaunch<P, Source>::replay_se_grad(dim3(blocks_for(n_slots, 1 << ray_shift)), stream, all, *opt,
                                                                   (float*)grad, (float*)hess, ws, ray_shift,
                                                                   lobes_of(tree, opt)));
    rc = check_launch("se_grad");
    if (rc) return rc;
    launch_se_grad<Source, float>(tree, rest, opt, 3, color_ref, color_out, grad, hess, stream, ws.undone, ws.any_undone);
    return check_launch("se_grad");
}


}  // namespace

#pragma GCC visibility push(default)
extern "C" {

int svox_abi_version(void) { return SVOX_ABI_VERSION; }

const char* svox_last_error(void) { return g_error; }

const char* svox_status_string(int status) {
    switch (status) {
        case SVOX_OK: return "ok";
        case SVOX_ERR_NULL_POINTER: return "null pointer";
        case SVOX_ERR_BAD_SHAPE: return "bad shape";
        case SVOX_ERR_BAD_DTYPE: return "bad dtype";
        case SVOX_ERR_UNSUPPORTED: return "unsupported";
        case SVOX_ERR_LAUNCH: return "kernel launch failed";
        case SVOX_ERR_NO_DEVICE: return "no device";
        default: return "unknown status";
    }
}

// Debugging aid: bit 0 routes every call to the generic kernels.
void svox_set_debug_flags(int flags) { g_debug_flags = flags; }

int svox_out_data_dim(int32_t format, int32_t basis_dim, int32_t data_dim) {
    if (data_dim < 1) return -1;
    if (format != SVOX_FORMAT_RGBA) {
        if (basis_dim <= 0) return -1;
        return (data_dim - 1) / basis_dim;
    }
    return data_dim - 1;
}

int svox_query_vertical(const SvoxTreeSpec* tree, const void* indices, int64_t n_points, void* values_out,
                        int64_t* node_ids_out, void* stream) {
    return svox_query_vertical_ws(tree, indices, n_points, values_out, node_ids_out, nullptr, 0, stream);
}

int64_t svox_query_vertical_workspace_bytes(const SvoxTreeSpec* tree, int64_t n_points) {
    if (check_tree(tree, false) || n_points <= 0 || !walk_copy_pays(tree, n_points)) return 0;
    return tree->capacity * 32;
}

int svox_query_vertical_ws(const SvoxTreeSpec* tree, const void* indices, int64_t n_points, void* values_out,
                           int64_t* node_ids_out, void* workspace, int64_t workspace_bytes, void* stream) {
    int rc = check_tree(tree, true);
    if (rc) return rc;
    if (n_points < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative point count");
    if (n_points == 0) return SVOX_OK;
    if (!indices || !values_out || !node_ids_out) return fail(SVOX_ERR_NULL_POINTER, "indices / values_out / node_ids_out is NULL");
    const bool copy = workspace && ((uintptr_t)workspace & 3u) == 0 && ((uintptr_t)tree->child & 15u) == 0 &&
                      workspace_bytes >= tree->capacity * 32 && walk_copy_pays(tree, n_points);
    if (tree->dtype == SVOX_F32)
        return launch_query<float, kQueryGather>(tree, indices, n_points, values_out, nullptr, node_ids_out,
                                                 tree->data_dim, (hipStream_t)stream, "query_vertical",
                                                 copy ? (int32_t*)workspace : nullptr);
    return launch_query<double, kQueryGather>(tree, indices, n_points, values_out, nullptr, node_ids_out,
                                              tree->data_dim, (hipStream_t)stream, "query_vertical");
}

int svox_query_vertical_backward(const SvoxTreeSpec* tree, const void* indices, int64_t n_points,
                                 const void* grad_output, int32_t grad_dim, void* grad_data_out,
                                 int32_t accumulate, void* stream) {
    return svox_query_vertical_backward_ws(tree, indices, n_points, grad_output, grad_dim, grad_data_out, accumulate, nullptr,
                                           0, stream);
}

int64_t svox_query_vertical_backward_workspace_bytes(const SvoxTreeSpec* tree, int64_t n_points, int32_t grad_dim) {
    Partition part;
    if (check_tree(tree, false) || n_points <= 0 || grad_dim < 1) return 0;
    return plan_partition(tree, n_points, grad_dim, &part);
}

int svox_query_vertical_backward_ws(const SvoxTreeSpec* tree, const void* indices, int64_t n_points,
                                    const void* grad_output, int32_t grad_dim, void* grad_data_out, int32_t accumulate,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
    return svox_query_vertical_backward_ids(tree, indices, nullptr, n_points, grad_output, grad_dim, grad_data_out, accumulate,
                                            workspace, workspace_bytes, stream);
}

int svox_query_vertical_backward_ids(const SvoxTreeSpec* tree, const void* indices, const int64_t* node_ids, int64_t n_points,
                                     const void* grad_output, int32_t grad_dim, void* grad_data_out, int32_t accumulate,
                                     void* workspace, int64_t workspace_bytes, void* stream) {
    int rc = check_tree(tree, false);
    if (rc) return rc;
    if (n_points < 0 || grad_dim < 1) return fail(SVOX_ERR_BAD_SHAPE, "negative point count or grad_dim < 1");
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    if (!grad_data_out) return fail(SVOX_ERR_NULL_POINTER, "grad_data_out is NULL");
    if (!accumulate && workspace && ((uintptr_t)workspace & 7u) == 0 && n_points > 0 && indices && grad_output) {
        Partition part;
        const int64_t need = plan_partition(tree, n_points, grad_dim, &part);
        if (need > 0 && need <= workspace_bytes)
            return launch_partition(tree, part, (const float*)indices, node_ids, (const float*)grad_output, grad_dim,
                                    (float*)grad_data_out, workspace, (hipStream_t)stream);
    }
    const int64_t esz = tree->dtype == SVOX_F32 ? 4 : 8;
    if (!accumulate) {
        rc = zero_fill(grad_data_out, tree->capacity * tree->N * tree->N * tree->N * grad_dim * esz,
                       (hipStream_t)stream);
        if (rc) return rc;
    }
    if (n_points == 0) return SVOX_OK;
    if (!indices || !grad_output) return fail(SVOX_ERR_NULL_POINTER, "indices / grad_output is NULL");
    if (tree->dtype == SVOX_F32)
        return launch_query<float, kQueryScatterAdd>(tree, indices, n_points, (void*)grad_output, grad_data_out,
                                                     (int64_t*)node_ids, grad_dim, (hipStream_t)stream,
                                                     "query_vertical_backward");
    return launch_query<double, kQueryScatterAdd>(tree, indices, n_points, (void*)grad_output, grad_data_out,
                                                  (int64_t*)node_ids, grad_dim, (hipStream_t)stream,
                                                  "query_vertical_backward");
}

int svox_assign_vertical(const SvoxTreeSpec* tree, const void* indices, int64_t n_points, const void* values,
                         int32_t value_dim, void* stream) {
    int rc = check_tree(tree, true);
    if (rc) return rc;
    if (n_points < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative point count");
    if (value_dim < 1 || value_dim > tree->data_dim)
        return fail(SVOX_ERR_BAD_SHAPE, "value_dim %d outside [1, data_dim=%d]", value_dim, tree->data_dim);
    if (n_points == 0) return SVOX_OK;
    if (!indices || !values) return fail(SVOX_ERR_NULL_POINTER, "indices / values is NULL");
    if (tree->dtype == SVOX_F32)
        return launch_query<float, kQueryAssign>(tree, indices, n_points, (void*)values, nullptr, nullptr,
                                                 value_dim, (hipStream_t)stream, "assign_vertical");
    return launch_query<double, kQueryAssign>(tree, indices, n_points, (void*)values, nullptr, nullptr, value_dim,
                                              (hipStream_t)stream, "assign_vertical");
}

int svox_calc_corners(const SvoxTreeSpec* tree, const int64_t* indexer, int64_t n_leaves, void* corners_out,
                      void* stream) {
    int rc = check_tree(tree, false);
    if (rc) return rc;
    if (n_leaves < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative leaf count");
    if (n_leaves == 0) return SVOX_OK;
    if (!indexer || !corners_out) return fail(SVOX_ERR_NULL_POINTER, "indexer / corners_out is NULL");
    const unsigned blocks = (unsigned)((n_leaves + kQueryThreads - 1) / kQueryThreads);
    if (tree->dtype == SVOX_F32)
        hipLaunchKernelGGL((corners_kernel<float>), dim3(blocks), dim3(kQueryThreads), 0, (hipStream_t)stream,
                           tree->parent_depth, tree->N, tree->capacity, indexer, n_leaves, (float*)corners_out);
    else
        hipLaunchKernelGGL((corners_kernel<double>), dim3(blocks), dim3(kQueryThreads), 0, (hipStream_t)stream,
                           tree->parent_depth, tree->N, tree->capacity, indexer, n_leaves, (double*)corners_out);
    return check_launch("calc_corners");
}

// The forward pass of a training step: the picture of svox_volume_render, and in the workspace the notes
// svox_volume_render_backward_noted works from (where noted_ok() allows; else the plain forward pass).
int svox_volume_render_noted(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt,
                             void* out, void* workspace, int64_t workspace_bytes, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_rays(rays);
    if (rc) return rc;
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    if (rays->n_rays == 0) return SVOX_OK;
    if (!out) return fail(SVOX_ERR_NULL_POINTER, "out is NULL");
    if (!noted_ok(tree, opt, rays->n_rays, workspace, workspace_bytes))
        return svox_volume_render(tree, rays, opt, out, stream);
    const NoteStamp stamp = stamp_of(tree, rays, opt);
    rc = launch_noted(tree, batch_source<float>(rays, false), opt, out, workspace, workspace_bytes, rays->n_rays, stamp,
                      (hipStream_t)stream);
    if (rc) return rc;
    return check_launch("volume_render_noted");
}

int svox_volume_render_backward_noted(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays,
                                      const SvoxRenderOptions* opt, const void* grad_output, void* grad_data_out,
                                      int32_t accumulate, void* workspace, int64_t workspace_bytes, void* stream) {
    return svox_volume_render_backward_noted_with(tree, rays, opt, grad_output, grad_data_out, accumulate, workspace,
                                                  workspace_bytes, nullptr, stream);
}

int svox_volume_render_backward_noted_with(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays,
                                           const SvoxRenderOptions* opt, const void* grad_output, void* grad_data_out,
                                           int32_t accumulate, void* workspace, int64_t workspace_bytes,
                                           const SvoxNotesExtras* extras, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_rays(rays);
    if (rc) return rc;
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    if (!noted_ok(tree, opt, rays->n_rays, workspace, workspace_bytes))
        return svox_volume_render_backward_ws(tree, rays, opt, grad_output, grad_data_out, accumulate, workspace,
                                              workspace_bytes, stream);
    if (!grad_data_out) return fail(SVOX_ERR_NULL_POINTER, "grad_data_out is NULL");
    if (!accumulate) {
        rc = zero_fill(grad_data_out, data_bytes(tree), (hipStream_t)stream);
        if (rc) return rc;
    }
    if (rays->n_rays == 0) return SVOX_OK;
    if (!grad_output) return fail(SVOX_ERR_NULL_POINTER, "grad_output is NULL");
    const BatchSource<float> all = batch_source<float>(rays, true);
    return backward_from_notes(tree, all, all, opt, grad_output, grad_data_out, workspace, workspace_bytes,
                               rays->n_rays, stamp_of(tree, rays, opt), (hipStream_t)stream, false,
                               extras ? extras->report : nullptr);
}

int svox_volume_render_images_noted(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                                    int64_t pose_stride, const SvoxRenderOptions* opt, void* out, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_camera(cam, n_images, pose_stride);
    if (rc) return rc;
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    if (cam->width == 0 || cam->height == 0 || n_images == 0) return SVOX_OK;
    if (!out) return fail(SVOX_ERR_NULL_POINTER, "out is NULL");
    const int64_t n_slots = (int64_t)n_images * cam->width * cam->height;
    if (!noted_ok(tree, opt, n_slots, workspace, workspace_bytes))
        return svox_volume_render_images(tree, cam, n_images, pose_stride, opt, out, stream);
    const NoteStamp stamp = stamp_of_image(tree, cam, n_images, opt);
    rc = launch_noted(tree, image_source<float>(cam, n_images, pose_stride, opt), opt, out, workspace, workspace_bytes,
                      n_slots, stamp, (hipStream_t)stream);
    if (rc) return rc;
    return check_launch("volume_render_images_noted");
}

int svox_volume_render_images_backward_noted(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                                             int64_t pose_stride, const SvoxRenderOptions* opt,
                                             const void* grad_output, void* grad_data_out, int32_t accumulate,
                                             void* workspace, int64_t workspace_bytes, void* stream) {
    return svox_volume_render_images_backward_noted_with(tree, cam, n_images, pose_stride, opt, grad_output, grad_data_out,
                                                         accumulate, workspace, workspace_bytes, nullptr, stream);
}

int svox_volume_render_images_backward_noted_with(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                                                  int64_t pose_stride, const SvoxRenderOptions* opt,
                                                  const void* grad_output, void* grad_data_out, int32_t accumulate,
                                                  void* workspace, int64_t workspace_bytes, const SvoxNotesExtras* extras,
                                                  void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_camera(cam, n_images, pose_stride);
    if (rc) return rc;
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    const int64_t n_slots = (int64_t)n_images * cam->width * cam->height;
    if (!noted_ok(tree, opt, n_slots, workspace, workspace_bytes))
        return svox_volume_render_images_backward_ws(tree, cam, n_images, pose_stride, opt, grad_output, grad_data_out,
                                                     accumulate, workspace, workspace_bytes, stream);
    if (!grad_data_out) return fail(SVOX_ERR_NULL_POINTER, "grad_data_out is NULL");
    if (!accumulate) {
        rc = zero_fill(grad_data_out, data_bytes(tree), (hipStream_t)stream);
        if (rc) return rc;
    }
    if (n_slots == 0) return SVOX_OK;
    if (!grad_output) return fail(SVOX_ERR_NULL_POINTER, "grad_output is NULL");
    const ImageSource<float> all = image_source<float>(cam, n_images, pose_stride, opt);
    return backward_from_notes(tree, all, all, opt, grad_output, grad_data_out, workspace, workspace_bytes, n_slots,
                               stamp_of_image(tree, cam, n_images, opt), (hipStream_t)stream, false,
                               extras ? extras->report : nullptr);
}

int svox_volume_render(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt, void* out,
                       void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_rays(rays);
    if (rc) return rc;
    if (rays->n_rays == 0) return SVOX_OK;
    if (!out) return fail(SVOX_ERR_NULL_POINTER, "out is NULL");
    if (tree->dtype == SVOX_F32)
        launch_forward<BatchSource<float>, float>(tree, batch_source<float>(rays), opt, od, out,
                                                  (hipStream_t)stream);
    else
        launch_forward<BatchSource<double>, double>(tree, batch_source<double>(rays), opt, od, out,
                                                    (hipStream_t)stream);
    return check_launch("volume_render");
}

int svox_volume_render_images(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                              int64_t pose_stride, const SvoxRenderOptions* opt, void* out, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_camera(cam, n_images, pose_stride);
    if (rc) return rc;
    if (cam->width == 0 || cam->height == 0 || n_images == 0) return SVOX_OK;
    if (!out) return fail(SVOX_ERR_NULL_POINTER, "out is NULL");
    if (tree->dtype == SVOX_F32) {
        const auto src = image_source<float>(cam, n_images, pose_stride, opt);
        launch_forward<ImageSource<float>, float>(tree, src, opt, od, out, (hipStream_t)stream);
    } else {
        const auto src = image_source<double>(cam, n_images, pose_stride, opt);
        launch_forward<ImageSource<double>, double>(tree, src, opt, od, out, (hipStream_t)stream);
    }
    return check_launch("volume_render_image");
}

int svox_volume_render_image(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, const SvoxRenderOptions* opt,
                             void* out, void* stream) {
    return svox_volume_render_images(tree, cam, 1, 12, opt, out, stream);
}

int svox_volume_render_backward(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt,
                                const void* grad_output, void* grad_data_out, int32_t accumulate, void* stream) {
    return svox_volume_render_backward_ws(tree, rays, opt, grad_output, grad_data_out, accumulate, nullptr, 0,
                                          stream);
}

int svox_notes_pool_info(int64_t n_rays, int64_t workspace_bytes, int64_t* counter_offset, int64_t* pool_stocks) {
    if (!counter_offset || !pool_stocks) return fail(SVOX_ERR_NULL_POINTER, "svox_notes_pool_info: NULL output");
    ReplaySpace ws;
    // (any 16-byte aligned address does for the arithmetic)
    char* const base = (char*)(uintptr_t)4096;
    if (!carve_workspace(base, workspace_bytes, n_rays, list_at_end(n_rays), &ws))
        return fail(SVOX_ERR_BAD_SHAPE, "svox_notes_pool_info: the workspace does not hold a chunk per ray");
    *counter_offset = (int64_t)((char*)ws.stocks_taken - base);
    *pool_stocks = ws.n_stocks;
    return SVOX_OK;
}

int64_t svox_volume_render_backward_workspace_bytes(int64_t n_rays, int32_t records_per_ray) {
    if (n_rays <= 0 || records_per_ray <= 0) return 0;
    const int64_t chunks_per_ray = (records_per_ray + kChunkRecords - 1) / kChunkRecords;
    return n_rays * chunks_per_ray * kChunkBytes + bitmap_bytes(n_rays) + kTailBytes;
}

int svox_volume_render_backward_ws(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt,
                                   const void* grad_output, void* grad_data_out, int32_t accumulate,
                                   void* workspace, int64_t workspace_bytes, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_rays(rays);
    if (rc) return rc;
    if (!grad_data_out) return fail(SVOX_ERR_NULL_POINTER, "grad_data_out is NULL");
    if (tree->dtype == SVOX_F32 && workspace && workspace_bytes >= 0 && rays->n_rays > 0 && grad_output) {
        const BatchSource<float> all = batch_source<float>(rays, true);
        rc = backward_by_noting(tree, all, all, opt, grad_output, grad_data_out, workspace, workspace_bytes,
                                rays->n_rays, stamp_of(tree, rays, opt), accumulate != 0, (hipStream_t)stream);
        if (rc <= 0) return rc;
    }
    if (!accumulate) {
        rc = zero_fill(grad_data_out, data_bytes(tree), (hipStream_t)stream);
        if (rc) return rc;
    }
    if (rays->n_rays == 0) return SVOX_OK;
    if (!grad_output) return fail(SVOX_ERR_NULL_POINTER, "grad_output is NULL");
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    if (tree->dtype == SVOX_F32)
        launch_backward<BatchSource<float>, float>(tree, batch_source<float>(rays, true), opt, od, grad_output,
                                                   grad_data_out, (hipStream_t)stream);
    else
        launch_backward<BatchSource<double>, double>(tree, batch_source<double>(rays, true), opt, od, grad_output,
                                                     grad_data_out, (hipStream_t)stream);
    return check_launch("volume_render_backward");
}

// svox_volume_render_backward_ws on the library's own array: no allocation anywhere on the way (the
// stock counter in the array's tail is cleared by the fill kernel of launch_noted before the noting
// launch; everything else in the array is written by that launch before the launches after it read it).
int svox_volume_render_backward_static(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays,
                                       const SvoxRenderOptions* opt, const void* grad_output, void* grad_data_out,
                                       int32_t accumulate, void* stream) {
    int rc = check_rays(rays);
    if (rc) return rc;
    if (rays->n_rays > SVOX_STATIC_RAYS_MAX)
        return fail(SVOX_ERR_BAD_SHAPE,
                    "svox.volume_render_backward_static: %lld rays exceed the %d rays the library's fixed "
                    "workspace serves per call; split the batch (accumulate = 1 from the second part on) or "
                    "call svox_volume_render_backward_ws with a workspace of your own",
                    (long long)rays->n_rays, (int)SVOX_STATIC_RAYS_MAX);
    static DeviceAddress workspace_at;
    void* const ws = workspace_at.get(HIP_SYMBOL(scratch));
    if (!ws) return fail(SVOX_ERR_NO_DEVICE, "svox.volume_render_backward_static: no usable current device");
    return svox_volume_render_backward_ws(tree, rays, opt, grad_output, grad_data_out, accumulate, ws,
                                          (int64_t)SVOX_STATIC_WORKSPACE_BYTES, stream);
}

int svox_volume_render_images_backward(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                                       int64_t pose_stride, const SvoxRenderOptions* opt,
                                       const void* grad_output, void* grad_data_out, int32_t accumulate,
                                       void* stream) {
    return svox_volume_render_images_backward_ws(tree, cam, n_images, pose_stride, opt, grad_output, grad_data_out,
                                                 accumulate, nullptr, 0, stream);
}

int svox_volume_render_images_backward_ws(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, int32_t n_images,
                                          int64_t pose_stride, const SvoxRenderOptions* opt,
                                          const void* grad_output, void* grad_data_out, int32_t accumulate,
                                          void* workspace, int64_t workspace_bytes, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    rc = check_camera(cam, n_images, pose_stride);
    if (rc) return rc;
    if (!grad_data_out) return fail(SVOX_ERR_NULL_POINTER, "grad_data_out is NULL");
    const int64_t n_slots = (int64_t)n_images * cam->width * cam->height;
    if (tree->dtype == SVOX_F32 && workspace && workspace_bytes >= 0 && n_slots > 0 && grad_output) {
        const auto src = image_source<float>(cam, n_images, pose_stride, opt);
        rc = backward_by_noting(tree, src, src, opt, grad_output, grad_data_out, workspace, workspace_bytes, n_slots,
                                stamp_of_image(tree, cam, n_images, opt), accumulate != 0, (hipStream_t)stream);
        if (rc <= 0) return rc;
    }
    if (!accumulate) {
        rc = zero_fill(grad_data_out, data_bytes(tree), (hipStream_t)stream);
        if (rc) return rc;
    }
    if (cam->width == 0 || cam->height == 0 || n_images == 0) return SVOX_OK;
    if (!grad_output) return fail(SVOX_ERR_NULL_POINTER, "grad_output is NULL");
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    if (tree->dtype == SVOX_F32) {
        const auto src = image_source<float>(cam, n_images, pose_stride, opt);
        launch_backward<ImageSource<float>, float>(tree, src, opt, od, grad_output, grad_data_out, (hipStream_t)stream);
    } else {
        const auto src = image_source<double>(cam, n_images, pose_stride, opt);
        launch_backward<ImageSource<double>, double>(tree, src, opt, od, grad_output, grad_data_out, (hipStream_t)stream);
    }
    return check_launch("volume_render_image_backward");
}

int svox_volume_render_image_backward(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam,
                                      const SvoxRenderOptions* opt, const void* grad_output, void* grad_data_out,
                                      int32_t accumulate, void* stream) {
    return svox_volume_render_images_backward(tree, cam, 1, 12, opt, grad_output, grad_data_out, accumulate, stream);
}

int svox_se_grad(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt,
                 const void* color_ref, void* color_out, void* grad_out, void* hessdiag_out, void* stream) {
    int od;
    int rc = check_rays(rays);
    if (rc) return rc;
    rc = se_grad_prepare(tree, opt, grad_out, hessdiag_out, &od, (hipStream_t)stream);
    if (rc) return rc;
    if (rays->n_rays == 0) return SVOX_OK;
    if (!color_ref || !color_out) return fail(SVOX_ERR_NULL_POINTER, "color_ref / color_out is NULL");
    if (tree->dtype == SVOX_F32)
        launch_se_grad<BatchSource<float>, float>(tree, batch_source<float>(rays, true), opt, od, color_ref,
                                                  color_out, grad_out, hessdiag_out, (hipStream_t)stream);
    else
        launch_se_grad<BatchSource<double>, double>(tree, batch_source<double>(rays, true), opt, od, color_ref,
                                                    color_out, grad_out, hessdiag_out, (hipStream_t)stream);
    return check_launch("se_grad");
}

int svox_se_grad_image(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, const SvoxRenderOptions* opt,
                       const void* color_ref, void* color_out, void* grad_out, void* hessdiag_out, void* stream) {
    int od;
    int rc = check_camera(cam, 1, 12);
    if (rc) return rc;
    rc = se_grad_prepare(tree, opt, grad_out, hessdiag_out, &od, (hipStream_t)stream);
    if (rc) return rc;
    if (cam->width == 0 || cam->height == 0) return SVOX_OK;
    if (!color_ref || !color_out) return fail(SVOX_ERR_NULL_POINTER, "color_ref / color_out is NULL");
    if (tree->dtype == SVOX_F32) {
        const auto src = image_source<float>(cam, 1, 12, opt);
        launch_se_grad<ImageSource<float>, float>(tree, src, opt, od, color_ref, color_out, grad_out, hessdiag_out,
                                                  (hipStream_t)stream);
    } else {
        const auto src = image_source<double>(cam, 1, 12, opt);
        launch_se_grad<ImageSource<double>, double>(tree, src, opt, od, color_ref, color_out, grad_out,
                                                    hessdiag_out, (hipStream_t)stream);
    }
    return check_launch("se_grad_persp");
}

int svox_se_grad_ws(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxRenderOptions* opt,
                    const void* color_ref, void* color_out, void* grad_out, void* hessdiag_out, void* workspace,
                    int64_t workspace_bytes, void* stream) {
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    int od;
    int rc = check_rays(rays);
    if (rc) return rc;
    rc = check_render(tree, opt, &od);
    if (rc) return rc;
    const SvoxRenderOptions plain = without_thresholds(opt);
    if (od != 3 || rays->n_rays == 0 || !color_ref || !color_out ||
        !noted_ok(tree, &plain, rays->n_rays, workspace, workspace_bytes))
        return svox_se_grad(tree, rays, opt, color_ref, color_out, grad_out, hessdiag_out, stream);
    const bool apart = !clears_on_the_way(tree, rays->n_rays, grad_out, hessdiag_out);
    rc = se_grad_prepare(tree, opt, grad_out, hessdiag_out, &od, (hipStream_t)stream, apart);
    if (rc) return rc;
    const BatchSource<float> all = batch_source<float>(rays, true);
    return se_grad_from_notes(tree, all, all, &plain, color_ref, color_out, grad_out, hessdiag_out, workspace,
                              workspace_bytes, rays->n_rays, stamp_of(tree, rays, &plain), (hipStream_t)stream);
}

int svox_se_grad_image_ws(const SvoxTreeSpec* tree, const SvoxCameraSpec* cam, const SvoxRenderOptions* opt,
                          const void* color_ref, void* color_out, void* grad_out, void* hessdiag_out,
                          void* workspace, int64_t workspace_bytes, void* stream) {
    if (workspace_bytes < 0) return fail(SVOX_ERR_BAD_SHAPE, "negative workspace size");
    int od;
    int rc = check_camera(cam, 1, 12);
    if (rc) return rc;
    rc = check_render(tree, opt, &od);
    if (rc) return rc;
    const SvoxRenderOptions plain = without_thresholds(opt);
    const int64_t n_slots = (int64_t)cam->width * cam->height;
    if (od != 3 || n_slots == 0 || !color_ref || !color_out ||
        !noted_ok(tree, &plain, n_slots, workspace, workspace_bytes))
        return svox_se_grad_image(tree, cam, opt, color_ref, color_out, grad_out, hessdiag_out, stream);
    const bool apart = !clears_on_the_way(tree, n_slots, grad_out, hessdiag_out);
    rc = se_grad_prepare(tree, opt, grad_out, hessdiag_out, &od, (hipStream_t)stream, apart);
    if (rc) return rc;
    const ImageSource<float> all = image_source<float>(cam, 1, 12, opt);
    return se_grad_from_notes(tree, all, all, &plain, color_ref, color_out, grad_out, hessdiag_out, workspace,
                              workspace_bytes, n_slots, stamp_of_image(tree, cam, 1, &plain), (hipStream_t)stream);
}

int svox_mark_leaves_below(const SvoxTreeSpec* tree, float sigma_thresh, int32_t density_softplus, int32_t* marks_out,
                           void* stream) {
    int rc = check_tree(tree, true);
    if (rc) return rc;
    if (!marks_out) return fail(SVOX_ERR_NULL_POINTER, "marks_out is NULL");
    if (!(sigma_thresh >= 0.0f)) return fail(SVOX_ERR_BAD_SHAPE, "marks need a sigma_thresh >= 0, got %g", (double)sigma_thresh);
    const int64_t cells = tree->capacity * tree->N * tree->N * tree->N;
    if (cells == 0) return SVOX_OK;
    const unsigned blocks = blocks_for(cells, 256);
    if (tree->dtype == SVOX_F32)
        hipLaunchKernelGGL((mark_leaves_kernel<float>), dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (const float*)tree->data, tree->child, cells, tree->data_dim, sigma_thresh,
                           density_softplus != 0, marks_out);
    else
        hipLaunchKernelGGL((mark_leaves_kernel<double>), dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (const double*)tree->data, tree->child, cells, tree->data_dim, (double)sigma_thresh,
                           density_softplus != 0, marks_out);
    return check_launch("mark_leaves_below");
}

int64_t svox_walk_table_bytes(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int64_t n_rays, int32_t image,
                              int32_t every_positive_leaf) {
    int od;
    if (n_rays <= 0 || check_render(tree, opt, &od) || !walk_table_pays(tree, opt, n_rays, image != 0, every_positive_leaf != 0)) return 0;
    return tree->capacity * 32;
}

int svox_walk_table(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt, int32_t every_positive_leaf, int32_t* table_out,
                    SvoxTreeSpec* with_table_out, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    if (!table_out || !with_table_out) return fail(SVOX_ERR_NULL_POINTER, "table_out / with_table_out is NULL");
    if (tree->N != 2 || tree->capacity > (int64_t)kWalkNodes) return fail(SVOX_ERR_BAD_SHAPE, "walk tables are for octrees of fewer than 2^22 nodes");
    if (has_walk_table(tree)) return fail(SVOX_ERR_BAD_SHAPE, "child_marks is a walk table already");
    const int32_t* const from = walk_source(tree, opt, every_positive_leaf != 0);
    if (!from) return fail(SVOX_ERR_BAD_SHAPE, "a walk table is made from a table that begins at a multiple of 16 bytes");
    const bool marked = from != tree->child;
    hipLaunchKernelGGL(walk_table_kernel, dim3((unsigned)((tree->capacity * 8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, from,
                       (int32_t)tree->capacity, (uint32_t*)table_out);
    *with_table_out = *tree;
    with_table_out->child_marks = table_out;
    with_table_out->child_marks_softplus = !marked ? SVOX_MARKS_WALK | SVOX_MARKS_NONE : tree->child_marks_softplus ? SVOX_MARKS_WALK | 1 : SVOX_MARKS_WALK;
    with_table_out->child_marks_thresh = walk_thresh(marked ? tree->child_marks_thresh : 0.0f);
    return check_launch("walk_table");
}

int svox_mark_empty_leaves(const SvoxTreeSpec* tree, int32_t* marks_out, void* stream) {
    return svox_mark_leaves_below(tree, 0.0f, 0, marks_out, stream);
}

int svox_grid_weight_render(const void* data, int32_t reso, int32_t dtype, const SvoxCameraSpec* cam,
                            const SvoxRenderOptions* opt, const void* offset, const void* scaling,
                            void* grid_weight_out, void* grid_hit_out, void* stream) {
    if (!data || !opt || !offset || !scaling || !grid_weight_out || !grid_hit_out)
        return fail(SVOX_ERR_NULL_POINTER, "grid_weight_render: NULL argument");
    if (dtype != SVOX_F32 && dtype != SVOX_F64) return fail(SVOX_ERR_BAD_DTYPE, "dtype must be SVOX_F32 or SVOX_F64");
    // cell ids are 32-bit, as in the reference (reso^3 < 2^31)
    if (reso < 1 || reso > 1290) return fail(SVOX_ERR_BAD_SHAPE, "grid resolution must be in [1, 1290]");
    int rc = check_camera(cam, 1, 12);
    if (rc) return rc;
    const int64_t bytes = (int64_t)reso * reso * reso * (dtype == SVOX_F32 ? 4 : 8);
    rc = zero_fill(grid_weight_out, bytes, (hipStream_t)stream);
    if (rc) return rc;
    rc = zero_fill(grid_hit_out, bytes, (hipStream_t)stream);
    if (rc) return rc;
    if (cam->width == 0 || cam->height == 0) return SVOX_OK;
    if (dtype == SVOX_F32) {
        const auto src = image_source<float>(cam, 1, 12, opt);
        hipLaunchKernelGGL((grid_weight_kernel<float>), dim3(blocks_for(total_items_of(src), kMarchThreads)),
                           dim3(kMarchThreads), 0, (hipStream_t)stream, (const float*)data, reso, src, *opt,
                           (const float*)offset, (const float*)scaling, (float*)grid_weight_out,
                           (float*)grid_hit_out);
    } else {
        const auto src = image_source<double>(cam, 1, 12, opt);
        hipLaunchKernelGGL((grid_weight_kernel<double>), dim3(blocks_for(total_items_of(src), kMarchThreads)),
                           dim3(kMarchThreads), 0, (hipStream_t)stream, (const double*)data, reso, src, *opt,
                           (const double*)offset, (const double*)scaling, (double*)grid_weight_out,
                           (double*)grid_hit_out);
    }
    return check_launch("grid_weight_render");
}

int svox_volume_render_stats(const SvoxTreeSpec* tree, const SvoxRaysSpec* rays, const SvoxCameraSpec* cam,
                             const SvoxRenderOptions* opt, SvoxMarchStats* stats_out, void* stream) {
    int od;
    int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    if (!stats_out) return fail(SVOX_ERR_NULL_POINTER, "stats_out is NULL");
    if ((rays != nullptr) == (cam != nullptr))
        return fail(SVOX_ERR_BAD_SHAPE, "exactly one of rays and cam must be given");
    unsigned long long* st = (unsigned long long*)stats_out;
    if (rays) {
        rc = check_rays(rays);
        if (rc) return rc;
        if (rays->n_rays == 0) return SVOX_OK;
        const unsigned blocks = blocks_for(rays->n_rays, kMarchThreads);
        if (tree->dtype == SVOX_F32)
            hipLaunchKernelGGL((render_stats_kernel<float, BatchSource<float>>), dim3(blocks), dim3(kMarchThreads), 0,
                               (hipStream_t)stream, make_tree<float>(tree), batch_source<float>(rays), *opt, st);
        else
            hipLaunchKernelGGL((render_stats_kernel<double, BatchSource<double>>), dim3(blocks), dim3(kMarchThreads),
                               0, (hipStream_t)stream, make_tree<double>(tree), batch_source<double>(rays), *opt, st);
    } else {
        rc = check_camera(cam);
        if (rc) return rc;
        if (cam->width == 0 || cam->height == 0) return SVOX_OK;
        if (tree->dtype == SVOX_F32) {
            const auto src = image_source<float>(cam, 1, 12, opt);
            const unsigned blocks = blocks_for(total_items_of(src), kMarchThreads);
            hipLaunchKernelGGL((render_stats_kernel<float, ImageSource<float>>), dim3(blocks), dim3(kMarchThreads), 0,
                               (hipStream_t)stream, make_tree<float>(tree), src, *opt, st);
        } else {
            const auto src = image_source<double>(cam, 1, 12, opt);
            const unsigned blocks = blocks_for(total_items_of(src), kMarchThreads);
            hipLaunchKernelGGL((render_stats_kernel<double, ImageSource<double>>), dim3(blocks), dim3(kMarchThreads),
                               0, (hipStream_t)stream, make_tree<double>(tree), src, *opt, st);
        }
    }
    return check_launch("volume_render_stats");
}

int svox_octree_kernels_serve(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt) {
    int od;
    const int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    return fast_basis(tree, opt) >= 0 ? 1 : 0;
}

int svox_notes_serve(const SvoxTreeSpec* tree, const SvoxRenderOptions* opt) {
    int od;
    const int rc = check_render(tree, opt, &od);
    if (rc) return rc;
    return notes_possible(tree, opt) ? 1 : 0;
}

int svox_give_up_count(int64_t* count_out) {
    if (!count_out) return fail(SVOX_ERR_NULL_POINTER, "count_out is NULL");
    unsigned int n = 0;
    hipError_t err = hipDeviceSynchronize();
    if (err == hipSuccess) err = hipMemcpyFromSymbol(&n, HIP_SYMBOL(split_give_ups), sizeof(n), 0, hipMemcpyDeviceToHost);
    if (err != hipSuccess) return fail(SVOX_ERR_LAUNCH, "svox.give_up_count: %s", hipGetErrorString(err));
    *count_out = (int64_t)n;
    return SVOX_OK;
}

}  // extern "C"
#pragma GCC visibility pop
