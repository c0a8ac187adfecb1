// march_kernels.h -- ray marching through the leaves of the N^3 tree: forward rendering, its
// backward pass, the squared-error gradient / Hessian diagonal, the dense-grid weight render and
// the visit counters (reference: svox/csrc/rt_kernel.cu:189-1003).
//
// The tree kernels exist in two flavours that compute the same numbers:
//   GenericPolicy<T>   any branching factor, scalar type, data format, component range, softplus;
//                      the reference's floating-point walk from the root for every sample.
//   OctreePolicy<FMT,D> fp32 trees of three colours (RGBA, or SH and lobes with D in {1,4,9,16,25}):
//                      record length and basis size known at compile time, a wavefront to 64 rays that
//                      share their work; octrees walk on integer coordinates, restarted from the
//                      previous path (OctreeCursor), other branching factors as above.
// (Small batches through fp64 octrees have kernels of their own: group_kernels.h.)
#pragma once

#include <cstddef>
#include <type_traits>

#include "basis.h"
#include "tree_walk.h"

namespace svox {

constexpr int kMarchThreads = 64;  // one wavefront per block: finished tiles free their slot at once

// Orders the LDS traffic of the block's single wavefront: what a lane wrote before is read by
// any lane after.  The hardware keeps a wavefront's LDS operations in order; this keeps the compiler
// from moving them across and waits for the LDS counter only.  (__syncthreads would also wait for
// every outstanding global load, store and atomic of the wavefront -- the gradient atomics, which
// nothing here has to wait for.)
__device__ __forceinline__ void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// __any without the detour through vector registers that the library's takes
__device__ __forceinline__ bool any_lane(bool b) { return __builtin_amdgcn_ballot_w64(b) != 0ull; }

// ------------------------------------------------------------------------------------------------
// ray sources
// ------------------------------------------------------------------------------------------------
template <typename T>
struct RayBatch {
    const T* origins;
    const T* dirs;
    const T* vdirs;
    int64_t n_rays;
};

template <typename T>
struct Camera {
    const T* c2w;
    float fx, fy;
    int width, height;
};

// _dda_unit, rt_kernel.cu:203-220: the segment of the ray inside the unit cube
template <typename T>
__device__ __forceinline__ void dda_unit(const T* cen, const T* invdir, T* tmin, T* tmax) {
    T lo = T(0), hi = T(1e9f);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const T t1 = -cen[i] * invdir[i];
        const T t2 = t1 + invdir[i];
        lo = max_(lo, min_(t1, t2));
        hi = min_(hi, max_(t1, t2));
    }
    *tmin = lo;
    *tmax = hi;
}

// _dda_unit for a point inside the unit cube -- the leaf-local position of a sample, every coordinate in [0, 1) --
// as the octree walk uses it: the length tmax - tmin of the segment.  There the entry distance is 0 (on every axis
// t1 = -c * inv and t2 = t1 + inv lie on either side of 0, so min(t1, t2) <= 0), and the larger of t1 and t2 is t2
// where inv > 0 and t1 elsewhere, i.e. t1 + max(inv, 0): the same roundings and the same value as dda_unit gives
// (an axis whose inv is NaN drops out of both), in half the instructions of the walk's innermost turn.
__device__ __forceinline__ float leaf_exit(const float* cen, const float* invdir) {
    float hi = 1e9f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float t1 = -cen[i] * invdir[i];
        hi = min_(hi, t1 + max_(invdir[i], 0.0f));
    }
    return hi;
}

// cam2world_ray, rt_kernel.cu:758-772: pixel corner (no half-pixel offset), camera looking down
// -z with +y up.  x and y are formed in double and rounded; the radicand is widened for `+ 1.0`.
template <typename T>
__device__ __forceinline__ void cam2world_ray(int ix, int iy, const Camera<T>& cam, T* dir, T* origin) {
    T x = (T)(((double)ix - 0.5 * (double)cam.width) / (double)cam.fx);
    T y = (T)(-((double)iy - 0.5 * (double)cam.height) / (double)cam.fy);
    T z = (T)__builtin_sqrtf((float)((double)fma_(x, x, y * y) + 1.0));
    x /= z;
    y /= z;
    z = (T)(-1.0f / z);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const T* row = cam.c2w + r * 4;
        dir[r] = fma_(row[2], z, fma_(row[0], x, row[1] * y));
        origin[r] = row[3];
    }
}

// maybe_world2ndc, rt_kernel.cu:775-796 with near = 1
template <typename T>
__device__ __forceinline__ void maybe_world2ndc(const SvoxRenderOptions& opt, T* dir, T* cen) {
    if (opt.ndc_width < 0) return;
    const T near = T(1);
    const T t = -(near + cen[2]) / dir[2];
#pragma unroll
    for (int i = 0; i < 3; ++i) cen[i] = fma_(t, dir[i], cen[i]);
    const float two_f = 2 * opt.ndc_focal;
    const T kx = (T)(two_f / (float)opt.ndc_width);
    const T ky = (T)(two_f / (float)opt.ndc_height);
    dir[0] = -kx * (dir[0] / dir[2] - cen[0] / cen[2]);
    dir[1] = -ky * (dir[1] / dir[2] - cen[1] / cen[2]);
    dir[2] = T(-2) * near / cen[2];
    cen[0] = -kx * (cen[0] / cen[2]);
    cen[1] = -ky * (cen[1] / cen[2]);
    cen[2] = T(1) + T(2) * near / cen[2];
    const T n = norm3(dir);
    dir[0] /= n;
    dir[1] /= n;
    dir[2] /= n;
}

// Ray sources.  The rays of a launch are numbered 0 .. total()-1 ("items"); a wavefront owns the
// `per_wave` consecutive items of chunk chunk_of_block(blockIdx.x) and feeds them to its 64 lanes.
//   Batch: item i is ray i.
//   Image: items are numbered so that 64 consecutive items are one 8x8 pixel tile and 256
//          consecutive items one 16x16 block (four tiles), image after image: the rays a wavefront
//          holds at any time stay close in the tree, and the dispatcher starts the next image's
//          blocks as the previous image's last ones drain.  Items that fall outside the image
//          (sizes that are not multiples of 16) have no ray.  The blocks of an image are counted
//          row by row or (inside_out) ring by ring from the middle of the image: a launch lasts as
//          long as its longest rays, a camera that looks at an object has them in the middle of
//          the picture, and counted from there they start first instead of after the dispatcher
//          has gone through the upper half of the image.
// fetch_item returns the output slot of the item (ray index / pixel index) or -1, and the ray in
// tree coordinates.
template <typename T>
struct BatchSource {
    static constexpr bool kGated = false;
    RayBatch<T> rays;
    int per_wave;
    int refill_at;   // idle lanes that trigger taking new rays
    int xcd_group;   // see chunk_of_block; 1 for unrelated rays
    // > 0 (per_wave a power of two): the wavefront that owns items [w * per_wave, (w + 1) * per_wave)
    // takes the groups of four rays w, w + n_waves, w + 2 * n_waves, ... of the batch instead of one
    // contiguous range.  A batch in some coherent order (the rays of an image, row by row) keeps its
    // long rays together, and the wavefronts that own them would finish long after the others (1M
    // rays of 8 images in tile order: 3x the time of the same rays shuffled, backward 5x); dealt
    // out like this every wavefront gets its share whatever the order, at 2-3 % for a shuffled batch
    // (groups of four keep the reads of the rays in whole 48-byte pieces; single rays cost 14 %).
    int64_t n_waves;
    __device__ __forceinline__ int64_t total() const { return n_waves > 0 ? n_waves * per_wave : rays.n_rays; }
    // rays are numbered as they lie in the batch; with n_waves == 0 item i is ray i
    static constexpr bool kItemsAreSlots = true;
    __device__ __forceinline__ int64_t n_slots() const { return rays.n_rays; }
    __device__ __forceinline__ void view_dir(int64_t slot, T* vdir) const {
#pragma unroll
        for (int k = 0; k < 3; ++k) vdir[k] = rays.vdirs[slot * 3 + k];
    }
    __device__ __forceinline__ int64_t fetch_item(int64_t i, const SvoxRenderOptions&, const T* offset,
                                                  const T* scaling, T* origin, T* dir, T* vdir) const {
        if (n_waves > 0) {
            const int shift = __builtin_ctz((unsigned)per_wave);
            const int64_t j = i & (per_wave - 1), w = i >> shift;
            i = ((((j >> 2) * n_waves + w) << 2) | (j & 3));
        }
        if (i >= rays.n_rays) return -1;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            origin[k] = rays.origins[i * 3 + k];
            dir[k] = rays.dirs[i * 3 + k];
            vdir[k] = rays.vdirs[i * 3 + k];
        }
        transform_coord(origin, offset, scaling);
        return i;
    }
};

// Rays of a batch that meet the cube, for noting passes (list_hits_kernel): item i is ray list[i].  And the batch as it is, where that is
// one of the shapes such a pass is launched in (kGated, ReplaySpace::chosen; a kernel of their own, as the look at the gate costs others 1 to
// 2 %: dense 128^3 SH1, 28 456 rays with notes 435.3 -> 443.7 us).
struct ListedSource : BatchSource<float> {
    static constexpr bool kGated = true;
    const int32_t* list;
    const unsigned long long* n_listed;
    __device__ __forceinline__ int64_t total() const { return (int64_t)*n_listed; }
    __device__ __forceinline__ int64_t fetch_item(int64_t i, const SvoxRenderOptions& opt, const float* offset,
                                                  const float* scaling, float* origin, float* dir, float* vdir) const {
        return BatchSource<float>::fetch_item(list[i], opt, offset, scaling, origin, dir, vdir);
    }
};
struct WholeSource : BatchSource<float> {
    static constexpr bool kGated = true;
};

__host__ __device__ inline int blocks16_of(int extent) { return (extent + 15) / 16; }

// Which chunk of items the wavefront of block `b` (of gridDim.x) works on.  Workgroups are handed
// to the 8 XCDs in turn (block b runs on XCD b mod 8), and every XCD has its own L2.  With
// group > 1, runs of `group` consecutive chunks go to one XCD, so neighbouring image tiles, whose
// rays read the same child rows and leaf records, share that L2; the runs themselves still rotate
// over the XCDs, which keeps the load balanced.  A bijection on [0, gridDim.x).
__device__ __forceinline__ int64_t chunk_of_block(unsigned b, unsigned n_blocks, int group) {
    constexpr unsigned kXcds = 8;
    if (group <= 1) return b;
    const unsigned span = kXcds * (unsigned)group;
    const unsigned full = n_blocks / span * span;
    if (b >= full) return b;
    const unsigned xcd = b % kXcds, j = b / kXcds;
    return (int64_t)((j / group) * kXcds + xcd) * group + j % group;
}

// Block `rank` of an nbx x nby grid of blocks counted from the middle outwards: the innermost
// rectangle first, then ring after ring (each ring clockwise from its top left corner).
__device__ __forceinline__ void block_inside_out(int rank, int nbx, int nby, int& bx, int& by) {
    int p = (min(nbx, nby) - 1) / 2;
    while (p > 0 && rank >= (nbx - 2 * p) * (nby - 2 * p)) --p;
    const int w = nbx - 2 * p, h = nby - 2 * p;
    const int inner = (w > 2 && h > 2) ? (w - 2) * (h - 2) : 0;
    const int k = rank - inner;
    if (h == 1) {
        bx = p + k; by = p;
    } else if (w == 1) {
        bx = p; by = p + k;
    } else if (k < w) {
        bx = p + k; by = p;
    } else if (k < w + h - 1) {
        bx = p + w - 1; by = p + (k - w + 1);
    } else if (k < 2 * w + h - 2) {
        bx = p + w - 1 - (k - (w + h - 2)); by = p + h - 1;
    } else {
        bx = p; by = p + h - 1 - (k - (2 * w + h - 3));
    }
}

template <typename T>
struct ImageSource {
    static constexpr bool kGated = false;
    Camera<T> cam;          // cam.c2w: pose of image 0
    int n_images;
    int64_t pose_stride;    // scalars between consecutive poses
    int per_wave;           // 64 (one 8x8 tile) or 256 (one 16x16 block)
    int refill_at;          // idle lanes that trigger taking new rays
    int xcd_group;          // see chunk_of_block
    int run;                // > 0: the images advance together, `run` 16x16 blocks at a time
    int inside_out;         // != 0: the blocks of an image are counted from its middle outwards
    // pixels are numbered image by image, row by row; the items run through the tiles instead
    static constexpr bool kItemsAreSlots = false;
    __device__ __forceinline__ int64_t n_slots() const { return (int64_t)n_images * cam.height * cam.width; }
    __device__ __forceinline__ void view_dir(int64_t slot, T* vdir) const {
        const int64_t per_image = (int64_t)cam.height * cam.width;
        const int64_t image = slot / per_image;
        const int pixel = (int)(slot - image * per_image);
        const int iy = pixel / cam.width, ix = pixel - iy * cam.width;
        Camera<T> c = cam;
        c.c2w = cam.c2w + image * pose_stride;
        T origin[3];
        cam2world_ray(ix, iy, c, vdir, origin);
    }
    __device__ __forceinline__ int64_t total() const {
        const int64_t per_image = (int64_t)blocks16_of(cam.width) * blocks16_of(cam.height);
        const int64_t padded = run > 0 ? (per_image + run - 1) / run * run : per_image;
        return (int64_t)n_images * padded * 256;
    }
    __device__ __forceinline__ int64_t fetch_item(int64_t i, const SvoxRenderOptions& opt, const T* offset,
                                                  const T* scaling, T* origin, T* dir, T* vdir) const {
        const int nbx = blocks16_of(cam.width), nby = blocks16_of(cam.height);
        const int64_t block = i >> 8;
        const int within = (int)(i & 255);
        int image, b;
        if (run > 0) {
            // runs of `run` blocks, image after image, then the next run of every image
            const int64_t r = block / run;
            const int64_t round = r / n_images;
            image = (int)(r - round * n_images);
            b = (int)(round * run + (block - r * run));
            if (b >= nbx * nby) return -1;
        } else {
            image = (int)(block / (nbx * nby));
            if (image >= n_images) return -1;
            b = (int)(block - (int64_t)image * (nbx * nby));
        }
        int by = b / nbx, bx = b - by * nbx;
        if (inside_out) block_inside_out(b, nbx, nby, bx, by);
        const int sub = within >> 6, pos = within & 63;
        const int ix = bx * 16 + (sub & 1) * 8 + (pos & 7);
        const int iy = by * 16 + (sub >> 1) * 8 + (pos >> 3);
        if (ix >= cam.width || iy >= cam.height) return -1;
        return fetch_pixel(image, ix, iy, opt, offset, scaling, origin, dir, vdir);
    }
    __device__ __forceinline__ int64_t fetch_pixel(int image, int ix, int iy, const SvoxRenderOptions& opt, const T* offset,
                                                   const T* scaling, T* origin, T* dir, T* vdir) const {
        Camera<T> c = cam;
        c.c2w = cam.c2w + (int64_t)image * pose_stride;
        cam2world_ray(ix, iy, c, dir, origin);
#pragma unroll
        for (int k = 0; k < 3; ++k) vdir[k] = dir[k];
        maybe_world2ndc(opt, dir, origin);
        transform_coord(origin, offset, scaling);
        return ((int64_t)image * cam.height + iy) * cam.width + ix;
    }
    // the pixel of a number as the pixels are numbered, of which there are n_slots()
    __device__ __forceinline__ int64_t fetch_slot(int64_t slot, const SvoxRenderOptions& opt, const T* offset, const T* scaling,
                                                  T* origin, T* dir, T* vdir) const {
        const int64_t per_image = (int64_t)cam.height * cam.width;
        const int image = (int)(slot / per_image);
        const int pixel = (int)(slot - image * per_image);
        const int iy = pixel / cam.width;
        return fetch_pixel(image, pixel - iy * cam.width, iy, opt, offset, scaling, origin, dir, vdir);
    }
};

// Pixels of pictures that meet the cube, for noting passes, as ListedSource has the rays of a batch; and the pictures as they are, where that
// is the shape such a pass is launched in.  (One kernel for both, which looks at the number, took 1.15 to 2 times as long where most pixels do.)
struct ListedImageSource : ImageSource<float> {
    static constexpr bool kGated = true;
    const int32_t* list;
    const unsigned long long* n_listed;
    __device__ __forceinline__ int64_t total() const { return (int64_t)*n_listed; }
    __device__ __forceinline__ int64_t fetch_item(int64_t i, const SvoxRenderOptions& opt, const float* offset,
                                                  const float* scaling, float* origin, float* dir, float* vdir) const {
        return fetch_slot(list[i], opt, offset, scaling, origin, dir, vdir);
    }
};
struct WholeImageSource : ImageSource<float> {
    static constexpr bool kGated = true;
};

// ------------------------------------------------------------------------------------------------
// per-ray march state
// ------------------------------------------------------------------------------------------------
template <typename T>
struct RayState {
    T o[3], d[3], inv[3];
    T t, tmax, dscale;
};

// rt_kernel.cu:228-247: scale and normalise the direction, reciprocal in double, clip to the cube
template <typename T>
__device__ __forceinline__ bool setup_ray(RayState<T>& r, const T* origin, const T* dir, const T* scaling) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        r.o[i] = origin[i];
        r.d[i] = dir[i] * scaling[i];
    }
    const T s = T(1) / norm3(r.d);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        r.d[i] *= s;
        r.inv[i] = (T)(1.0 / ((double)r.d[i] + 1e-9));
    }
    r.dscale = s;
    T tmin, tmax;
    dda_unit(r.o, r.inv, &tmin, &tmax);
    r.t = tmin;
    r.tmax = tmax;
    return !(tmax < T(0) || tmin > tmax);
}

// t += delta_t.  If t cannot advance any more (a delta below the spacing of floats at t, or NaN), the
// reference's `while (t < tmax)` loop would never end; the ray is ended after this sample instead.
template <typename T>
__device__ __forceinline__ void advance(RayState<T>& r, T delta_t) {
    const T t_next = r.t + delta_t;
    r.t = t_next > r.t ? t_next : r.tmax;
}

struct Visit {
    int64_t leaf;  // cell index node*N^3 + cell; -1 ends the ray (malformed tree)
    int levels;
};

// Child entries one lane reads per turn of the octree walk (OctreeCursor::turn).  A lane that needs
// more (its ray crossed the boundary of a large cell and has to descend many levels) goes on in its
// next turn, so that the other lanes of the wavefront do not wait for it: measured, the lanes need
// 2.0 entries per leaf on average, but the slowest lane of a wavefront 4.8.  (Budgets of 1 and 3, and
// extra turns per round for the interrupted lanes, were measured slower.)
constexpr int kSeekBudget = 2;

// One sample with the reference's walk: position, leaf, step length.  rt_kernel.cu:262-275.
template <typename T>
__device__ __forceinline__ Visit step_generic(const TreeDev<T>& tr, const RayState<T>& r, T step_size,
                                              T* delta_t) {
    T pos[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) pos[j] = fma_(r.t, r.d[j], r.o[j]);
    T cube;
    Visit v;
    v.leaf = descend_generic<T>(tr.child, tr.capacity, tr.N, pos, &cube, &v.levels);
    T s0, s1;
    dda_unit(pos, r.inv, &s0, &s1);
    *delta_t = (s1 - s0) / cube + step_size;
    return v;
}

// The child table of an octree as the march reads it: through a buffer descriptor, so that a read which a lane has no need for, or which a
// malformed tree leads out of the table, costs neither a branch nor a request -- beyond the last byte it gives 0.  (The table is smaller than
// 4 GiB, checked on the host.)
struct ChildTable {
    __amdgpu_buffer_rsrc_t entries;
    uint32_t last_cell;
    bool octree, words;   // words: it is a walk table
    static constexpr uint32_t kNowhere = 0xffffffe0u;   // a row beyond the largest table
    template <typename T>
    __device__ __forceinline__ explicit ChildTable(const TreeDev<T>& tr) {
        const uint32_t cells = (uint32_t)tr.capacity << 3;
        octree = tr.N == 2;
        last_cell = cells - 1u;
        words = octree && tr.walk != nullptr;
        entries = __builtin_amdgcn_make_buffer_rsrc((void*)(words ? tr.walk : tr.child), 0, octree ? cells << 2 : 0u, 0x00020000);
    }
    // The table for a wavefront whose first rays are these, before any of them begins.  Rays that run close together find the rows they read in L1, and
    // the turns of a walk on a walk table that only descend then cost more than the reads it saves: it stays with the child table where most
    // neighbours enter the cube less than 0.7 of the square root of 1/nodes apart -- of a surface 0.4 of its leaves -- unless marks went into the walk table,
    // which the child table has not.  (Pictures, us, child table / walk table, by that distance over the square root: 128^3 shell RGBA 0.34 175 / 198, 0.38 147 / 173,
    // 0.48 117 / 131, 0.64 114 / 116, 0.69 118 / 111, SH9 0.38 175 / 197, 0.43 173 / 166; 256^3 RGBA 0.48 345 / 387, 0.68 228 / 247, 0.77 203 / 219, 0.86 189 / 181, SH9 0.6 299 / 318, 0.68
    // 260 / 272, 0.77 241 / 248, 0.86 229 / 215; 512^3 RGBA 0.6 465 / 514, 0.96 410 / 446, 1.2 323 / 337, 1.5 266 / 254, SH9 0.6 605 / 596, 0.96 629 / 578; 128^3 grid SH4 0.6
    // 384 / 411, 1.2 281 / 293, 1.6 267 / 244.)
    template <typename T>
    __device__ __forceinline__ void settle(const TreeDev<T>& tr, const RayState<T>& r, bool active) {
        if (!words || tr.walk_marked) return;
        T apart = T(0);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const T at = active ? fma_(r.t, r.d[i], r.o[i]) : T(0);
            const T by = at - neighbour(at);
            apart = fma_(by, by, apart);
        }
        const unsigned long long rays = __builtin_amdgcn_ballot_w64(active), odd = 0x5555555555555555ull;
        const unsigned long long pairs = rays & ((rays >> 1 & odd) | (rays & odd) << 1);
        const unsigned long long close = __builtin_amdgcn_ballot_w64(apart * (T)tr.capacity < T(0.5)) & pairs;
        if (2 * __popcll(close) > __popcll(pairs)) {
            words = false;
            entries = __builtin_amdgcn_make_buffer_rsrc((void*)tr.child, 0, (last_cell + 1u) << 2, 0x00020000);
        }
    }
    // the value of the lane beside, of each pair
    static __device__ __forceinline__ float neighbour(float v) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
    }
    __device__ __forceinline__ int32_t read(uint32_t at) const { return (int32_t)__builtin_amdgcn_raw_buffer_load_b32(entries, (int)at, 0, 0); }
    __device__ __forceinline__ uint32_t cell(uint32_t number) const { return min(number, last_cell); }
};

// (a << n) | b in one instruction: in plain C++ the compiler orders the three below so that it takes four
template <int n>
__device__ __forceinline__ uint32_t shift_or(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_lshl_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "n"(n), "v"(b));
    return r;
}
// which cell of its node a sample lies in, `up` levels above the finest that its integer coordinates hold
__device__ __forceinline__ uint32_t octant_of(uint32_t ix, uint32_t iy, uint32_t iz, int up) {
    const unsigned bx = __builtin_amdgcn_ubfe(ix, (unsigned)up, 1u), by = __builtin_amdgcn_ubfe(iy, (unsigned)up, 1u),
                   bz = __builtin_amdgcn_ubfe(iz, (unsigned)up, 1u);
    return shift_or<1>(shift_or<1>(bx, by), bz);
}

// The walk of one lane's ray through the tree, sample after sample.  A sample's integer coordinates (24 bits an axis)
// say which cell it lies in at every level, and those it shares with the sample before say how far up the next search
// has to start: where the child rows of the previous path begin is kept in LDS, one column per lane (`path`, laid out
// [kPathLevels + 2][64], the root's row last; the first two rows are a dump for the levels below, which no search resumes from).
//
// The march waits for this chain -- position, coordinates, path, child reads, step -- once per leaf, and where no other
// wavefront fills the gaps what counts are its instructions: a lone wavefront issues one every 7 to 9 cycles, takes 30 to 40 for a
// branch, 160 for a read that hits L1.  So the ray's origin and direction are kept
// times 2^24 (exact: the coordinates need no further product), the sample is looked up in the path as soon as it is
// known (aim) rather than when its turn comes, the levels are counted from below, so that the level to resume from is the highest
// bit of what the samples differ in, and a lane that has no read to make is turned away by the bounds of the buffer (ChildTable) and not by
// a branch.  A turn is 75 vector instructions and one branch (110 and five where the reads, the level found and the malformed were each
// a branch; 145 with selects over pending and finished searches).  A wavefront alone, child table in L2, ns a leaf: 625 to 830 -> 530 to 690 on one
// wavefront per tile, 705 to 890 -> 460 to 590 on two (by how far the rays are apart).  800x800 picture of a 512^3 SH16 shell 314 -> 270 us, 8 such pictures
// 762 -> 743, an NDC picture 563 -> 541; squared error of 200 003 rays 481 -> 433, training step of 1 Mi rays 1242 -> 1209.
// (Keeping whole child rows of the last four levels in LDS as well, so that a
// step costs one read instead of two, made the two-wavefront kernel 3 to 8 % faster where it runs alone on a CU, and
// everything else up to 45 % slower.)
struct OctreeCursor {
    int32_t* rows;         // the lane's column of the path: rows[64 * (1 + max(up, kPathUp))]
    float m[3];            // the sample, clamped, times -2^24
    uint32_t ix, iy, iz;   // its integer coordinates
    int up;                // where the search for its leaf stands, in levels above the finest the coordinates hold (kCoordBits
                           // minus the level; negative: the sample lies deeper): the child row to look into ...
    uint32_t row;          // ... begins at this byte of the table
    static constexpr int kPathUp = kCoordBits - kPathLevels - 1;   // of the path's upper dump row; the other lies below it

    // `lane_path`: this lane's column
    __device__ __forceinline__ void reset(int32_t* lane_path) {
        rows = lane_path - kPathUp * kMarchThreads;
        rows[kCoordBits * kMarchThreads] = 0;
        m[0] = m[1] = m[2] = 0.0f;
        ix = iy = iz = 0;
        up = kCoordBits - 1;
        row = 0;
    }
    // the first sample of a ray fresh from setup_ray
    __device__ __forceinline__ void begin(RayState<float>& r) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            r.o[i] *= 16777216.0f;
            r.d[i] *= 16777216.0f;
        }
        aim(r, kCoordBits - 1);
    }
    // the sample at r.t; leaf_up: where the leaf of the sample before it lies (kCoordBits - 1: the path says nothing of it)
    __device__ __forceinline__ void aim(const RayState<float>& r, int leaf_up) {
        // (clamp01, times -2^24: of a coordinate that is no number, as 0 times an infinite direction is, clamp01 makes the upper bound, and fmed3 the
        // least of the other two.  The asm keeps the compiler from taking the signs out again.)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            m[i] = __builtin_amdgcn_fmed3f(-fma_(r.t, r.d[i], r.o[i]), 0.0f, -__uint_as_float(0x3F7FFFEFu) * 16777216.0f);
            asm("" : "+v"(m[i]));
        }
        const uint32_t nx = (uint32_t)-m[0], ny = (uint32_t)-m[1], nz = (uint32_t)-m[2];
        // the first level the two samples differ at is that of the highest bit they differ in; not below the leaf, nor the path
        const uint32_t diff = (ix ^ nx) | (iy ^ ny) | (iz ^ nz) | 1u << leaf_up | 1u << (kPathUp + 1);
        up = 31 - __builtin_clz(diff);
        row = (uint32_t)rows[(up + 1) * kMarchThreads];
        ix = nx;
        iy = ny;
        iz = nz;
    }
    // which cell of its node the sample lies in
    __device__ __forceinline__ uint32_t octant() const { return octant_of(ix, iy, iz, up); }
    // the byte of the table that holds the child entry to look at, in the row that begins at `from`
    __device__ __forceinline__ uint32_t entry(uint32_t from) const { return shift_or<2>(octant(), from); }
    // One turn of the lanes with `go`: up to kSeekBudget child reads, and if the leaf is found its index (with
    // kEmptyLeafBit if it is marked empty) in slot_leaf, the step of the sample in slot_dt, and the ray moved on; else
    // both are left as they are.  A lane whose sample lies deeper than the coordinates resolve is left with a negative `up`.
    __device__ __forceinline__ void turn(RayState<float>& r, bool go, const ChildTable& child, float step_size, int32_t& slot_leaf,
                                         float& slot_dt) {
        static_assert(kSeekBudget == 2, "two reads, written out");
        const uint32_t first = entry(go ? row : ChildTable::kNowhere);
        const int32_t skip1 = child.read(first);
        const bool below = skip1 > 0;
        const uint32_t next = row + ((uint32_t)skip1 << 5);
        // (of a lane that stays where it is the second row means nothing, and is read by nobody)
        int32_t* const at = rows + max(up, kPathUp) * kMarchThreads;
        at[kMarchThreads] = (int32_t)row;
        at[0] = (int32_t)next;
        up -= below ? 1 : 0;
        const uint32_t second = entry(below ? next : ChildTable::kNowhere);
        row = below ? next : row;
        const int32_t skip2 = child.read(second);
        const int32_t skip = min(skip1, skip2);   // (the second is 0 where there was no need for it)
        const int leaf_up = up;
        row += (uint32_t)max(skip2, 0) << 5;
        up -= skip2 > 0 ? 1 : 0;
        if (go & (skip <= 0) & (leaf_up >= 0)) {
            up = leaf_up;
            take(r, (int32_t)child.cell((below ? second : first) >> 2) | (skip >> 1 & kEmptyLeafBit), step_out(r, leaf_up, step_size), slot_leaf, slot_dt);
        }
    }
    // The same on a walk table, `row` a word of it: one read, and none where the sample lies in a node that has leaves only (a second read in
    // the turn, which every wavefront would wait for for the sake of a few lanes, costs as much as the turns it saves).
    // The step is worked out for both of the levels the leaf may lie at while the read is on its way (squared error of 200 003 rays, the
    // march 219 -> 207 us, 8 pictures 692 -> 686, 1 Mi rays with notes 664 -> 649).  A turn of a wavefront alone with its tile takes 1000 cycles where the table
    // is in L2 (1500 on the child table), 1400 where it is not (2150).
    __device__ __forceinline__ void turn_words(RayState<float>& r, bool go, const ChildTable& child, float step_size, int32_t& slot_leaf,
                                               float& slot_dt) {
        const uint32_t word = row;
        uint32_t cell = octant();
        const int32_t skip = child.read(shift_or<2>(cell, go & (word < (uint32_t)kLastNodeBit) ? word << 5 : ChildTable::kNowhere));
        int32_t* const at = rows + max(up, kPathUp) * kMarchThreads;
        at[kMarchThreads] = (int32_t)word;
        const uint32_t up_bits = (uint32_t)up << 23;
        const float to_leaf = __uint_as_float((383u << 23) - up_bits);
        const float inv_cube = __uint_as_float(((uint32_t)(127 - kCoordBits) << 23) + up_bits);
        float here[3], below_it[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const float s = m[j] * to_leaf;
            here[j] = __builtin_amdgcn_fractf(s);
            below_it[j] = __builtin_amdgcn_fractf(s + s);
        }
        float dt = leaf_exit(here, r.inv) * inv_cube + step_size, dt_below = leaf_exit(below_it, r.inv) * (inv_cube * 0.5f) + step_size;
        up -= 1;
        uint32_t cell_below = octant();
        asm volatile("" : "+v"(dt), "+v"(dt_below), "+v"(cell_below));   // (not after the read)
        const bool below = skip > 0;
        row = word + ((uint32_t)skip & 0x7fffffffu);
        at[0] = (int32_t)row;
        up += below ? 0 : 1;
        cell = below ? cell_below : cell;
        dt = below ? dt_below : dt;
        if (go & (up >= 0) & !(below & (row < (uint32_t)kLastNodeBit))) {
            const uint32_t empty = __builtin_amdgcn_ubfe(row, kWalkNodeBits + cell, 1u);
            take(r, (int32_t)(child.cell((row & kWalkNodes) << 3 | cell) | empty << 30), dt, slot_leaf, slot_dt);
        }
    }
    // the step to the far side of the leaf the sample lies in
    __device__ __forceinline__ float step_out(const RayState<float>& r, int leaf_up, float step_size) const {
        // -2^-up and 2^(up - 24): dividing by the power of two is the multiplication by its reciprocal
        const uint32_t up_bits = (uint32_t)leaf_up << 23;
        const float to_leaf = __uint_as_float((383u << 23) - up_bits);
        const float inv_cube = __uint_as_float(((uint32_t)(127 - kCoordBits) << 23) + up_bits);
        // leaf-local position frac(pos * 2^levels): s - floor(s), exact for the non-negative s of a clamped
        // coordinate, in one instruction
        float local[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) local[j] = __builtin_amdgcn_fractf(m[j] * to_leaf);
        return leaf_exit(local, r.inv) * inv_cube + step_size;
    }
    // the sample's leaf is found, at the level `up` says: on to the next sample
    __device__ __forceinline__ void take(RayState<float>& r, int32_t leaf, float dt, int32_t& slot_leaf, float& slot_dt) {
        slot_leaf = leaf;
        slot_dt = dt;
        const float t_next = r.t + slot_dt;
        r.t = t_next > r.t ? t_next : r.tmax;   // (advance())
        aim(r, up);
    }
};

// A sample of the lanes with `go` by the reference's walk from the root: what lies deeper than the integer coordinates hold, and
// trees with another branching factor, which have no exact integer formulation.  `broken`: the tree is malformed, the ray ends here.
__device__ __forceinline__ void walk_from_root(const TreeDev<float>& tr, RayState<float>& r, OctreeCursor& cur, float step_size, bool go,
                                               bool& broken, int32_t& slot_leaf, float& slot_dt) {
    if (!go) return;
    float local[3], cells_per_axis;
    int levels;
#pragma unroll
    for (int j = 0; j < 3; ++j) local[j] = -cur.m[j] * (1.0f / 16777216.0f);
    slot_leaf = (int32_t)descend_generic<float>(tr.child, tr.capacity, tr.N, local, &cells_per_axis, &levels, true);
    if (slot_leaf >= 0) {
        // (rt_kernel.cu:274 divides by the cell count; for a power of two the product with the reciprocal is
        // the same number)
        const float segment = leaf_exit(local, r.inv);
        slot_dt = (tr.N == 2 ? segment * (1.0f / cells_per_axis) : segment / cells_per_axis) + step_size;
        const float t_next = r.t + slot_dt;
        r.t = t_next > r.t ? t_next : r.tmax;
        cur.aim(r, kCoordBits - 1);
    } else {
        broken = true;
    }
}

// ------------------------------------------------------------------------------------------------
// policies
// ------------------------------------------------------------------------------------------------
template <typename T>
struct GenericPolicy {
    using scalar = T;
    static constexpr bool kOctree = false;
};

template <int FMT, int D>
struct OctreePolicy {
    using scalar = float;
    static constexpr bool kOctree = true;
    static constexpr int kFormat = FMT;                                // RGBA, SH, or SG for both kinds of lobes
    static constexpr int kBasis = D;                                   // 0 for RGBA
    static constexpr int kRecord = (FMT == SVOX_FORMAT_RGBA) ? 4 : 3 * D + 1;
    // SH: the basis is a closed form of the view direction, cheap enough to evaluate again wherever a
    // colour is formed; lobes (SG, ASG): D exponentials, evaluated once per ray and kept as a row in LDS
    static constexpr bool kForwardRows = FMT == SVOX_FORMAT_SG;
};

// The table of lobes of a tree of spherical gaussians (TreeSpec.extra_data: basis_dim rows [lambda, mu])
// or anisotropic ones ([lambda_x, lambda_y, x-axis, y-axis, z-axis]), and which of the two it is: the two
// formats differ in nothing but the basis of a ray, which is evaluated once per ray, so one set of
// kernels (OctreePolicy<SVOX_FORMAT_SG, D>) serves both and looks at `format` there.
struct Lobes {
    const float* table;
    int cols;
    int format;
};
// A launch that renders only the components [min_comp, max_comp] of the basis (rt_kernel.cu:286-288: the loops over
// the coefficients run over that range) runs on the kernels that keep a ray's basis as a row in LDS (the lobe
// policy, whatever the format: its rows are made by precalc_basis, which knows spherical harmonics too), with the
// row zero outside the range: the full-length colour sums then add 0 * coefficient = 0 for the terms the reference
// leaves out, which leaves the running sum as it is -- the same bits for every finite coefficient (a coefficient
// that is infinite or NaN outside the range would show here and not in the reference) -- and the gradient terms
// of those components are zeros added to zeros.
template <int D>
__device__ __forceinline__ bool partial_range(const SvoxRenderOptions& opt) {
    return opt.min_comp > 0 || opt.max_comp < D - 1;   // (uniform: the same for every lane of the launch)
}
template <int D>
__device__ __forceinline__ void keep_range(const SvoxRenderOptions& opt, float* x) {
#pragma unroll
    for (int i = 0; i < D; ++i) x[i] = (i >= opt.min_comp && i <= opt.max_comp) ? x[i] : 0.0f;
}

// The basis of one ray (maybe_precalc_basis, rt_kernel.cu:111-187) for the policy's format, zero outside the
// launch's component range.
template <class P>
__device__ __forceinline__ void policy_basis(const Lobes& lobes, const SvoxRenderOptions& opt, const float* vdir,
                                             float* out) {
    if constexpr (P::kFormat == SVOX_FORMAT_SH) {
        sh_basis<float>(P::kBasis, vdir, out);
    } else {
        precalc_basis<float>(lobes.format, P::kBasis, lobes.table, lobes.cols, vdir, out);
    }
    if (partial_range<P::kBasis>(opt)) keep_range<P::kBasis>(opt, out);
}

// atomicMax of the reference (common.cuh:152-172): compare-and-swap loop around fmaxf
__device__ __forceinline__ void atomic_max_float(float* addr, float value) {
    unsigned* a = (unsigned*)addr;
    unsigned old = *a, assumed;
    do {
        assumed = old;
        old = atomicCAS(a, assumed, __float_as_uint(max_(value, __uint_as_float(assumed))));
    } while (old != assumed);
}
__device__ __forceinline__ void atomic_max_float(double* addr, double value) {
    unsigned long long* a = (unsigned long long*)addr;
    unsigned long long old = *a, assumed;
    do {
        assumed = old;
        const double m = (double)max_((float)value, (float)__longlong_as_double((long long)assumed));
        old = atomicCAS(a, assumed, (unsigned long long)__double_as_longlong(m));
    } while (old != assumed);
}

// ------------------------------------------------------------------------------------------------
// forward
// ------------------------------------------------------------------------------------------------
// trace_ray, rt_kernel.cu:222-321, generic flavour.  `basis` and `acc` are this lane's columns of two LDS arrays
// laid out [index][lane] (stride kMarchThreads): the reference's loops index them at run time, and as register
// arrays they would live in scratch memory.
template <typename T>
__device__ void trace_generic(const TreeDev<T>& tr, const SvoxRenderOptions& opt, const T* origin,
                              const T* dir, const T* vdir, const T* scaling, int out_dim, T* out, T* basis, T* acc) {
    constexpr int S = kMarchThreads;
    RayState<T> r;
    if (!setup_ray(r, origin, dir, scaling)) {
        for (int j = 0; j < out_dim; ++j) out[j] = (T)opt.background_brightness;
        return;
    }
    for (int j = 0; j < out_dim; ++j) acc[j * S] = T(0);
    if (opt.format != SVOX_FORMAT_RGBA) {
        T b[SVOX_MAX_BASIS_DIM];
        precalc_basis<T>(opt.format, opt.basis_dim, tr.extra, tr.extra_cols, vdir, b);
#pragma unroll
        for (int i = 0; i < SVOX_MAX_BASIS_DIM; ++i)
            if (i < opt.basis_dim) basis[i * S] = b[i];
    }
    T light = T(1);
    const T pad = (T)opt.rgb_padding;
    const T d_rgb_pad = (T)(1 + 2 * opt.rgb_padding);
    bool stopped = false;
    while (r.t < r.tmax) {
        T delta_t;
        const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
        if (v.leaf < 0) break;
        const T* val = tr.data + v.leaf * tr.K;
        T sigma = val[tr.K - 1];
        if (opt.density_softplus) sigma = softplus_m1(sigma);
        if (sigma > (T)opt.sigma_thresh) {
            const T att = exp_sp<T>(-delta_t * r.dscale * sigma);
            const T weight = light * (T(1) - att);
            if (opt.format != SVOX_FORMAT_RGBA) {
                for (int c = 0; c < out_dim; ++c) {
                    const int off = c * opt.basis_dim;
                    T tmp = T(0);
                    for (int i = opt.min_comp; i <= opt.max_comp; ++i) tmp = fma_(basis[i * S], val[off + i], tmp);
                    acc[c * S] = fma_(weight, fma_(sigmoid_(tmp), d_rgb_pad, -pad), acc[c * S]);
                }
            } else {
                for (int c = 0; c < out_dim; ++c)
                    acc[c * S] = fma_(weight, fma_(sigmoid_(val[c]), d_rgb_pad, -pad), acc[c * S]);
            }
            light *= att;
            if (tr.weight_accum) {
                if (tr.weight_accum_max)
                    atomic_max_float(tr.weight_accum + v.leaf, weight);
                else
                    atomicAdd(tr.weight_accum + v.leaf, weight);
            }
            if (light <= (T)opt.stop_thresh) {
                const T scale = (T)(1.0 / (1.0 - (double)light));
                for (int j = 0; j < out_dim; ++j) acc[j * S] *= scale;
                stopped = true;
                break;
            }
        }
        advance(r, delta_t);
    }
    if (!stopped)
        for (int j = 0; j < out_dim; ++j) acc[j * S] = fma_(light, (T)opt.background_brightness, acc[j * S]);
    for (int j = 0; j < out_dim; ++j) out[j] = acc[j * S];
}

// number of set bits of `mask` below this lane
__device__ __forceinline__ int rank_in(unsigned long long mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// trace_ray for the generic policy: one ray per lane, no sharing of work between lanes
template <typename T>
__host__ __device__ inline size_t generic_forward_lds_bytes(int basis_dim, int out_dim) {
    return (size_t)kMarchThreads * (size_t)(basis_dim + out_dim) * sizeof(T);
}
template <typename T, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_forward_generic_kernel(TreeDev<T> tr, Source src,
                                                                               SvoxRenderOptions opt, int out_dim,
                                                                               T* __restrict__ out) {
    // dynamic LDS: (basis_dim + out_dim) scalars of T per lane, generic_forward_lds_bytes
    extern __shared__ __align__(16) unsigned char generic_lds[];
    T* const sh_basis = (T*)generic_lds;
    T* const sh_acc = sh_basis + kMarchThreads * (opt.format == SVOX_FORMAT_RGBA ? 1 : opt.basis_dim);
    T offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    T origin[3], dir[3], vdir[3];
    const int64_t item = blockIdx.x * (int64_t)kMarchThreads + threadIdx.x;
    const int64_t slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
    if (slot < 0) return;
    trace_generic<T>(tr, opt, origin, dir, vdir, scaling, out_dim, out + slot * out_dim, sh_basis + threadIdx.x,
                     sh_acc + threadIdx.x);
}

constexpr int kQueue = 4;  // leaves a lane walks ahead before the wavefront shades them
static_assert(kQueue <= 4, "ShadeShared::who packs the queue slot into two bits");

// Shade list shared by the wavefront: the (lane, slot) pairs of one round whose leaf has to be
// shaded, compacted so that consecutive lanes can take consecutive entries.  kRows: the basis of
// every lane's ray is kept as a row (needed where other lanes multiply with it); otherwise only
// the view direction is kept and the basis is re-evaluated where it is used.
template <int D, bool kRows>
struct ShadeShared;
template <int D>
struct ShadeShared<D, true> {
    float basis[kMarchThreads * D];             // [lane][coefficient]
    float colour[kQueue * kMarchThreads * 3];   // [slot][lane][channel]: sigmoid(basis . coefficients)
    int32_t leaf[kQueue * kMarchThreads];       // leaf cell index of entry e
    uint8_t who[kQueue * kMarchThreads];        // owner lane | slot << 6
};
template <int D>
struct ShadeShared<D, false> {
    float vdir[kMarchThreads * 3];              // [lane][xyz]
    float colour[kQueue * kMarchThreads * 3];
    int32_t leaf[kQueue * kMarchThreads];
    uint8_t who[kQueue * kMarchThreads];
};
// The LDS of a wavefront that walks and shades in turn.  The lowest row of its path, a dump, is `who`, which lives from a shade list to the end of its
// round: 256 bytes more are a granule more for some, and two wavefronts fewer on a compute unit (march without notes of 200 000 rays, 81^3 SH16, 3 797 us instead of
// 3 130; forward pass of 200 000 rays of a 128^3 shell with 16 lobes 414 instead of 321, of 285 000 rays of a 512^3 SH16 shell 890 instead of 754).
template <int D, bool kRows>
struct MarchShared {
    ShadeShared<D, kRows> sh;
    int32_t path[(kPathLevels + 1) * kMarchThreads];
    __device__ __forceinline__ int32_t* lane_path(int lane) { return (int32_t*)((char*)this + offsetof(MarchShared, path)) - kMarchThreads + lane; }
};
static_assert(sizeof(((ShadeShared<1, true>*)nullptr)->who) == sizeof(int32_t) * kMarchThreads, "the row before the path is `who`");

// Colours of all list entries, computed by the whole wavefront: item p = 3 * entry + channel goes to
// lane p mod 64.  One item is the reference's dot product for one channel, evaluated in the
// reference's order (coefficient 0 first) from 16-byte loads of the leaf record and the owner
// lane's basis, followed by the sigmoid.
// kWithSigma: the densities of the entries are not known yet (a launch whose marks say that every leaf on the list
// is shaded): the lane of an entry's last channel also reads the density, the scalar after its coefficients, and
// leaves it in sigma_out[slot * 64 + owner].
template <class P, bool kRows, bool kWithSigma = false>
__device__ __forceinline__ void shade_entries(const float* __restrict__ data,
                                              ShadeShared<(P::kBasis > 0 ? P::kBasis : 1), kRows>& sh,
                                              int n_entries, int lane, float* sigma_out = nullptr) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    const int n_items = n_entries * 3;
    for (int p = lane; p < n_items; p += kMarchThreads) {
        const int e = p / 3, c = p - 3 * e;
        const int32_t leaf = sh.leaf[e];
        const int who = sh.who[e];
        const int owner = who & 63, slot = who >> 6;
        const float* rec = data + (int64_t)leaf * K;
        float density = 0.0f;
        if constexpr (kWithSigma) {
            if (c == 2) density = rec[K - 1];
        }
        float s;
        if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
            s = sigmoid_(rec[c]);
        } else {
            const float* co = rec + c * D;
            // the coefficients are asked for first: the basis is evaluated while they arrive
            float cv[D];
#pragma unroll
            for (int i = 0; i < D; ++i) cv[i] = co[i];
            float b[D];
            if constexpr (kRows) {
#pragma unroll
                for (int i = 0; i < D; ++i) b[i] = sh.basis[owner * D + i];
            } else {
                const float vd[3] = {sh.vdir[owner * 3], sh.vdir[owner * 3 + 1], sh.vdir[owner * 3 + 2]};
                sh_basis<float>(P::kBasis, vd, b);
            }
            float tmp = 0.0f;
#pragma unroll
            for (int i = 0; i < D; ++i) tmp = fma_(b[i], cv[i], tmp);
            s = sigmoid_(tmp);
        }
        sh.colour[(slot * kMarchThreads + owner) * 3 + c] = s;
        if constexpr (kWithSigma) {
            if (c == 2) sigma_out[slot * kMarchThreads + owner] = density;
        }
    }
}

// ---- phases of a round shared by the octree kernels --------------------------------------------
// Refill: once `refill_at` lanes are idle and the wavefront's range [next, end) is not used up, the
// idle lanes take the next items, ranked by ballot.  Returns kRoundRefilled (look again), kRoundDone
// (every lane idle, range used up) or kRoundWork.
enum RoundState { kRoundWork, kRoundRefilled, kRoundDone };
template <class Start>
__device__ __forceinline__ RoundState refill_lanes(bool active, int64_t& next, int64_t end, int refill_at,
                                                   Start&& start) {
    const unsigned long long idle = __ballot(!active);
    const int n_idle = __popcll(idle);
    if (next < end && n_idle >= refill_at) {
        if (!active) {
            const int64_t item = next + rank_in(idle);
            if (item < end) start(item);
        }
        next += n_idle;
        return kRoundRefilled;
    }
    return n_idle == kMarchThreads ? kRoundDone : kRoundWork;
}

// Walk: kQueue turns; slot q receives the leaf found in turn q and its step length, or -1 (no live
// ray, or a descent still under way).  `broken` reports a malformed tree: the ray ends there.
__device__ __forceinline__ void walk_turns(const TreeDev<float>& tr, const ChildTable& child, RayState<float>& r, OctreeCursor& cur,
                                           float step, bool active, bool& broken, int32_t* q_leaf, float* q_dt) {
    broken = false;
    if (__builtin_expect(!child.octree, 0)) {
#pragma unroll
        for (int q = 0; q < kQueue; ++q) {
            q_leaf[q] = -1;
            q_dt[q] = 0.0f;
            walk_from_root(tr, r, cur, step, active && !broken && r.t < r.tmax, broken, q_leaf[q], q_dt[q]);
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < kQueue; ++q) {
        q_leaf[q] = -1;
        q_dt[q] = 0.0f;
    }
    if (child.words) {
#pragma unroll
        for (int q = 0; q < kQueue; ++q) cur.turn_words(r, active & (r.t < r.tmax), child, step, q_leaf[q], q_dt[q]);
    } else {
#pragma unroll
        for (int q = 0; q < kQueue; ++q) cur.turn(r, active & (r.t < r.tmax), child, step, q_leaf[q], q_dt[q]);
    }
    // (a descent that has come below the last level the coordinates hold waits for the end of the round)
    const bool deep = active && cur.up < 0 && r.t < r.tmax;
    if (__builtin_expect(any_lane(deep), 0)) walk_from_root(tr, r, cur, step, deep, broken, q_leaf[kQueue - 1], q_dt[kQueue - 1]);
}

// Sigma: the densities of the queued leaves, fetched together (the last scalar of each record).
template <int K>
__device__ __forceinline__ void fetch_sigma(const float* __restrict__ data, const int32_t* q_leaf, float* q_sigma) {
#pragma unroll
    for (int q = 0; q < kQueue; ++q) {
        // no leaf in the slot (-1) or a leaf marked empty (kEmptyLeafBit): nothing to read
        q_sigma[q] = (uint32_t)q_leaf[q] < (uint32_t)kEmptyLeafBit ? data[(int64_t)q_leaf[q] * K + (K - 1)] : 0.0f;
    }
}

// density_softplus (rt_kernel.cu:276-277): the march works on log(1 + exp(sigma - 1)) of the stored density.
// q_sigma: in the stored densities of the queued leaves, out the densities the march uses; q_raw keeps the stored
// ones (the gradient's chain factor sigmoid(raw - 1), rt_kernel.cu:471-474, and the notes need them).  A slot
// without a leaf, or with a leaf marked empty, stays at 0.
__device__ __forceinline__ void soften_sigma(bool softplus, const int32_t* q_leaf, float* q_sigma, float* q_raw) {
#pragma unroll
    for (int q = 0; q < kQueue; ++q) q_raw[q] = q_sigma[q];
    if (softplus) {
#pragma unroll
        for (int q = 0; q < kQueue; ++q)
            q_sigma[q] = (uint32_t)q_leaf[q] < (uint32_t)kEmptyLeafBit ? softplus_m1(q_raw[q]) : 0.0f;
    }
}

// Shade list: the (lane, slot) pairs with sigma > thresh, compacted by ballot and prefix count
// (`skip`: none of this lane's).  Returns the number of entries.
template <class Shared>
__device__ __forceinline__ int build_shade_list(Shared& sh, const int32_t* q_leaf, const float* q_sigma,
                                                float thresh, int lane, bool skip = false) {
    int n_entries = 0;
#pragma unroll
    for (int q = 0; q < kQueue; ++q) {
        const bool want = !skip && q_leaf[q] >= 0 && q_sigma[q] > thresh;
        const unsigned long long m = __ballot(want);
        if (want) {
            const int e = n_entries + rank_in(m);
            sh.leaf[e] = q_leaf[q];
            sh.who[e] = (uint8_t)(lane | (q << 6));
        }
        n_entries += __popcll(m);
    }
    return n_entries;
}

// The same list where the marks of the launch say that every leaf they let through is shaded (the marks were made
// with the launch's own sigma_thresh): every queued leaf that is not marked joins, its density still unread.
template <class Shared>
__device__ __forceinline__ int build_shade_list_all(Shared& sh, const int32_t* q_leaf, int lane) {
    int n_entries = 0;
#pragma unroll
    for (int q = 0; q < kQueue; ++q) {
        const bool want = (uint32_t)q_leaf[q] < (uint32_t)kEmptyLeafBit;
        const unsigned long long m = __ballot(want);
        if (want) {
            const int e = n_entries + rank_in(m);
            sh.leaf[e] = q_leaf[q];
            sh.who[e] = (uint8_t)(lane | (q << 6));
        }
        n_entries += __popcll(m);
    }
    return n_entries;
}

// Workspace of the replaying backward: chunks of kChunkRecords records of 3 float2 (leaf and step
// length, density and first sigmoid, the other two sigmoids) followed by one float2 whose x
// holds the index of the ray's next chunk.  Ray number i starts in chunk i; further chunks come
// from the rest of the workspace, of which a wavefront takes a stock of 64 chunks at a time through
// one atomic counter (a heavy image tile needs hundreds, most tiles none); the lanes that need a
// chunk in the same step are ranked by ballot.  (Rays in pieces take as many as they need through a second
// counter, and keep the first in step: take_chunks.)
constexpr int kStampWords = 6;   // ray count; tree data, child; ray origins, directions; step size and threshold
struct ReplaySpace {
    float2* base;          // chunk c starts at base + c * kChunkFloat2
    int64_t first_shared;  // chunks [0, first_shared) are the rays' first chunks
    int64_t n_chunks;      // chunks [first_shared, n_chunks) are handed out
    unsigned long long* stocks_taken;   // counters, zero when the launch starts: stocks handed out; chunks handed out one by one; rays listed
    // the noting forward kernels write `stamp` (what the notes belong to) to stamp_at; replay_backward_kernel uses
    // the notes only if it finds its own stamp there
    unsigned long long* stamp_at;
    unsigned long long stamp[kStampWords];
    // one bit per ray (ray i: bit i % 64 of word i / 64).  replay_backward_kernel sets the bits of the
    // rays it could not do from their notes; a launch of render_backward_kernel that is given the
    // bitmap as `only` does those rays and no others
    unsigned long long* undone;
    const unsigned long long* only;
    // not zero if any bit is set: the launch for those rays, which most passes have none of, then need not look for them (training step of an 800x800 picture 899 -> 887 us)
    unsigned long long* any_undone;
    // > 0: the looks in a row after which a waiting wavefront of render_forward_split_kernel gives up, in place of
    // kSpinLimit (set by a debug flag, so that a test can see what a give-up leaves behind)
    int32_t spin_limit;
    // where replay_backward_kernel reports how full the notes ran, for the caller to look at whenever it likes (host
    // memory the device can write, or nullptr): stocks asked for in the upper half, stocks there are in the lower
    unsigned long long* report;
    uint32_t n_stocks;
    // counts the wavefronts of render_forward_split_kernel that gave up waiting (svox_give_up_count)
    unsigned int* give_ups;
    int32_t* list;         // room for a number per ray, behind the chunks or in the first stocks (ListedSource, ListedImageSource), or nullptr
    uint32_t list_stocks;  // of the stocks, those that a launch which fills the list takes for it
    // a noting launch: the blocks that march; those beyond clear these arrays of clear_words words each
    uint32_t march_blocks;
    uint32_t* clear_at[2];
    int64_t clear_words;
    // A pass of which only the device knows how many rays it has (list_hits_kernel) is launched in several shapes: this launch does its
    // work if there are at least, and at most, as many as it is made for (sources that are kGated).
    const unsigned long long* n_listed;
    int64_t least, most;
    __device__ __forceinline__ bool chosen() const { return (int64_t)*n_listed >= least && (int64_t)*n_listed <= most; }
};

// The arrays a gradient is going to be added to are cleared by further blocks of the launch that takes the notes for it: that one waits
// for the chains of its longest rays, with the way to memory all but idle, and the blocks behind its last tile fill the places of those
// that have ended.  (Two arrays of 172 MB, 200 003 rays: the squared error 524 us, 471 with them cleared on the way.)  Written past L2, which holds what the rays read.
constexpr int64_t kClearWords = 16384;   // a block's share of an array
static __device__ __forceinline__ void clear_share(const ReplaySpace& ws) {
    typedef uint32_t Words4 __attribute__((ext_vector_type(4)));
    const int64_t from = (int64_t)(blockIdx.x - ws.march_blocks) * kClearWords;
    const int64_t n = ws.clear_words - from < kClearWords ? ws.clear_words - from : kClearWords;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (!ws.clear_at[k]) continue;
        uint32_t* const at = ws.clear_at[k] + from;
        for (int64_t i = threadIdx.x; i < n / 4; i += blockDim.x) __builtin_nontemporal_store(Words4{0, 0, 0, 0}, (Words4*)at + i);
        for (int64_t i = n / 4 * 4 + threadIdx.x; i < n; i += blockDim.x) at[i] = 0;
    }
}

// whether the workspace carries the stamp this launch expects
__device__ __forceinline__ bool stamp_matches(const ReplaySpace& ws) {
    bool same = true;
#pragma unroll
    for (int i = 0; i < kStampWords; ++i) same = same && ws.stamp_at[i] == ws.stamp[i];
    return same;
}

// The first ray at or after `next` (a wavefront-uniform ray number below `end`) whose 64-ray word of
// the bitmap `only` is not zero, found 64 words at a time; a value >= end if there is none.
__device__ __forceinline__ int64_t skip_clear_words(const unsigned long long* __restrict__ only, int64_t next,
                                                    int64_t end, int lane) {
    while (next < end) {
        const int64_t word = next >> 6, last_word = (end - 1) >> 6;
        const bool some = word + lane <= last_word && only[word + lane] != 0ull;
        const unsigned long long nz = __ballot(some);
        if (nz == 0ull) {
            next = (word + kMarchThreads) << 6;
            continue;
        }
        const int64_t first = (word + __builtin_ctzll(nz)) << 6;
        if (first > next) next = first;
        break;
    }
    return next;
}

// What a launch of render_backward_kernel does:
//   kBackwardPlain   both marches walk the tree;
//   kBackwardSecond  only the second march: the first was made by a noting forward kernel.
// (Notes are taken by render_forward_kernel and render_forward_split_kernel with kNoted and used by
// replay_backward_kernel; render_backward_kernel serves the rays that have none.)
enum BackwardMode { kBackwardPlain = 0, kBackwardSecond = 1 };

// Head of a ray's notes, kept in the spare floats of its first chunk (after the 15 records): the
// link to the next chunk, the number of notes (-1: they did not fit; 0 also for a ray that misses
// the tree), the ray's delta_scale (rt_kernel.cu:228), a flag (1.0f: the ray misses the tree, 2.0f:
// its walk broke off in a malformed tree, 3.0f: the launch gave up on the ray -- count -1, no sum --, else 0.0f)
// and the sum of the backward pass's first march where the noting pass could form it (NoteTaker::finish).
constexpr int kChunkRecords = 15;
constexpr int kChunkFloat2 = (kChunkRecords + 1) * 3;   // 384 bytes
constexpr int kHeadFloat2 = kChunkRecords * 3;          // float2 index of {link, count}, then {delta_scale, -}
constexpr int kChunkStock = 64;   // further chunks a wavefront takes at a time (at most 64 lanes ask at once)

// The notes of one lane's ray while they are taken (by the forward kernels, for replay_backward_kernel
// and replay_se_grad_kernel): every leaf with sigma > 0, in the order the ray meets them, up to where nothing shines through
// any more (opaque_light).
struct NoteTaker {
    int count, pos;     // notes so far; place in the chunk being written
    bool lost;          // the workspace ran out: the backward pass of this ray will march
    float2* first;      // the ray's own chunk, which also holds the head of its notes
    float2* chunk;      // the chunk being written

    __device__ __forceinline__ void begin(const ReplaySpace& ws, int64_t slot) {
        count = 0;
        pos = 0;
        lost = false;
        first = ws.base + slot * kChunkFloat2;
        chunk = first;
    }
    // A ray that misses the tree: no notes, flagged as a miss.
    static __device__ __forceinline__ void missed(const ReplaySpace& ws, int64_t slot) {
        ws.base[slot * kChunkFloat2 + kHeadFloat2] = make_float2(0.0f, __int_as_float(0));
        ws.base[slot * kChunkFloat2 + kHeadFloat2 + 1] = make_float2(0.0f, 1.0f);
    }
    // Called by all lanes of the wavefront together; `note`: this lane has a leaf to note.  Lanes whose
    // chunk is full take the next chunks of the wavefront's stock [shared_next, shared_end), in lane
    // order; a new stock costs one atomic on the workspace's counter (what is left of the old one is
    // given up).
    __device__ __forceinline__ void take(const ReplaySpace& ws, int64_t& shared_next, int64_t& shared_end, int lane,
                                         bool note, int32_t leaf, float dt, float sigma, const float* s) {
        const bool need = note && !lost && pos == kChunkRecords;
        const unsigned long long m = __ballot(need);
        if (m) {
            if (shared_next + __popcll(m) > shared_end) {
                unsigned long long t = 0;
                if (lane == 0) t = atomicAdd(ws.stocks_taken, 1ull);
                const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)t);
                const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(t >> 32));
                const int64_t stock = (int64_t)(((unsigned long long)hi << 32) | lo);
                shared_next = ws.first_shared + stock * kChunkStock;
                shared_end = shared_next + kChunkStock < ws.n_chunks ? shared_next + kChunkStock : ws.n_chunks;
                if (shared_next > shared_end) shared_next = shared_end;
            }
            const int64_t mine = shared_next + rank_in(m);
            if (need) {
                if (mine < shared_end) {
                    chunk[kHeadFloat2] = make_float2(__int_as_float((int32_t)mine), 0.0f);
                    chunk = ws.base + mine * kChunkFloat2;
                    pos = 0;
                } else {
                    lost = true;
                }
            }
            shared_next += __popcll(m);
        }
        if (note) {
            if (!lost) {
                float2* e = chunk + pos * 3;
                e[0] = make_float2(__int_as_float(leaf), dt);
                e[1] = make_float2(sigma, s[0]);
                e[2] = make_float2(s[1], s[2]);
                pos += 1;
            }
            count += 1;
        }
    }
    // The head of the notes: the count beside the link (written when the first chunk filled up), -1 if
    // the notes are incomplete; then the ray's delta_scale and 2.0f if the walk broke off in a
    // malformed tree; then, from a noting pass that had the gradient of the picture at hand, the sum
    // the backward pass forms in its first march (render_backward_kernel<kBackwardSecond> starts from it).
    // The notes of a ray whose launch gave up on it (the bounded wait of render_forward_split_kernel ran out): no
    // count and no sum of the first march (flag 3.0f): the backward pass marches this ray twice.
    __device__ __forceinline__ void give_up(float dscale) {
        ((float*)(first + kHeadFloat2))[1] = __int_as_float(-1);
        first[kHeadFloat2 + 1] = make_float2(dscale, 3.0f);
        first[kHeadFloat2 + 2] = make_float2(0.0f, 0.0f);
    }
    __device__ __forceinline__ void finish(bool broken, float dscale, float march1_sum = 0.0f) {
        ((float*)(first + kHeadFloat2))[1] = __int_as_float(lost || broken ? -1 : count);
        first[kHeadFloat2 + 1] = make_float2(dscale, broken ? 2.0f : 0.0f);
        first[kHeadFloat2 + 2] = make_float2(march1_sum, 0.0f);
    }
    // The end of a ray of a pass that takes the notes for replay_se_grad_kernel: its pixel, whose colour and light in
    // front of the background are acc and light, as se_grad_kernel's first march leaves it (rt_kernel.cu:560-563,
    // 635-637, 711-713), and in the head, in place of flag and sum, the residual against the reference colour.
    __device__ __forceinline__ void finish_residual(bool broken, float dscale, const float* acc, float light, float bg,
                                                    const float* __restrict__ color_ref, float* __restrict__ pixel) {
        float resid[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            resid[c] = acc[c] + fma_(light, bg, -color_ref[c]);
            pixel[c] = resid[c] + color_ref[c];
        }
        ((float*)(first + kHeadFloat2))[1] = __int_as_float(lost || broken ? -1 : count);
        first[kHeadFloat2 + 1] = make_float2(dscale, resid[0]);
        first[kHeadFloat2 + 2] = make_float2(resid[1], resid[2]);
    }
};

// A noting pass follows a ray beyond the early stop of its picture, but not beyond the leaf behind which the transmittance of what it
// shades is zero: every weight further on is zero there, whatever the gradient of the picture is scaled by, and the picture stops there
// by itself.  (Not where it never stops, stop_thresh < 0: such a picture is composed to the end of its rays.)  Three things that the
// reference's gradient has of such leaves are not there, though passes without notes and rays whose notes found no room add them: the
// rounding that is left of `accum` in their density gradients, where the exact term is zero; a NaN that 0 * NaN makes of a coefficient
// that is none; and the end of a ray in a malformed tree, where it lies behind.  (Up to kQueue - 1 leaves behind the last that counts
// are still noted, those of its round: leaving them out, a comparison for every leaf, costs the step below 8 us.)
// The chain of a batch's longest rays is what such a pass waits for, and those that graze a surface are long because of what they pass
// through: 50 001 rays of a 256^3 SH9 shell with softplus, training step 342 -> 208 us.  A bound of 2^-126, below which a weight has
// lost digits, ends them hardly sooner (207 us), and leaves out terms that a large gradient of the picture makes count.
// Marches on two wavefronts are 1 % longer with SH9 and RGBA than before rays ended here (50 000 rays of a 256^3 SH9 shell 314.4 -> 317.9 us,
// dense 64^3 RGBA, 30 000 rays 187.3 -> 189.4), as long with SH1 and SH4, and 0.6 % shorter with SH16 -- though not for the look at the light:
// without it they measure the same.
__device__ __forceinline__ float opaque_light(const SvoxRenderOptions& opt, const float* out) {
    return opt.stop_thresh >= 0.0f || out == nullptr ? 0.0f : -1.0f;   // (light is never below zero)
}

// What a noting pass that has the gradient of the picture at hand accumulates per ray beside its notes:
// the sum the backward pass forms in its first march (rt_kernel.cu:358-419; the same expressions, in
// the same order, as march 1 of render_backward_kernel), so that a ray whose notes do not fit needs
// only the second march afterwards.
struct March1Sum {
    float go[3], light, accum;
    __device__ __forceinline__ void begin(const float* __restrict__ grad_out, int64_t slot) {
        go[0] = grad_out[slot * 3];
        go[1] = grad_out[slot * 3 + 1];
        go[2] = grad_out[slot * 3 + 2];
        light = 1.0f;
        accum = 0.0f;
    }
    // a leaf with sigma > 0 and the sigmoids s of its colour
    __device__ __forceinline__ void leaf(float dt, float sigma, float dscale, const float* s, float d_rgb_pad, float pad) {
        const float att = expf_fixed(-dt * sigma * dscale);
        const float weight = light * (1.0f - att);
        float total_color = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; ++c) total_color = fma_(fma_(s[c], d_rgb_pad, -pad), go[c], total_color);
        light *= att;
        accum = fma_(weight, total_color, accum);
    }
    __device__ __forceinline__ float end(float bg) const {
        const float total_grad = (go[0] + go[1]) + go[2];
        return fma_(light * bg, total_grad, accum);
    }
};

// trace_ray, octree flavour: a persistent wavefront working in rounds.
//
//   refill    lanes whose ray has ended take the next rays of the wavefront's range (ranked by
//             ballot among the idle lanes) once `refill_at` lanes are idle: rays differ wildly in
//             length, and a finished lane does not wait for the longest ray of the wavefront;
//   walk      kQueue turns; in a turn every live lane advances its ray by one leaf and remembers
//             (leaf, step length), or, if the descent needs more than kSeekBudget child reads,
//             goes on with it in its next turn.  The next position depends only on the tree, not
//             on the leaf's contents, so this phase waits for child-table reads only;
//   sigma     the densities of the remembered leaves are fetched together (kQueue loads in flight);
//   shade     the leaves with sigma > sigma_thresh of all lanes form one list, and the wavefront
//             evaluates their colours together (shade_entries), all 64 lanes busy whatever the
//             number of rays that hit something;
//   composite every lane folds its leaves, in order, into its colour and transmittance, stops at
//             stop_thresh and writes the pixel when the ray ends.
// A ray that stops early has walked at most kQueue - 1 leaves too far; the values are the same as
// when every leaf is shaded on the spot.
// kAccum: the compositing weight of every shaded leaf is also added to (or maximised into)
// tr.weight_accum at the leaf's cell index (rt_kernel.cu:298-304).
// kRefill: the wavefront owns more than 64 rays and refills idle lanes; without it the 64 rays are
// set up once before the loop, and nothing the set-up needs stays live inside it.
// kNoted: the forward pass of a training step.  The picture is composed as without it; beside it the
// launch leaves in the workspace the notes the backward pass works from (NoteTaker): every leaf with
// sigma > 0 up to where nothing shines through any more (opaque_light), so a ray is walked on after its
// picture stopped early, and the colours of the leaves at or below sigma_thresh are evaluated too.  With out == nullptr only the
// notes are taken (the backward pass without a forward pass before it); kGrad: that backward pass's
// grad_out is given, and the sum of its first march is formed on the way (March1Sum).  A pass that takes notes for
// replay_se_grad_kernel (not kGrad, stop_thresh 0) is given the reference colours in grad_out's place
// (NoteTaker::finish_residual).
// kAllShaded: tr.child is a marked copy of the child table made with this launch's sigma_thresh (and softplus
// setting): a leaf that is not marked has sigma > sigma_thresh, so the round has no density phase -- every
// unmarked leaf goes on the shade list and its density arrives with its coefficients (one round trip to memory
// per round instead of two that wait for one another).
// (Noting passes of up to 16 lobes: room for four wavefronts on a SIMD, which 132 registers leave no room for.)
template <class P, class Source, bool kAccum, bool kRefill, bool kNoted = false, bool kGrad = false,
          bool kAllShaded = false>
__global__ __launch_bounds__(kMarchThreads, kNoted && P::kForwardRows && P::kBasis <= 16 ? 4 : 1) void render_forward_kernel(TreeDev<float> tr, Source src,
                                                                       SvoxRenderOptions opt,
                                                                       float* __restrict__ out, ReplaySpace ws,
                                                                       const float* __restrict__ grad_out = nullptr) {
    static_assert(!kAllShaded || (!kNoted && !kAccum), "notes and weights look at leaves the marks may hide");
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    __shared__ MarchShared<D, P::kForwardRows> lds;
    auto& sh = lds.sh;
    __shared__ float sh_sigma[kAllShaded ? kQueue * kMarchThreads : 1];
    // Wavefronts that take new rays, with 16 functions: four to a SIMD, not the five that 94 registers leave room for.  A batch of 1 Mi rays is 4 096 of them, four to
    // a SIMD, and where five find room some SIMDs have five and others three: 1 Mi rays drawn from pictures of a 512^3 SH16 shell 395 us with room for five, 367 for
    // four.  (launch_bounds has a say in the least only.)
    if constexpr (kRefill && !kNoted && P::kFormat == SVOX_FORMAT_SH && P::kBasis == 16) asm volatile("" ::: "v103");
    if constexpr (kNoted) {
        if constexpr (Source::kGated) {
            if (!ws.chosen()) return;
        }
        if (blockIdx.x >= ws.march_blocks) return clear_share(ws);
    }
    const int lane = threadIdx.x;
    float offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    const float step = opt.step_size, sigma_thresh = opt.sigma_thresh, stop_thresh = opt.stop_thresh;
    const float opaque = opaque_light(opt, out);

    int64_t next = chunk_of_block(blockIdx.x, kNoted ? ws.march_blocks : gridDim.x, src.xcd_group) * (int64_t)src.per_wave;
    const int64_t total = src.total();
    const int64_t end = next + src.per_wave < total ? next + src.per_wave : total;

    if constexpr (kNoted) {
        if (blockIdx.x == 0 && lane < kStampWords) ws.stamp_at[lane] = ws.stamp[lane];
    }

    RayState<float> r;
    float acc[3] = {0.f, 0.f, 0.f};
    float light = 1.0f;
    int64_t slot = -1;
    bool active = false;
    bool painted = false;   // kNoted: the ray's picture is finished (early stop), its notes go on
    NoteTaker notes;
    March1Sum sum1;
    int64_t shared_next = 0, shared_end = 0;   // the wavefront's stock of chunks for notes (uniform)
    OctreeCursor cur;
    cur.reset(lds.lane_path(lane));
    ChildTable child(tr);

    // takes ray `item` into this lane: a miss is answered at once, a hit becomes the lane's ray
    auto start = [&](int64_t item) {
        float origin[3], dir[3], vdir[3];
        slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
        if (slot < 0) return;
        if (setup_ray(r, origin, dir, scaling)) {
            if constexpr (P::kFormat == SVOX_FORMAT_SH) {
                sh.vdir[lane * 3] = vdir[0];
                sh.vdir[lane * 3 + 1] = vdir[1];
                sh.vdir[lane * 3 + 2] = vdir[2];
            } else if constexpr (P::kForwardRows) {
                float basis[D];
                policy_basis<P>(Lobes{tr.extra, tr.extra_cols, opt.format}, opt, vdir, basis);
#pragma unroll
                for (int i = 0; i < D; ++i) sh.basis[lane * D + i] = basis[i];
            }
            acc[0] = acc[1] = acc[2] = 0.0f;
            light = 1.0f;
            if constexpr (kRefill) cur.begin(r);
            active = true;
            if constexpr (kNoted) {
                painted = out == nullptr;   // no picture asked for: nothing to compose
                notes.begin(ws, slot);
                if constexpr (kGrad) sum1.begin(grad_out, slot);
            }
        } else {
            if (!kNoted || out) {
                out[slot * 3] = bg;
                out[slot * 3 + 1] = bg;
                out[slot * 3 + 2] = bg;
            }
            if constexpr (kNoted) NoteTaker::missed(ws, slot);
        }
    };
    if constexpr (!kRefill) {
        if (next + lane < end) start(next + lane);
        child.settle(tr, r, active);
        if (active) cur.begin(r);
    }

    while (true) {
        if constexpr (kRefill) {
            const RoundState state = refill_lanes(active, next, end, src.refill_at, start);
            if (state == kRoundRefilled) continue;
            if (state == kRoundDone) break;
        } else {
            if (!any_lane(active)) break;
        }

        // ---- walk
        int32_t q_leaf[kQueue];
        float q_dt[kQueue];
        bool broken;
        walk_turns(tr, child, r, cur, step, active, broken, q_leaf, q_dt);
        // ---- sigma
        float q_sigma[kQueue], q_raw[kQueue];   // (q_raw: what the notes keep, the stored density)
        int n_entries;
        if constexpr (kAllShaded) {
            n_entries = build_shade_list_all(sh, q_leaf, lane);
        } else {
            fetch_sigma<K>(tr.data, q_leaf, q_sigma);
            soften_sigma(opt.density_softplus, q_leaf, q_sigma, q_raw);
            // ---- shade list
            n_entries = build_shade_list(sh, q_leaf, q_sigma, kNoted ? 0.0f : sigma_thresh, lane);
        }
        bool stopped = false;
        if (n_entries > 0) {   // most rounds of a ray pass through empty space: nothing to shade
            wave_lds_sync();   // list and view directions are visible to every lane
            shade_entries<P, P::kForwardRows, kAllShaded>(tr.data, sh, n_entries, lane, sh_sigma);
            wave_lds_sync();
            if constexpr (kAllShaded) {
#pragma unroll
                for (int q = 0; q < kQueue; ++q) {
                    const bool listed = (uint32_t)q_leaf[q] < (uint32_t)kEmptyLeafBit;
                    const float raw = sh_sigma[q * kMarchThreads + lane];
                    q_sigma[q] = listed ? (opt.density_softplus ? softplus_m1(raw) : raw) : 0.0f;
                }
            }
            // ---- composite
            // the attenuations and padded colours of the four slots do not depend on one another: they
            // are evaluated side by side, and only the products with the transmittance form a chain
            float q_att[kQueue], q_rgb[kQueue][3], q_s[kQueue][3];
#pragma unroll
            for (int q = 0; q < kQueue; ++q) {
                q_att[q] = expf_fixed(-q_dt[q] * r.dscale * q_sigma[q]);
                const float* s = sh.colour + (q * kMarchThreads + lane) * 3;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    q_s[q][c] = s[c];
                    q_rgb[q][c] = fma_(s[c], d_rgb_pad, -pad);
                }
            }
#pragma unroll
            for (int q = 0; q < kQueue; ++q) {
                // (the light of a ray whose picture is finished goes on: opaque_light)
                const bool shade = active && q_leaf[q] >= 0 && !stopped && q_sigma[q] > sigma_thresh;
                const bool take = shade && !painted;
                const float weight = light * (1.0f - q_att[q]);
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[c] = take ? fma_(weight, q_rgb[q][c], acc[c]) : acc[c];
                light = shade ? light * q_att[q] : light;
                if constexpr (kAccum) {
                    if (take) {
                        if (tr.weight_accum_max)
                            atomic_max_float(tr.weight_accum + q_leaf[q], weight);
                        else
                            atomicAdd(tr.weight_accum + q_leaf[q], weight);
                    }
                }
                stopped = stopped || (take && light <= stop_thresh);
                if constexpr (kNoted) {
                    const bool note = active && q_leaf[q] >= 0 && q_sigma[q] > 0.0f;
                    notes.take(ws, shared_next, shared_end, lane, note, q_leaf[q], q_dt[q], q_raw[q], q_s[q]);
                    if constexpr (kGrad) {
                        if (note) sum1.leaf(q_dt[q], q_sigma[q], r.dscale, q_s[q], d_rgb_pad, pad);
                    }
                }
            }
        }
        if (active) {
            if (stopped) {
                // rt_kernel.cu:306-313: rescale and leave without the background (done here, once
                // per round, with the transmittance the ray stopped at)
                const float scale = (float)(1.0 / (1.0 - (double)light));
                out[slot * 3] = acc[0] * scale;
                out[slot * 3 + 1] = acc[1] * scale;
                out[slot * 3 + 2] = acc[2] * scale;
                if constexpr (kNoted)
                    painted = true;   // the notes go on
                else
                    active = false;
            }
            if (active && (broken || !(r.t < r.tmax) || (kNoted && light <= opaque))) {
                if (kNoted && !kGrad && grad_out) {
                    notes.finish_residual(broken, r.dscale, acc, light, bg, grad_out + slot * 3, out + slot * 3);
                } else {
                    if (!painted) {
                        out[slot * 3] = fma_(light, bg, acc[0]);
                        out[slot * 3 + 1] = fma_(light, bg, acc[1]);
                        out[slot * 3 + 2] = fma_(light, bg, acc[2]);
                    }
                    if constexpr (kNoted) notes.finish(broken, r.dscale, kGrad ? sum1.end(bg) : 0.0f);
                }
                active = false;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// backward
// ------------------------------------------------------------------------------------------------
// trace_ray_backward, rt_kernel.cu:323-477, generic flavour: one ray per lane, the reference's two marches --
// <render, grad_out> and the colour gradient in the first, the density gradient in the second; both test
// sigma > 0 and never stop early.  The colour terms are the reference's products (basis[i] * tmp2) but are not
// scattered lane by lane: a lane whose sample has density leaves its factors (tmp2 per channel) and the offset of its
// leaf in LDS, the lanes of a step that did so are listed, and the wavefront adds the listed records flat -- scalar f
// of the list from lane f mod 64, so that consecutive scalars of a record go out together, one request per 64 bytes
// instead of one per scalar (the memory system takes atomic adds at a fixed rate of requests).  For that the lanes
// of a wavefront stay in the loop of the first march until the last of them is through.  The basis of a ray and its
// grad_out sit in LDS as well, where the runtime-indexed loops of the reference can address them (in registers such
// arrays end up in scratch memory).
// Dynamic LDS, in scalars of T per lane: basis_dim (1 for RGBA) made odd, so that the lanes' rows start in different
// banks, + 2 * out_dim, then 8 bytes (leaf offset) and 1 byte (list) per lane: generic_backward_lds_bytes.
template <typename T>
__host__ __device__ inline size_t generic_backward_lds_bytes(int basis_dim, int out_dim) {
    return (size_t)kMarchThreads * ((size_t)((basis_dim | 1) + 2 * out_dim) * sizeof(T) + sizeof(int64_t) + 1);
}

template <typename T, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_backward_generic_kernel(
    TreeDev<T> tr, Source src, SvoxRenderOptions opt, int out_dim, const T* __restrict__ grad_out,
    T* __restrict__ grad_data) {
    extern __shared__ __align__(16) unsigned char generic_lds[];
    const int lane = threadIdx.x;
    const bool rgba = opt.format == SVOX_FORMAT_RGBA;
    const int bd = (rgba ? 1 : opt.basis_dim) | 1;                          // row length, odd
    T* const sh_basis = (T*)generic_lds;                                    // [lane * bd + i]
    T* const sh_go = sh_basis + kMarchThreads * bd;                         // [c * 64 + lane]: grad_out of the ray
    T* const sh_factor = sh_go + kMarchThreads * out_dim;                   // [c * 64 + lane]: tmp2 of the sample
    int64_t* const sh_base = (int64_t*)(sh_factor + kMarchThreads * out_dim);   // [lane]: leaf * K
    uint8_t* const sh_list = (uint8_t*)(sh_base + kMarchThreads);           // lanes with a record in this step

    T offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    T origin[3], dir[3], vdir[3];
    const int64_t item = blockIdx.x * (int64_t)kMarchThreads + lane;
    const int64_t slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
    RayState<T> r;
    bool alive = slot >= 0 && setup_ray(r, origin, dir, scaling);
    if (alive) {
        if (!rgba) {
            T basis[SVOX_MAX_BASIS_DIM];
            precalc_basis<T>(opt.format, opt.basis_dim, tr.extra, tr.extra_cols, vdir, basis);
#pragma unroll
            for (int i = 0; i < SVOX_MAX_BASIS_DIM; ++i)
                if (i < opt.basis_dim) sh_basis[lane * bd + i] = basis[i];
        }
        for (int j = 0; j < out_dim; ++j) sh_go[j * kMarchThreads + lane] = grad_out[slot * out_dim + j];
    }
    wave_lds_sync();
    const T* const my_basis = sh_basis + lane * bd;
    const T pad = (T)opt.rgb_padding;
    const T d_rgb_pad = (T)(1 + 2 * opt.rgb_padding);
    const int lo = rgba ? 0 : opt.min_comp;
    const int n_comp = rgba ? 1 : (opt.max_comp - opt.min_comp + 1 > 0 ? opt.max_comp - opt.min_comp + 1 : 0);
    const int per_record = out_dim * n_comp;
    const T tmin = alive ? r.t : T(0);
    T accum = T(0);
    {
        T light = T(1);
        while (any_lane(alive && r.t < r.tmax)) {
            bool emit = false;
            if (alive && r.t < r.tmax) {
                T delta_t;
                const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
                if (v.leaf < 0) {
                    alive = false;   // a broken tree: the reference leaves the ray here, second march included
                } else {
                    const int64_t base = v.leaf * tr.K;
                    const T* val = tr.data + base;
                    T sigma = val[tr.K - 1];
                    if (opt.density_softplus) sigma = softplus_m1(sigma);
                    if (sigma > T(0)) {
                        const T att = exp_sp<T>(-delta_t * sigma * r.dscale);
                        const T weight = light * (T(1) - att);
                        T total_color = T(0);
                        for (int c = 0; c < out_dim; ++c) {
                            const T go_c = sh_go[c * kMarchThreads + lane];
                            T sg;
                            if (!rgba) {
                                const int off = c * opt.basis_dim;
                                T tmp = T(0);
                                for (int i = opt.min_comp; i <= opt.max_comp; ++i)
                                    tmp = fma_(my_basis[i], val[off + i], tmp);
                                sg = sigmoid_(tmp);
                                sh_factor[c * kMarchThreads + lane] =
                                    (T)((double)(weight * sg) * (1.0 - (double)sg) * (double)go_c * (double)d_rgb_pad);
                            } else {
                                sg = sigmoid_(val[c]);
                                sh_factor[c * kMarchThreads + lane] = weight * sg * (T(1) - sg) * go_c * d_rgb_pad;
                            }
                            total_color = fma_(fma_(sg, d_rgb_pad, -pad), go_c, total_color);
                        }
                        sh_base[lane] = base;
                        emit = per_record > 0;
                        light *= att;
                        accum = fma_(weight, total_color, accum);
                    }
                    advance(r, delta_t);
                }
            }
            // the records of this step, added by the whole wavefront
            const unsigned long long m = __ballot(emit);
            if (m != 0) {
                if (emit) sh_list[rank_in(m)] = (uint8_t)lane;
                wave_lds_sync();
                const int n_scalars = __popcll(m) * per_record;
                for (int f = lane; f < n_scalars; f += kMarchThreads) {
                    const int rec = f / per_record, e = f - rec * per_record;
                    const int c = e / n_comp, i = lo + (e - c * n_comp);
                    const int owner = sh_list[rec];
                    const T factor = sh_factor[c * kMarchThreads + owner];
                    if (rgba)
                        atomicAdd(grad_data + sh_base[owner] + c, factor);
                    else
                        atomicAdd(grad_data + sh_base[owner] + c * opt.basis_dim + i, sh_basis[owner * bd + i] * factor);
                }
                wave_lds_sync();
            }
        }
        if (alive) {
            T total_grad = T(0);
            for (int j = 0; j < out_dim; ++j) total_grad += sh_go[j * kMarchThreads + lane];
            accum = fma_(light * (T)opt.background_brightness, total_grad, accum);
        }
    }
    if (alive) {
        T light = T(1);
        r.t = tmin;
        while (r.t < r.tmax) {
            T delta_t;
            const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
            if (v.leaf < 0) break;
            const int64_t base = v.leaf * tr.K;
            const T* val = tr.data + base;
            T sigma = val[tr.K - 1];
            const T raw_sigma = sigma;
            if (opt.density_softplus) sigma = softplus_m1(sigma);
            if (sigma > T(0)) {
                const T att = exp_sp<T>(-delta_t * sigma * r.dscale);
                const T weight = light * (T(1) - att);
                T total_color = T(0);
                for (int c = 0; c < out_dim; ++c) {
                    const T go_c = sh_go[c * kMarchThreads + lane];
                    T sg;
                    if (!rgba) {
                        const int off = c * opt.basis_dim;
                        T tmp = T(0);
                        for (int i = opt.min_comp; i <= opt.max_comp; ++i) tmp = fma_(my_basis[i], val[off + i], tmp);
                        sg = sigmoid_(tmp);
                    } else {
                        sg = sigmoid_(val[c]);
                    }
                    total_color = fma_(fma_(sg, d_rgb_pad, -pad), go_c, total_color);
                }
                light *= att;
                accum = fma_(-weight, total_color, accum);
                const T chain = opt.density_softplus ? sigmoid_(raw_sigma - T(1)) : T(1);
                atomicAdd(grad_data + base + tr.K - 1, delta_t * r.dscale * fma_(total_color, light, -accum) * chain);
            }
            advance(r, delta_t);
        }
    }
}

// value of `v` in lane `k` (k uniform across the wavefront)
__device__ __forceinline__ float read_lane(float v, int k) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// trace_ray_backward, octree flavour: a persistent wavefront working in the forward kernel's rounds
// (refill, walk, sigma, shade, composite).
//
// A lane runs its ray twice.  March 1 accumulates <render, grad_out> and writes nothing.  March 2
// replays the ray and produces, per visited leaf with sigma > 0, the reference's gradient record:
// basis[i] * tmp2[c] for the colour coefficients and the density term.  The records are not
// scattered lane by lane: the records of a round are listed in LDS (RecordList) and added by the
// whole wavefront, and where several rays of the wavefront sit in the same leaf their records are
// summed first (group_by_leaf), so that the leaf receives one atomic per element instead of one per
// ray.  The per-term products are the reference's; only the order in which they are added up differs.
// Both marches test sigma > 0 and never stop early (rt_kernel.cu:377, 441).
//
// Gradient records of a round.  A record is the K-long vector (basis[i] * tmp2[c] for the colour
// coefficients, g_sigma last) of a lane, to be added at a leaf.  The records of the queue slots are
// collected in LDS -- in the shade list's storage, which is dead once the colours are evaluated --
// and added together.  The list is flushed when it is full and at the end of the round.  Two forms:
//   flat        the n * K scalars of the list, scalar f from lane f mod 64, so that every atomic
//               instruction covers 64 consecutive scalars whatever K is;
//   by record   the lanes tied to elements (add_records_by_leaf): the list is cut into 64 / K slices
//               of consecutive records and lane l serves element l % K of slice l / K (of every
//               record, in two or more steps, if K > 64).  Which element a lane serves never changes,
//               so an addition costs about half the instructions of running over the flat list; the
//               price is idle lanes where K does not divide 64.  Consecutive records of the same leaf
//               are summed in registers and added once.  term(rec, e, t) gives the NV values of
//               element e of record rec, emit(leaf, e, sum) adds them.
// Records longer than half a wavefront (K > 32: one record at a time either way) are added by
// RecordList::add_held in both forms: the by-record scheme with the values of a record handed round by
// readlane instead of read through LDS one after the other.
// Before either, group_by_leaf looks for leaves that several records of the list share; if enough do,
// the list is put in an order that brings the records of a leaf together and added by record.

// Scratch of group_by_leaf, in LDS that is dead while records are added.
struct GroupScratch {
    uint8_t table[256];              // hash of a leaf -> some record of the list with that hash
    uint8_t order[kMarchThreads];    // position in the grouped order -> record
    int32_t leaf[kMarchThreads];     // position in the grouped order -> its leaf
};
// The list is regrouped if at least one record in kMergeMinShare repeats the leaf of another one.
// Where rays do not share leaves (a shuffled training batch) looking for repeats is pure cost, so a
// wavefront that found too few looks again only kMergeRecheck flushes later; one that found enough
// looks at every flush (the look is small beside the regrouping it decides on).
constexpr int kMergeMinShare = 2;
constexpr int kMergeRecheck = 8;
struct MergeState {
    int skip = 0;   // flushes left before the next look (wavefront-uniform)
};

// n <= 64 records; record r's leaf is leaves[r] (visible to every lane).  Estimates how many records
// repeat the leaf of another record: every record writes its number at its leaf's hash, reads the
// number that stayed there and compares leaves (a record that reads its own number repeats nothing it
// can see; two leaves with one hash hide each other's repeats, which only makes the estimate low).
// If they are too few, returns false.  Otherwise fills gs.order / gs.leaf with the records grouped by
// leaf (groups in the order of their first record, records of a group in list order) and returns true.
__device__ __forceinline__ bool group_by_leaf(GroupScratch& gs, MergeState& state, const int32_t* leaves, int n,
                                              int lane) {
    if (state.skip > 0) {
        state.skip -= 1;
        return false;
    }
    const bool mine = lane < n;
    const int32_t leaf = mine ? leaves[lane] : -1;
    const unsigned h = ((uint32_t)leaf * 2654435761u) >> 24;
    if (mine) gs.table[h] = (uint8_t)lane;
    wave_lds_sync();
    bool repeat = false;
    if (mine) {
        const int j = gs.table[h];
        repeat = j != lane && leaves[j] == leaf;
    }
    if (__popcll(__ballot(repeat)) * kMergeMinShare < n) {
        state.skip = kMergeRecheck;
        return false;
    }
    unsigned long long todo = __ballot(mine);
    int base = 0, pos = 0;
    while (todo) {
        const int lead = __builtin_ctzll(todo);
        const int32_t l = __builtin_amdgcn_readlane(leaf, lead);
        const unsigned long long same = __ballot(mine && leaf == l);
        if ((same >> lane) & 1ull) pos = base + rank_in(same);
        base += __popcll(same);
        todo &= ~same;
    }
    if (mine) {
        gs.order[pos] = (uint8_t)lane;
        gs.leaf[pos] = leaf;
    }
    wave_lds_sync();
    return true;
}

template <int K, int NV, class Term, class Emit>
__device__ __forceinline__ void add_records_by_leaf(int n, int lane, const int32_t* leaves, Term&& term,
                                                    Emit&& emit) {
    constexpr int kPer = K <= kMarchThreads ? kMarchThreads / K : 1;
    const int r = K <= kMarchThreads ? lane / K : 0;
    if (r >= kPer) return;
    const int per = (n + kPer - 1) / kPer;
    const int lo = r * per;
    const int hi = lo + per < n ? lo + per : n;
    for (int e = K <= kMarchThreads ? lane - r * K : lane; e < K; e += kMarchThreads) {
        int32_t cur = -1;
        float acc[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = 0.0f;
        for (int rec = lo; rec < hi; ++rec) {
            const int32_t leaf = leaves[rec];
            if (leaf != cur) {
                if (cur >= 0) emit(cur, e, acc);
                cur = leaf;
#pragma unroll
                for (int v = 0; v < NV; ++v) acc[v] = 0.0f;
            }
            float t[NV];
            term(rec, e, t);
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] += t[v];
        }
        if (cur >= 0) emit(cur, e, acc);
    }
}

// One record per lane of a wavefront: a step in which all 64 lanes emit fills the list once.  Leaves,
// density terms and colour factors (20 bytes a record) fill ShadeShared::leaf and ::who exactly; the
// owners follow the GroupScratch in ShadeShared::colour.
constexpr int kEmitCap = kMarchThreads;
// (kByRecord: the replay kernel's list, in ReplayShared.)
constexpr int kReplayRows = 32;   // rays of a batch at most (more would cost wavefronts per CU in LDS)
template <int D>
struct ReplayShared {
    int32_t leaf[kEmitCap];
    float factor[kEmitCap * 4];
    uint8_t owner[kEmitCap];
    uint8_t start[kMarchThreads];    // ReplayRays::take
    GroupScratch group;
    float basis[kReplayRows * D];
};
template <class P, int D, bool kByRecord = false>
struct RecordList {
    static constexpr int K = P::kRecord;
    std::conditional_t<kByRecord, ReplayShared<D>, ShadeShared<D, true>>& sh;
    float* grad_data;
    int lane;
    MergeState& merge;
    int n = 0;   // wavefront-uniform

    __device__ __forceinline__ int32_t* leaves() const { return sh.leaf; }
    // per record four factors: the three colour factors tmp2[c], then the density term
    __device__ __forceinline__ float* factors() const {
        if constexpr (kByRecord)
            return sh.factor;
        else
            return (float*)(sh.leaf + kEmitCap);
    }
    __device__ __forceinline__ uint8_t* owners() const {
        if constexpr (kByRecord)
            return sh.owner;
        else
            return (uint8_t*)sh.colour + sizeof(GroupScratch);
    }

    // element e of record rec: basis[i] * tmp2[c] for a colour coefficient, g_sigma for the density
    __device__ __forceinline__ float element(int rec, int e) const {
        const int c = P::kFormat == SVOX_FORMAT_RGBA ? e : e / D;
        if (c < 3) {
            const float v = factors()[rec * 4 + c];
            return P::kFormat == SVOX_FORMAT_RGBA ? v : sh.basis[owners()[rec] * D + (e - c * D)] * v;
        }
        return factors()[rec * 4 + 3];
    }

    // The colours of the round are in registers by the time records are added: their LDS is free.
    __device__ __forceinline__ GroupScratch& scratch() const {
        if constexpr (kByRecord)
            return sh.group;
        else
            return *(GroupScratch*)sh.colour;
    }

    // add_records_by_leaf for records longer than half a wavefront (one record at a time, lane e on
    // element e).  What the lanes need to find a record's values -- its place in the list, its leaf,
    // its owner -- is first taken into registers, record r by lane r, and then handed round by
    // readlane: per record that leaves two LDS reads (the factor of the lane's channel, the owner's
    // basis value) whose addresses come from scalars, so the reads of kHeldBlock records are in flight
    // together.  (Through LDS alone a record costs three reads that wait for one another: place, owner,
    // basis.)  order: the records' adding order (grouped by leaf), or nullptr for the list's own.
    static constexpr bool kHeld = K > kMarchThreads / 2;
    static constexpr int kHeldBlock = 4;
    __device__ __forceinline__ void add_held(const uint8_t* order) {
        const bool mine = lane < n;
        const int rec = mine ? (order ? order[lane] : lane) : 0;
        const int my_rec = rec;
        const int my_leaf = leaves()[rec];
        const int my_owner = owners()[rec];
        // readlane looks into other lanes, so every lane must hold its record and must stay in step with the
        // others: the loop below is one every lane runs (its trip count depends on K alone), and a lane whose
        // element lies beyond the record only leaves out the additions.
        for (int e0 = 0; e0 < K; e0 += kMarchThreads) {
            const int e = e0 + lane;
            const bool on = e < K;
            const int c_raw = P::kFormat == SVOX_FORMAT_RGBA ? e : e / D;
            const int c = c_raw < 3 ? c_raw : 3;                              // (3: the density element, and lanes that are not `on`)
            const int i = P::kFormat == SVOX_FORMAT_RGBA || c == 3 ? 0 : e - c * D;
            const bool with_basis = P::kFormat != SVOX_FORMAT_RGBA && c < 3;
            int32_t cur = -1;
            float acc = 0.0f;
            for (int at = 0; at < n; at += kHeldBlock) {
                int32_t leaf[kHeldBlock];
                float val[kHeldBlock], leaf_basis[kHeldBlock];
#pragma unroll
                for (int u = 0; u < kHeldBlock; ++u) {
                    const int a = at + u < n ? at + u : n - 1;   // (past the end: the last record again, unused)
                    leaf[u] = __builtin_amdgcn_readlane(my_leaf, a);
                    const int owner = __builtin_amdgcn_readlane(my_owner, a);
                    const float t = factors()[__builtin_amdgcn_readlane(my_rec, a) * 4 + c];
                    // (every lane reads, also the lane of the density element, whose i is 0: a read under a
                    // condition would be waited for on the spot)
                    float basis_value = 1.0f;
                    if constexpr (P::kFormat != SVOX_FORMAT_RGBA) basis_value = sh.basis[owner * D + i];
                    leaf_basis[u] = basis_value;
                    val[u] = t;
                }
#pragma unroll
                for (int u = 0; u < kHeldBlock; ++u) val[u] = with_basis ? leaf_basis[u] * val[u] : val[u];
#pragma unroll
                for (int u = 0; u < kHeldBlock; ++u) {
                    if (at + u < n) {
                        if (leaf[u] != cur) {
                            if (on && cur >= 0) atomicAdd(grad_data + (int64_t)cur * K + e, acc);
                            cur = leaf[u];
                            acc = 0.0f;
                        }
                        acc += val[u];
                    }
                }
            }
            if (on && cur >= 0) atomicAdd(grad_data + (int64_t)cur * K + e, acc);
        }
    }

    // Adds the list with the records of every leaf summed first, if enough records share a leaf.
    __device__ __forceinline__ bool flush_grouped() {
        GroupScratch& gs = scratch();
        if (!group_by_leaf(gs, merge, leaves(), n, lane)) return false;
        if constexpr (kHeld) {
            add_held(gs.order);
        } else {
            add_records_by_leaf<K, 1>(
                n, lane, gs.leaf, [&](int at, int e, float* t) { t[0] = element(gs.order[at], e); },
                [&](int32_t leaf, int e, const float* sum) { atomicAdd(grad_data + (int64_t)leaf * K + e, sum[0]); });
        }
        wave_lds_sync();
        n = 0;
        return true;
    }

    __device__ __forceinline__ void flush() {
        if constexpr (kByRecord) {
            flush_by_record();
            return;
        }
        if (n == 0) return;
        wave_lds_sync();
        if (flush_grouped()) return;
        if constexpr (kHeld) {
            // long records: one at a time with its values handed round by readlane (measured on the
            // marching backward of an 800x800 image: 2.55 -> 2.38 ms, with a workspace 2.07 -> 1.80 ms;
            // for records of up to 32 scalars the flat form below is as fast)
            add_held(nullptr);
            wave_lds_sync();
            n = 0;
            return;
        }
        const int total = n * K;
        for (int f = lane; f < total; f += kMarchThreads) {
            const int rec = f / K, e = f - rec * K;
            float val;
            if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
                val = factors()[rec * 4 + e];
            } else {
                if (e < 3 * D) {
                    const int c = e / D;
                    val = sh.basis[owners()[rec] * D + (e - c * D)] * factors()[rec * 4 + c];
                } else {
                    val = factors()[rec * 4 + 3];
                }
            }
            atomicAdd(grad_data + (int64_t)leaves()[rec] * K + e, val);
        }
        wave_lds_sync();
        n = 0;
    }

    // The same additions by add_records_by_leaf.  (Measured: 12 % off replay_backward_kernel, whose
    // time is mostly these additions; nothing for render_backward_kernel.)
    __device__ __forceinline__ void flush_by_record() {
        if (n == 0) return;
        wave_lds_sync();
        if (flush_grouped()) return;
        if constexpr (kHeld) {
            add_held(nullptr);
        } else {
            add_records_by_leaf<K, 1>(
                n, lane, leaves(), [&](int rec, int e, float* t) { t[0] = element(rec, e); },
                [&](int32_t leaf, int e, const float* sum) { atomicAdd(grad_data + (int64_t)leaf * K + e, sum[0]); });
        }
        wave_lds_sync();
        n = 0;
    }

    // the record of every lane with `emit` set joins the list (in lane order)
    __device__ __forceinline__ void append(bool emit, int32_t leaf, const float* tmp2, float g_sigma) {
        unsigned long long todo = __ballot(emit);
        while (todo) {
            if (n == kEmitCap) flush();
            const bool pending = (todo >> lane) & 1ull;
            const int slot = n + rank_in(todo);
            const bool take = pending && slot < kEmitCap;
            if (take) {
                leaves()[slot] = leaf;
                owners()[slot] = (uint8_t)lane;
                factors()[slot * 4] = tmp2[0];
                factors()[slot * 4 + 1] = tmp2[1];
                factors()[slot * 4 + 2] = tmp2[2];
                factors()[slot * 4 + 3] = g_sigma;
            }
            const unsigned long long taken = __ballot(take);
            n += __popcll(taken);
            todo &= ~taken;
        }
    }
};
static_assert(5 * kEmitCap * 4 <= kQueue * kMarchThreads * 5, "record list exceeds the shade list");
static_assert(kEmitCap <= kMarchThreads, "group_by_leaf holds one record per lane");
static_assert(sizeof(GroupScratch) + kEmitCap <= sizeof(float) * kQueue * kMarchThreads * 3,
              "GroupScratch and the owners live in ShadeShared::colour");
using ShadeSharedProbe = ShadeShared<1, true>;
static_assert(offsetof(ShadeSharedProbe, who) - offsetof(ShadeSharedProbe, leaf) == sizeof(int32_t) * kQueue * kMarchThreads,
              "the record list runs from ShadeShared::leaf into ShadeShared::who");


// ------------------------------------------------------------------------------------------------
// forward, walk and shading on two wavefronts
// ------------------------------------------------------------------------------------------------
// The round of render_forward_kernel is one chain per wavefront: four turns of the walk (child reads
// that hit in L2), then the densities and the records of the leaves found (reads that go to HBM), then
// the colours, then the next walk.  The walk does not depend on what the leaves hold, but a
// wavefront's loads come back in the order they were issued, so within one wavefront the next walk
// cannot run while the records are on their way.  Here a block is two wavefronts that share the 64
// rays of a tile: the first only walks and hands every leaf it finds (that is not marked empty) to
// the second through a ring in LDS, a few leaves per lane deep; the second takes the leaves as they
// come, fetches densities and records, evaluates colours and composites exactly as
// render_forward_kernel does, and tells the walk which rays have stopped.  Same arithmetic, same
// pictures.  Each wavefront sets the rays up for itself (the same instructions give the same rays).
// A wavefront that finds nothing to do sleeps a few cycles and looks again; after kSpinLimit looks in a
// row it gives up, so that a launch ends whatever happens.
//
// kNoted: as in render_forward_kernel, the launch also leaves the notes of every ray for the backward
// pass: every leaf with sigma > 0 up to where nothing shines through any more, so the walk goes on after the picture's early stop,
// and the colours of leaves below sigma_thresh are evaluated too; the picture itself is composed as
// without notes.
constexpr int kSplitThreads = 2 * kMarchThreads;
constexpr int64_t kBeyondL2 = 131072;  // nodes of whose child rows an L2 cache has room for
constexpr int kWalkTurns = 4;          // of the walk, between looks at the rays that have ended
constexpr int kRing = 8;               // leaves a lane's walk may be ahead of its shading (a power of two)
constexpr int kSpinLimit = 1 << 22;
constexpr int32_t kEndedBit = 1 << 30;   // in SplitBox::taken: the ray wants no more leaves

// A place of the ring is one 64-bit word that carries everything the walk hands over: the leaf in bits 0 to 29, the round
// of the ring it was written in (its parity, counted from 1) in bit 30, and the step length in the upper half.  With bit 31
// set there is no leaf: the walk of the ray is over, with bit 0 because the tree is malformed.  The shading sees from the
// parity whether a place has been written since it last took it, so the walk publishes a leaf with a single store and waits
// for nothing (a count beside the ring, released after the entries it covers: 800x800 picture 343 instead of 331 us,
// 50 001 rays with notes 241 instead of 225).
constexpr uint32_t kRoundBit = 1u << 30, kOverBit = 1u << 31;
struct SplitBox {
    unsigned long long place[kRing * kMarchThreads];   // [place in the ring][lane]
    int32_t path[(kPathLevels + 2) * kMarchThreads];   // of the walk (OctreeCursor); its two dump rows are also the ring's, for what is no leaf
    int32_t taken[kMarchThreads];                      // set by the shading: places taken so far (| kEndedBit)
};
static_assert(offsetof(SplitBox, path) == sizeof(unsigned long long) * kRing * kMarchThreads, "a row of places behind the ring is two of the path");
__device__ __forceinline__ uint32_t ring_round(int32_t n) { return ((uint32_t)n / kRing & 1u) ? kRoundBit : 0u; }

// Places and counts are read and written as atomics of the workgroup (unlike a volatile access, which the compiler leaves on
// the generic address path -- a flat instruction with a wait for every store --, it still knows that they live in LDS and
// issues plain LDS reads and writes).  A count is published with release order, after the places it covers were read; the
// walk writes to a place only if the count it has read says so, and nothing the store depends on can come after it.
__device__ __forceinline__ unsigned long long ring_read(const unsigned long long* at) {
    return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void ring_write(unsigned long long* at, uint32_t code, float dt) {
    __hip_atomic_store(at, (unsigned long long)__float_as_uint(dt) << 32 | code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int32_t taken_read(const int32_t* at) {
    return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void taken_write(int32_t* at, int32_t value) {
    __hip_atomic_store(at, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// (The density phase stays also where the marks of a launch say that every leaf they let through is shaded,
// render_forward_kernel's kAllShaded: here the walk is the critical path, and the density read of a leaf brings the
// last line of its record into L2 ahead of the coefficient reads.)
template <class P, class Source, bool kNoted = false, bool kGrad = false>
__global__ __launch_bounds__(kSplitThreads) void render_forward_split_kernel(TreeDev<float> tr, Source src,
                                                                             SvoxRenderOptions opt,
                                                                             float* __restrict__ out, ReplaySpace ws,
                                                                             const float* __restrict__ grad_out = nullptr) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    __shared__ ShadeShared<D, P::kForwardRows> sh;
    __shared__ SplitBox box;
    if constexpr (kNoted) {
        if constexpr (Source::kGated) {
            if (!ws.chosen()) return;
        }
        if (blockIdx.x >= ws.march_blocks) return clear_share(ws);
        if (blockIdx.x == 0 && threadIdx.x < kStampWords) ws.stamp_at[threadIdx.x] = ws.stamp[threadIdx.x];
    }
    const int lane = threadIdx.x & (kMarchThreads - 1);
    const bool walks = threadIdx.x < kMarchThreads;   // uniform in a wavefront
    float offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    const float step = opt.step_size, sigma_thresh = opt.sigma_thresh, stop_thresh = opt.stop_thresh;
    const float opaque = opaque_light(opt, out);
    const int spin_limit = ws.spin_limit > 0 ? ws.spin_limit : kSpinLimit;

    const int64_t item = chunk_of_block(blockIdx.x, kNoted ? ws.march_blocks : gridDim.x, src.xcd_group) * (int64_t)kMarchThreads + lane;
    RayState<float> r;
    int64_t slot = -1;
    bool active = false;
    {
        float origin[3], dir[3], vdir[3];
        if (item < src.total()) slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
        if (slot >= 0) active = setup_ray(r, origin, dir, scaling);
        if (!walks) {
            if (slot >= 0 && !active) {
                if (!kNoted || out) {
                    out[slot * 3] = bg;
                    out[slot * 3 + 1] = bg;
                    out[slot * 3 + 2] = bg;
                }
                if constexpr (kNoted) NoteTaker::missed(ws, slot);
            }
            if constexpr (P::kFormat == SVOX_FORMAT_SH) {
                if (active) {
                    sh.vdir[lane * 3] = vdir[0];
                    sh.vdir[lane * 3 + 1] = vdir[1];
                    sh.vdir[lane * 3 + 2] = vdir[2];
                }
            } else if constexpr (P::kForwardRows) {
                if (active) {
                    float basis[D];
                    policy_basis<P>(Lobes{tr.extra, tr.extra_cols, opt.format}, opt, vdir, basis);
#pragma unroll
                    for (int i = 0; i < D; ++i) sh.basis[lane * D + i] = basis[i];
                }
            }
        }
    }
    if (!any_lane(active)) return;   // (both wavefronts see the same rays: both leave or both stay)
    if (walks) {
#pragma unroll
        for (int i = 0; i < kRing; ++i) box.place[i * kMarchThreads + lane] = kRoundBit;   // (not the first round)
    } else {
        box.taken[lane] = active ? 0 : kEndedBit;
    }
    __syncthreads();

    if (walks) {
        // ---- the walk: one leaf per live lane and turn, into the ring
        OctreeCursor cur;
        cur.reset(box.path + lane);
        ChildTable child(tr);
        child.settle(tr, r, active);
        if (active) cur.begin(r);
        // (counts of places in bytes of the ring)
        constexpr uint32_t kPlace = kMarchThreads * 8, kPlaces = kRing * kPlace;
        uint32_t written = 0, taken = 0;
        bool live = active, broken = false;
        int spins = 0;
        if (!active) r.t = r.tmax = 0.0f;
        auto room = [&]() { return written - taken < kPlaces; };
        auto hand_over = [&](bool found, uint32_t code, float dt) {
            // (a lane without one writes to the row behind the ring)
            unsigned char* const at = (unsigned char*)&box + lane * 8 + (found ? written & (kPlaces - 1) : kPlaces);
            ring_write((unsigned long long*)at, code | (written << 18 & kRoundBit), dt);
            written += found ? kPlace : 0u;
        };
        static_assert(kPlaces << 18 == kRoundBit, "the bit of a count that says which round it is");
        // The walk is the longest chain of a tile: it goes first where wavefronts share a SIMD, on trees whose child rows lie beyond L2 for all batches, on others
        // for batches of up to 147 000 rays without notes, in normalised device coordinates, and on trees of other branching factors, whose walk is the reference's.  Where many tiles run, rays of a picture or notes to write, it keeps the shading from its
        // turns, and every ring is full.  (us, walk first / as they come.  Batches, 100 000 rays: 128^3 shell SH9 165 / 174, 18 % hit 118 / 127, 32^3 SH9 94 / 101,
        // 190 000: 128^3 shell RGBA 264 / 215, SH9 266 / 259, 150 000: 512^3 shell SH9 403 / 425, 222 / 245; with notes, the gradient, 100 000: 128^3 shell SH9
        // 201 / 188, 150 000: 512^3 368 / 384.  Pictures of 800x800: 512^3 SH16 354 / 350, 64^3 RGBA from close up 424 / 352, 128^3 shell SH9 432 / 346, eight of 400x400 416 / 351.
        // Pictures in normalised device coordinates, all of whose tiles are long, 504x378: blobs 128^3 SH16 93 / 98, 256^3 114 / 127, SH4 of 512^3 167 / 179, SH25 290 / 285.  N = 3, 81^3 SH9,
        // 800x800 193 / 215, four of 400x400 298 / 370, training step of 60 000 rays 894 / 919.)
        if (opt.ndc_width > 0 || !child.octree || (Source::kItemsAreSlots && (tr.capacity >= kBeyondL2 || (!kNoted && gridDim.x <= 2304u)))) __builtin_amdgcn_s_setprio(3);
        while (true) {
            // asked for here, looked at after the turns: not waited for.  (Four turns to a look: one wavefront alone 620 ns a leaf, with two turns and
            // looks at the rays that are over 770, with a look at everything in every turn 870.)
            const int32_t taken_next = taken_read(&box.taken[lane]);
            if (child.words) {
#pragma unroll
                for (int k = 0; k < kWalkTurns; ++k) {
                    int32_t leaf = -1;
                    float dt = 0.0f;
                    cur.turn_words(r, (r.t < r.tmax) & room(), child, step, leaf, dt);
                    hand_over((uint32_t)leaf < (uint32_t)kEmptyLeafBit, (uint32_t)leaf, dt);
                }
            } else if (child.octree) {
#pragma unroll
                for (int k = 0; k < kWalkTurns; ++k) {
                    int32_t leaf = -1;
                    float dt = 0.0f;
                    cur.turn(r, (r.t < r.tmax) & room(), child, step, leaf, dt);
                    hand_over((uint32_t)leaf < (uint32_t)kEmptyLeafBit, (uint32_t)leaf, dt);
                }
            }
            taken = (uint32_t)(taken_next & ~kEndedBit) * kPlace;
            if (taken_next & kEndedBit) {
                live = false;
                r.tmax = r.t;
            }
            const bool go = (r.t < r.tmax) & room(), deep = go & (cur.up < 0 || !child.octree);
            if (__builtin_expect(any_lane(deep), 0)) {
                int32_t leaf = -1;
                float dt = 0.0f;
                walk_from_root(tr, r, cur, step, deep, broken, leaf, dt);
                if (broken) r.tmax = r.t;
                hand_over((uint32_t)leaf < (uint32_t)kEmptyLeafBit, (uint32_t)leaf, dt);
            }
            spins += 1;
            if (any_lane(go)) {
                spins = 0;
                continue;
            }
            // nobody can go on: the rays that are over say so, once, and where every ring is full the shading is behind
            const bool over = live & !(r.t < r.tmax) & room();
            hand_over(over, kOverBit | (broken ? 1u : 0u), 0.0f);
            live = live & !over;
            if (!any_lane(live)) break;
            if (spins > spin_limit) {
                if (lane == 0) atomicAdd(ws.give_ups, 1u);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        return;
    }

    // ---- the shading: takes up to kQueue leaves per lane at a time, as render_forward_kernel's round
    float acc[3] = {0.f, 0.f, 0.f};
    float light = 1.0f;
    int32_t taken = 0;
    int spins = 0;
    // kNoted: the picture of a ray may be finished (early stop) while its notes go on; without `out`
    // there is no picture to compose
    bool painted = kNoted && out == nullptr;
    NoteTaker notes;
    March1Sum sum1;
    int64_t shared_next = 0, shared_end = 0;   // the wavefront's stock of chunks for notes (uniform)
    if constexpr (kNoted) notes.begin(ws, active ? slot : 0);
    if constexpr (kNoted && kGrad) sum1.begin(grad_out, active ? slot : 0);
    while (true) {
        // the next places of the lane's ring, as far as the walk has written them
        unsigned long long place[kQueue];
#pragma unroll
        for (int q = 0; q < kQueue; ++q) place[q] = ring_read(&box.place[((taken + q) & (kRing - 1)) * kMarchThreads + lane]);
        int n_take = 0;
        const bool ended = kNoted && light <= opaque;   // nothing behind the leaves seen so far counts any more
        bool run = active && !ended;
#pragma unroll
        for (int q = 0; q < kQueue; ++q) {
            const uint32_t code = (uint32_t)place[q];
            run = run && (code & kRoundBit) == ring_round(taken + q) && !(code & kOverBit);
            n_take += run ? 1 : 0;
        }
        const uint32_t next = (uint32_t)place[0];
        const bool over = (next & kOverBit) && (next & kRoundBit) == ring_round(taken);
        if (active && (over || ended)) {
            // the ray left the tree: the background shows through what is left of the light
            if (kNoted && !over) taken_write(&box.taken[lane], taken | kEndedBit);   // (or the walk may stop)
            const bool broken = over && (next & 1u) != 0;
            if (kNoted && !kGrad && grad_out) {
                notes.finish_residual(broken, r.dscale, acc, light, bg, grad_out + slot * 3, out + slot * 3);
            } else {
                if (!painted) {
                    out[slot * 3] = fma_(light, bg, acc[0]);
                    out[slot * 3 + 1] = fma_(light, bg, acc[1]);
                    out[slot * 3 + 2] = fma_(light, bg, acc[2]);
                }
                if constexpr (kNoted) notes.finish(broken, r.dscale, kGrad ? sum1.end(bg) : 0.0f);
            }
            active = false;
        }
        if (!any_lane(active)) break;
        // (waiting for fuller hands -- two or four leaves per lane, a few looks of patience -- and a ring
        // of 16 were measured: no gain, the larger ring costs LDS)
        if (!any_lane(n_take > 0)) {   // the walk has found nothing new yet
            if (++spins > spin_limit) {
                // Cannot happen while the walk runs.  If it ever does, nothing plausible is left behind: the pixel
                // is NaN, the ray's notes say "march me" (the backward pass then does, twice), and the library's
                // give-up counter tells the host (svox_give_up_count).
                if (active && out && !painted)
                    out[slot * 3] = out[slot * 3 + 1] = out[slot * 3 + 2] = __int_as_float(0x7fc00000);
                if constexpr (kNoted) {
                    if (active) notes.give_up(r.dscale);
                }
                if (lane == 0) atomicAdd(ws.give_ups, 1u);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        spins = 0;
        int32_t q_leaf[kQueue];
        float q_dt[kQueue];
#pragma unroll
        for (int q = 0; q < kQueue; ++q) {
            q_leaf[q] = q < n_take ? (int32_t)((uint32_t)place[q] & (kRoundBit - 1u)) : -1;
            q_dt[q] = q < n_take ? __uint_as_float((uint32_t)(place[q] >> 32)) : 0.0f;
        }
        taken += n_take;
        if (n_take > 0) taken_write(&box.taken[lane], taken);
        float q_sigma[kQueue], q_raw[kQueue];
        fetch_sigma<K>(tr.data, q_leaf, q_sigma);
        soften_sigma(opt.density_softplus, q_leaf, q_sigma, q_raw);
        const int n_entries = build_shade_list(sh, q_leaf, q_sigma, kNoted ? 0.0f : sigma_thresh, lane);
        bool stopped = false;
        if (n_entries > 0) {
            wave_lds_sync();
            shade_entries<P, P::kForwardRows>(tr.data, sh, n_entries, lane);
            wave_lds_sync();
            float q_att[kQueue], q_rgb[kQueue][3], q_s[kQueue][3];
#pragma unroll
            for (int q = 0; q < kQueue; ++q) {
                q_att[q] = expf_fixed(-q_dt[q] * r.dscale * q_sigma[q]);
                const float* s = sh.colour + (q * kMarchThreads + lane) * 3;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    q_s[q][c] = s[c];
                    q_rgb[q][c] = fma_(s[c], d_rgb_pad, -pad);
                }
            }
#pragma unroll
            for (int q = 0; q < kQueue; ++q) {
                // (the light of a ray whose picture is finished goes on: opaque_light)
                const bool shade = active && q_leaf[q] >= 0 && !stopped && q_sigma[q] > sigma_thresh;
                const bool take = shade && !painted;
                const float weight = light * (1.0f - q_att[q]);
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[c] = take ? fma_(weight, q_rgb[q][c], acc[c]) : acc[c];
                light = shade ? light * q_att[q] : light;
                stopped = stopped || (take && light <= stop_thresh);
                if constexpr (kNoted) {
                    const bool note = active && q_leaf[q] >= 0 && q_sigma[q] > 0.0f;
                    notes.take(ws, shared_next, shared_end, lane, note, q_leaf[q], q_dt[q], q_raw[q], q_s[q]);
                    if constexpr (kGrad) {
                        if (note) sum1.leaf(q_dt[q], q_sigma[q], r.dscale, q_s[q], d_rgb_pad, pad);
                    }
                }
            }
            wave_lds_sync();   // the colours are read before the next list overwrites them
        }
        if (active && stopped) {
            // rt_kernel.cu:306-313: rescale and leave without the background; the walk may stop
            const float scale = (float)(1.0 / (1.0 - (double)light));
            out[slot * 3] = acc[0] * scale;
            out[slot * 3 + 1] = acc[1] * scale;
            out[slot * 3 + 2] = acc[2] * scale;
            if constexpr (kNoted) {
                painted = true;   // the picture is done; the notes go on
            } else {
                active = false;
                taken_write(&box.taken[lane], taken | kEndedBit);
            }
        }
    }
}

// kMode: kBackwardPlain runs both marches; kBackwardSecond runs only the second, for rays whose first
// march a noting forward kernel has already made (with grad_out at hand: NoteTaker keeps the sum of
// march 1 in the head of the ray's notes) but whose notes did not fit the workspace.
// (RGBA: room for five wavefronts on a SIMD, which is two registers fewer than the compiler takes by itself: 285 000 rays that all hit a 128^3 shell, without notes,
// 847 -> 697 us, a 64^3 grid 1 231 -> 1 008.  Lobes: for four.)
template <class P, class Source, bool kRefill, int kMode>
__global__ __launch_bounds__(kMarchThreads, P::kFormat == SVOX_FORMAT_RGBA ? 5 : P::kForwardRows && P::kBasis <= 16 ? 4 : 1) void render_backward_kernel(TreeDev<float> tr, Source src,
                                                                        SvoxRenderOptions opt,
                                                                        const float* __restrict__ grad_out,
                                                                        float* __restrict__ grad_data,
                                                                        ReplaySpace ws) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    __shared__ MarchShared<D, true> lds;
    auto& sh = lds.sh;
    if (ws.only && *ws.any_undone == 0) return;
    const int lane = threadIdx.x;
    float offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    const float step = opt.step_size;

    int64_t next = chunk_of_block(blockIdx.x, gridDim.x, src.xcd_group) * (int64_t)src.per_wave;
    const int64_t total = src.total();
    const int64_t end = next + src.per_wave < total ? next + src.per_wave : total;

    enum { kMarch1 = 0, kMarch2 = 1 };
    RayState<float> r;
    float go[3] = {0.f, 0.f, 0.f};
    float light = 1.0f, accum = 0.0f, tmin = 0.0f;
    bool active = false;
    int phase = kMarch1;
    MergeState merge;
    OctreeCursor cur;
    cur.reset(lds.lane_path(lane));
    const ChildTable child(tr);

    // takes ray `item` into this lane if it hits the tree
    auto start = [&](int64_t item) {
        float origin[3], dir[3], vdir[3];
        // (with a bitmap a batch launch does not deal its rays out: its items are ray numbers)
        if (Source::kItemsAreSlots && ws.only && !((ws.only[item >> 6] >> (item & 63)) & 1ull)) return;
        const int64_t slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
        if (!Source::kItemsAreSlots && ws.only && slot >= 0 && !((ws.only[slot >> 6] >> (slot & 63)) & 1ull)) return;
        if (slot >= 0 && setup_ray(r, origin, dir, scaling)) {
            float march1_sum = 0.0f;
            bool first_march_too = false;
            if constexpr (kMode == kBackwardSecond) {
                const float2* head = ws.base + slot * kChunkFloat2 + kHeadFloat2;
                // (a walk that broke off in a malformed tree: the reference adds nothing for such a ray)
                if (head[1].y == 2.0f) return;
                // (a ray the noting launch gave up on has no sum: both marches)
                first_march_too = head[1].y == 3.0f;
                march1_sum = first_march_too ? 0.0f : head[2].x;
            }
            if constexpr (P::kFormat != SVOX_FORMAT_RGBA) {
                float basis[D];
                policy_basis<P>(Lobes{tr.extra, tr.extra_cols, opt.format}, opt, vdir, basis);
#pragma unroll
                for (int i = 0; i < D; ++i) sh.basis[lane * D + i] = basis[i];
            }
            go[0] = grad_out[slot * 3];
            go[1] = grad_out[slot * 3 + 1];
            go[2] = grad_out[slot * 3 + 2];
            light = 1.0f;
            accum = march1_sum;
            tmin = r.t;
            cur.begin(r);
            phase = kMode == kBackwardSecond && !first_march_too ? kMarch2 : kMarch1;
            active = true;
        }
    };
    if constexpr (!kRefill) {
        if (next + lane < end) start(next + lane);
    }

    while (true) {
        if constexpr (kRefill) {
            if (Source::kItemsAreSlots && ws.only) next = skip_clear_words(ws.only, next, end, lane);
            const RoundState state = refill_lanes(active, next, end, src.refill_at, start);
            if (state == kRoundRefilled) continue;
            if (state == kRoundDone) break;
        } else {
            if (!any_lane(active)) break;
        }

        // ---- walk
        int32_t q_leaf[kQueue];
        float q_dt[kQueue];
        bool broken;
        float q_sigma[kQueue];
        walk_turns(tr, child, r, cur, step, active, broken, q_leaf, q_dt);
        // ---- sigma
        float q_raw[kQueue];
        fetch_sigma<K>(tr.data, q_leaf, q_sigma);
        soften_sigma(opt.density_softplus, q_leaf, q_sigma, q_raw);
        // ---- shade list: every leaf with density
        const int n_entries = build_shade_list(sh, q_leaf, q_sigma, 0.0f, lane);
        wave_lds_sync();
        if (n_entries > 0) shade_entries<P, true>(tr.data, sh, n_entries, lane);
        wave_lds_sync();
        // ---- composite slot by slot; the gradient records of the round are added together
        RecordList<P, D> records{sh, grad_data, lane, merge};
        // what does not depend on the transmittance is evaluated for the four slots side by side
        float q_att[kQueue], q_total[kQueue], q_s[kQueue][3];
#pragma unroll
        for (int q = 0; q < kQueue; ++q) {
            q_att[q] = expf_fixed(-q_dt[q] * q_sigma[q] * r.dscale);
            const float* s = sh.colour + (q * kMarchThreads + lane) * 3;
            float total_color = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                q_s[q][c] = s[c];
                total_color = fma_(fma_(s[c], d_rgb_pad, -pad), go[c], total_color);
            }
            q_total[q] = total_color;
        }
#pragma unroll
        for (int q = 0; q < kQueue; ++q) {
            bool emit = false;
            float tmp2[3] = {0.f, 0.f, 0.f};
            float g_sigma = 0.f;
            if (active && q_leaf[q] >= 0 && q_sigma[q] > 0.0f) {
                const float att = q_att[q];
                const float weight = light * (1.0f - att);
                const float* s = q_s[q];
                const float total_color = q_total[q];
                light *= att;
                if (phase == kMarch1) {
                    accum = fma_(weight, total_color, accum);
                } else {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
                            tmp2[c] = weight * s[c] * (1.0f - s[c]) * go[c] * d_rgb_pad;
                        } else {
                            tmp2[c] = (float)((double)(weight * s[c]) * (1.0 - (double)s[c]) * (double)go[c] *
                                              (double)d_rgb_pad);
                        }
                    }
                    accum = fma_(-weight, total_color, accum);
                    g_sigma = q_dt[q] * r.dscale * fma_(total_color, light, -accum);
                    if (opt.density_softplus) g_sigma *= sigmoid_(q_raw[q] - 1.0f);   // rt_kernel.cu:471-474
                    emit = true;
                }
            }
            records.append(emit, q_leaf[q], tmp2, g_sigma);
        }
        records.flush();
        // ---- end of a march
        if (active && (broken || !(r.t < r.tmax))) {
            if (phase == kMarch1 && !broken) {
                const float total_grad = (go[0] + go[1]) + go[2];
                accum = fma_(light * bg, total_grad, accum);
                light = 1.0f;
                phase = kMarch2;
                r.t = tmin;
                cur.aim(r, kCoordBits - 1);
            } else {
                active = false;
            }
        }
    }
}

// ---- notes read back ---------------------------------------------------------------------------
// The replay kernels give every NOTE a lane.  A block of four wavefronts owns 2^ray_shift rays (16 to 64) and lists
// those that have notes; then its wavefronts take from the list, each time as many rays as fit with all their notes
// into 64 lanes, lane l the l-th note: exponentials, colours and factors of 64 leaves at a time.  What has to be formed
// one leaf after the other -- the transmittance in front of a leaf, the colour that lies behind it -- is passed from
// lane to lane (each_in_turn).  A ray with more than 64 notes is taken alone, 64 notes at a time, once for its sum and
// once for its records.
// Neighbours that share leaves are taken first, and in slices: 64 / 2^k notes of each of up to 16 rays, so that
// records of one leaf stand in the same batch and leave the wavefront as one (a ray passes a leaf once: rays taken
// alone, or packed end to end, have next to none to add together).  It pays where the atomic additions bound the
// kernel, and costs two passes over the notes instead of one, so it goes by what neighbours have in common: half of
// the rays of a piece of 16 begin in the leaf of the one to their left.  Steps of training (forward and backward pass,
// us), 800x800 pictures unless stated, with the rays packed or alone -> with slices: dense 128^3 SH9, from 1.2 of its
// edges away 9 090 -> 5 680, from 2 5 030 -> 4 050, from 4 1 480 -> 1 475; 64^3 RGBA from 1.2 2 480 -> 1 465; 64^3
// SH16 from 2 3 800 -> 1 830; N = 3, 81^3 SH9 from 2 3 360 -> 2 035; a 256^3 SH9 shell from 1.5 1 690 -> 1 470, from 4
// 685 -> 655, 50 001 rays of it 650 -> 638; 65 536 scattered rays of 64^3 RGBA with softplus 725 -> 722; 262 144 of
// 128^3 SH9 5 190 -> 5 140.  (The line at a third: the same; at three quarters the pictures from 2 away are lost to
// it.)
// (One lane per ray, as the march has it, is the wrong shape here: where one ray in five meets the scene, and those
// differ in length, 60 to 95 % of the lanes idle, and every ray's notes are read twice, first for the sum of the first
// march.  replay_backward_kernel from that to this: 4 096 rays of a 16^3 RGBA tree 22.6 -> 9.1 us, 50 001 rays of a
// 256^3 SH9 shell with softplus 244 -> 82 us, 1 Mi rays of a 512^3 SH16 shell 457 -> 378 us, an 800x800 picture of
// it 414 -> 296 us; replay_se_grad_kernel, 200 003 rays, 256^3 SH9: 199 -> 111 us.  What is left of the large cases is the
// rate of the atomic additions, about 16 requests of 64 bytes a nanosecond: without them 159 and 151 us.)
// A ray whose notes are incomplete, or every ray if the workspace carries another stamp, is marked in the bitmap for a
// launch of the marching kernel.
constexpr int kReplayMaxShift = 6;
constexpr int kReplayWaves = 4;
constexpr int kReplayThreads = kReplayWaves * kMarchThreads;

// one ray of the list; link: its second chunk, or, if `known`, where ReplayRays::chunks has its chunks from the second on
struct ReplayRay {
    int32_t ray;
    uint32_t known : 1;
    int32_t count : 31;
    int32_t link;
    float dscale;
};
// one lane's note
struct ReplayNote {
    bool valid;
    int owner;      // row of the ray in LDS
    int32_t ray;
    int p, count;   // place among the notes of the ray that are in this batch, and their number
    int last;       // lane of the last of them
    int32_t leaf;
    float dt, raw, s[3], dscale;
};
// What a wavefront keeps of a ray from one slice of its notes to the next, in LDS, by the ray's row: the transmittance
// in front of the slice, N running sums, and where the notes go on.
template <int N>
struct ReplayCarry {
    static constexpr int kRows = 16;
    float through[kRows], run[N][kRows];
    int32_t chunk[kRows], index[kRows];
    __device__ __forceinline__ void begin(int row, int32_t ray) {
        through[row] = 1.0f;
        chunk[row] = 0;
        index[row] = ray;
    }
};
struct ReplayRays {
    // The chunks of a ray's notes are a chain, and to follow it is one trip to memory after the other.  The rays of the
    // list follow theirs all at once, before the first note is read, as long as there is room to keep what they find.
    static constexpr int kChunks = 512;
    ReplayRay list[1 << kReplayMaxShift];
    int32_t chunks[kChunks];
    int n, cursor;                 // of the list: rays, and rays taken
    int n_shared, shared_cursor;   // ... of those that come first, which share leaves with their neighbours
    int n_chunks;

    // Lists the rays of block `block` of `blocks` that have notes and writes its part of the bitmap of undone rays.
    // The rays are dealt out in pieces of 16 neighbours: neighbouring pixels share leaves, whose records are added
    // together.  They are also all long or all short together, so the pieces of a block come from all over the launch:
    // piece number b of the k-th `blocks` pieces goes to block b - k * 0.618 blocks (without the turn a block would get
    // pieces below one another wherever the width of a picture divides `blocks`).
    __device__ __forceinline__ void gather(const ReplaySpace& ws, bool stamped, int64_t n_slots, int block, int blocks,
                                           int ray_shift) {
        static_assert(1 << kReplayMaxShift <= kMarchThreads, "one wavefront looks the rays up");
        const int lane = threadIdx.x;
        if (lane < kMarchThreads) {
            if (lane == 0) shared_cursor = n_chunks = 0;
            const unsigned k = (unsigned)lane >> 4, turn = (unsigned)((float)blocks * 0.618f);
            const int64_t ray = (((int64_t)k * blocks + ((unsigned)block + k * turn) % (unsigned)blocks) << 4) + (lane & 15);
            const bool seated = lane < (1 << ray_shift) && ray < n_slots;
            int32_t count = 0, link = 0, leaf = -1;
            float dscale = 0.0f;
            if (seated) {
                const float2* first = ws.base + ray * kChunkFloat2;
                const float2 head = first[kHeadFloat2], tail = first[kHeadFloat2 + 1];
                link = __float_as_int(head.x);
                count = stamped ? __float_as_int(head.y) : -1;
                dscale = tail.x;
                if (count > 0) leaf = __float_as_int(first[0].x);
            }
            const unsigned long long undone = __ballot(count < 0), m = __ballot(count > 0);
            if ((lane & 15) == 0 && seated) ((uint16_t*)ws.undone)[ray >> 4] = (uint16_t)(undone >> lane);
            if (lane == 0 && undone) *ws.any_undone = 1;
            if (lane == 0) n = __popcll(m);
            wave_lds_sync();
            bool known = false;
            int place = 0;
            if (count > 0) {
                const int more = (count - 1) / kChunkRecords;
                const int to = more > 0 && more <= kChunks ? atomicAdd(&n_chunks, more) : 0;
                known = more > 0 && more <= kChunks && to + more <= kChunks;
                place = to;
                if (known) {
                    int32_t index = link;
                    for (int at = 0; at < more; ++at) {
                        if (at > 0) index = __float_as_int(ws.base[(int64_t)index * kChunkFloat2 + kHeadFloat2].x);
                        chunks[to + at] = index;
                    }
                }
            }
            // Neighbours share leaves if half of them begin in the leaf of the one to their left (16 of them are two
            // rows of 8 pixels).
            const int32_t left = __shfl_up(leaf, 1);
            const unsigned long long alike = __ballot(leaf >= 0 && leaf == left && (lane & 7) != 0);
            const unsigned like_left = (unsigned)(alike >> (lane & 48)) & 0xffffu;
            const unsigned with_notes = (unsigned)(m >> (lane & 48)) & 0xffffu;
            const unsigned long long shared = __ballot(count > 0 && 2 * __popc(like_left) >= __popc(with_notes));
            if (lane == 0) cursor = n_shared = __popcll(shared);
            if (count > 0) {
                const bool first = (shared >> lane & 1ull) != 0;
                list[first ? rank_in(shared) : __popcll(shared) + rank_in(m & ~shared)] =
                    ReplayRay{(int32_t)ray, known ? 1u : 0u, count, known ? place : link, dscale};
            }
        }
        __syncthreads();
    }

    // reads note i of ray r; chunk, index: number and place of a chunk at or before the note's (0 and the first chunk
    // if nothing is known), moved on to the note's
    __device__ __forceinline__ void read(const ReplaySpace& ws, const ReplayRay& r, int i, int& chunk, int32_t& index,
                                         ReplayNote& g) const {
        const int want = i / kChunkRecords;
        const bool known = r.known != 0;
        if (g.valid && want > 0) {
            if (known) index = chunks[r.link + want - 1];
            if (known) chunk = want;
        }
        while (any_lane(g.valid && chunk < want)) {
            if (g.valid && chunk < want) {
                index = chunk == 0 ? r.link : __float_as_int(ws.base[(int64_t)index * kChunkFloat2 + kHeadFloat2].x);
                chunk += 1;
            }
        }
        if (g.valid) {
            const float2* e = ws.base + (int64_t)index * kChunkFloat2 + (i - want * kChunkRecords) * 3;
            const float2 a = e[0], b = e[1], c = e[2];
            g.leaf = __float_as_int(a.x);
            g.dt = a.y;
            g.raw = b.x;
            g.s[0] = b.y;
            g.s[1] = c.x;
            g.s[2] = c.y;
        }
    }

    // Takes the next rays of the list whose notes fit into the wavefront: `at` receives the first of them (n: the list
    // is used up), g each lane's note.  Returns how many rays these are; 0: one ray that has more than 64 notes.
    __device__ __forceinline__ int take(const ReplaySpace& ws, uint8_t* start, int lane, int& at, ReplayNote& g) {
        int rays, sum, count;
        bool fits;
        at = __builtin_amdgcn_readfirstlane(__atomic_load_n(&cursor, __ATOMIC_RELAXED));
        while (true) {
            if (at >= n) return 0;
            count = at + lane < n ? list[at + lane].count : 0;
            sum = count <= kMarchThreads ? count : kMarchThreads + 1;
#pragma unroll
            for (int off = 1; off < kMarchThreads; off <<= 1) {
                const int other = __shfl_up(sum, off);
                if (lane >= off) sum += other;
            }
            fits = at + lane < n && sum <= kMarchThreads && lane < kReplayRows;
            rays = __popcll(__ballot(fits));
            int seen = at;
            if (lane == 0) seen = atomicCAS(&cursor, at, at + (rays > 0 ? rays : 1));
            seen = __builtin_amdgcn_readfirstlane(seen);
            if (seen == at) break;
            at = seen;   // (another wavefront was faster)
        }
        if (rays == 0) return 0;
        const int n_notes = __builtin_amdgcn_readlane(sum, rays - 1);
        start[lane] = 0;
        wave_lds_sync();
        if (fits) start[sum - count] = 1;
        wave_lds_sync();
        const unsigned long long starts = __ballot(start[lane] != 0);
        const unsigned long long upto = starts & (~0ull >> (63 - lane));
        g.valid = lane < n_notes;
        g.owner = __popcll(upto) - 1;
        const int first = 63 - __builtin_clzll(upto);
        g.p = lane - first;
        const ReplayRay r = list[at + g.owner];
        g.ray = r.ray;
        g.count = r.count;
        g.last = first + r.count - 1;
        g.dscale = r.dscale;
        int chunk = 0;
        int32_t index = r.ray;
        read(ws, r, g.p, chunk, index, g);
        return rays;
    }

    // Takes the next neighbours that share leaves, 16 at most and not more than a wavefront's part of all: `at` receives
    // the first of them.  Returns how many; 0: all are taken.
    __device__ __forceinline__ int take_shared(int lane, int& at) {
        at = __builtin_amdgcn_readfirstlane(__atomic_load_n(&shared_cursor, __ATOMIC_RELAXED));
        while (at < n_shared) {
            const int piece = list[at + lane < n_shared ? at + lane : n_shared - 1].ray >> 4;
            const bool with_first = piece == __builtin_amdgcn_readfirstlane(piece) && at + lane < n_shared;
            const bool its_part = lane * kReplayWaves < n_shared && lane < ReplayCarry<1>::kRows;
            const int rays = __builtin_ctzll(~__ballot(with_first && its_part));
            int seen = at;
            if (lane == 0) seen = atomicCAS(&shared_cursor, at, at + rays);
            seen = __builtin_amdgcn_readfirstlane(seen);
            if (seen == at) return rays;
            at = seen;   // (another wavefront was faster)
        }
        return 0;
    }

    // Slice number k of the `taken` rays from entry `at` on: as many notes of each, one after the other, as there are
    // lanes for (a power of two).  Returns whether any ray has notes in it.
    template <int N>
    __device__ __forceinline__ bool take_slice(const ReplaySpace& ws, int at, int taken, int k, int lane,
                                               ReplayCarry<N>& carry, ReplayNote& g) {
        const int shift = taken > 1 ? 6 - (32 - __builtin_clz((unsigned)taken - 1u)) : 6, wide = 1 << shift;
        const bool seated = lane >> shift < taken;
        g.owner = seated ? lane >> shift : 0;
        const ReplayRay r = list[at + g.owner];
        const int left = seated ? r.count - (k << shift) : 0;
        g.ray = r.ray;
        g.p = lane & (wide - 1);
        g.count = left < wide ? left : wide;
        g.valid = g.p < g.count;
        g.last = lane - g.p + g.count - 1;
        g.dscale = r.dscale;
        if (!any_lane(g.valid)) return false;
        int chunk = carry.chunk[g.owner];
        int32_t index = carry.index[g.owner];
        read(ws, r, (k << shift) + g.p, chunk, index, g);
        if (g.valid && lane == g.last) {
            carry.chunk[g.owner] = chunk;
            carry.index[g.owner] = index;
        }
        return true;
    }

    // notes [64 * segment, 64 * segment + 64) of entry `at`; chunk, index: where the segment before it left off
    __device__ __forceinline__ void take_segment(const ReplaySpace& ws, int at, int segment, int lane, int& chunk,
                                                 int32_t& index, ReplayNote& g) {
        const ReplayRay r = list[at];
        if (segment == 0) {
            chunk = 0;
            index = r.ray;
        }
        const int i = segment * kMarchThreads + lane;
        g.valid = i < r.count;
        g.owner = 0;
        g.ray = r.ray;
        g.p = lane;
        g.count = r.count - segment * kMarchThreads < kMarchThreads ? r.count - segment * kMarchThreads : kMarchThreads;
        g.last = g.count - 1;
        g.dscale = r.dscale;
        read(ws, r, i, chunk, index, g);
        chunk = __builtin_amdgcn_readlane(chunk, __builtin_amdgcn_readfirstlane(g.last));
        index = __builtin_amdgcn_readlane(index, __builtin_amdgcn_readfirstlane(g.last));
    }
};

// The march's running values over the lanes of every ray: each lane applies its leaf to the value of the lane before it
// (the first lane of a ray to `seed`), over and over; after k turns the first k lanes of every ray hold their final
// values.  In this order, and not as prefix sums of fewer turns, because what lies behind a leaf is a difference of
// sums: the rounding of the reference's order is part of small gradients.
// A turn is two or three instructions for all rays of the batch.
template <class Step>
__device__ __forceinline__ void each_in_turn(const ReplayNote& g, Step&& step) {
    for (int turn = 0; any_lane(g.valid && g.p >= turn); turn += 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) step();
    }
}
__device__ __forceinline__ float lane_before(float v) {
    constexpr int kWaveShiftRight1 = 0x138;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kWaveShiftRight1, 0xf, 0xf, false));
}
// transmittance in front of the lane's leaf (first leaf of a ray: seed)
__device__ __forceinline__ float light_before(const ReplayNote& g, float att, float seed) {
    float before = seed, after = 0.0f;
    each_in_turn(g, [&]() {
        const float neighbour = lane_before(after);   // (read by every lane, whatever it does with it)
        before = g.p == 0 ? seed : neighbour;
        after = before * att;
    });
    return before;
}
// running sums of weight * value[i], the lane's own included, into sum
template <int N>
__device__ __forceinline__ void running_sums(const ReplayNote& g, float weight, const float (&value)[N],
                                             const float (&seed)[N], float (&sum)[N]) {
    float run[N];
#pragma unroll
    for (int i = 0; i < N; ++i) run[i] = 0.0f;
    each_in_turn(g, [&]() {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float neighbour = lane_before(run[i]);
            run[i] = fma_(weight, value[i], g.p == 0 ? seed[i] : neighbour);
        }
    });
#pragma unroll
    for (int i = 0; i < N; ++i) sum[i] = run[i];
}

// Wavefronts per SIMD that the replay kernels' registers are cut to.  The loop over slices would else take one step
// more of them than the loops beside it do without it: replay_backward_kernel, SH9 rays, 79 without that loop, 78
// uncut, 74 cut; none spills.
template <class P, class Source>
constexpr int replay_waves(bool squared_error) {
    if (P::kFormat == SVOX_FORMAT_SG || P::kBasis > 16) return 3;
    if (std::is_same_v<Source, ImageSource<float>>) return 5;
    return squared_error && P::kBasis > 9 ? 5 : 6;
}
// The backward pass from the notes a noting forward kernel left (NoteTaker), trace_ray_backward's second march
// (rt_kernel.cu:358-475: the sum of the first march, then the records of the second).
template <class P, class Source>
__global__ __launch_bounds__(kReplayThreads, (replay_waves<P, Source>(false))) void replay_backward_kernel(
    Source src, SvoxRenderOptions opt, const float* __restrict__ grad_out, float* __restrict__ grad_data, ReplaySpace ws,
    int ray_shift, Lobes lobes) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    __shared__ ReplayShared<D> shared[kReplayWaves];
    __shared__ ReplayCarry<1> carries[kReplayWaves];
    __shared__ ReplayRays rays;
    const int lane = threadIdx.x & (kMarchThreads - 1);
    ReplayShared<D>& sh = shared[threadIdx.x / kMarchThreads];
    ReplayCarry<1>& carry = carries[threadIdx.x / kMarchThreads];
    const bool stamped = stamp_matches(ws);
    if (ws.report && stamped && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(ws.report, *ws.stocks_taken << 32 | ws.n_stocks, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    rays.gather(ws, stamped, src.n_slots(), (int)blockIdx.x, (int)gridDim.x, ray_shift);

    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    MergeState merge;
    RecordList<P, D, true> records{sh, grad_data, lane, merge};
    // the basis rows of the rays of a batch (entry at + lane by lane)
    auto set_rows = [&](int at, int n_rays) {
        if constexpr (P::kFormat != SVOX_FORMAT_RGBA) {
            if (lane < n_rays) {
                float vdir[3];
                src.view_dir(rays.list[at + lane].ray, vdir);
                float basis[D];
                policy_basis<P>(lobes, opt, vdir, basis);
#pragma unroll
                for (int i = 0; i < D; ++i) sh.basis[lane * D + i] = basis[i];
            }
        }
    };
    float go[3];
    float att, total_color[1];   // of the lane's leaf
    auto look = [&](const ReplayNote& g) {
        go[0] = go[1] = go[2] = 0.0f;
        att = 1.0f;
        total_color[0] = 0.0f;
        if (g.valid) {
#pragma unroll
            for (int c = 0; c < 3; ++c) go[c] = grad_out[(int64_t)g.ray * 3 + c];
            const float sigma = opt.density_softplus ? softplus_m1(g.raw) : g.raw;
            att = expf_fixed(-g.dt * sigma * g.dscale);
#pragma unroll
            for (int c = 0; c < 3; ++c) total_color[0] = fma_(fma_(g.s[c], d_rgb_pad, -pad), go[c], total_color[0]);
        }
    };
    // the records of a batch; behind: what lies behind the lane's leaf
    auto add = [&](const ReplayNote& g, float light, float behind) {
        const unsigned long long m = __ballot(g.valid);
        const int place = rank_in(m);
        if (g.valid) {
            const float weight = light * (1.0f - att);
            sh.leaf[place] = g.leaf;
            records.owners()[place] = (uint8_t)g.owner;
            float* const f = records.factors() + place * 4;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
                    f[c] = weight * g.s[c] * (1.0f - g.s[c]) * go[c] * d_rgb_pad;
                } else {
                    f[c] = (float)((double)(weight * g.s[c]) * (1.0 - (double)g.s[c]) * (double)go[c] * (double)d_rgb_pad);
                }
            }
            float g_sigma = g.dt * g.dscale * fma_(total_color[0], light * att, -behind);
            if (opt.density_softplus) g_sigma *= sigmoid_(g.raw - 1.0f);   // rt_kernel.cu:471-474
            f[3] = g_sigma;
        }
        records.n = __popcll(m);
        records.flush();
    };
    // neighbours that share leaves: slice by slice, once for the sum of the first march, once for the records
    int at, n_rays;
    while ((n_rays = rays.take_shared(lane, at)) > 0) {
        ReplayNote g;
        set_rows(at, n_rays);
        if (lane < n_rays) {
            carry.run[0][lane] = 0.0f;
            carry.begin(lane, rays.list[at + lane].ray);
        }
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            wave_lds_sync();
#pragma unroll 1
            for (int k = 0; rays.take_slice(ws, at, n_rays, k, lane, carry, g); ++k) {
                look(g);
                const float light = light_before(g, att, carry.through[g.owner]);
                const float weight = light * (1.0f - att);
                float run[1] = {carry.run[0][g.owner]};
                running_sums(g, pass == 0 ? weight : -weight, total_color, run, run);
                if (g.valid && lane == g.last) {
                    carry.through[g.owner] = light * att;
                    carry.run[0][g.owner] = run[0];
                }
                if (pass == 1) add(g, light, run[0]);
                wave_lds_sync();
            }
            if (pass == 0 && lane < n_rays) {
                // the background behind the last leaf
                const int32_t ray = rays.list[at + lane].ray;
                const float* const grad = grad_out + (int64_t)ray * 3;
                carry.run[0][lane] = fma_(carry.through[lane] * bg, (grad[0] + grad[1]) + grad[2], carry.run[0][lane]);
                carry.begin(lane, ray);
            }
        }
    }
    while (true) {
        ReplayNote g;
        const int taken = rays.take(ws, sh.start, lane, at, g);
        if (at >= rays.n) break;
        if (taken > 0) {
            set_rows(at, taken);
            look(g);
            const float light = light_before(g, att, 1.0f);
            const float weight = light * (1.0f - att);
            float run[1] = {0.0f};
            running_sums(g, weight, total_color, run, run);
            const int last = g.valid ? g.last : lane;
            run[0] = fma_(__shfl(light * att, last) * bg, (go[0] + go[1]) + go[2], __shfl(run[0], last));
            running_sums(g, -weight, total_color, run, run);
            add(g, light, run[0]);
            continue;
        }
        set_rows(at, 1);
        const int segments = (rays.list[at].count + kMarchThreads - 1) / kMarchThreads;
        float run[1] = {0.0f};
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            float through = 1.0f;   // transmittance in front of the segment
            int chunk = 0;
            int32_t index = 0;
            for (int k = 0; k < segments; ++k) {
                rays.take_segment(ws, at, k, lane, chunk, index, g);
                look(g);
                const float light = light_before(g, att, through);
                const float weight = light * (1.0f - att);
                float behind[1];
                running_sums(g, pass == 0 ? weight : -weight, total_color, run, behind);
                run[0] = __shfl(behind[0], g.last);
                through = __shfl(light * att, g.last);
                if (pass == 1) add(g, light, behind[0]);
            }
            if (pass == 0) run[0] = fma_(through * bg, __shfl((go[0] + go[1]) + go[2], 0), run[0]);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// squared-error gradient and Gauss-Newton Hessian diagonal
// ------------------------------------------------------------------------------------------------
// sigmoid(basis . coefficients) of channel c, rt_kernel.cu:541-547
template <typename T>
__device__ __forceinline__ T channel_sigmoid(const SvoxRenderOptions& opt, const T* basis, const T* val, int c) {
    if (opt.format == SVOX_FORMAT_RGBA) return sigmoid_(val[c]);
    const int off = c * opt.basis_dim;
    T tmp = T(0);
    for (int i = opt.min_comp; i <= opt.max_comp; ++i) tmp = fma_(basis[i], val[off + i], tmp);
    return sigmoid_(tmp);
}

// trace_ray_se_grad_hess, rt_kernel.cu:479-715, generic flavour: one ray per lane, three marches (residual; colour
// gradients and the rendered colour as a running suffix; density gradients), all with sigma > 0 and
// no early stop.  The attenuation argument is spelled -delta_t * delta_scale * sigma in the first
// march and -delta_t * sigma * delta_scale in the other two, as in the reference.  The reference's
// out_dim atomics per sample on the density entry are summed first and added once.  The colour terms of the second
// march are added by the whole wavefront, flat over the records of the lanes that have one in the step, as in
// render_backward_generic_kernel (same LDS layout: the second block of out_dim scalars per lane holds the ray's
// residual instead of grad_out), into both arrays.
template <typename T, class Source>
__global__ __launch_bounds__(kMarchThreads) void se_grad_generic_kernel(TreeDev<T> tr, Source src,
                                                                        SvoxRenderOptions opt, int out_dim,
                                                                        const T* __restrict__ color_ref,
                                                                        T* __restrict__ color_out,
                                                                        T* __restrict__ grad, T* __restrict__ hess) {
    extern __shared__ __align__(16) unsigned char generic_lds[];
    const int lane = threadIdx.x;
    const bool rgba = opt.format == SVOX_FORMAT_RGBA;
    const int bd = (rgba ? 1 : opt.basis_dim) | 1;                          // row length, odd
    T* const sh_basis = (T*)generic_lds;                                    // [lane * bd + i]
    T* const sh_resid = sh_basis + kMarchThreads * bd;                      // [c * 64 + lane]: residual of the ray
    T* const sh_factor = sh_resid + kMarchThreads * out_dim;                // [c * 64 + lane]: grad_ci of the sample
    int64_t* const sh_base = (int64_t*)(sh_factor + kMarchThreads * out_dim);   // [lane]: leaf * K
    uint8_t* const sh_list = (uint8_t*)(sh_base + kMarchThreads);           // lanes with a record in this step

    T offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    T origin[3], dir[3], vdir[3];
    const int64_t item = blockIdx.x * (int64_t)kMarchThreads + lane;
    const int64_t slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
    const T bg = (T)opt.background_brightness;
    RayState<T> r;
    bool alive = slot >= 0 && setup_ray(r, origin, dir, scaling);
    if (slot >= 0 && !alive) {
        for (int j = 0; j < out_dim; ++j) color_out[slot * out_dim + j] = bg;
    }
    if (alive && !rgba) {
        T basis[SVOX_MAX_BASIS_DIM];
        precalc_basis<T>(opt.format, opt.basis_dim, tr.extra, tr.extra_cols, vdir, basis);
#pragma unroll
        for (int i = 0; i < SVOX_MAX_BASIS_DIM; ++i)
            if (i < opt.basis_dim) sh_basis[lane * bd + i] = basis[i];
    }
    wave_lds_sync();
    const T* const my_basis = sh_basis + lane * bd;
    const T pad = (T)opt.rgb_padding;
    const T d_rgb_pad = (T)(1 + 2 * opt.rgb_padding);
    const int lo = rgba ? 0 : opt.min_comp;
    const int n_comp = rgba ? 1 : (opt.max_comp - opt.min_comp + 1 > 0 ? opt.max_comp - opt.min_comp + 1 : 0);
    const int per_record = out_dim * n_comp;
    const T tmin = alive ? r.t : T(0);
    T resid[4] = {T(0), T(0), T(0), T(0)};
    if (alive) {
        T light = T(1);
        while (r.t < r.tmax) {
            T delta_t;
            const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
            if (v.leaf < 0) break;
            const T* val = tr.data + v.leaf * tr.K;
            T sigma = val[tr.K - 1];
            if (opt.density_softplus) sigma = softplus_m1(sigma);
            if (sigma > T(0)) {
                const T att = exp_sp<T>(-delta_t * r.dscale * sigma);
                const T weight = light * (T(1) - att);
                for (int c = 0; c < out_dim; ++c)
                    resid[c] = fma_(weight, fma_(channel_sigmoid(opt, my_basis, val, c), d_rgb_pad, -pad), resid[c]);
                light *= att;
            }
            advance(r, delta_t);
        }
        for (int j = 0; j < out_dim; ++j) {
            resid[j] += fma_(light, bg, -color_ref[slot * out_dim + j]);
            sh_resid[j * kMarchThreads + lane] = resid[j];
        }
    }
    wave_lds_sync();
    T color_accum[4] = {T(0), T(0), T(0), T(0)};
    {
        T light = T(1);
        if (alive) r.t = tmin;
        bool marching = alive;   // (a broken tree ends this march, not the ray: the reference breaks out of the loop)
        while (any_lane(marching && r.t < r.tmax)) {
            bool emit = false;
            if (marching && r.t < r.tmax) {
                T delta_t;
                const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
                if (v.leaf < 0) {
                    marching = false;
                } else {
                    const int64_t base = v.leaf * tr.K;
                    const T* val = tr.data + base;
                    T sigma = val[tr.K - 1];
                    if (opt.density_softplus) sigma = softplus_m1(sigma);
                    if (sigma > T(0)) {
                        const T att = exp_sp<T>(-delta_t * sigma * r.dscale);
                        const T weight = light * (T(1) - att);
                        for (int c = 0; c < out_dim; ++c) {
                            const T sg = channel_sigmoid(opt, my_basis, val, c);
                            sh_factor[c * kMarchThreads + lane] =
                                rgba ? weight * sg * (T(1) - sg) * d_rgb_pad
                                     : (T)((double)(weight * sg) * (1.0 - (double)sg) * (double)d_rgb_pad);
                            color_accum[c] = fma_(weight, fma_(sg, d_rgb_pad, -pad), color_accum[c]);
                        }
                        sh_base[lane] = base;
                        emit = per_record > 0;
                        light *= att;
                    }
                    advance(r, delta_t);
                }
            }
            const unsigned long long m = __ballot(emit);
            if (m != 0) {
                if (emit) sh_list[rank_in(m)] = (uint8_t)lane;
                wave_lds_sync();
                const int n_scalars = __popcll(m) * per_record;
                for (int f = lane; f < n_scalars; f += kMarchThreads) {
                    const int rec = f / per_record, e = f - rec * per_record;
                    const int c = e / n_comp, i = lo + (e - c * n_comp);
                    const int owner = sh_list[rec];
                    const T grad_ci = sh_factor[c * kMarchThreads + owner];
                    const T grad_wi = rgba ? grad_ci : sh_basis[owner * bd + i] * grad_ci;
                    const int64_t at = sh_base[owner] + (rgba ? c : c * opt.basis_dim + i);
                    atomicAdd(grad + at, grad_wi * sh_resid[c * kMarchThreads + owner]);
                    atomicAdd(hess + at, grad_wi * grad_wi);
                }
                wave_lds_sync();
            }
        }
        if (alive)
            for (int j = 0; j < out_dim; ++j) color_accum[j] = fma_(light, bg, color_accum[j]);
    }
    if (!alive) return;
    {
        T light = T(1);
        r.t = tmin;
        while (r.t < r.tmax) {
            T delta_t;
            const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
            if (v.leaf < 0) break;
            const int64_t base = v.leaf * tr.K;
            const T* val = tr.data + base;
            const T raw_sigma = val[tr.K - 1];
            const T sigma = opt.density_softplus ? softplus_m1(raw_sigma) : raw_sigma;
            if (sigma > T(0)) {
                const T att = exp_sp<T>(-delta_t * sigma * r.dscale);
                const T weight = light * (T(1) - att);
                T color_curr[4];
                for (int c = 0; c < out_dim; ++c) {
                    color_curr[c] = fma_(channel_sigmoid(opt, my_basis, val, c), d_rgb_pad, -pad);
                    color_accum[c] = fma_(-weight, color_curr[c], color_accum[c]);
                }
                light *= att;
                T g = T(0), h = T(0);
                for (int j = 0; j < out_dim; ++j) {
                    const T grad_sigma = delta_t * r.dscale * fma_(color_curr[j], light, -color_accum[j]);
                    const T grad2_sigma = grad_sigma * grad_sigma;
                    if (opt.density_softplus) {
                        const T sg = sigmoid_(raw_sigma - T(1));
                        const T d_sg = sg * (T(1) - sg);
                        g += grad_sigma * resid[j] * sg;
                        h += fma_(grad2_sigma * sg, sg, grad_sigma * d_sg);
                    } else {
                        g += grad_sigma * resid[j];
                        h += grad2_sigma;
                    }
                }
                atomicAdd(grad + base + tr.K - 1, g);
                atomicAdd(hess + base + tr.K - 1, h);
            }
            advance(r, delta_t);
        }
    }
    for (int j = 0; j < out_dim; ++j) color_out[slot * out_dim + j] = resid[j] + color_ref[slot * out_dim + j];
}

// trace_ray_se_grad_hess, octree flavour: the backward kernel's persistent wavefront and rounds.
// Two marches instead of three: march 1 forms the residual with the first spelling of the
// attenuation and, beside it, the rendered colour with the second spelling (what the reference's
// second march accumulates); march 2 then produces, per leaf with sigma > 0, both the colour terms
// (the reference's second march) and the density terms (its third).  Every term has the reference's
// value; records are added cooperatively, one coalesced atomic instruction per record element and
// output array, after summing the lanes whose rays sit in the same leaf.
// (Room for five wavefronts on a SIMD with up to four functions, 2 to 6 registers fewer than the compiler takes by itself; lobes on wavefronts that take new rays: for
// four.  285 000 rays that all hit, four wavefronts / five: 64^3 grid RGBA 3 282 / 2 602, SH4 4 197 / 3 263 us, 128^3 shell 1 440 / 1 176, 1 675 / 1 300, 512^3
// 1 816 / 1 473, 2 326 / 1 801; 700 000, 128^3 shell, 9 lobes, three / four 2 527 / 2 357.)
template <class P, class Source, bool kRefill>
__global__ __launch_bounds__(kMarchThreads, !kRefill && P::kBasis <= 4 ? 5 : P::kForwardRows && P::kBasis <= 9 ? 4 : 1) void se_grad_kernel(TreeDev<float> tr, Source src, SvoxRenderOptions opt,
                                                                const float* __restrict__ color_ref,
                                                                float* __restrict__ color_out,
                                                                float* __restrict__ grad_data,
                                                                float* __restrict__ hess_data,
                                                                const unsigned long long* __restrict__ only,
                                                               const unsigned long long* __restrict__ any_undone) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    __shared__ MarchShared<D, true> lds;
    auto& sh = lds.sh;
    if (only && *any_undone == 0) return;
    const int lane = threadIdx.x;
    float offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    const float step = opt.step_size;

    int64_t next = chunk_of_block(blockIdx.x, gridDim.x, src.xcd_group) * (int64_t)src.per_wave;
    const int64_t total = src.total();
    const int64_t end = next + src.per_wave < total ? next + src.per_wave : total;

    RayState<float> r;
    float ref[3] = {0.f, 0.f, 0.f};
    float resid[3] = {0.f, 0.f, 0.f};    // march 1: colour so far; afterwards the residual
    float caccum[3] = {0.f, 0.f, 0.f};   // rendered colour not yet passed (second spelling)
    float light = 1.0f, light1 = 1.0f, tmin = 0.0f;
    int64_t slot = -1;
    bool active = false, second = false;
    OctreeCursor cur;
    cur.reset(lds.lane_path(lane));
    const ChildTable child(tr);

    // takes ray `item` into this lane: a miss is answered at once, a hit becomes the lane's ray
    // (with a bitmap `only` the launch does the rays whose bit is set and no others; a batch launch
    // then does not deal its rays out: its items are ray numbers)
    auto start = [&](int64_t item) {
        float origin[3], dir[3], vdir[3];
        if (Source::kItemsAreSlots && only && !((only[item >> 6] >> (item & 63)) & 1ull)) return;
        slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
        if (slot < 0) return;
        if (!Source::kItemsAreSlots && only && !((only[slot >> 6] >> (slot & 63)) & 1ull)) return;
        if (setup_ray(r, origin, dir, scaling)) {
            if constexpr (P::kFormat != SVOX_FORMAT_RGBA) {
                float basis[D];
                policy_basis<P>(Lobes{tr.extra, tr.extra_cols, opt.format}, opt, vdir, basis);
#pragma unroll
                for (int i = 0; i < D; ++i) sh.basis[lane * D + i] = basis[i];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                ref[c] = color_ref[slot * 3 + c];
                resid[c] = 0.0f;
                caccum[c] = 0.0f;
            }
            light = light1 = 1.0f;
            tmin = r.t;
            cur.begin(r);
            second = false;
            active = true;
        } else {
            color_out[slot * 3] = bg;
            color_out[slot * 3 + 1] = bg;
            color_out[slot * 3 + 2] = bg;
        }
    };
    if constexpr (!kRefill) {
        if (next + lane < end) start(next + lane);
    }

    while (true) {
        if constexpr (kRefill) {
            if (Source::kItemsAreSlots && only) next = skip_clear_words(only, next, end, lane);
            const RoundState state = refill_lanes(active, next, end, src.refill_at, start);
            if (state == kRoundRefilled) continue;
            if (state == kRoundDone) break;
        } else {
            if (!any_lane(active)) break;
        }

        // ---- walk
        int32_t q_leaf[kQueue];
        float q_dt[kQueue];
        bool broken;
        walk_turns(tr, child, r, cur, step, active, broken, q_leaf, q_dt);
        // ---- sigma
        float q_sigma[kQueue], q_raw[kQueue];
        fetch_sigma<K>(tr.data, q_leaf, q_sigma);
        soften_sigma(opt.density_softplus, q_leaf, q_sigma, q_raw);
        // ---- shade list
        const int n_entries = build_shade_list(sh, q_leaf, q_sigma, 0.0f, lane);
        wave_lds_sync();
        shade_entries<P, true>(tr.data, sh, n_entries, lane);
        wave_lds_sync();
        // ---- composite and emit, slot by slot
#pragma unroll
        for (int q = 0; q < kQueue; ++q) {
            bool emit = false;
            float gci[3] = {0.f, 0.f, 0.f};
            float g_sigma = 0.f, h_sigma = 0.f;
            if (active && q_leaf[q] >= 0 && q_sigma[q] > 0.0f) {
                const float att = expf_fixed(-q_dt[q] * q_sigma[q] * r.dscale);
                const float weight = light * (1.0f - att);
                const float* s = sh.colour + (q * kMarchThreads + lane) * 3;
                float col[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) col[c] = fma_(s[c], d_rgb_pad, -pad);
                light *= att;
                if (!second) {
                    const float att1 = expf_fixed(-q_dt[q] * r.dscale * q_sigma[q]);
                    const float weight1 = light1 * (1.0f - att1);
                    light1 *= att1;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        resid[c] = fma_(weight1, col[c], resid[c]);
                        caccum[c] = fma_(weight, col[c], caccum[c]);
                    }
                } else {
                    // (density_softplus: the chain factor of rt_kernel.cu:693-703; 1 and 0 without it)
                    const float sg = opt.density_softplus ? sigmoid_(q_raw[q] - 1.0f) : 1.0f;
                    const float d_sg = sg * (1.0f - sg);
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
                            gci[c] = weight * s[c] * (1.0f - s[c]) * d_rgb_pad;
                        } else {
                            gci[c] = (float)((double)(weight * s[c]) * (1.0 - (double)s[c]) * (double)d_rgb_pad);
                        }
                        caccum[c] = fma_(-weight, col[c], caccum[c]);
                        const float gs = q_dt[q] * r.dscale * fma_(col[c], light, -caccum[c]);
                        if (opt.density_softplus) {
                            g_sigma += gs * resid[c] * sg;
                            h_sigma += fma_(gs * gs * sg, sg, gs * d_sg);
                        } else {
                            g_sigma += gs * resid[c];
                            h_sigma += gs * gs;
                        }
                    }
                    emit = true;
                }
            }
            unsigned long long todo = __ballot(emit);
            while (todo) {
                const int leader = __ffsll((long long)todo) - 1;
                const int32_t leaf_l = __builtin_amdgcn_readlane(q_leaf[q], leader);
                const unsigned long long same = __ballot(emit && q_leaf[q] == leaf_l);
                todo &= ~same;
                float* g = grad_data + (int64_t)leaf_l * K;
                float* h = hess_data + (int64_t)leaf_l * K;
#pragma unroll
                for (int e0 = 0; e0 < K; e0 += 64) {
                    const int e = e0 + lane;
                    float g_val = 0.0f, h_val = 0.0f;
                    unsigned long long members = same;
                    while (members) {
                        const int k = __ffsll((long long)members) - 1;
                        members &= members - 1;
                        const float t0 = read_lane(gci[0], k), t1 = read_lane(gci[1], k), t2 = read_lane(gci[2], k);
                        const float r0 = read_lane(resid[0], k), r1 = read_lane(resid[1], k),
                                    r2 = read_lane(resid[2], k);
                        const float gs = read_lane(g_sigma, k), hs = read_lane(h_sigma, k);
                        float g_term, h_term;
                        if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
                            const float tc = e == 0 ? t0 : e == 1 ? t1 : t2;
                            const float rc = e == 0 ? r0 : e == 1 ? r1 : r2;
                            g_term = e < 3 ? tc * rc : gs;
                            h_term = e < 3 ? tc * tc : hs;
                        } else {
                            const int c = e / D;
                            const float b = e < 3 * D ? sh.basis[k * D + (e - c * D)] : 0.0f;
                            const float gw = b * (c == 0 ? t0 : c == 1 ? t1 : t2);
                            const float rc = c == 0 ? r0 : c == 1 ? r1 : r2;
                            g_term = e < 3 * D ? gw * rc : gs;
                            h_term = e < 3 * D ? gw * gw : hs;
                        }
                        g_val += g_term;
                        h_val += h_term;
                    }
                    if (e < K) {
                        atomicAdd(g + e, g_val);
                        atomicAdd(h + e, h_val);
                    }
                }
            }
        }
        // ---- end of a march
        if (active && (broken || !(r.t < r.tmax))) {
            if (!second && !broken) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    resid[c] += fma_(light1, bg, -ref[c]);
                    caccum[c] = fma_(light, bg, caccum[c]);
                }
                light = 1.0f;
                r.t = tmin;
                cur.aim(r, kCoordBits - 1);
                second = true;
            } else {
#pragma unroll
                for (int c = 0; c < 3; ++c) color_out[slot * 3 + c] = resid[c] + ref[c];
                active = false;
            }
        }
    }
}

// se_grad from the notes a noting forward kernel left (NoteTaker; taken with both thresholds at zero, the colours
// written and the residuals left in the heads by finish_residual): the records of march 2 of se_grad_kernel, term by
// term the same values, a note to a lane (ReplayRays).  A ray whose notes are incomplete, or every ray if the workspace
// carries another stamp, is marked in the bitmap for a launch of se_grad_kernel.
template <int D>
struct ReplaySeShared : ReplayShared<D> {
    float hess_sigma[kEmitCap];             // the density term of the Hessian (factor[3]: that of the gradient)
    float resid[kReplayRows * 3];
};
template <class P, class Source>
__global__ __launch_bounds__(kReplayThreads, (replay_waves<P, Source>(true))) void replay_se_grad_kernel(
    Source src, SvoxRenderOptions opt, float* __restrict__ grad_data, float* __restrict__ hess_data, ReplaySpace ws,
    int ray_shift, Lobes lobes) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    constexpr bool kRgba = P::kFormat == SVOX_FORMAT_RGBA;
    __shared__ ReplaySeShared<D> shared[kReplayWaves];
    __shared__ ReplayCarry<3> carries[kReplayWaves];
    __shared__ ReplayRays rays;
    const int lane = threadIdx.x & (kMarchThreads - 1);
    ReplaySeShared<D>& sh = shared[threadIdx.x / kMarchThreads];
    ReplayCarry<3>& carry = carries[threadIdx.x / kMarchThreads];
    rays.gather(ws, stamp_matches(ws), src.n_slots(), (int)blockIdx.x, (int)gridDim.x, ray_shift);

    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    MergeState merge;
    auto flush = [&](int n) {
        wave_lds_sync();
        // where enough records share a leaf, the records of a leaf are brought together first
        const bool grouped = group_by_leaf(sh.group, merge, sh.leaf, n, lane);
        auto emit = [&](int32_t leaf, int e, const float* sum) {
            const int64_t at = (int64_t)leaf * K + e;
            atomicAdd(grad_data + at, sum[0]);
            atomicAdd(hess_data + at, sum[1]);
        };
        if constexpr (K > kMarchThreads / 2) {
            // One record at a time, lane e on element e; place, leaf and owner of the records are held
            // in registers, record r by lane r, and handed round by readlane, so that the LDS reads of a
            // record have their addresses from scalars and those of four records are in flight together
            // (RecordList::add_held).
            const bool mine = lane < n;
            const int my_rec = mine ? (grouped ? sh.group.order[lane] : lane) : 0;
            const int my_leaf = sh.leaf[my_rec];
            const int my_owner = sh.owner[my_rec];
            constexpr int kBlock = 4;
            // (a loop every lane runs, so that every lane holds its record when readlane looks: see add_held)
            for (int e0 = 0; e0 < K; e0 += kMarchThreads) {
                const int e = e0 + lane;
                const bool on = e < K;
                const int c_raw = kRgba ? e : e / D;
                const int c = c_raw < 3 ? c_raw : 3;
                const int i = kRgba || c == 3 ? 0 : e - c * D;
                const int cc = c < 3 ? c : 0;
                int32_t cur = -1;
                float acc[2] = {0.0f, 0.0f};
                for (int at = 0; at < n; at += kBlock) {
                    int32_t leaf[kBlock];
                    float f[kBlock], b[kBlock], rs[kBlock], hs[kBlock];
#pragma unroll
                    for (int u = 0; u < kBlock; ++u) {
                        const int a = at + u < n ? at + u : n - 1;   // (past the end: the last record again, unused)
                        const int rec = __builtin_amdgcn_readlane(my_rec, a);
                        const int owner = __builtin_amdgcn_readlane(my_owner, a);
                        leaf[u] = __builtin_amdgcn_readlane(my_leaf, a);
                        f[u] = sh.factor[rec * 4 + c];
                        b[u] = kRgba ? 1.0f : sh.basis[owner * D + i];
                        rs[u] = sh.resid[owner * 3 + cc];
                        hs[u] = sh.hess_sigma[rec];
                    }
#pragma unroll
                    for (int u = 0; u < kBlock; ++u) {
                        if (at + u < n) {
                            if (leaf[u] != cur) {
                                if (on && cur >= 0) emit(cur, e, acc);
                                cur = leaf[u];
                                acc[0] = acc[1] = 0.0f;
                            }
                            const float gw = kRgba ? f[u] : b[u] * f[u];
                            acc[0] += c < 3 ? gw * rs[u] : f[u];
                            acc[1] += c < 3 ? gw * gw : hs[u];
                        }
                    }
                }
                if (on && cur >= 0) emit(cur, e, acc);
            }
        } else {
            add_records_by_leaf<K, 2>(
                n, lane, grouped ? sh.group.leaf : sh.leaf,
                // element e of a record: colour coefficient (c, i) or, last, the density
                [&](int at, int e, float* t) {
                    const int rec = grouped ? sh.group.order[at] : at;
                    const int c = kRgba ? e : e / D;
                    if (c < 3) {
                        const int owner = sh.owner[rec];
                        const float v = sh.factor[rec * 4 + c];
                        const float gw = kRgba ? v : sh.basis[owner * D + (e - c * D)] * v;
                        t[0] = gw * sh.resid[owner * 3 + c];
                        t[1] = gw * gw;
                    } else {
                        t[0] = sh.factor[rec * 4 + 3];
                        t[1] = sh.hess_sigma[rec];
                    }
                },
                emit);
        }
        wave_lds_sync();
    };
    // what the march of a ray starts from, entry at + lane by lane
    auto set_rows = [&](int at, int n_rays) {
        if (lane < n_rays) {
            const int64_t ray = rays.list[at + lane].ray;
            const float2* head = ws.base + ray * kChunkFloat2 + kHeadFloat2;
            const float2 r = head[2];
            sh.resid[lane * 3] = head[1].y;
            sh.resid[lane * 3 + 1] = r.x;
            sh.resid[lane * 3 + 2] = r.y;
            if constexpr (!kRgba) {
                float vdir[3];
                src.view_dir(ray, vdir);
                float basis[D];
                policy_basis<P>(lobes, opt, vdir, basis);
#pragma unroll
                for (int i = 0; i < D; ++i) sh.basis[lane * D + i] = basis[i];
            }
        }
        wave_lds_sync();
    };
    float att, col[3];   // of the lane's leaf
    auto look = [&](const ReplayNote& g) {
        const float sigma = opt.density_softplus ? softplus_m1(g.raw) : g.raw;
        att = g.valid ? expf_fixed(-g.dt * sigma * g.dscale) : 1.0f;
#pragma unroll
        for (int c = 0; c < 3; ++c) col[c] = g.valid ? fma_(g.s[c], d_rgb_pad, -pad) : 0.0f;
    };
    // the records of a batch; behind: the colour that lies behind the lane's leaf
    auto add = [&](const ReplayNote& g, float light, const float* behind) {
        const unsigned long long m = __ballot(g.valid);
        const int place = rank_in(m);
        if (g.valid) {
            const float weight = light * (1.0f - att), after = light * att;
            const float sg = opt.density_softplus ? sigmoid_(g.raw - 1.0f) : 1.0f;
            const float d_sg = sg * (1.0f - sg);
            float g_sigma = 0.0f, h_sigma = 0.0f;
            sh.leaf[place] = g.leaf;
            sh.owner[place] = (uint8_t)g.owner;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if constexpr (kRgba) {
                    sh.factor[place * 4 + c] = weight * g.s[c] * (1.0f - g.s[c]) * d_rgb_pad;
                } else {
                    sh.factor[place * 4 + c] =
                        (float)((double)(weight * g.s[c]) * (1.0 - (double)g.s[c]) * (double)d_rgb_pad);
                }
                const float gs = g.dt * g.dscale * fma_(col[c], after, -behind[c]);
                const float resid = sh.resid[g.owner * 3 + c];
                if (opt.density_softplus) {
                    g_sigma += gs * resid * sg;
                    h_sigma += fma_(gs * gs * sg, sg, gs * d_sg);
                } else {
                    g_sigma += gs * resid;
                    h_sigma += gs * gs;
                }
            }
            sh.factor[place * 4 + 3] = g_sigma;
            sh.hess_sigma[place] = h_sigma;
        }
        flush(__popcll(m));
    };
    // neighbours that share leaves: slice by slice, once for the ray's colour, once for the records
    int at, n_rays;
    while ((n_rays = rays.take_shared(lane, at)) > 0) {
        ReplayNote g;
        set_rows(at, n_rays);
        if (lane < n_rays) {
#pragma unroll
            for (int c = 0; c < 3; ++c) carry.run[c][lane] = 0.0f;
            carry.begin(lane, rays.list[at + lane].ray);
        }
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            wave_lds_sync();
#pragma unroll 1
            for (int k = 0; rays.take_slice(ws, at, n_rays, k, lane, carry, g); ++k) {
                look(g);
                const float light = light_before(g, att, carry.through[g.owner]);
                const float weight = light * (1.0f - att);
                float run[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) run[c] = carry.run[c][g.owner];
                running_sums(g, pass == 0 ? weight : -weight, col, run, run);
                if (g.valid && lane == g.last) {
                    carry.through[g.owner] = light * att;
#pragma unroll
                    for (int c = 0; c < 3; ++c) carry.run[c][g.owner] = run[c];
                }
                if (pass == 1) add(g, light, run);
                wave_lds_sync();
            }
            if (pass == 0 && lane < n_rays) {
                // the background behind the last leaf
#pragma unroll
                for (int c = 0; c < 3; ++c) carry.run[c][lane] = fma_(carry.through[lane], bg, carry.run[c][lane]);
                carry.begin(lane, rays.list[at + lane].ray);
            }
        }
    }
    while (true) {
        ReplayNote g;
        const int taken = rays.take(ws, sh.start, lane, at, g);
        if (at >= rays.n) break;
        if (taken > 0) {
            set_rows(at, taken);
            look(g);
            const float light = light_before(g, att, 1.0f);
            const float weight = light * (1.0f - att);
            const int last = g.valid ? g.last : lane;
            const float through = __shfl(light * att, last);
            float run[3] = {0.0f, 0.0f, 0.0f};
            running_sums(g, weight, col, run, run);
#pragma unroll
            for (int c = 0; c < 3; ++c) run[c] = fma_(through, bg, __shfl(run[c], last));
            running_sums(g, -weight, col, run, run);
            add(g, light, run);
            continue;
        }
        set_rows(at, 1);
        const int segments = (rays.list[at].count + kMarchThreads - 1) / kMarchThreads;
        float run[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            float through = 1.0f;   // transmittance in front of the segment
            int chunk = 0;
            int32_t index = 0;
            for (int k = 0; k < segments; ++k) {
                rays.take_segment(ws, at, k, lane, chunk, index, g);
                look(g);
                const float light = light_before(g, att, through);
                const float weight = light * (1.0f - att);
                float behind[3];
                running_sums(g, pass == 0 ? weight : -weight, col, run, behind);
#pragma unroll
                for (int c = 0; c < 3; ++c) run[c] = __shfl(behind[c], g.last);
                through = __shfl(light * att, g.last);
                if (pass == 1) add(g, light, behind);
            }
            if (pass == 0) {
#pragma unroll
                for (int c = 0; c < 3; ++c) run[c] = fma_(through, bg, run[c]);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// dense-grid weight render
// ------------------------------------------------------------------------------------------------
// grid_trace_ray + grid_weight_render_kernel, rt_kernel.cu:898-1003: one pixel ray per lane through a
// dense reso^3 density grid; per cell with sigma > sigma_thresh the largest compositing weight any
// ray gave it and the number of visits.
template <typename T>
__global__ __launch_bounds__(kMarchThreads) void grid_weight_kernel(const T* __restrict__ data, int reso,
                                                                    ImageSource<T> src, SvoxRenderOptions opt,
                                                                    const T* __restrict__ offset_p,
                                                                    const T* __restrict__ scaling_p,
                                                                    T* __restrict__ grid_weight,
                                                                    T* __restrict__ grid_hit) {
    T offset[3], scaling[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        offset[i] = offset_p[i];
        scaling[i] = scaling_p[i];
    }
    T origin[3], dir[3], vdir[3];
    const int64_t item = blockIdx.x * (int64_t)kMarchThreads + threadIdx.x;
    if (src.fetch_item(item, opt, offset, scaling, origin, dir, vdir) < 0) return;
    RayState<T> r;
    if (!setup_ray(r, origin, dir, scaling)) return;
    const T cube_sz = (T)reso;
    T light = T(1);
    while (r.t < r.tmax) {
        T pos[3];
        int32_t uvw[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            pos[j] = clamp01(fma_(r.t, r.d[j], r.o[j])) * cube_sz;
            uvw[j] = (int32_t)floor_(pos[j]);
            pos[j] -= (T)uvw[j];
        }
        const int32_t node_id = uvw[0] * reso * reso + uvw[1] * reso + uvw[2];
        T s0, s1;
        dda_unit(pos, r.inv, &s0, &s1);
        const T delta_t = (s1 - s0) / cube_sz + (T)opt.step_size;
        const T sigma = data[node_id];
        if (sigma > (T)opt.sigma_thresh) {
            const T att = exp_sp<T>(-delta_t * r.dscale * sigma);
            const T weight = light * (T(1) - att);
            light *= att;
            atomic_max_float(grid_weight + node_id, weight);
            atomicAdd(grid_hit + node_id, T(1));
        }
        advance(r, delta_t);
    }
}

// ------------------------------------------------------------------------------------------------
// visit counters
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned lo = __shfl_down((unsigned)(v & 0xffffffffull), off);
        const unsigned hi = __shfl_down((unsigned)(v >> 32), off);
        v += ((unsigned long long)hi << 32) | lo;
    }
    return v;
}

// Counts, with the reference's walk, what the forward march (thresholds, early stop) and one
// backward march (sigma > 0, no stop) of every ray visit.
template <typename T, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_stats_kernel(TreeDev<T> tr, Source src,
                                                                     SvoxRenderOptions opt,
                                                                     unsigned long long* __restrict__ stats) {
    T offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    T origin[3], dir[3], vdir[3];
    const int64_t slot = src.fetch_item(blockIdx.x * (int64_t)kMarchThreads + threadIdx.x, opt, offset, scaling,
                                        origin, dir, vdir);
    unsigned long long c_rays = 0, c_hit = 0, c_samples = 0, c_shaded = 0, c_bwd = 0, c_bwd_pos = 0, c_levels = 0;
    unsigned long long c_tail = 0;
    if (slot >= 0) {
        c_rays = 1;
        RayState<T> r;
        if (setup_ray(r, origin, dir, scaling)) {
            c_hit = 1;
            T light = T(1);
            bool fwd_live = true;
            unsigned since_shaded = 0;   // forward visits since the ray's last shaded leaf
            while (r.t < r.tmax) {
                T delta_t;
                const Visit v = step_generic<T>(tr, r, (T)opt.step_size, &delta_t);
                if (v.leaf < 0) break;
                T sigma = tr.data[v.leaf * tr.K + tr.K - 1];
                if (opt.density_softplus) sigma = softplus_m1(sigma);
                c_bwd += 1;
                if (sigma > T(0)) c_bwd_pos += 1;
                if (fwd_live) {
                    c_samples += 1;
                    c_levels += (unsigned)v.levels;
                    since_shaded += 1;
                    if (sigma > (T)opt.sigma_thresh) {
                        c_shaded += 1;
                        since_shaded = 0;
                        light *= exp_sp<T>(-delta_t * r.dscale * sigma);
                        if (light <= (T)opt.stop_thresh) fwd_live = false;
                    }
                }
                advance(r, delta_t);
            }
            c_tail = since_shaded;
        }
    }
    // every lane reaches the reductions
    c_rays = wave_sum(c_rays);
    c_hit = wave_sum(c_hit);
    c_samples = wave_sum(c_samples);
    c_shaded = wave_sum(c_shaded);
    c_bwd = wave_sum(c_bwd);
    c_bwd_pos = wave_sum(c_bwd_pos);
    c_levels = wave_sum(c_levels);
    c_tail = wave_sum(c_tail);
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(stats + 0, c_rays);
        atomicAdd(stats + 1, c_hit);
        atomicAdd(stats + 2, c_samples);
        atomicAdd(stats + 3, c_shaded);
        atomicAdd(stats + 4, c_bwd);
        atomicAdd(stats + 5, c_bwd_pos);
        atomicAdd(stats + 6, c_levels);
        atomicAdd(stats + 7, c_tail);
    }
}

}  // namespace svox
