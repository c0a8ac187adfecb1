// group_kernels.h -- the march through double-precision octrees, four lanes to a ray.
//
// A double-precision call is rarely large (a gradient check, a reference run), so it lasts as long as its longest ray,
// and what a ray waits for is its chain: descent, record, colour, step.  One ray per lane (the generic kernels) leaves
// that chain to one lane: six dependent child reads from the root, then one channel's dot product after the other.  Here
// four lanes share a ray: they walk it together (the same addresses, one request), each doing one axis' arithmetic, and
// start from the previous leaf's path as the single-precision kernels do (OctreeCursor); lane c of the group evaluates
// channel c; the record of a leaf is asked for before the next step of the walk and used after it.  16 rays to a
// wavefront also spread a small batch over four times the wavefronts (8 or 16 lanes to a ray: 2 000 rays 11 and 17 %
// faster, 100 000 rays 46 and 120 % slower).  The values are those of the generic kernels bit for bit: the same
// expressions in the same order; multiplying by 2^-levels is dividing by 2^levels.
// Measured (20 000 rays through a dense 64^3 SH4 tree): forward 580 -> 306 us, gradient 1372 -> 445 us; 200 rays
// 449 -> 232 and 1196 -> 392 us; 100 000 rays 816 -> 597 and 1954 -> 1505 us.
#pragma once

#include "march_kernels.h"

namespace svox {

constexpr int kGroupLanes = 4;
constexpr int kGroupSeekBudget = 2;   // child reads in a turn of the walk
constexpr int kGroupRays = kMarchThreads / kGroupLanes;

// value of lane k of the caller's group of four (every lane of the group takes part)
template <int k>
__device__ __forceinline__ int from_group(int v) {
    return __builtin_amdgcn_mov_dpp(v, k * 0x55, 0xf, 0xf, true);
}
template <int k>
__device__ __forceinline__ double from_group(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = from_group<k>((int)(b & 0xffffffffll)), hi = from_group<k>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The march of one ray.  Lane c of the group keeps axis c of the ray (lane 3 axis 0 again) and the group puts the three
// together where all are needed: double-precision arithmetic is what a turn consists of.  A turn makes at most
// kGroupSeekBudget child reads; a longer descent goes on in the next turn, so that the other rays of the wavefront do not
// wait for it.
struct GroupWalk {
    double o, d, inv, up;      // this lane's axis, o and d times 2^24; up = max(inv, 0), see leaf_exit
    double t, tmax, dscale;
    double p;                  // the sample's clamped coordinate on this lane's axis, times 2^24
    int32_t* rows;             // this lane's column of the path, counted from level 1 (OctreeCursor)
    uint32_t nx, ny, nz;       // integer cell coordinates of the sample
    int levels;                // of the previous leaf (1: none)
    int level;                 // where the search for the sample's leaf stands
    int32_t node;

    __device__ __forceinline__ void begin(const RayState<double>& r, int axis, int32_t* lane_path) {
        o = (axis == 1 ? r.o[1] : axis == 2 ? r.o[2] : r.o[0]) * 16777216.0;
        d = (axis == 1 ? r.d[1] : axis == 2 ? r.d[2] : r.d[0]) * 16777216.0;
        inv = axis == 1 ? r.inv[1] : axis == 2 ? r.inv[2] : r.inv[0];
        up = max_(inv, 0.0);
        t = r.t;
        tmax = r.tmax;
        dscale = r.dscale;
        rows = lane_path - kMarchThreads;
        rows[kMarchThreads] = 0;
        nx = ny = nz = 0;
        levels = 1;
    }
    __device__ __forceinline__ bool ended() const { return !(t < tmax); }

    // the sample at t: its position, and the deepest node of the previous path it still lies in
    __device__ __forceinline__ void aim() {
        p = max_(0.0, min_((1.0 - 1e-6) * 16777216.0, fma_(t, d, o)));   // (clamp01, times 2^24)
        const int n = (int)(uint32_t)p;
        const uint32_t mx = (uint32_t)from_group<0>(n), my = (uint32_t)from_group<1>(n), mz = (uint32_t)from_group<2>(n);
        const uint32_t diff = (nx ^ mx) | (ny ^ my) | (nz ^ mz);
        const uint32_t first_diff = (diff ? (uint32_t)__builtin_clz(diff) : 0xffffffffu) - (31 - kCoordBits);
        level = (int)min(min(first_diff, (uint32_t)levels), (uint32_t)kPathLevels);
        node = rows[level * kMarchThreads];
        nx = mx;
        ny = my;
        nz = mz;
    }

    // One turn of the search.  True: the leaf is found (its cell index, -1 in a malformed tree), delta_t is the step of
    // the sample and the ray stands at the next one (aim() is still to be called).  rt_kernel.cu:262-275, 315.
    __device__ __forceinline__ bool turn(const TreeDev<double>& tr, double step_size, int64_t& leaf, double& delta_t) {
        int32_t cell = 0, skip = 1;
#pragma unroll
        for (int it = 0; it < kGroupSeekBudget; ++it) {
            if (skip > 0 && level <= kCoordBits) {
                rows[min(level, kPathLevels + 1) * kMarchThreads] = node;
                cell = (node << 3) | cell_at(nx, ny, nz, level);
                skip = tr.child[cell];
                // (negative: no entry of a well-formed tree; the walk from the root says what comes of it)
                const bool down = skip != 0;
                node += skip;
                level = down ? ((uint32_t)node >= (uint32_t)tr.capacity ? kCoordBits + 1 : level + 1) : level;
                skip = down ? 1 : 0;
            }
        }
        if (skip > 0 && level <= kCoordBits) return false;
        double segment;
        leaf = cell;
        if (skip == 0) {
            levels = level;
            // (dda_unit for a point inside the cube: the entry distance is 0, see leaf_exit)
            const double e = -__builtin_amdgcn_fract(p * __longlong_as_double((long long)(1023 - kCoordBits + level) << 52)) * inv + up;
            const double hi = min_(min_(min_((double)1e9f, from_group<0>(e)), from_group<1>(e)), from_group<2>(e));
            segment = hi * __longlong_as_double((long long)(1023 - level) << 52);
        } else {
            // more levels than the integer coordinates hold, or a malformed tree
            levels = 1;
            const double q = p * (1.0 / 16777216.0);
            double local[3] = {from_group<0>(q), from_group<1>(q), from_group<2>(q)};
            const double all_inv[3] = {from_group<0>(inv), from_group<1>(inv), from_group<2>(inv)};
            double cells_per_axis, s0, s1;
            int levels_f;
            leaf = descend_generic<double>(tr.child, tr.capacity, tr.N, local, &cells_per_axis, &levels_f);
            dda_unit(local, all_inv, &s0, &s1);
            segment = (s1 - s0) / cells_per_axis;
        }
        delta_t = segment + step_size;
        const double t_next = t + delta_t;
        t = t_next > t ? t_next : tmax;    // (advance())
        return true;
    }
};

// What a lane of a group asks for of a leaf: the density and its channel's coefficients.
template <int D>
struct GroupRecord {
    static constexpr int kCoefficients = D > 0 ? D : 1;
    static constexpr int K = D > 0 ? 3 * D + 1 : 4;
    double raw, co[kCoefficients];
    __device__ __forceinline__ void ask(const double* __restrict__ data, int64_t leaf, int channel) {
        const double* rec = data + leaf * K;
        raw = rec[K - 1];
#pragma unroll
        for (int i = 0; i < kCoefficients; ++i) co[i] = channel < 3 ? rec[channel * kCoefficients + i] : 0.0;
    }
    // rt_kernel.cu:286-297
    __device__ __forceinline__ double colour(const SvoxRenderOptions& opt, const double* basis) const {
        if constexpr (D == 0) {
            return sigmoid_(co[0]);
        } else {
            double tmp = 0.0;
#pragma unroll
            for (int i = 0; i < D; ++i)
                if (i >= opt.min_comp && i <= opt.max_comp) tmp = fma_(basis[i], co[i], tmp);
            return sigmoid_(tmp);
        }
    }
};

// Set-up common to both kernels: the group's ray; its basis in LDS, one row per ray.
template <int D, class Source>
__device__ __forceinline__ int64_t group_ray(const TreeDev<double>& tr, const Source& src, const SvoxRenderOptions& opt, int lane,
                                             int32_t* path, double* basis_rows, GroupWalk& walk, bool& hit) {
    double offset[3], scaling[3], origin[3], dir[3], vdir[3];
    load_transform(tr, offset, scaling);
    const int64_t item = blockIdx.x * (int64_t)kGroupRays + lane / kGroupLanes;
    int64_t slot = -1;
    if (item < src.total()) slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
    RayState<double> r;
    hit = slot >= 0 && setup_ray(r, origin, dir, scaling);
    if (hit) walk.begin(r, lane & (kGroupLanes - 1), path + lane);
    if constexpr (D > 0) {
        if (hit && (lane & (kGroupLanes - 1)) == 0) {
            double b[D];
            precalc_basis<double>(opt.format, D, tr.extra, tr.extra_cols, vdir, b);
#pragma unroll
            for (int i = 0; i < D; ++i) basis_rows[lane / kGroupLanes * D + i] = b[i];
        }
    }
    wave_lds_sync();
    return slot;
}

// trace_ray, rt_kernel.cu:222-321
template <int D, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_forward_group_kernel(TreeDev<double> tr, Source src,
                                                                             SvoxRenderOptions opt, double* __restrict__ out) {
    __shared__ int32_t path[(kPathLevels + 1) * kMarchThreads];
    __shared__ double basis_rows[kGroupRays * (D > 0 ? D : 1)];
    const int lane = threadIdx.x, channel = lane & (kGroupLanes - 1);
    GroupWalk walk;
    bool live;
    const int64_t slot = group_ray<D>(tr, src, opt, lane, path, basis_rows, walk, live);
    if (slot < 0) return;
    const double bg = (double)opt.background_brightness;
    if (!live) {
        if (channel < 3) out[slot * 3 + channel] = bg;
        return;
    }
    const double* const basis = basis_rows + lane / kGroupLanes * (D > 0 ? D : 1);
    const double pad = (double)opt.rgb_padding, d_rgb_pad = (double)(1 + 2 * opt.rgb_padding);
    double acc = 0.0, light = 1.0;
    bool stopped = false, waiting = false;   // waiting: the record of a leaf is on its way
    double dt = 0.0;
    GroupRecord<D> rec;
    bool walking = !walk.ended();
    if (walking) walk.aim();
    while (walking || waiting) {
        // the next leaf is looked up while the record of the one before it is on its way
        int64_t leaf = -1;
        double next_dt = 0.0;
        if (walking && !walk.turn(tr, (double)opt.step_size, leaf, next_dt)) continue;
        const bool more = walking && leaf >= 0;
        walking = more && !walk.ended();
        if (walking) walk.aim();
        if (waiting) {
            const double sigma = opt.density_softplus ? softplus_m1(rec.raw) : rec.raw;
            if (sigma > (double)opt.sigma_thresh) {
                const double att = exp_sp<double>(-dt * walk.dscale * sigma);
                const double weight = light * (1.0 - att);
                acc = fma_(weight, fma_(rec.colour(opt, basis), d_rgb_pad, -pad), acc);
                light *= att;
                if (light <= (double)opt.stop_thresh) {
                    acc *= (double)(1.0 / (1.0 - light));
                    stopped = true;
                    break;
                }
            }
        }
        waiting = more;
        dt = next_dt;
        if (more) rec.ask(tr.data, leaf, channel);
    }
    if (!stopped) acc = fma_(light, bg, acc);
    if (channel < 3) out[slot * 3 + channel] = acc;
}

// trace_ray_backward, rt_kernel.cu:323-477.  The first march sums <render, grad_out> and keeps the leaves with density
// it met, as far as they fit (kGroupKept to a ray); the second forms the records of the gradient from that list, and
// walks on only where the list was full.  The wavefront adds the records of a step together: scalar f from lane
// f mod 64, so that the scalars of a record go out in requests of 64 bytes (the memory system takes a fixed number of
// those per microsecond).
constexpr int kGroupKept = 96;

template <int D, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_backward_group_kernel(TreeDev<double> tr, Source src,
                                                                              SvoxRenderOptions opt,
                                                                              const double* __restrict__ grad_out,
                                                                              double* __restrict__ grad_data) {
    constexpr int K = GroupRecord<D>::K;
    constexpr int DD = D > 0 ? D : 1;
    __shared__ int32_t path[(kPathLevels + 1) * kMarchThreads];
    __shared__ double basis_rows[kGroupRays * DD];
    __shared__ double kept_dt[kGroupKept * kGroupRays];     // [place][ray]
    __shared__ int32_t kept_leaf[kGroupKept * kGroupRays];
    __shared__ double factors[kGroupRays * 4];       // of the ray's record: the three colour factors, the density term
    __shared__ int32_t leaves[kGroupRays];           // where the record goes
    __shared__ uint8_t listed[kGroupRays];           // rays with a record in this step
    const int lane = threadIdx.x, channel = lane & (kGroupLanes - 1), ray = lane / kGroupLanes;
    GroupWalk walk;
    bool live;
    const int64_t slot = group_ray<D>(tr, src, opt, lane, path, basis_rows, walk, live);
    if (!__any(live)) return;
    const double* const basis = basis_rows + ray * DD;
    const double pad = (double)opt.rgb_padding, d_rgb_pad = (double)(1 + 2 * opt.rgb_padding);
    double go[3] = {0.0, 0.0, 0.0};
    if (live) {
#pragma unroll
        for (int j = 0; j < 3; ++j) go[j] = grad_out[slot * 3 + j];
    }
    const double my_go = channel == 0 ? go[0] : channel == 1 ? go[1] : go[2];
    double accum = 0.0, light = 1.0;
    double resume_t = 0.0;     // where the second march walks on
    int n_kept = 0;
    bool full = false;
    // one leaf with density: attenuation, weight and <colour, grad_out>
    auto shade = [&](const GroupRecord<D>& rec, double sigma, double dt, double& weight, double& sg) {
        const double att = exp_sp<double>(-dt * sigma * walk.dscale);
        weight = light * (1.0 - att);
        sg = rec.colour(opt, basis);
        const double col = fma_(sg, d_rgb_pad, -pad);
        double total_color = fma_(from_group<0>(col), go[0], 0.0);
        total_color = fma_(from_group<1>(col), go[1], total_color);
        total_color = fma_(from_group<2>(col), go[2], total_color);
        light *= att;
        return total_color;
    };
    // ---- first march
    bool whole = live;         // false also for a ray that leaves a malformed tree: no second march (the reference's return)
    if (live) {
        bool waiting = false, walking = !walk.ended();
        double dt = 0.0, at_t = 0.0;       // (at_t: the parameter of the leaf whose record is on its way)
        int32_t waiting_leaf = 0;
        GroupRecord<D> rec;
        if (walking) walk.aim();
        while (walking || waiting) {
            int64_t leaf = -1;
            double next_dt = 0.0;
            const double next_t = walk.t;
            if (walking && !walk.turn(tr, (double)opt.step_size, leaf, next_dt)) continue;
            const bool more = walking && leaf >= 0;
            if (walking && !more) whole = false;
            walking = more && !walk.ended();
            if (walking) walk.aim();
            if (waiting) {
                const double sigma = opt.density_softplus ? softplus_m1(rec.raw) : rec.raw;
                if (sigma > 0.0) {
                    double weight, sg;
                    const double total_color = shade(rec, sigma, dt, weight, sg);
                    accum = fma_(weight, total_color, accum);
                    if (n_kept < kGroupKept) {
                        if (channel == 0) {
                            kept_dt[n_kept * kGroupRays + ray] = dt;
                            kept_leaf[n_kept * kGroupRays + ray] = waiting_leaf;
                        }
                        n_kept += 1;
                    } else if (!full) {
                        full = true;
                        resume_t = at_t;
                    }
                }
            }
            waiting = more;
            waiting_leaf = (int32_t)leaf;
            dt = next_dt;
            at_t = next_t;
            if (more) rec.ask(tr.data, leaf, channel);
        }
    }
    wave_lds_sync();
    if (whole) accum = fma_(light * (double)opt.background_brightness, (go[0] + go[1]) + go[2], accum);
    // ---- second march
    light = 1.0;
    int at = 0;
    bool waiting = false, walking = false;
    double dt = 0.0;
    int32_t waiting_leaf = 0;
    GroupRecord<D> rec;
    auto ask_kept = [&]() {
        waiting = whole && at < n_kept;
        if (waiting) {
            waiting_leaf = kept_leaf[at * kGroupRays + ray];
            dt = kept_dt[at * kGroupRays + ray];
            rec.ask(tr.data, waiting_leaf, channel);
            at += 1;
        } else if (whole && full) {
            full = false;                   // the list is used up: the rest of the ray is walked again
            walk.t = resume_t;
            walking = true;
            walk.aim();
        }
    };
    ask_kept();
    while (__any(waiting || walking)) {
        bool emit = false;
        bool turned = true;                 // this ray takes part in the step (its search for a leaf is not under way)
        int64_t leaf = -1;
        double next_dt = 0.0;
        if (walking) {
            turned = walk.turn(tr, (double)opt.step_size, leaf, next_dt);
            if (turned) {
                walking = leaf >= 0 && !walk.ended();
                if (walking) walk.aim();
            }
        }
        if (turned && waiting) {
            const double raw = rec.raw;
            const double sigma = opt.density_softplus ? softplus_m1(raw) : raw;
            if (sigma > 0.0) {
                double weight, sg;
                const double total_color = shade(rec, sigma, dt, weight, sg);
                accum = fma_(-weight, total_color, accum);
                double f = D == 0 ? weight * sg * (1.0 - sg) * my_go * d_rgb_pad
                                  : (weight * sg) * (1.0 - sg) * my_go * d_rgb_pad;
                if (channel == 3) {
                    const double chain = opt.density_softplus ? sigmoid_(raw - 1.0) : 1.0;
                    f = dt * walk.dscale * fma_(total_color, light, -accum) * chain;
                }
                factors[ray * 4 + channel] = f;
                if (channel == 0) leaves[ray] = waiting_leaf;
                emit = true;
            }
        }
        if (turned) {
            waiting = leaf >= 0;
            if (waiting) {
                waiting_leaf = (int32_t)leaf;
                dt = next_dt;
                rec.ask(tr.data, leaf, channel);
            } else if (!walking) {
                ask_kept();
            }
        }
        // the records of this step, added by the whole wavefront
        const unsigned long long m = __ballot(emit && channel == 0);
        if (m != 0) {
            if (emit && channel == 0) listed[rank_in(m)] = (uint8_t)ray;
            wave_lds_sync();
            const int n_scalars = __popcll(m) * K;
            for (int f = lane; f < n_scalars; f += kMarchThreads) {
                const int rec_at = f / K, e = f - rec_at * K;
                const int owner = listed[rec_at];
                const int c = e / DD < 3 ? e / DD : 3;
                double v = factors[owner * 4 + c];
                if constexpr (D > 0) {
                    const int i = e - c * DD;
                    if (c < 3) {
                        if (i < opt.min_comp || i > opt.max_comp) continue;
                        v = basis_rows[owner * DD + i] * v;
                    }
                }
                atomicAdd(grad_data + (int64_t)leaves[owner] * K + e, v);
            }
            wave_lds_sync();
        }
    }
}

// ---- launches (march_double.hip).  D: 0 for RGBA, else the basis size (1, 4, 9, 16 or 25)
template <class Source>
void launch_group_forward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                          const SvoxRenderOptions& opt, double* out);
template <class Source>
void launch_group_backward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                           const SvoxRenderOptions& opt, const double* grad_out, double* grad_data);

}  // namespace svox
