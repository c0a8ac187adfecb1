// group_kernels.h -- the march through double-precision octrees, several lanes to a ray.
//
// A double-precision call is rarely large (a gradient check, a reference run), so it lasts as long as its longest ray,
// and what a ray waits for is its chain: descent, density, colour, step.  One ray per lane (the generic kernels) leaves
// that chain to one lane.  Here every ray is walked in 4 to 64 pieces at once, a lane to each, as cut_kernel.h does it: the lanes of a
// piece walk until their samples are, bit for bit, those of the next one, and list the leaves with density in LDS; the lists are
// put in the ray's order, and its entries are evaluated by all lanes together (a lane to an entry) and composed one after the
// other.  The gradient forms its records from the same lists, and walks a second time only where one round did not hold all of
// a ray.  The values are those of the generic kernels bit for bit: the same expressions in the same order; multiplying by 2^-levels
// is dividing by 2^levels.
// Bound by the chain of a turn (two child reads, the density, some 150 double-precision instructions: 1 to 1.3 us) up to 20 000 rays, by
// how many wavefronts LDS has room for beyond: with 592 entries nine to a compute unit up to SH4, eight to SH16 (GroupBlock; seven and six where
// everything had its own place: dense 64^3 SH4, 65 536 rays, gradient 986 us instead of 596, 256^3 shell SH16 1527 instead of 1161; 20 000 rays 250 instead of 245).
// Measured, four lanes that walk a ray together, from end to end / pieces, forward pass and gradient, us (more: group_cut):
//   64^3 SH4, half of the leaves empty  1 000 rays 226, 383 / 51, 72    20 000 278, 553 / 144, 245
//   no leaf empty                       1 000 rays 232, 541 / 54, 124   20 000 285, 686 / 220, 518
// The lanes of a ray that walk it together are the kernels for more rays than find room in pieces (below).
#pragma once

#include "cut_kernel.h"

namespace svox {

constexpr int kGroupSeekBudget = 2;    // child reads in a turn of the walk
constexpr int kGroupRays = 16;         // of a wavefront, at most
constexpr int kGroupEntries = 592;     // leaves the lists of a wavefront have room for
constexpr int kGroupReserve = kGroupRays;   // of them kept for the pieces that the rays stand in
constexpr int kGroupHeads = 8;         // samples of a piece that the piece before can go on from

// The march of one piece.  A turn makes at most kGroupSeekBudget child reads; a longer descent goes on in the next turn, so that
// the other lanes of the wavefront do not wait for it.
struct GroupWalk {
    double o[3], d[3], inv[3]; // o and d times 2^24
    double t, tmax;
    double p[3];               // the sample's clamped coordinates, times 2^24
    int32_t* rows;             // this lane's column of the path, counted from level 1 (OctreeCursor)
    uint32_t nx, ny, nz;       // integer cell coordinates of the sample
    int levels;                // of the previous leaf (1: none)
    int level;                 // where the search for the sample's leaf stands
    int32_t node;

    __device__ __forceinline__ void begin(int32_t* lane_path) {
        rows = lane_path - kMarchThreads;
        nx = ny = nz = 0;
        from_root();
    }
    // the path is lost: the next aim() starts at the root
    __device__ __forceinline__ void from_root() {
        rows[kMarchThreads] = 0;
        levels = 1;
    }
    __device__ __forceinline__ bool ended() const { return !(t < tmax); }

    // the sample at t: its position, and the deepest node of the previous path it still lies in
    __device__ __forceinline__ void aim() {
#pragma unroll
        for (int j = 0; j < 3; ++j) p[j] = max_(0.0, min_((1.0 - 1e-6) * 16777216.0, fma_(t, d[j], o[j])));   // (clamp01, times 2^24)
        const uint32_t mx = (uint32_t)p[0], my = (uint32_t)p[1], mz = (uint32_t)p[2];
        const uint32_t diff = (nx ^ mx) | (ny ^ my) | (nz ^ mz);
        const uint32_t first_diff = (diff ? (uint32_t)__builtin_clz(diff) : 0xffffffffu) - (31 - kCoordBits);
        level = (int)min(min(first_diff, (uint32_t)levels), (uint32_t)kPathLevels);
        node = rows[level * kMarchThreads];
        nx = mx;
        ny = my;
        nz = mz;
    }

    // One turn of the search.  True: the leaf is found (its cell index, -1 in a malformed tree), delta_t is the step of
    // the sample and the piece stands at the next one (aim() is still to be called).  rt_kernel.cu:262-275, 315.
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
            const double scale = __longlong_as_double((long long)(1023 - kCoordBits + level) << 52);
            double hi = (double)1e9f;
#pragma unroll
            for (int j = 0; j < 3; ++j) hi = min_(hi, -__builtin_amdgcn_fract(p[j] * scale) * inv[j] + max_(inv[j], 0.0));
            segment = hi * __longlong_as_double((long long)(1023 - level) << 52);
        } else {
            // more levels than the integer coordinates hold, or a malformed tree
            levels = 1;
            double local[3], cells_per_axis, s0, s1;
            int levels_f;
#pragma unroll
            for (int j = 0; j < 3; ++j) local[j] = p[j] * (1.0 / 16777216.0);
            leaf = descend_generic<double>(tr.child, tr.capacity, tr.N, local, &cells_per_axis, &levels_f);
            dda_unit(local, inv, &s0, &s1);
            segment = (s1 - s0) / cells_per_axis;
        }
        delta_t = segment + step_size;
        const double t_next = t + delta_t;
        t = t_next > t ? t_next : tmax;    // (advance())
        return true;
    }
};

// What a lane has found, and the ray's order (CutLists): of the end of a lane's list, which of the piece's first samples are listed
// (bits 0 to 7), the sample (8 to 10) of the lane (11 to 16) the ray goes on with.
constexpr uint32_t kGroupLinked = 1u << 20, kGroupOver = 1u << 21, kGroupBroken = 1u << 22;

// trace_ray, rt_kernel.cu:222-321 (result: the picture), and trace_ray_backward, rt_kernel.cu:323-477 (result: grad_data).  The
// gradient's first pass sums <render, grad_out>, its second forms the records, whose scalars the wavefront adds together: scalar f
// from lane f mod 64, so that they go out in requests of 64 bytes (the memory system takes a fixed number of those per microsecond).
//
// LDS says how many wavefronts a compute unit holds (granules of 1 280 bytes), so what is not needed at the same time lies in the same place: what a block of
// entries evaluates and what puts the lists in order lies where the walk keeps its path, which starts at the root again in a round after one that
// was composed (few rays have one); the rays' order fills the list of free entries from behind.
template <bool kBackward>
struct GroupBlock {
    // of the entries of a block: the colour, then the factors of the coefficients' gradient; the attenuation, then the weight;
    // <colour, grad_out>, then the density's gradient
    union {
        double colour[kMarchThreads * 3];
        uint32_t end[kMarchThreads];       // (before there is one) of a lane's list: how it ends
    };
    double attenuation[kMarchThreads], total[kBackward ? kMarchThreads : 1];
    // of a lane's list: how many there are, from which on and how many are composed now, and where in the ray's order
    uint16_t count[kMarchThreads], from[kMarchThreads], taken[kMarchThreads], place[kMarchThreads];
};
// (With 25 functions the coefficients of an entry take 150 registers: the compiler is told to leave room for two wavefronts on a SIMD, which costs 20 to 28
// bytes of scratch.  Forward pass and gradient of 20 000 rays, one / two: 64^3 SH25 289, 912 / 203, 683 us, no leaf empty 483, 1934 / 335, 1432, 256^3 shell
// 435, 974 / 271, 752.)
template <int D, class Source, bool kBackward>
__global__ __launch_bounds__(kMarchThreads, D > 16 ? 2 : 1) void render_group_kernel(TreeDev<double> tr, Source src, SvoxRenderOptions opt,
                                                                     const double* __restrict__ grad_out, double* __restrict__ result,
                                                                     int per_wave, int most_cut) {
    constexpr int DD = D > 0 ? D : 1;
    constexpr int K = D > 0 ? 3 * D + 1 : 4;
    __shared__ union {
        int32_t path[(kPathLevels + 1) * kMarchThreads];
        GroupBlock<kBackward> block;
    } sh;
    __shared__ PieceHeads<double, kGroupHeads> heads;          // (-1: not known yet)
    // the leaves found, and the one after each in its lane's list; the entries that are free
    __shared__ double list_dt[kGroupEntries];
    __shared__ int32_t list_leaf[kGroupEntries];
    __shared__ uint16_t list_next[kGroupEntries];
    // from the front the entries that are free, from behind those of every ray in its order, ray by ray (each once, and none that is free)
    __shared__ uint16_t spare[kGroupEntries];
    auto order = [&](int place) -> uint16_t& { return spare[kGroupEntries - 1 - place]; };
    double* const colour = sh.block.colour;
    double* const attenuation = sh.block.attenuation;
    double* const total = sh.block.total;
    uint16_t* const list_count = sh.block.count;
    uint16_t* const list_from = sh.block.from;
    uint16_t* const list_taken = sh.block.taken;
    uint16_t* const list_place = sh.block.place;
    uint32_t* const list_end = sh.block.end;
    __shared__ double ray_basis[kGroupRays * DD], ray_go[kBackward ? kGroupRays * 3 : 1], ray_dscale[kGroupRays];
    __shared__ int32_t ray_count[kGroupRays], ray_at[kGroupRays], ray_lane[kGroupRays];
    constexpr double kUnknown = -1.0;
    const double kNone = __longlong_as_double(0x7ff0000000000000ll);
    const int lane = threadIdx.x;
    const double step = (double)opt.step_size;
    const double bg = (double)opt.background_brightness;
    const double pad = (double)opt.rgb_padding, d_rgb_pad = (double)(1 + 2 * opt.rgb_padding);
    const double list_thresh = kBackward ? 0.0 : (double)opt.sigma_thresh;

    // ---- the wavefront's rays: lane k of the first per_wave looks at the k-th of them
    RayState<double> r{};
    int64_t slot = -1;
    bool hit = false;
    {
        double offset[3], scaling[3], origin[3], dir[3], vdir[3];
        load_transform(tr, offset, scaling);
        const int64_t item = (int64_t)lane * gridDim.x + blockIdx.x;
        if (lane < per_wave && item < src.total()) slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
        hit = slot >= 0 && setup_ray(r, origin, dir, scaling);
        if (!kBackward && slot >= 0 && !hit) {
#pragma unroll
            for (int j = 0; j < 3; ++j) result[slot * 3 + j] = bg;
        }
        const int row = rank_in(__ballot(hit));
        if (hit) {
            ray_lane[row] = lane;
            ray_dscale[row] = r.dscale;
            if constexpr (D > 0) {
                double b[D];
                precalc_basis<double>(opt.format, D, tr.extra, tr.extra_cols, vdir, b);
#pragma unroll
                for (int i = 0; i < D; ++i) ray_basis[row * D + i] = b[i];
            }
            if constexpr (kBackward) {
#pragma unroll
                for (int j = 0; j < 3; ++j) ray_go[row * 3 + j] = grad_out[slot * 3 + j];
            }
        }
    }
    const int n_rays = __popcll(__ballot(hit));
    if (n_rays == 0) return;
    wave_lds_sync();
    // ---- 2^cut lanes to each of those that meet the cube
    const int cut = min(most_cut, __builtin_clz((unsigned)n_rays) - 25 - ((n_rays & (n_rays - 1)) != 0 ? 1 : 0));   // 2^cut * n_rays <= 64
    const int pieces = 1 << cut, ray = lane >> cut, piece = lane & (pieces - 1), leader = lane - piece;
    hit = ray < n_rays;
    const int row = hit ? ray : 0;
    GroupWalk walk;
    double t0;
    {
        const int from = ray_lane[row];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            walk.o[j] = __shfl(r.o[j], from) * 16777216.0;
            walk.d[j] = __shfl(r.d[j], from) * 16777216.0;
            walk.inv[j] = __shfl(r.inv[j], from);
        }
        t0 = __shfl(r.t, from);
        walk.tmax = __shfl(r.tmax, from);
        slot = (int64_t)__shfl((long long)slot, from);
    }
    walk.begin(sh.path + lane);
    const double length = walk.tmax - t0, part = 1.0 / (double)pieces;
    auto begin_of = [&](int k) { return k < pieces ? fma_((double)k * part, length, t0) : kNone; };

    // the ray (the same in all its lanes)
    bool whole = hit;                  // not in a malformed tree: no gradient (the reference's return)
    double light = 1.0, accum = 0.0;   // accum: the channel of this lane, or the sum over the three of <render, grad_out>
    const int channel = min(piece, 2);
    double go_sum = 0.0;
    if constexpr (kBackward) go_sum = (ray_go[row * 3] + ray_go[row * 3 + 1]) + ray_go[row * 3 + 2];

    // The entries [0, ray_count) of every ray in its order, evaluated and composed in blocks of one to a lane.  add: with their gradient.
    auto compose = [&](bool active, int n_order, bool& ended, bool add) {
        for (int base = 0; any_lane(active && !ended && base < n_order); base += pieces) {
            auto entry_of = [&](int e, int& of_ray) {      // entry e of the block, -1: there is none
                of_ray = e >> cut;
                const int k = base + (e & (pieces - 1));
                return of_ray < n_rays && k < ray_count[of_ray] ? (int)order(ray_at[of_ray] + k) : -1;
            };
            // (a lane to an entry: what it reads of a record is asked for at once; a lane to a channel waited three times, and once more for the density.
            // Forward pass, gradient step of 20 000 rays: 64^3 SH4 177, 467 -> 161, 414 us, no leaf empty 267, 897 -> 235, 797; 128^3 SH4 359, 992 -> 330, 901;
            // 64^3 SH16 202, 777 -> 183, 702; 16^3 SH4 57, 156 -> 51, 138.)
            int of_ray;
            const int mine = entry_of(lane, of_ray);
            double raw = 0.0;
            if (mine >= 0) {
                const double* const rec = tr.data + (int64_t)list_leaf[mine] * K;
                raw = rec[K - 1];
                double s[3];
                if constexpr (D == 0) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) s[c] = rec[c];
                } else {
                    double co[3 * DD];
#pragma unroll
                    for (int i = 0; i < 3 * DD; ++i) co[i] = rec[i];
#pragma unroll
                    for (int c = 0; c < 3; ++c) s[c] = 0.0;
#pragma unroll
                    for (int i = 0; i < DD; ++i) {
                        if (i >= opt.min_comp && i <= opt.max_comp) {
#pragma unroll
                            for (int c = 0; c < 3; ++c) s[c] = fma_(ray_basis[of_ray * DD + i], co[c * DD + i], s[c]);
                        }
                    }
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    s[c] = sigmoid_(s[c]);
                    colour[lane * 3 + c] = s[c];
                }
                const double sigma = opt.density_softplus ? softplus_m1(raw) : raw;
                if constexpr (kBackward) {
                    attenuation[lane] = exp_sp<double>(-list_dt[mine] * sigma * ray_dscale[of_ray]);
                    double sum = 0.0;
#pragma unroll
                    for (int j = 0; j < 3; ++j) sum = fma_(fma_(s[j], d_rgb_pad, -pad), ray_go[of_ray * 3 + j], sum);
                    total[lane] = sum;
                } else {
                    attenuation[lane] = exp_sp<double>(-list_dt[mine] * ray_dscale[of_ray] * sigma);
                }
            }
            wave_lds_sync();
            const int n_here = active && !ended ? min(pieces, n_order - base) : 0;
            for (int k = 0; any_lane(k < n_here); k += 4) {
                double q_att[4], q_value[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int e = min(leader + k + q, kMarchThreads - 1);
                    q_att[q] = attenuation[e];
                    q_value[q] = kBackward ? total[e] : colour[e * 3 + channel];
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (k + q < n_here && !ended) {
                        const double weight = light * (1.0 - q_att[q]);
                        if constexpr (kBackward) {
                            light *= q_att[q];
                            accum = fma_(add ? -weight : weight, q_value[q], accum);
                            if (add && piece == 0) {
                                attenuation[leader + k + q] = weight;
                                total[leader + k + q] = fma_(q_value[q], light, -accum);
                            }
                        } else {
                            accum = fma_(weight, fma_(q_value[q], d_rgb_pad, -pad), accum);
                            light *= q_att[q];
                            if (light <= (double)opt.stop_thresh) {
                                // rt_kernel.cu:306-313: rescale and leave without the background
                                accum *= (double)(1.0 / (1.0 - light));
                                ended = true;
                            }
                        }
                    }
                }
            }
            wave_lds_sync();
            if (kBackward && add) {
                if (mine >= 0) {
                    const double weight = attenuation[lane];
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        const double sg = colour[lane * 3 + j];
                        colour[lane * 3 + j] = weight * sg * (1.0 - sg) * ray_go[of_ray * 3 + j] * d_rgb_pad;
                    }
                    const double chain = opt.density_softplus ? sigmoid_(raw - 1.0) : 1.0;
                    total[lane] = list_dt[mine] * ray_dscale[of_ray] * total[lane] * chain;
                }
                wave_lds_sync();
                for (int f = lane; f < kMarchThreads * K; f += kMarchThreads) {
                    int of_ray;
                    const int e = f / K, i = f - e * K, of = entry_of(e, of_ray);
                    if (of < 0) continue;
                    double v;
                    if constexpr (D > 0) {
                        const int c = i / DD, b = i - c * DD;
                        if (c < 3 && (b < opt.min_comp || b > opt.max_comp)) continue;
                        v = c < 3 ? ray_basis[of_ray * DD + b] * colour[e * 3 + c] : total[e];
                    } else {
                        v = i < 3 ? colour[e * 3 + i] : total[e];
                    }
                    atomicAdd(result + (int64_t)list_leaf[of] * K + i, v);
                }
                wave_lds_sync();
            }
        }
    };

    bool again = false;                // the second march of a gradient
    while (true) {
        // ---- this lane's piece
        walk.t = piece > 0 ? begin_of(piece) : t0;
        bool active = whole;
        bool walking = active && !walk.ended();
        bool fresh = true;             // the sample at walk.t has not been looked at
        int next = piece + 1, head = 0;    // the piece ahead, and its next sample to compare with
        double next_at = begin_of(next);
        int patience = 32;                 // turns the lane may yet spend on waiting for the piece ahead (256: 128^3 shell, 2 000 rays 84 -> 227 us)
        int sample = 0, count = 0;
        uint32_t end = walking ? 0u : kGroupOver;
#pragma unroll
        for (int i = 0; i < kGroupHeads; ++i) heads.write(i, lane, walking ? (i == 0 ? walk.t : kUnknown) : kNone);
        wave_lds_sync();
        int at_lane = leader, at = 0;      // where the ray's composition stands
        int first = 0, last = 0;           // of this lane's list
        int n_spare = kGroupEntries;
        for (int i = lane; i < kGroupEntries; i += kMarchThreads) spare[i] = (uint16_t)i;
        wave_lds_sync();
        int rounds = 0, n_order = 0;
        while (true) {
            rounds += 1;
            walk.from_root();
            if (!fresh) walk.aim();    // (a search that was under way)
            // ---- walk; the density of a leaf is looked at a turn after the leaf was found
            int32_t leaf_before = -1;
            double dt_before = 0.0, raw_before = 0.0;
            int number_before = 0;
            // (the nearer a piece is to where its ray stands, the more of the room it may take: what a round has listed should be complete.  20 000 rays
            // of a 64^3 grid without empty leaves 328 -> 262 us)
            const int room_for = lane == at_lane ? kGroupReserve : kMarchThreads + kGroupReserve + ((lane - at_lane) * 160 >> cut);
            while (true) {
                // (an entry is left for every leaf that is under way, and some for those who alone can free others)
                const int room = n_spare - __popcll(__ballot(leaf_before >= 0));
                bool go = walking && room >= room_for;
                if (!any_lane(go || leaf_before >= 0)) break;
                const bool ahead = go && fresh && walk.t >= next_at;
                if (any_lane(ahead)) {
                    if (ahead) {
                        // on the ground of the piece ahead: is this one of its samples?
                        double there = kUnknown;
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            if (k > 0 && there != kUnknown && there < walk.t && head < kGroupHeads - 1) head += 1;
                            there = heads.read(head, leader + next);
                        }
                        if (there == walk.t) {
                            end |= kGroupLinked | (uint32_t)head << 8 | (uint32_t)(leader + next) << 11;
                            walking = go = false;
                        } else if (there == kNone || there < walk.t) {
                            // it has none after the one here, tells of none, or may not walk on: the one after it; otherwise its next
                            // sample is not known yet, or not looked at (one that lies ahead is walked to)
                            if (there == kNone || (there != kUnknown && head == kGroupHeads - 1) || room < kMarchThreads + kGroupReserve ||
                                --patience < 0) {
                                next += 1;
                                next_at = begin_of(next);
                                head = 0;
                            }
                            go = false;
                        }
                    }
                }
                int64_t leaf = -1;
                double dt = 0.0;
                bool found = false;
                if (go) {
                    if (fresh) walk.aim();
                    fresh = false;
                    found = walk.turn(tr, step, leaf, dt);
                }
                const bool listed = leaf_before >= 0 && (opt.density_softplus ? softplus_m1(raw_before) : raw_before) > list_thresh;
                const unsigned long long m = __ballot(listed);
                if (listed) {
                    if (number_before < kGroupHeads) end |= 1u << number_before;
                    const int id = spare[n_spare - 1 - rank_in(m)];
                    list_leaf[id] = leaf_before;
                    list_dt[id] = dt_before;
                    if (count == 0) first = id;
                    else list_next[last] = (uint16_t)id;
                    last = id;
                    count += 1;
                }
                n_spare -= __popcll(m);
                leaf_before = -1;
                if (found) {
                    if (leaf < 0) {
                        walking = false;
                        end |= kGroupOver | kGroupBroken;
                    } else {
                        leaf_before = (int32_t)leaf;
                        dt_before = dt;
                        raw_before = tr.data[leaf * K + K - 1];
                        number_before = sample;
                        sample += 1;
                        fresh = true;
                        if (walk.ended()) {
                            walking = false;
                            end |= kGroupOver;
                        } else if (sample < kGroupHeads) {
                            heads.write(sample, lane, walk.t);
                        }
                    }
                }
                if (!walking && (end & (kGroupLinked | kGroupOver)) != 0) {
                    // the piece before is to see that there are no more (a sample that links, or breaks off, is one still)
                    const int from = (end & (kGroupLinked | kGroupBroken)) != 0 ? sample + 1 : sample;
#pragma unroll
                    for (int i = 0; i < kGroupHeads; ++i)
                        if (i >= from) heads.write(i, lane, kNone);
                }
            }
            wave_lds_sync();
            list_count[lane] = (uint16_t)count;
            list_end[lane] = end;
            list_taken[lane] = 0;
            wave_lds_sync();
            // ---- the rays' order, as far as it is listed
            bool over = false, broken = false, going = active;
            n_order = 0;
            while (any_lane(going)) {
                if (going) {
                    const int have = list_count[at_lane];
                    const uint32_t e = list_end[at_lane];
                    if (piece == 0) {
                        list_from[at_lane] = (uint16_t)at;
                        list_taken[at_lane] = (uint16_t)(have - at);
                        list_place[at_lane] = (uint16_t)n_order;
                    }
                    n_order += have - at;
                    if (e & kGroupLinked) {
                        at_lane = (int)(e >> 11 & 63u);
                        at = __popc(list_end[at_lane] & ((1u << (e >> 8 & 7u)) - 1u));
                    } else {
                        over = (e & kGroupOver) != 0;
                        broken = (e & kGroupBroken) != 0;
                        at = 0;
                        going = false;
                    }
                }
            }
            if (piece == 0 && hit) ray_count[ray] = n_order;
            wave_lds_sync();
            {
                int to = 0;
                for (int i = 0; i < n_rays; ++i) to += i < ray ? ray_count[i] : 0;
                if (piece == 0 && hit) ray_at[ray] = to;
                const int taken = list_taken[lane], from = taken > 0 ? (int)list_from[lane] : 0;
                to += list_place[lane] - from;
                int id = first;
                for (int i = 0; any_lane(i < from + taken); ++i) {
                    if (i < from + taken) {
                        if (i >= from) order(to + i) = (uint16_t)id;
                        id = list_next[id];
                    }
                }
            }
            wave_lds_sync();
            bool ended = false;  // the ray ends before its order does
            compose(active, n_order, ended, again);
            if (active && (over || ended)) {
                if constexpr (kBackward) {
                    whole = whole && !broken;
                } else if (piece < 3) {
                    result[slot * 3 + channel] = ended ? accum : fma_(light, bg, accum);
                }
                active = false;
            }
            if (!any_lane(active)) break;
            // the lists that were used up (or passed over), and the rays that are over
            if (!active || lane < at_lane) walking = false;
            const int freed = !active || lane <= at_lane ? count : 0;
            for (int i = 0; any_lane(i < freed); ++i) {
                const unsigned long long m = __ballot(i < freed);
                if (i < freed) {
                    spare[n_spare + rank_in(m)] = (uint16_t)first;
                    first = list_next[first];
                }
                n_spare += __popcll(m);
            }
            if (freed > 0) count = 0;
            wave_lds_sync();
        }
        if (!kBackward || again) break;
        // ---- the gradient's second pass: from the lists, if they hold the rays from end to end
        if (whole) accum = fma_(light * bg, go_sum, accum);
        light = 1.0;
        again = true;
        if (rounds == 1) {
            bool ended = false;
            if (piece == 0 && hit && !whole) ray_count[ray] = 0;
            wave_lds_sync();
            compose(whole, n_order, ended, true);
            break;
        }
    }
}

// ---- more rays than the pieces of find room on the GPU, or in their lists (group_cut): four lanes walk a ray together (the same addresses, one
// request), each doing one axis' arithmetic, lane c evaluates channel c, and the record of a leaf is asked for before the next step
// of the walk and used after it.  (What both take, and the lines between them: group_cut.)
constexpr int kSharedLanes = 4;
constexpr int kSharedRays = kMarchThreads / kSharedLanes;

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
struct SharedWalk {
    double o, d, inv, far;     // this lane's axis, o and d times 2^24; far = max(inv, 0), see leaf_exit
    double t, tmax, dscale;
    double p;                  // the sample's clamped coordinate on this lane's axis, times 2^24
    int32_t* rows;             // this lane's column of the path (OctreeCursor)
    uint32_t nx, ny, nz;       // integer cell coordinates of the sample
    int up;                    // where the search for its leaf stands
    uint32_t row;
    int leaf_up;               // of the previous leaf (kCoordBits - 1: the path says nothing of it)

    __device__ __forceinline__ void begin(const RayState<double>& r, int axis, int32_t* lane_path) {
        o = (axis == 1 ? r.o[1] : axis == 2 ? r.o[2] : r.o[0]) * 16777216.0;
        d = (axis == 1 ? r.d[1] : axis == 2 ? r.d[2] : r.d[0]) * 16777216.0;
        inv = axis == 1 ? r.inv[1] : axis == 2 ? r.inv[2] : r.inv[0];
        far = max_(inv, 0.0);
        t = r.t;
        tmax = r.tmax;
        dscale = r.dscale;
        rows = lane_path - OctreeCursor::kPathUp * kMarchThreads;
        rows[kCoordBits * kMarchThreads] = 0;
        nx = ny = nz = 0;
        leaf_up = kCoordBits - 1;
    }
    __device__ __forceinline__ bool ended() const { return !(t < tmax); }

    // the sample at t: its position, and the deepest row of the previous path it still lies in
    __device__ __forceinline__ void aim() {
        p = max_(0.0, min_((1.0 - 1e-6) * 16777216.0, fma_(t, d, o)));   // (clamp01, times 2^24)
        const int n = (int)(uint32_t)p;
        const uint32_t mx = (uint32_t)from_group<0>(n), my = (uint32_t)from_group<1>(n), mz = (uint32_t)from_group<2>(n);
        const uint32_t diff = (nx ^ mx) | (ny ^ my) | (nz ^ mz) | 1u << leaf_up | 1u << (OctreeCursor::kPathUp + 1);
        up = 31 - __builtin_clz(diff);
        row = (uint32_t)rows[(up + 1) * kMarchThreads];
        nx = mx;
        ny = my;
        nz = mz;
    }

    // One turn of the search.  True: the leaf is found (its cell index, -1 in a malformed tree), delta_t is the step of
    // the sample and the ray stands at the next one (aim() is still to be called).  rt_kernel.cu:262-275, 315.
    __device__ __forceinline__ bool turn(const TreeDev<double>& tr, const ChildTable& child, double step_size, int64_t& leaf, double& delta_t) {
        static_assert(kGroupSeekBudget == 2, "two reads, written out");
        const uint32_t first = shift_or<2>(octant_of(nx, ny, nz, up), row);
        const int32_t skip1 = child.read(first);
        const bool below = skip1 > 0;
        const uint32_t next = row + ((uint32_t)skip1 << 5);
        int32_t* const at = rows + max(up, OctreeCursor::kPathUp) * kMarchThreads;
        at[kMarchThreads] = (int32_t)row;
        at[0] = (int32_t)next;
        up -= below ? 1 : 0;
        const uint32_t second = shift_or<2>(octant_of(nx, ny, nz, up), below ? next : ChildTable::kNowhere);
        row = below ? next : row;
        const int32_t skip2 = child.read(second);
        const int32_t skip = min(skip1, skip2);
        const uint32_t cell = (below ? second : first) >> 2;
        const bool found = skip <= 0;
        // (a negative entry, of which a well-formed tree has none, and a cell beyond the table: the walk from the root says what comes of it)
        const bool deep = up < 0 || (found & (skip < 0 || cell > child.last_cell));
        const int here = up;
        row += (uint32_t)max(skip2, 0) << 5;
        up -= skip2 > 0 ? 1 : 0;
        if (!found && !deep) return false;
        double segment;
        leaf = cell;
        if (!deep) {
            leaf_up = here;
            // (dda_unit for a point inside the cube: the entry distance is 0, see leaf_exit)
            const double e = -__builtin_amdgcn_fract(p * __longlong_as_double((long long)(1023 - here) << 52)) * inv + far;
            const double hi = min_(min_(min_((double)1e9f, from_group<0>(e)), from_group<1>(e)), from_group<2>(e));
            segment = hi * __longlong_as_double((long long)(1023 - kCoordBits + here) << 52);
        } else {
            // more levels than the integer coordinates hold, or a malformed tree
            leaf_up = kCoordBits - 1;
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
struct SharedRecord {
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

// The group's ray; its basis in LDS, one row per ray.
template <int D, class Source>
__device__ __forceinline__ int64_t shared_ray(const TreeDev<double>& tr, const Source& src, const SvoxRenderOptions& opt, int lane,
                                             int32_t* path, double* basis_rows, SharedWalk& walk, bool& hit) {
    double offset[3], scaling[3], origin[3], dir[3], vdir[3];
    load_transform(tr, offset, scaling);
    const int64_t item = blockIdx.x * (int64_t)kSharedRays + lane / kSharedLanes;
    int64_t slot = -1;
    if (item < src.total()) slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
    RayState<double> r;
    hit = slot >= 0 && setup_ray(r, origin, dir, scaling);
    if (hit) walk.begin(r, lane & (kSharedLanes - 1), path + lane);
    if constexpr (D > 0) {
        if (hit && (lane & (kSharedLanes - 1)) == 0) {
            double b[D];
            precalc_basis<double>(opt.format, D, tr.extra, tr.extra_cols, vdir, b);
#pragma unroll
            for (int i = 0; i < D; ++i) basis_rows[lane / kSharedLanes * D + i] = b[i];
        }
    }
    wave_lds_sync();
    return slot;
}

// trace_ray, rt_kernel.cu:222-321
template <int D, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_forward_shared_kernel(TreeDev<double> tr, Source src,
                                                                             SvoxRenderOptions opt, double* __restrict__ out) {
    __shared__ int32_t path[(kPathLevels + 2) * kMarchThreads];
    __shared__ double basis_rows[kSharedRays * (D > 0 ? D : 1)];
    const int lane = threadIdx.x, channel = lane & (kSharedLanes - 1);
    SharedWalk walk;
    const ChildTable child(tr);
    bool live;
    const int64_t slot = shared_ray<D>(tr, src, opt, lane, path, basis_rows, walk, live);
    if (slot < 0) return;
    const double bg = (double)opt.background_brightness;
    if (!live) {
        if (channel < 3) out[slot * 3 + channel] = bg;
        return;
    }
    const double* const basis = basis_rows + lane / kSharedLanes * (D > 0 ? D : 1);
    const double pad = (double)opt.rgb_padding, d_rgb_pad = (double)(1 + 2 * opt.rgb_padding);
    double acc = 0.0, light = 1.0;
    bool stopped = false, waiting = false;   // waiting: the record of a leaf is on its way
    double dt = 0.0;
    SharedRecord<D> rec;
    bool walking = !walk.ended();
    if (walking) walk.aim();
    while (walking || waiting) {
        // the next leaf is looked up while the record of the one before it is on its way
        int64_t leaf = -1;
        double next_dt = 0.0;
        if (walking && !walk.turn(tr, child, (double)opt.step_size, leaf, next_dt)) continue;
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
// it met, as far as they fit (kSharedKept to a ray); the second forms the records of the gradient from that list, and
// walks on only where the list was full.  The wavefront adds the records of a step together: scalar f from lane
// f mod 64, so that the scalars of a record go out in requests of 64 bytes (the memory system takes a fixed number of
// those per microsecond).
// (Few, as LDS has room for the more wavefronts: 96 / 64 / 48 / 32, gradient of 131 072 rays, no leaf empty, 128^3 SH4 6 304 / 5 515 / 4 796 / 4 686 us,
// half of them 4 372 / 4 180 / 3 762 / 3 669, 256^3 shell SH16 6 278 / 5 557 / 5 175 / 5 033.)
constexpr int kSharedKept = 32;

template <int D, class Source>
__global__ __launch_bounds__(kMarchThreads) void render_backward_shared_kernel(TreeDev<double> tr, Source src,
                                                                              SvoxRenderOptions opt,
                                                                              const double* __restrict__ grad_out,
                                                                              double* __restrict__ grad_data) {
    constexpr int K = SharedRecord<D>::K;
    constexpr int DD = D > 0 ? D : 1;
    __shared__ int32_t path[(kPathLevels + 2) * kMarchThreads];
    __shared__ double basis_rows[kSharedRays * DD];
    __shared__ double kept_dt[kSharedKept * kSharedRays];     // [place][ray]
    __shared__ int32_t kept_leaf[kSharedKept * kSharedRays];
    __shared__ double factors[kSharedRays * 4];       // of the ray's record: the three colour factors, the density term
    __shared__ int32_t leaves[kSharedRays];           // where the record goes
    __shared__ uint8_t listed[kSharedRays];           // rays with a record in this step
    const int lane = threadIdx.x, channel = lane & (kSharedLanes - 1), ray = lane / kSharedLanes;
    SharedWalk walk;
    const ChildTable child(tr);
    bool live;
    const int64_t slot = shared_ray<D>(tr, src, opt, lane, path, basis_rows, walk, live);
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
    auto shade = [&](const SharedRecord<D>& rec, double sigma, double dt, double& weight, double& sg) {
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
        SharedRecord<D> rec;
        if (walking) walk.aim();
        while (walking || waiting) {
            int64_t leaf = -1;
            double next_dt = 0.0;
            const double next_t = walk.t;
            if (walking && !walk.turn(tr, child, (double)opt.step_size, leaf, next_dt)) continue;
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
                    if (n_kept < kSharedKept) {
                        if (channel == 0) {
                            kept_dt[n_kept * kSharedRays + ray] = dt;
                            kept_leaf[n_kept * kSharedRays + ray] = waiting_leaf;
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
    SharedRecord<D> rec;
    auto ask_kept = [&]() {
        waiting = whole && at < n_kept;
        if (waiting) {
            waiting_leaf = kept_leaf[at * kSharedRays + ray];
            dt = kept_dt[at * kSharedRays + ray];
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
            turned = walk.turn(tr, child, (double)opt.step_size, leaf, next_dt);
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
                          const SvoxRenderOptions& opt, double* out, int per_wave, int most_cut);
template <class Source>
void launch_shared_forward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                           const SvoxRenderOptions& opt, double* out);
template <class Source>
void launch_group_backward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                           const SvoxRenderOptions& opt, const double* grad_out, double* grad_data, int per_wave, int most_cut);
template <class Source>
void launch_shared_backward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                            const SvoxRenderOptions& opt, const double* grad_out, double* grad_data);

}  // namespace svox
