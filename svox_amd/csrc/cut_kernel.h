// cut_kernel.h -- forward passes of few rays: every ray is walked in several pieces at once.
//
// A launch of the march kernels lasts as long as its longest ray: up to 300 leaves, one after the other, at half a
// microsecond and more each, with most of the GPU idle where the rays are few.  The walk does not depend on what the leaves
// hold, and hardly on where it started: a sample's step leads to the far side of its leaf, so two walks of one ray that begin at
// different places are on the same sample, to the bit, once they have met in a leaf and their roundings have agreed (after
// two leaves in half of the cases, after seven in 99.8 %).  So a ray's way through the cube is cut into 2^cut pieces of equal
// length, a lane walks each from where it begins, and goes on past its end until its sample is, bit for bit, one that the lane of
// the next piece had; the rest of the ray is that lane's.  What is composed are the samples of the walk from the ray's beginning, exactly.
//
// A wavefront is dealt a few rays from all over the launch and gives those that meet the cube, be they one or all, the same number of
// pieces, as many as it has lanes for.  It works in rounds: the lanes walk and list the leaves they find with density above the
// pass's threshold, in LDS, until all have come to their pieces' ends or have no room for more; the colours and attenuations of the
// new entries are evaluated by all lanes together (shade_entries' dot products); the entries of every ray are put in the ray's
// order, up to the first piece that is not complete, whose list is then empty again; the first lane of the ray composes them and all
// lanes write the notes.
#pragma once

#include "march_kernels.h"

namespace svox {

// Leaves a lane has room for.  (us, 12 / 16: pictures and rays without notes 64^3 SH9, 16 000 rays 146 / 183, 128^3 SH9, 200x200
// 100 / 109: more wavefronts at once; with notes 64^3 SH4, 4 000 rays 78 / 61, 128^3 SH9, 4 000 rays 151 / 137: fewer rounds.)
constexpr int cut_listed(bool noted) { return noted ? 16 : 12; }
constexpr int kCutTurns = kQueue; // of the walk, between looks at the densities of the leaves found
constexpr int kCutHeads = 8;      // samples of a piece that the piece before can go on from
constexpr int kCutMostRays = 8;   // of a wavefront

// Where the first samples of every piece are.  The lanes write and look at them in the same loop, with nothing between that would make the
// compiler read again or write at once, so both are atomics of the workgroup (ring_read), and nothing else can reach them.
template <class T, int kHeads>
class PieceHeads {
    T at[kHeads * kMarchThreads];

public:
    __device__ __forceinline__ T read(int head, int lane) const {
        return __hip_atomic_load(&at[head * kMarchThreads + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void write(int head, int lane, T t) {
        __hip_atomic_store(&at[head * kMarchThreads + lane], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

// n chunks from those that all rays share, one after the other: the number of the first.  The counter of the stocks handed out is
// kept in step with the one of chunks, beside it, that they are taken from here.
__device__ __forceinline__ unsigned long long take_chunks(const ReplaySpace& ws, int n) {
    const unsigned long long t = atomicAdd(ws.stocks_taken + 1, (unsigned long long)n);
    const unsigned long long stocks = (t + n + kChunkStock - 1) / kChunkStock;
    if (t == 0 || stocks != (t + kChunkStock - 1) / kChunkStock) atomicMax(ws.stocks_taken, stocks);
    return t;
}

// One lane's list, [place][lane], and where it ends.
template <int kListed>
struct CutLists {
    int32_t leaf[kListed * kMarchThreads];
    float dt[kListed * kMarchThreads];
    float raw[kListed * kMarchThreads];      // stored density
    float colour[kListed * kMarchThreads * 3];
    int32_t count[kMarchThreads];
    // what is composed in this round: from which entry on, how many, and from which place in the ray's order on
    // (16 bits: with 26 880 bytes of LDS six wavefronts run on a compute unit, with more five; 8 000 rays of a 128^3 SH4 grid 174 / 193 us)
    int16_t from[kMarchThreads], taken[kMarchThreads], place[kMarchThreads];
    // which of the piece's first samples are listed (bits 0 to 7); the sample (8 to 10) of the lane (11 to 16) the ray goes on
    // with, if it does (kLinked), or whether it ends here (kOver), in a malformed tree (kBroken)
    uint32_t end[kMarchThreads];
};
constexpr uint32_t kCutLinked = 1u << 20, kCutOver = 1u << 21, kCutBroken = 1u << 22;

template <class P, class Source, bool kNoted, bool kGrad>
__global__ __launch_bounds__(kMarchThreads) void render_forward_cut_kernel(TreeDev<float> tr, Source src, SvoxRenderOptions opt,
                                                                           float* __restrict__ out, ReplaySpace ws,
                                                                           const float* __restrict__ grad_out, int per_wave, int most_cut) {
    constexpr int D = P::kBasis > 0 ? P::kBasis : 1;
    constexpr int K = P::kRecord;
    constexpr int kListed = cut_listed(kNoted);
    constexpr int kMostRays = kCutMostRays;
    __shared__ int32_t path[(kPathLevels + 2) * kMarchThreads];
    __shared__ PieceHeads<float, kCutHeads + 1> heads;       // (-1: not known yet; the last row is for what is to be kept from nobody)
    __shared__ CutLists<kListed> lists;
    __shared__ float atts[kNoted ? kListed * kMarchThreads : 1];      // attenuations (without notes: in lists.dt)
    float* const att_of = kNoted ? atts : lists.dt;
    // entries (lane | place << 6): first those whose colours are to be evaluated, then, in equal shares, those of every ray in its order
    __shared__ __align__(8) uint16_t order[kListed * kMarchThreads];
    // where the notes of a ray go: how many it has, the number and place of the chunk the last of them is in, the place of the next
    __shared__ int32_t ray_noted[kNoted ? kMostRays : 1], ray_limit[kNoted ? kMostRays : 1], ray_chunk[kNoted ? kMostRays : 1],
        ray_more[kNoted ? kMostRays : 1];
    __shared__ int32_t ray_lane[kMostRays];
    __shared__ float ray_dscale[kMostRays];
    __shared__ float ray_basis[kMostRays * (P::kForwardRows ? D : 3)];   // the basis of a ray, or its view direction
    constexpr float kUnknown = -1.0f;
    const float kNone = __int_as_float(0x7f800000);
    if constexpr (kNoted) {
        if (blockIdx.x >= ws.march_blocks) return clear_share(ws);
        if (blockIdx.x == 0 && threadIdx.x < kStampWords) ws.stamp_at[threadIdx.x] = ws.stamp[threadIdx.x];
    }
    const int lane = threadIdx.x;
    float offset[3], scaling[3];
    load_transform(tr, offset, scaling);
    const float bg = opt.background_brightness;
    const float pad = opt.rgb_padding;
    const float d_rgb_pad = 1 + 2 * opt.rgb_padding;
    const float step = opt.step_size, sigma_thresh = opt.sigma_thresh, stop_thresh = opt.stop_thresh;
    const float opaque = opaque_light(opt, out);
    const float list_thresh = kNoted ? 0.0f : sigma_thresh;

    // ---- the wavefront's rays: lane k of the first per_wave looks at the k-th of them
    RayState<float> r{};
    int64_t slot = -1;
    bool hit = false;
    {
        float origin[3], dir[3], vdir[3];
        const int64_t item = (int64_t)lane * (kNoted ? ws.march_blocks : gridDim.x) + blockIdx.x;
        if (lane < per_wave && item < src.total()) slot = src.fetch_item(item, opt, offset, scaling, origin, dir, vdir);
        if (slot >= 0) hit = setup_ray(r, origin, dir, scaling);
        if (slot >= 0 && !hit) {
            if (!kNoted || out) {
                out[slot * 3] = bg;
                out[slot * 3 + 1] = bg;
                out[slot * 3 + 2] = bg;
            }
            if constexpr (kNoted) NoteTaker::missed(ws, slot);
        }
        const int row = rank_in(__ballot(hit));
        if (hit) {
            ray_lane[row] = lane;
            ray_dscale[row] = r.dscale;
            if constexpr (P::kForwardRows) {
                float basis[D];
                policy_basis<P>(Lobes{tr.extra, tr.extra_cols, opt.format}, opt, vdir, basis);
#pragma unroll
                for (int i = 0; i < D; ++i) ray_basis[row * D + i] = basis[i];
            } else {
#pragma unroll
                for (int i = 0; i < 3; ++i) ray_basis[row * 3 + i] = vdir[i];
            }
        }
    }
    const int n_rays = __popcll(__ballot(hit));
    if (n_rays == 0) return;
    wave_lds_sync();
    // ---- 2^cut lanes to each of those that meet the cube
    const int cut = min(most_cut, __builtin_clz((unsigned)n_rays) - 25 - ((n_rays & (n_rays - 1)) != 0 ? 1 : 0));   // 2^cut * n_rays <= 64
    const int pieces = 1 << cut, ray = lane >> cut, piece = lane & (pieces - 1), leader = lane - piece;
    {
        const int from = ray_lane[ray < n_rays ? ray : 0];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            r.o[i] = __shfl(r.o[i], from);
            r.d[i] = __shfl(r.d[i], from);
            r.inv[i] = __shfl(r.inv[i], from);
        }
        r.t = __shfl(r.t, from);
        r.tmax = __shfl(r.tmax, from);
        r.dscale = __shfl(r.dscale, from);
        slot = (int64_t)__shfl((long long)slot, from);
        hit = ray < n_rays;
    }

    // ---- this lane's piece
    const float t0 = r.t, length = r.tmax - r.t, share = 1.0f / (float)pieces;
    auto begin_of = [&](int k) { return k < pieces ? fma_((float)k * share, length, t0) : kNone; };
    if (piece > 0) r.t = begin_of(piece);
    bool walking = hit && r.t < r.tmax;
    int next = piece + 1, head = 0;    // the piece ahead, and its next sample to compare with
    float next_at = begin_of(next);
    int patience = 256;                // turns the lane may yet spend on waiting for the piece ahead
    int sample = 0, count = 0, shaded = 0;
    uint32_t end = 0;
#pragma unroll
    for (int i = 0; i < kCutHeads; ++i) heads.write(i, lane, walking ? (i == 0 ? r.t : kUnknown) : kNone);
    if (!walking) end = kCutOver;
    OctreeCursor cur;
    cur.reset(path + lane);
    const ChildTable child(tr);
    if (walking) cur.begin(r);
    wave_lds_sync();

    // ---- the ray, in its leader
    bool active = hit && piece == 0;
    int at_lane = lane, at = 0;        // where its composition stands
    float acc[3] = {0.f, 0.f, 0.f};
    float light = 1.0f;
    bool painted = kNoted && out == nullptr;
    NoteTaker notes;
    March1Sum sum1;
    if constexpr (kNoted) notes.begin(ws, active ? slot : 0);
    int64_t chunk = active ? slot : 0;  // the one its last note is in
    if constexpr (kNoted && kGrad) sum1.begin(grad_out, active ? slot : 0);

    while (true) {
        // ---- walk
        while (any_lane(walking && count <= kListed - kCutTurns)) {
            const bool room = count <= kListed - kCutTurns;
            int32_t q_leaf[kCutTurns];
            float q_dt[kCutTurns];
            int number = sample;       // of the sample the next leaf found belongs to
            // the sample of a lane with `found` is looked at, the next one stands at r.t
            auto arrive = [&](bool found) {
                sample += found ? 1 : 0;
                const bool over = found & !(r.t < r.tmax);
                walking = walking & !over;
                end |= over ? kCutOver : 0u;
                heads.write(found & !over ? min(sample, kCutHeads) : kCutHeads, lane, r.t);
            };
#pragma unroll
            for (int q = 0; q < kCutTurns; ++q) {
                bool go = walking & room;
                const bool ahead = go & (r.t >= next_at);
                if (any_lane(ahead)) {
                    if (ahead) {
                        // on the ground of the piece ahead: is this one of its samples?
                        float there = kUnknown;
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            if (k > 0 && there != kUnknown && there < r.t && head < kCutHeads - 1) head += 1;
                            there = heads.read(head, leader + next);
                        }
                        if (there == r.t) {
                            end |= kCutLinked | (uint32_t)head << 8 | (uint32_t)(leader + next) << 11;
                            walking = go = false;
                        } else if (there == kNone || there < r.t) {
                            // it has none after the one here, or tells of none: the one after it; otherwise its next sample is not
                            // known yet, or not looked at (one that lies ahead is walked to)
                            if (there == kNone || (there != kUnknown && head == kCutHeads - 1) || --patience < 0) {
                                next += 1;
                                next_at = begin_of(next);
                                head = 0;
                            }
                            go = false;
                        }
                    }
                }
                q_leaf[q] = -1;
                q_dt[q] = 0.0f;
                if (child.octree) {
                    cur.turn(r, go, child, step, q_leaf[q], q_dt[q]);
                    arrive(q_leaf[q] >= 0);
                }
                // (lanes whose sample lies deeper than the coordinates wait for the last turn)
                if (q == kCutTurns - 1 || !child.octree) {
                    const bool deep = go & (cur.up < 0 || !child.octree);
                    if (__builtin_expect(any_lane(deep), 0)) {
                        bool broken = false;
                        walk_from_root(tr, r, cur, step, deep, broken, q_leaf[q], q_dt[q]);
                        if (broken) {
                            walking = false;
                            end |= kCutOver | kCutBroken;
                        }
                        arrive(deep & !broken);
                    }
                }
            }
            if (!walking && end != 0) {
                // the piece before is to see that there are no more (a sample that links, or breaks off, is one still)
                const int from = (end & (kCutLinked | kCutBroken)) != 0 ? sample + 1 : sample;
#pragma unroll
                for (int i = 0; i < kCutHeads; ++i)
                    if (i >= from) heads.write(i, lane, kNone);
            }
            float q_raw[kCutTurns];
            fetch_sigma<K>(tr.data, q_leaf, q_raw);
#pragma unroll
            for (int q = 0; q < kCutTurns; ++q) {
                if ((uint32_t)q_leaf[q] < (uint32_t)kEmptyLeafBit && (opt.density_softplus ? softplus_m1(q_raw[q]) : q_raw[q]) > list_thresh) {
                    if (number < kCutHeads) end |= 1u << number;
                    lists.leaf[count * kMarchThreads + lane] = q_leaf[q];
                    lists.dt[count * kMarchThreads + lane] = q_dt[q];
                    lists.raw[count * kMarchThreads + lane] = q_raw[q];
                    count += 1;
                }
                number += q_leaf[q] >= 0 ? 1 : 0;
            }
        }
        lists.count[lane] = count;
        lists.end[lane] = end;
        // ---- colours
        int n_fresh = 0;
        for (int i = 0; any_lane(shaded + i < count); ++i) {
            const bool want = shaded + i < count;
            const unsigned long long m = __ballot(want);
            if (want) order[n_fresh + rank_in(m)] = (uint16_t)(lane | (shaded + i) << 6);
            n_fresh += __popcll(m);
        }
        shaded = count;
        wave_lds_sync();
        // (a lane to an entry, all of whose record it asks for at once: a lane to a channel waited for memory three times as often.  8 000 rays, without notes and with:
        // 64^3 SH9 112, 117 -> 106, 109 us, no leaf empty 149, 190 -> 138, 176; 128^3 SH4 184, 264 -> 174, 251; 256^3 shell SH9 215, 242 -> 214, 243.)
        for (int e = lane; e < n_fresh; e += kMarchThreads) {
            const int of = order[e];
            const int at_ray = (of & 63) >> cut;
            const float* rec = tr.data + (int64_t)lists.leaf[of] * K;
            float s[3];
            if constexpr (P::kFormat == SVOX_FORMAT_RGBA) {
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c] = rec[c];
            } else {
                float co[3 * D];
#pragma unroll
                for (int i = 0; i < 3 * D; ++i) co[i] = rec[i];
                float b[D];
                if constexpr (P::kForwardRows) {
#pragma unroll
                    for (int i = 0; i < D; ++i) b[i] = ray_basis[at_ray * D + i];
                } else {
                    const float vd[3] = {ray_basis[at_ray * 3], ray_basis[at_ray * 3 + 1], ray_basis[at_ray * 3 + 2]};
                    sh_basis<float>(P::kBasis, vd, b);
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c] = 0.0f;
#pragma unroll
                for (int i = 0; i < D; ++i) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) s[c] = fma_(b[i], co[c * D + i], s[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) lists.colour[of * 3 + c] = sigmoid_(s[c]);
            const float raw = lists.raw[of];
            att_of[of] = expf_fixed(-lists.dt[of] * ray_dscale[at_ray] * (opt.density_softplus ? softplus_m1(raw) : raw));
        }
        wave_lds_sync();
        // ---- the rays' order, as far as it is listed
        constexpr int kShare = kListed;                       // (places of a ray: kShare << cut)
        int empty = -1;      // the lane whose list is used up though its piece is not
        int n_order = 0;
        bool over = false, broken = false;
        lists.taken[lane] = 0;
        wave_lds_sync();
        {
            bool going = active;
            while (any_lane(going)) {
                if (going) {
                    const int have = lists.count[at_lane];
                    const uint32_t e = lists.end[at_lane];
                    lists.from[at_lane] = (int16_t)at;
                    lists.taken[at_lane] = (int16_t)(have - at);
                    lists.place[at_lane] = (int16_t)n_order;
                    n_order += have - at;
                    if (e & kCutLinked) {
                        at_lane = (int)(e >> 11 & 63u);
                        at = __popc(lists.end[at_lane] & ((1u << (e >> 8 & 7u)) - 1u));
                    } else {
                        over = (e & kCutOver) != 0;
                        broken = (e & kCutBroken) != 0;
                        empty = at_lane;
                        at = 0;
                        going = false;
                    }
                }
            }
        }
        wave_lds_sync();
        {
            const int taken = lists.taken[lane], from = lists.from[lane], to = (ray * kShare << cut) + lists.place[lane];
            for (int i = 0; any_lane(i < taken); ++i)
                if (i < taken) order[to + i] = (uint16_t)(lane | (from + i) << 6);
        }
        wave_lds_sync();
        // ---- composition
        int limit = n_order;     // entries the ray takes note of
        bool ended = false;      // the ray ends before its order does
        for (int k = 0; any_lane(active && !ended && k < n_order); k += kQueue) {
            int of[kQueue];
            float q_att[kQueue], q_s[kQueue][3], q_sigma[kQueue], q_dt[kQueue];
            const int places = (ray * kShare << cut) + k;
#pragma unroll
            for (int q = 0; q < kQueue; ++q) of[q] = active && k + q < n_order ? order[places + q] : 0;
#pragma unroll
            for (int q = 0; q < kQueue; ++q) {
                q_att[q] = att_of[of[q]];
#pragma unroll
                for (int c = 0; c < 3; ++c) q_s[q][c] = lists.colour[of[q] * 3 + c];
                q_sigma[q] = 0.0f;
                q_dt[q] = 0.0f;
                if constexpr (kNoted) {
                    q_sigma[q] = opt.density_softplus ? softplus_m1(lists.raw[of[q]]) : lists.raw[of[q]];
                    if constexpr (kGrad) q_dt[q] = lists.dt[of[q]];
                }
            }
#pragma unroll
            for (int q = 0; q < kQueue; ++q) {
                const bool there = active && !ended && k + q < n_order;
                const bool shade = there && (!kNoted || q_sigma[q] > sigma_thresh);
                const float weight = light * (1.0f - q_att[q]);
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[c] = shade && !painted ? fma_(weight, fma_(q_s[q][c], d_rgb_pad, -pad), acc[c]) : acc[c];
                light = shade ? light * q_att[q] : light;
                if constexpr (kGrad) {
                    if (there) sum1.leaf(q_dt[q], q_sigma[q], r.dscale, q_s[q], d_rgb_pad, pad);
                }
                if (shade && !painted && light <= stop_thresh) {
                    // rt_kernel.cu:306-313: rescale and leave without the background
                    const float scale = (float)(1.0 / (1.0 - (double)light));
                    out[slot * 3] = acc[0] * scale;
                    out[slot * 3 + 1] = acc[1] * scale;
                    out[slot * 3 + 2] = acc[2] * scale;
                    painted = true;
                    if (!kNoted) ended = true;
                }
                if (kNoted && there && light <= opaque) {   // (nothing behind this leaf counts)
                    ended = true;
                    limit = k + q + 1;
                }
            }
        }
        if constexpr (kNoted) {
            // ---- notes
            const int before = notes.count, now = before + limit;
            const int have = before > 0 ? (before - 1) / kChunkRecords : 0;
            const int more = active && now > 0 && !notes.lost ? (now - 1) / kChunkRecords - have : 0;
            int sum = more;
#pragma unroll
            for (int off = 1; off < kMarchThreads; off <<= 1) {
                const int other = __shfl_up(sum, off);
                if (lane >= off) sum += other;
            }
            const int all = __builtin_amdgcn_readlane(sum, kMarchThreads - 1);
            if (all > 0) {
                // (as many as there are notes for, no stock: a wavefront of one ray would leave most of it unused, and the notes of
                // others that find no room cost far more: 1 000 rays, 128^3 SH9, gradient from notes 143 us, with stocks of 8 1240)
                unsigned long long t = 0;
                if (lane == 0) t = take_chunks(ws, all);
                const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)t);
                const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(t >> 32));
                const int64_t first_new = ws.first_shared + (int64_t)(((unsigned long long)hi << 32) | lo);
                if (more > 0) {
                    const int64_t mine = first_new + sum - more;
                    if (mine + more > ws.n_chunks) {
                        notes.lost = true;
                    } else {
                        for (int i = 0; i < more; ++i)
                            ws.base[(i == 0 ? chunk : mine + i - 1) * kChunkFloat2 + kHeadFloat2] =
                                make_float2(__int_as_float((int32_t)(mine + i)), 0.0f);
                        ray_more[ray] = (int32_t)mine;
                    }
                }
            }
            if (hit && piece == 0) {
                ray_noted[ray] = before;
                ray_limit[ray] = active && !notes.lost ? limit : 0;
                ray_chunk[ray] = (int32_t)chunk;
            }
            notes.count = now;
            if (more > 0 && !notes.lost) chunk = ray_more[ray] + more - 1;
            wave_lds_sync();
            const int taken = lists.taken[lane], from = lists.from[lane], place = lists.place[lane];
            const int row = ray < n_rays ? ray : 0, noted = ray_noted[row], in = noted > 0 ? (noted - 1) / kChunkRecords : 0;
            for (int i = 0; any_lane(i < taken && place + i < ray_limit[row]); ++i) {
                if (i < taken && place + i < ray_limit[row]) {
                    const int number = noted + place + i, c = number / kChunkRecords;
                    const int64_t to = c == in ? ray_chunk[row] : ray_more[row] + (c - in - 1);
                    float2* const e = ws.base + to * kChunkFloat2 + (number - c * kChunkRecords) * 3;
                    const int of = lane | (from + i) << 6;
                    e[0] = make_float2(__int_as_float(lists.leaf[of]), lists.dt[of]);
                    e[1] = make_float2(lists.raw[of], lists.colour[of * 3]);
                    e[2] = make_float2(lists.colour[of * 3 + 1], lists.colour[of * 3 + 2]);
                }
            }
            wave_lds_sync();
        }
        if (active && (over || ended)) {
            if (kNoted && !kGrad && grad_out) {
                notes.finish_residual(broken && !ended, r.dscale, acc, light, bg, grad_out + slot * 3, out + slot * 3);
            } else {
                if (!painted) {
                    out[slot * 3] = fma_(light, bg, acc[0]);
                    out[slot * 3 + 1] = fma_(light, bg, acc[1]);
                    out[slot * 3 + 2] = fma_(light, bg, acc[2]);
                }
                if constexpr (kNoted) notes.finish(broken && !ended, r.dscale, kGrad ? sum1.end(bg) : 0.0f);
            }
            active = false;
        }
        if (!any_lane(active)) break;
        // the lists that were used up, and the rays that are over
        // (every lane takes part in both: a shuffle reads nothing from lanes that are left out)
        const int used = __shfl(empty, leader), goes_on = __shfl(active ? 1 : 0, leader);
        if (used == lane) count = shaded = 0;
        if (!goes_on) walking = false;
    }
}

}  // namespace svox
