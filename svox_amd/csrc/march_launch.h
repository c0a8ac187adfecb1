// march_launch.h -- the launches of the wavefront-per-tile march kernels, one class per policy and ray source.
//
// The kernels of march_kernels.h are templates over the record's format and basis size.  Every policy is compiled in
// a translation unit of its own (march_policy.hip, once per format and basis size: build.py), so that a build takes
// as long as its slowest policy and not as long as their sum; svox_hip.hip picks the policy at run time
// (SVOX_DISPATCH_OCTREE) and calls these functions.
#pragma once

#include <type_traits>

#include "cut_kernel.h"
#include "march_kernels.h"

namespace svox {

template <class P, class Source>
struct MarchLaunch {
    // How many tiles of a forward launch (noting: one that takes notes; graded: with the gradient at hand) the GPU holds at once
    // with two wavefronts to a tile.
    static unsigned split_tiles_at_once(bool noting, bool graded);
    static void forward(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                        const SvoxRenderOptions& opt, float* out, const ReplaySpace& ws, bool split, bool accum, bool refill,
                        bool all_shaded);
    static void noting(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                       const SvoxRenderOptions& opt, float* out, const ReplaySpace& ws, const float* grad_out,
                       const float* color_ref, bool split, bool refill);
    // either of them with every ray cut into pieces (cut_kernel.h), per_wave rays to a wavefront, 2^most_cut pieces at most
    static void cut(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src, const SvoxRenderOptions& opt,
                    float* out, const ReplaySpace& ws, bool noted, const float* grad_out, const float* color_ref, int per_wave, int most_cut);
    static void backward(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                         const SvoxRenderOptions& opt, const float* grad_out, float* grad_data, const ReplaySpace& ws,
                         bool refill, bool second_only);
    static void replay_backward(dim3 blocks, hipStream_t stream, const Source& src, const SvoxRenderOptions& opt,
                                const float* grad_out, float* grad_data, const ReplaySpace& ws, int ray_shift,
                                const Lobes& lobes);
    static void se_grad(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                        const SvoxRenderOptions& opt, const float* color_ref, float* color_out, float* grad, float* hess,
                        const unsigned long long* only, const unsigned long long* any_undone, bool refill);
    static void replay_se_grad(dim3 blocks, hipStream_t stream, const Source& src, const SvoxRenderOptions& opt,
                               float* grad, float* hess, const ReplaySpace& ws, int ray_shift, const Lobes& lobes);
};

#ifdef SVOX_INSTANTIATE_POLICY
// What the runtime tells of the kernel's registers -- 12 tiles to a CU up to 80 of them, 10 up to 96, 8 up to 128 -- but not more
// than 12, which is all the LDS holds (12.25 KiB a tile and more).
template <class P, class Source>
unsigned MarchLaunch<P, Source>::split_tiles_at_once(bool noting, bool graded) {
    auto tiles = [](auto* kernel) {
        constexpr unsigned kCus = 256, kMost = 12;
        int blocks = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, kSplitThreads, 0) != hipSuccess) {
            (void)hipGetLastError();
            blocks = 8;
        }
        return kCus * ((unsigned)blocks < kMost ? (unsigned)blocks : kMost);
    };
    if (noting && graded) {
        static const unsigned n = tiles(render_forward_split_kernel<P, Source, true, true>);
        return n;
    }
    if (noting) {
        static const unsigned n = tiles(render_forward_split_kernel<P, Source, true, false>);
        return n;
    }
    static const unsigned n = tiles(render_forward_split_kernel<P, Source, false>);
    return n;
}

template <class P, class Source>
void MarchLaunch<P, Source>::forward(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                                     const SvoxRenderOptions& opt, float* out, const ReplaySpace& ws, bool split, bool accum,
                                     bool refill, bool all_shaded) {
    const float* const no_grad = nullptr;
#define SVOX_FORWARD(ACCUM, REFILL, ALL)                                                                              \
    hipLaunchKernelGGL((render_forward_kernel<P, Source, ACCUM, REFILL, false, false, ALL>), blocks,                  \
                       dim3(kMarchThreads), 0, stream, tr, src, opt, out, ws, no_grad)
    if (split)
        hipLaunchKernelGGL((render_forward_split_kernel<P, Source, false>), blocks, dim3(kSplitThreads), 0, stream, tr, src,
                           opt, out, ws, no_grad);
    else if (accum)
        SVOX_FORWARD(true, true, false);   // (accumulation is an analysis pass: one variant is enough)
    else if (refill && all_shaded)
        SVOX_FORWARD(false, true, true);
    else if (refill)
        SVOX_FORWARD(false, true, false);
    else if (all_shaded)
        SVOX_FORWARD(false, false, true);
    else
        SVOX_FORWARD(false, false, false);
#undef SVOX_FORWARD
}

template <class P, class Source>
void MarchLaunch<P, Source>::noting(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                                    const SvoxRenderOptions& opt, float* out, const ReplaySpace& ws, const float* grad_out,
                                    const float* color_ref, bool split, bool refill) {
    // (the colours take the gradient's place in the variants without it)
#define SVOX_NOTING(THREADS, ...)                                                                                        \
    hipLaunchKernelGGL((__VA_ARGS__), blocks, dim3(THREADS), 0, stream, tr, src, opt, out, ws, grad_out ? grad_out : color_ref)
    constexpr bool kListed = std::is_same<Source, ListedSource>::value;   // (marched tile by tile)
    constexpr bool kWhole = std::is_same<Source, WholeSource>::value;     // (on one wavefront per tile or chunk)
    constexpr bool kPixels = Source::kGated && !Source::kItemsAreSlots;   // (on two wavefronts per tile)
    if (split) {
        if constexpr (!kWhole) {
            if (grad_out)
                SVOX_NOTING(kSplitThreads, render_forward_split_kernel<P, Source, true, true>);
            else
                SVOX_NOTING(kSplitThreads, render_forward_split_kernel<P, Source, true, false>);
        }
    } else if constexpr (!kPixels) {
        if (refill) {
            if constexpr (!kListed) {
                if (grad_out)
                    SVOX_NOTING(kMarchThreads, render_forward_kernel<P, Source, false, true, true, true>);
                else
                    SVOX_NOTING(kMarchThreads, render_forward_kernel<P, Source, false, true, true, false>);
            }
        } else if (grad_out)
            SVOX_NOTING(kMarchThreads, render_forward_kernel<P, Source, false, false, true, true>);
        else
            SVOX_NOTING(kMarchThreads, render_forward_kernel<P, Source, false, false, true, false>);
    }
#undef SVOX_NOTING
}

template <class P, class Source>
void MarchLaunch<P, Source>::cut(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                                 const SvoxRenderOptions& opt, float* out, const ReplaySpace& ws, bool noted,
                                 const float* grad_out, const float* color_ref, int per_wave, int most_cut) {
#define SVOX_CUT(...)                                                                                                \
    hipLaunchKernelGGL((render_forward_cut_kernel<P, Source, __VA_ARGS__>), blocks, dim3(kMarchThreads), 0, stream, tr, src, opt, out, \
                       ws, grad_out ? grad_out : color_ref, per_wave, most_cut)
    if (noted && grad_out)
        SVOX_CUT(true, true);
    else if (noted)
        SVOX_CUT(true, false);
    else
        SVOX_CUT(false, false);
#undef SVOX_CUT
}

template <class P, class Source>
void MarchLaunch<P, Source>::backward(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                                      const SvoxRenderOptions& opt, const float* grad_out, float* grad_data,
                                      const ReplaySpace& ws, bool refill, bool second_only) {
#define SVOX_BACKWARD(REFILL, MODE)                                                                                   \
    hipLaunchKernelGGL((render_backward_kernel<P, Source, REFILL, MODE>), blocks, dim3(kMarchThreads), 0, stream, tr, \
                       src, opt, grad_out, grad_data, ws)
    if (refill && second_only)
        SVOX_BACKWARD(true, kBackwardSecond);
    else if (refill)
        SVOX_BACKWARD(true, kBackwardPlain);
    else if (second_only)
        SVOX_BACKWARD(false, kBackwardSecond);
    else
        SVOX_BACKWARD(false, kBackwardPlain);
#undef SVOX_BACKWARD
}

template <class P, class Source>
void MarchLaunch<P, Source>::replay_backward(dim3 blocks, hipStream_t stream, const Source& src,
                                             const SvoxRenderOptions& opt, const float* grad_out, float* grad_data,
                                             const ReplaySpace& ws, int ray_shift, const Lobes& lobes) {
    hipLaunchKernelGGL((replay_backward_kernel<P, Source>), blocks, dim3(kReplayThreads), 0, stream, src, opt, grad_out,
                       grad_data, ws, ray_shift, lobes);
}

template <class P, class Source>
void MarchLaunch<P, Source>::se_grad(dim3 blocks, hipStream_t stream, const TreeDev<float>& tr, const Source& src,
                                     const SvoxRenderOptions& opt, const float* color_ref, float* color_out, float* grad,
                                     float* hess, const unsigned long long* only, const unsigned long long* any_undone, bool refill) {
    if (refill)
        hipLaunchKernelGGL((se_grad_kernel<P, Source, true>), blocks, dim3(kMarchThreads), 0, stream, tr, src, opt,
                           color_ref, color_out, grad, hess, only, any_undone);
    else
        hipLaunchKernelGGL((se_grad_kernel<P, Source, false>), blocks, dim3(kMarchThreads), 0, stream, tr, src, opt,
                           color_ref, color_out, grad, hess, only, any_undone);
}

template <class P, class Source>
void MarchLaunch<P, Source>::replay_se_grad(dim3 blocks, hipStream_t stream, const Source& src,
                                            const SvoxRenderOptions& opt, float* grad, float* hess,
                                            const ReplaySpace& ws, int ray_shift, const Lobes& lobes) {
    hipLaunchKernelGGL((replay_se_grad_kernel<P, Source>), blocks, dim3(kReplayThreads), 0, stream, src, opt, grad, hess,
                       ws, ray_shift, lobes);
}
#endif  // SVOX_INSTANTIATE_POLICY

}  // namespace svox
