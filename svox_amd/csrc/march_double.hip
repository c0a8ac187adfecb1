// march_double.hip -- the double-precision march kernels of group_kernels.h and their launches.
#include <hip/hip_runtime.h>

#include "../../include/svox_hip.h"
#include "group_kernels.h"

namespace svox {

#define SVOX_GROUP_BASIS(D, ...)                              \
    switch (D) {                                              \
        case 0: { constexpr int kD = 0; __VA_ARGS__; } break; \
        case 1: { constexpr int kD = 1; __VA_ARGS__; } break; \
        case 4: { constexpr int kD = 4; __VA_ARGS__; } break; \
        case 9: { constexpr int kD = 9; __VA_ARGS__; } break; \
        case 16: { constexpr int kD = 16; __VA_ARGS__; } break; \
        default: { constexpr int kD = 25; __VA_ARGS__; } break; \
    }

template <class Source>
void launch_group_forward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                          const SvoxRenderOptions& opt, double* out, int per_wave, int most_cut) {
    SVOX_GROUP_BASIS(D, hipLaunchKernelGGL((render_group_kernel<kD, Source, false>), blocks, dim3(kMarchThreads), 0, stream, tr, src,
                                           opt, nullptr, out, per_wave, most_cut));
}
template <class Source>
void launch_shared_forward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                           const SvoxRenderOptions& opt, double* out) {
    SVOX_GROUP_BASIS(D, hipLaunchKernelGGL((render_forward_shared_kernel<kD, Source>), blocks, dim3(kMarchThreads), 0, stream, tr,
                                           src, opt, out));
}
template <class Source>
void launch_group_backward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                           const SvoxRenderOptions& opt, const double* grad_out, double* grad_data, int per_wave, int most_cut) {
    SVOX_GROUP_BASIS(D, hipLaunchKernelGGL((render_group_kernel<kD, Source, true>), blocks, dim3(kMarchThreads), 0, stream, tr, src,
                                           opt, grad_out, grad_data, per_wave, most_cut));
}

template <class Source>
void launch_shared_backward(int D, dim3 blocks, hipStream_t stream, const TreeDev<double>& tr, const Source& src,
                            const SvoxRenderOptions& opt, const double* grad_out, double* grad_data) {
    SVOX_GROUP_BASIS(D, hipLaunchKernelGGL((render_backward_shared_kernel<kD, Source>), blocks, dim3(kMarchThreads), 0, stream, tr,
                                           src, opt, grad_out, grad_data));
}

#define SVOX_GROUP_SOURCE(S)                                                                                               \
    template void launch_group_forward<S>(int, dim3, hipStream_t, const TreeDev<double>&, const S&, const SvoxRenderOptions&, \
                                          double*, int, int);                                                                        \
    template void launch_shared_forward<S>(int, dim3, hipStream_t, const TreeDev<double>&, const S&, const SvoxRenderOptions&, \
                                           double*);                                                                       \
    template void launch_group_backward<S>(int, dim3, hipStream_t, const TreeDev<double>&, const S&,                        \
                                           const SvoxRenderOptions&, const double*, double*, int, int);                    \
    template void launch_shared_backward<S>(int, dim3, hipStream_t, const TreeDev<double>&, const S&,                       \
                                            const SvoxRenderOptions&, const double*, double*);
SVOX_GROUP_SOURCE(BatchSource<double>)
SVOX_GROUP_SOURCE(ImageSource<double>)

}  // namespace svox
