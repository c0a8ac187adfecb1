// march_policy.hip -- the march kernels of one policy.  build.py compiles this file once per record format and basis
// size, with SVOX_POLICY_FORMAT (SVOX_FORMAT_RGBA, _SH or _SG) and SVOX_POLICY_BASIS defined.
#include <hip/hip_runtime.h>

#include "../../include/svox_hip.h"

#define SVOX_INSTANTIATE_POLICY
#include "march_launch.h"

namespace svox {
template struct MarchLaunch<OctreePolicy<SVOX_POLICY_FORMAT, SVOX_POLICY_BASIS>, BatchSource<float>>;
template struct MarchLaunch<OctreePolicy<SVOX_POLICY_FORMAT, SVOX_POLICY_BASIS>, ImageSource<float>>;
template void MarchLaunch<OctreePolicy<SVOX_POLICY_FORMAT, SVOX_POLICY_BASIS>, ListedSource>::noting(
    dim3, hipStream_t, const TreeDev<float>&, const ListedSource&, const SvoxRenderOptions&, float*, const ReplaySpace&, const float*,
    const float*, bool, bool);
template void MarchLaunch<OctreePolicy<SVOX_POLICY_FORMAT, SVOX_POLICY_BASIS>, WholeSource>::noting(
    dim3, hipStream_t, const TreeDev<float>&, const WholeSource&, const SvoxRenderOptions&, float*, const ReplaySpace&, const float*,
    const float*, bool, bool);
template void MarchLaunch<OctreePolicy<SVOX_POLICY_FORMAT, SVOX_POLICY_BASIS>, ListedImageSource>::noting(
    dim3, hipStream_t, const TreeDev<float>&, const ListedImageSource&, const SvoxRenderOptions&, float*, const ReplaySpace&, const float*,
    const float*, bool, bool);
template void MarchLaunch<OctreePolicy<SVOX_POLICY_FORMAT, SVOX_POLICY_BASIS>, WholeImageSource>::noting(
    dim3, hipStream_t, const TreeDev<float>&, const WholeImageSource&, const SvoxRenderOptions&, float*, const ReplaySpace&, const float*,
    const float*, bool, bool);
}  // namespace svox
