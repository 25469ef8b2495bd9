// Many-query attention launchers (kernels in attw_kernels.h).
#include "launch.h"
#include "attw_kernels.h"

namespace fl {

namespace {

template <int NP, int D>
hipError_t launch_one(hipStream_t st, const AttwArgs &a) {
    // three 64-key buffers, or the end's exchange of 4 x 64 x 34 floats
    constexpr size_t lds = std::max((size_t)3 * NP * 64 * D * 2, (size_t)34 * 256 * 4);
    const auto kern = k_attw<NP, D>;
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return attr;
    const int items = (a.M + 31) / 32 * a.group;
    hipLaunchKernelGGL(kern, dim3((unsigned)((items + 3) / 4 * a.nkv)), dim3(512), lds, st, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_attw(int planes, int D, hipStream_t st, const AttwArgs &a) {
    if (a.M < 1 || a.pos0 < 0 || a.nkv < 1 || a.group < 1 || a.slots < 32 || a.slots % 32 || a.pos0 + a.M > a.slots)
        return hipErrorInvalidValue;
    if (planes == 1) return D == 64 ? launch_one<1, 64>(st, a) : D == 128 ? launch_one<1, 128>(st, a) : hipErrorNotSupported;
    if (planes == 3) return D == 64 ? launch_one<3, 64>(st, a) : D == 128 ? launch_one<3, 128>(st, a) : hipErrorNotSupported;
    return hipErrorNotSupported;
}

hipError_t launch_attw_split(int kvfmt, int D, hipStream_t st, const AttwSplitArgs &a) {
    const dim3 grid((a.T + 31) / 32, a.nkv);
    if (a.T < 1 || (D != 64 && D != 128)) return hipErrorInvalidValue;
    if (kvfmt == KV_F32) {
        if (D == 64) hipLaunchKernelGGL((k_attw_split<0, 64>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_attw_split<0, 128>), grid, dim3(256), 0, st, a);
    } else if (kvfmt == KV_Q8) {
        if (D == 64) hipLaunchKernelGGL((k_attw_split<1, 64>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_attw_split<1, 128>), grid, dim3(256), 0, st, a);
    } else {
        return hipErrorNotSupported;
    }
    return hipGetLastError();
}

}  // namespace fl
