// Many-query attention launchers (kernels in attw_kernels.h).
#include "launch.h"
#include "attw_kernels.h"

namespace fl {

namespace {

template <int NP, int D, bool CAREFUL>
hipError_t launch_one(hipStream_t st, const AttwArgs &a) {
    // three 64-key buffers, or the end's exchange of 4 x 64 x 34 floats
    constexpr size_t lds = std::max((size_t)3 * NP * 64 * D * 2, (size_t)34 * 256 * 4);
    const auto kern = k_attw<NP, D, CAREFUL>;
    const int items = (a.M + 31) / 32 * a.group;
    hipLaunchKernelGGL(kern, dim3((unsigned)((items + 3) / 4 * a.nkv)), dim3(512), lds, st, a);
    return hipGetLastError();
}

template <int NP, int D>
hipError_t launch_form(hipStream_t st, const AttwArgs &a) {
    return a.flag ? launch_one<NP, D, false>(st, a) : launch_one<NP, D, true>(st, a);
}

template <int FMT, int D>
hipError_t launch_split(hipStream_t st, const AttwSplitArgs &a) {
    const dim3 grid((a.T + 31) / 32, a.nkv);
    if (a.careful) hipLaunchKernelGGL((k_attw_split<FMT, D, true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_attw_split<FMT, D, false>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_attw(int planes, int D, hipStream_t st, const AttwArgs &a) {
    if (a.M < 1 || a.pos0 < 0 || a.nkv < 1 || a.group < 1 || a.slots < 32 || a.slots % 32 || a.pos0 + a.M > a.slots)
        return hipErrorInvalidValue;
    if (planes == 1) return D == 64 ? launch_form<1, 64>(st, a) : D == 128 ? launch_form<1, 128>(st, a) : hipErrorNotSupported;
    if (planes == 3) return D == 64 ? launch_form<3, 64>(st, a) : D == 128 ? launch_form<3, 128>(st, a) : hipErrorNotSupported;
    return hipErrorNotSupported;
}

hipError_t launch_attw_split(int kvfmt, int D, hipStream_t st, const AttwSplitArgs &a) {
    if (a.T < 1 || (D != 64 && D != 128)) return hipErrorInvalidValue;
    if (kvfmt == KV_F32) return D == 64 ? launch_split<0, 64>(st, a) : launch_split<0, 128>(st, a);
    if (kvfmt == KV_Q8) return D == 64 ? launch_split<1, 64>(st, a) : launch_split<1, 128>(st, a);
    return hipErrorNotSupported;
}

}  // namespace fl
