// Many-query attention launchers (kernels in attw_kernels.h).
#include <cmath>

#include "launch.h"
#include "attw_kernels.h"

namespace fl {

namespace {

int workgroups(int M, int nkv, int group) { return ((M + 31) / 32 * group + 3) / 4 * nkv; }

template <int NP, int D, bool CAREFUL>
hipError_t launch_one(hipStream_t st, const AttwArgs &a) {
    // three 64-key buffers, or the end's exchange of 4 x 64 x 34 floats
    constexpr size_t lds = std::max((size_t)3 * NP * 64 * D * 2, (size_t)34 * 256 * 4);
    const int n = workgroups(a.M, a.nkv, a.group);
    if (a.ksplit <= 1) {
        hipLaunchKernelGGL((k_attw<NP, D, CAREFUL, false>), dim3((unsigned)n), dim3(512), lds, st, a);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_attw<NP, D, CAREFUL, true>), dim3((unsigned)(n * a.ksplit)), dim3(512), lds, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_attw_merge<D>, dim3(pack_grid(a.M, (a.qstride + 1023) / 1024)), dim3(256), 0, st, a);
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

// Splits of the keys, where the workgroups leave CUs idle (one fills a CU).  A
// 64-key tile takes 1.3 us (D = 64) or 2.0 (D = 128) of a chain; the merge costs
// a launch and ~0.2 us per split, so about 2 sqrt(tiles) splits, and none where
// they would save less than that.  Measured on MI355X, 24 Q4_K layers of 1024
// channels, 32 prompt tokens behind 500 / 8000: 1550 / 5210 us whole, 1436 /
// 1692 split, 1432 / 1825 in a short pass.  (With a slower merge, 1500 / 1795;
// sqrt(2 tiles) splits 1535 / 1797, a split per 4 tiles 1550 / 1835, per 3 1520 /
// 1885.)
int attw_ksplit(int M, int pos0, int nkv, int group, int &chunk) {
    const int nit = (pos0 + M + 63) / 64;
    const int want = std::min({kAttwSplitWgs / workgroups(M, nkv, group), (int)(2 * std::sqrt((double)nit)), kAttwMaxSplit});
    chunk = nit * want >= 32 && want > 1 ? (nit + want - 1) / want : nit;
    return (nit + chunk - 1) / chunk;
}

// A workgroup has 128 rows of one head, so kAttwSplitWgs of them bound this.
size_t attw_split_floats(int D) { return (size_t)kAttwSplitWgs * 128 * (D + 2); }

hipError_t launch_attw(int planes, int D, hipStream_t st, const AttwArgs &a) {
    if (a.M < 1 || a.pos0 < 0 || a.nkv < 1 || a.group < 1 || a.slots < 32 || a.slots % 32 || a.pos0 + a.M > a.slots)
        return hipErrorInvalidValue;
    if (a.ksplit > 1 && (!a.part || !a.ml || a.chunk < 1 || a.ksplit * workgroups(a.M, a.nkv, a.group) > kAttwSplitWgs ||
                         (long long)a.ksplit * a.chunk * 64 < a.pos0 + a.M))
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
