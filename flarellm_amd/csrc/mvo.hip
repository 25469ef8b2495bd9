// MFMA output projection (f32 input) launcher.
#include "launch.h"
#include "mvo_kernels.h"

namespace fl {

namespace {

constexpr size_t kMvoMaxLds = 160 * 1024, kMvoStaticLds = 2 * (kMvoThreads / 64) * 2 * 64 * 4 + 512;  // part and lb of k_mvo

template <int FMT, int KW>
hipError_t launch_one(hipStream_t st, const MvoArgs &a) {
    // 2M activation rows and, below 16, a zero row
    const size_t lds = (size_t)std::min(16, 2 * a.M + 1) * (a.W.cols + kMvoPad) * 2;
    if (lds + kMvoStaticLds > kMvoMaxLds && a.M > 4) {
        // rows too long for 8 tokens beside the partial sums: two launches
        MvoArgs b = a;
        b.M = 4;
        const hipError_t e = launch_one<FMT, KW>(st, b);
        if (e != hipSuccess) return e;
        b.M = a.M - 4;
        b.x = a.x + (size_t)4 * a.W.cols;
        if (a.out) b.out = a.out + (size_t)4 * a.W.rows;
        if (a.slots) b.slots = a.slots + 4;
        return launch_one<FMT, KW>(st, b);
    }
    constexpr int tiles = kMvoThreads / 64 / KW;  // per workgroup
    const auto kern = k_mvo<FMT, KW>;
    const int want = ((a.W.rows + 15) / 16 + tiles - 1) / tiles;
    hipLaunchKernelGGL(kern, dim3(resident_grid(kern, kMvoThreads, lds, want)), dim3(kMvoThreads), lds, st, a);
    return hipGetLastError();
}

// every wave of a tile gets units: KW at most the row's 256-value units
template <int FMT>
hipError_t launch_fmt(hipStream_t st, const MvoArgs &a) {
    const int nu = (a.W.cols + 255) / 256;
    if (nu >= 8) return launch_one<FMT, 8>(st, a);
    return nu >= 4 ? launch_one<FMT, 4>(st, a) : launch_one<FMT, 2>(st, a);
}

}  // namespace

hipError_t launch_mvo(int fmt, hipStream_t st, const MvoArgs &a) {
    if (a.M < 1 || a.M > kMvoMaxTokens) return hipErrorInvalidValue;
    if (fmt == F_Q6K) return a.W.cols % 256 ? hipErrorInvalidValue : launch_fmt<F_Q6K>(st, a);
    if (fmt == F_Q8_0) return a.W.cols % 32 ? hipErrorInvalidValue : launch_fmt<F_Q8_0>(st, a);
    return hipErrorNotSupported;
}

}  // namespace fl
