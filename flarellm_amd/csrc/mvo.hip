// MFMA output projection (f32 input) launcher.
#include "launch.h"
#include "mvo_kernels.h"

namespace fl {

namespace {

// dynamic LDS of a launch; beside it lie the partial sums and the keys
inline size_t mvo_lds(int M, int K) { return (size_t)2 * M * (K + kMvoPad) * 2; }
constexpr size_t kMvoDynLds = 160 * 1024 - (2 * (kMvoThreads / 64) * 2 * 64 * 4 + 256);

template <int FMT, int KW, bool LONG>
hipError_t launch_one(hipStream_t st, const MvoArgs &a) {
    constexpr int tiles = kMvoThreads / 64 / KW;  // per workgroup
    const auto kern = k_mvo<FMT, KW, LONG>;
    const size_t lds = LONG ? (size_t)a.W.cols * 4 : mvo_lds(a.M, a.W.cols);
    const int want = ((a.W.rows + 15) / 16 + tiles - 1) / tiles;
    hipLaunchKernelGGL(kern, dim3(resident_grid(kern, kMvoThreads, lds, want)), dim3(kMvoThreads), lds, st, a);
    return hipGetLastError();
}

// As many tokens per launch as the LDS holds rows of (8 up to 4848 columns, 4 up
// to 9704, 2 up to 19416), in pieces of even size: each reads the whole weight.
// One token of more than 38840 columns: LONG (up to 40816).
template <int FMT, int KW>
hipError_t launch_pieces(hipStream_t st, const MvoArgs &a) {
    int m = a.M;
    while (m > 1 && mvo_lds(m, a.W.cols) > kMvoDynLds) m--;
    const bool fits = mvo_lds(m, a.W.cols) <= kMvoDynLds;
    const int n = (a.M + m - 1) / m;
    MvoArgs b = a;
    for (int i = 0, t0 = 0; i < n; t0 += b.M, i++) {
        b.M = (a.M - t0 + n - i - 1) / (n - i);
        b.x = a.x + (size_t)t0 * a.W.cols;
        if (a.out) b.out = a.out + (size_t)t0 * a.W.rows;
        if (a.slots) b.slots = a.slots + t0;
        hipError_t e = hipErrorInvalidValue;
        if (fits) e = launch_one<FMT, KW, false>(st, b);
        else if (KW == 8 && a.W.cols <= 40816) e = launch_one<FMT, 8, true>(st, b);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// every wave of a tile gets units: KW at most the row's 256-value units
template <int FMT>
hipError_t launch_fmt(hipStream_t st, const MvoArgs &a) {
    const int nu = (a.W.cols + 255) / 256;
    if (nu >= 8) return launch_pieces<FMT, 8>(st, a);
    return nu >= 4 ? launch_pieces<FMT, 4>(st, a) : launch_pieces<FMT, 2>(st, a);
}

}  // namespace

hipError_t launch_mvo(int fmt, hipStream_t st, const MvoArgs &a) {
    if (a.M < 1 || a.M > kMvoMaxTokens || (a.epi != EPI_STORE && a.epi != EPI_ARGMAX)) return hipErrorInvalidValue;
    if (fmt == F_Q6K) return a.W.cols % 256 ? hipErrorInvalidValue : launch_fmt<F_Q6K>(st, a);
    if (fmt == F_Q8_0) return a.W.cols % 32 ? hipErrorInvalidValue : launch_fmt<F_Q8_0>(st, a);
    return hipErrorNotSupported;
}

}  // namespace fl
