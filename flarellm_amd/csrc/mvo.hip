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

// Waves per tile.  The time of a workgroup is its tiles (8 / kw at once, 256
// workgroups) times the values of its busiest wave, so a kw that leaves waves
// without a unit in the last round, or workgroups without a tile, loses.  The
// most waves that all get units (they read a row in one piece), unless another
// kw takes a tenth off.  Measured on MI355X, call time of 2 tokens with 8 (6
// units and less: 4, 3 and less: 2) waves against the kw taken: 64000 x 2304
// Q8_0 104.8 -> 84.0 us (1 wave), 100000 x 2304 Q6_K 104.6 -> 97.1 (2), 64000 x
// 3072 Q8_0 133.4 -> 114.2 (4), 64000 x 1536 Q8_0 88.8 -> 79.7 (2), 20000 x 576
// Q8_0 49.7 -> 47.8 (1), 8000 x 576 46.0 -> 44.8 (4).
int mvo_waves(int rows, int K) {
    const int tiles = (rows + 15) / 16, nu = (K + 255) / 256;
    if (mvo_lds(1, K) > kMvoDynLds) return 8;  // LONG
    auto cost = [&](int kw) {
        const int upw = (nu + kw - 1) / kw, slots = 256 * (8 / kw);
        const int values = (nu - 1) % kw ? upw * 256 : K - (nu - upw) * 256;  // of wave 0
        return (long long)((tiles + slots - 1) / slots) * values;
    };
    const int most = nu >= 8 ? 8 : nu >= 4 ? 4 : 2;
    int best = most;
    for (int kw : {8, 4, 2, 1})
        if (10 * cost(kw) <= 9 * cost(most) && cost(kw) < cost(best)) best = kw;
    return best;
}

template <int FMT>
hipError_t launch_fmt(hipStream_t st, const MvoArgs &a) {
    switch (mvo_waves(a.W.rows, a.W.cols)) {
    case 8: return launch_pieces<FMT, 8>(st, a);
    case 4: return launch_pieces<FMT, 4>(st, a);
    case 2: return launch_pieces<FMT, 2>(st, a);
    }
    return launch_pieces<FMT, 1>(st, a);
}

}  // namespace

hipError_t launch_mvo(int fmt, hipStream_t st, const MvoArgs &a) {
    if (a.M < 1 || a.M > kMvoMaxTokens || (a.epi != EPI_STORE && a.epi != EPI_ARGMAX)) return hipErrorInvalidValue;
    if (fmt == F_Q6K) return a.W.cols % 256 ? hipErrorInvalidValue : launch_fmt<F_Q6K>(st, a);
    if (fmt == F_Q8_0) return a.W.cols % 32 ? hipErrorInvalidValue : launch_fmt<F_Q8_0>(st, a);
    return hipErrorNotSupported;
}

}  // namespace fl
