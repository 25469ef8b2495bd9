// Large-batch GEMM launchers (kernels in bgemm_kernels.h).
#include "launch.h"
#include "bgemm_kernels.h"

namespace fl {

namespace {

template <int FMT, int TT, int NW>
hipError_t launch_one(hipStream_t st, const BgArgs &a) {
    constexpr size_t lds = (size_t)2 * TT * kPackRec + (FMT == F_Q4K ? NW * 32 * 4 : 0);
    const auto kern = k_bgemm<FMT, TT, NW>;
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.nrt * a.ntt * a.ksplit)), dim3(NW * 64), lds, st, a);
    return hipGetLastError();
}

template <int FMT>
hipError_t launch_tt(int tt, int nw, hipStream_t st, const BgArgs &a) {
    switch (10 * tt + nw) {
    case 14: return launch_one<FMT, 1, 4>(st, a);
    case 24: return launch_one<FMT, 2, 4>(st, a);
    case 28: return launch_one<FMT, 2, 8>(st, a);
    case 38: return launch_one<FMT, 3, 8>(st, a);
    case 48: return launch_one<FMT, 4, 8>(st, a);
    }
    return hipErrorInvalidValue;
}

}  // namespace

// The plan of least estimated time.  A workgroup of 8 waves (2 token tiles or
// more: with one, two workgroups of 4 waves always cost less), or two of 4 waves
// with at most 2 token tiles, fills a CU.  The costs are a least-squares fit to
// the times of all plans of 14 shapes on MI355X (576 x 576 to 14336 x 4096 and
// 4096 x 14336, 32 to 2048 tokens; 6 to 7 % mean error): per 256-value step,
// per round of the chip, and per MB of partial sums written; two workgroups of
// 4 waves are priced 10 % above the fit, which let them take near ties that
// they lose.  Split sums also cost their read (4 TB/s) and, unless the kernel
// behind sums them in any case (summed), a launch of 4 us.  Over those shapes
// and 15 others the plan taken is 1 to 2 % above the best; one cost per step
// for both formats and wave counts was 8 to 9 % above (4096 x 4096 Q4_K, 509
// tokens: 52 us unsplit where 33 are reached).
// Q8_0 sums every 32-block straight into its output, so a split holds at most
// kQ8Steps steps (7168 values: 1.4e-7 against 64 bits where 14336 in one chain
// had 2.0e-7).
constexpr int kQ8Steps = 28;
struct BgCost {
    double step8[3];  // 8 waves: us per step with 2..4 token tiles
    double step4[2];  // 4 waves, two workgroups on a CU
    double alone[2];  // 4 waves, one on a CU
    double round, mb;
};
constexpr BgCost kCostQ8{{4.27, 5.32, 6.71}, {3.34, 4.35}, {2.30, 3.21}, 2.3, 0.165};
constexpr BgCost kCostQ4{{3.52, 4.57, 5.81}, {2.43, 3.63}, {1.72, 2.53}, 1.6, 0.126};
BgPlan bgemm_plan(int fmt, int rows, int cols, int M, bool summed) {
    const BgCost &c = fmt == F_Q8_0 ? kCostQ8 : kCostQ4;
    const double mb = (double)M * rows * 4 / 1e6;
    const int tiles = (M + kPackTile - 1) / kPackTile, nst = (cols + 255) / 256;
    BgPlan best{};
    double best_us = 0;
    for (int tt = 1; tt <= std::min(4, tiles); tt++)
        for (int nw = tt == 1 ? 4 : 8; nw >= (tt <= 2 ? 4 : 8); nw /= 2)
            for (int want = 1; want <= std::min(nst, kBgMaxSplit); want++) {
                BgPlan p;
                p.tt = tt;
                p.nw = nw;
                p.ntt = (tiles + tt - 1) / tt;
                p.nrt = (rows + 32 * nw - 1) / (32 * nw);
                p.chunk = (nst + want - 1) / want;
                p.ksplit = (nst + p.chunk - 1) / p.chunk;
                if (p.ksplit != want || (fmt == F_Q8_0 && p.chunk > kQ8Steps)) continue;
                const long long wgs = (long long)p.nrt * p.ntt * p.ksplit, slots = nw == 8 ? 256 : 512;
                const double step = nw == 8 ? c.step8[tt - 2] : wgs <= 256 ? c.alone[tt - 1] : c.step4[tt - 1];
                double us = (double)((wgs + slots - 1) / slots) * (p.chunk * step + c.round) + p.ksplit * mb * c.mb;
                if (p.ksplit > 1) us += summed ? (p.ksplit - 1) * mb / 4 : 4.0 + p.ksplit * mb / 4;
                if (!best.tt || us < best_us) {
                    best = p;
                    best_us = us;
                }
            }
    return best;
}

hipError_t launch_bgemm(int fmt, hipStream_t st, const WDesc &W, const char *xp, int M, const BgPlan &p, float *part) {
    if (M < 1 || W.rows < 1 || W.cols % 32 || (fmt == F_Q4K && W.cols % 256)) return hipErrorInvalidValue;
    BgArgs a{};
    a.W = W;
    a.xp = xp;
    a.M = M;
    a.nst = (W.cols + 255) / 256;
    a.ksplit = p.ksplit;
    a.chunk = p.chunk;
    a.part = part;
    a.nrt = p.nrt;
    a.ntt = p.ntt;
    if (pack_bytes(M, W.cols) >> 32) return hipErrorInvalidValue;  // 32-bit offsets
    // every row, token and step belongs to a workgroup, every split has steps
    if ((long long)p.nrt * p.nw * 32 < W.rows || (long long)p.ntt * p.tt * kPackTile < M ||
        (long long)p.ksplit * p.chunk < a.nst || (long long)(p.ksplit - 1) * p.chunk >= a.nst)
        return hipErrorInvalidValue;
    if (fmt == F_Q4K) return launch_tt<F_Q4K>(p.tt, p.nw, st, a);
    if (fmt == F_Q8_0) return launch_tt<F_Q8_0>(p.tt, p.nw, st, a);
    return hipErrorNotSupported;
}

hipError_t launch_quant_pack(hipStream_t st, const float *x, int M, int K, char *xp) {
    if (M < 1 || K < 32 || K % 32) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_quant_pack, dim3((M + kPackTile - 1) / kPackTile, (K / 32 + 3) / 4), dim3(256), 0, st, x, M, K,
                       (K + 255) / 256, xp);
    return hipGetLastError();
}

hipError_t launch_b_resnorm(int pro, hipStream_t st, const float *part, int ksplit, int M, int H, float *x,
                            const float *w, float eps, char *xp) {
    if (H % 32 || H > kResnormMaxH || M < 1) return hipErrorInvalidValue;
    const auto kern = pro == PRO_NORMQ0 ? k_b_resnorm<PRO_NORMQ0> : k_b_resnorm<PRO_NORMQ1>;
    hipLaunchKernelGGL(kern, dim3(pack_grid(M, 1)), dim3(kResnormThreads), 0, st, part, ksplit, M, H, x, w, eps,
                       (H + 255) / 256, xp);
    return hipGetLastError();
}

hipError_t launch_b_residual_row(hipStream_t st, const float *part, int ksplit, size_t plane, int H, float *x) {
    hipLaunchKernelGGL(k_b_residual_row, dim3((H + 255) / 256), dim3(256), 0, st, part, ksplit, plane, H, x);
    return hipGetLastError();
}

hipError_t launch_b_silu(hipStream_t st, const float *part, int ksplit, int M, int F, char *xp) {
    if (F % 32 || M < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_b_silu, dim3(pack_grid(M, (F + 1023) / 1024)), dim3(256), 0, st, part, ksplit, M, F,
                       (F + 255) / 256, xp);
    return hipGetLastError();
}

}  // namespace fl
