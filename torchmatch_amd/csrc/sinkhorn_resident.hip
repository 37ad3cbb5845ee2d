// sinkhorn_resident.hip -- which solves run resident (sk_resident_kernel.h), on
// which tiles, and their launch.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include "../../include/torchmatch_amd.h"
#include "sk_resident.h"

namespace tmamd {
namespace {

constexpr int kCus = 256;
constexpr uint32_t kMaxPolls = 4u << 20;  // of 1 us or more each

// Words of the exchange buffer a problem in flight needs.
size_t xch_words(int G, int64_t Mp, bool f64) {
    const size_t xw = f64 ? 4 : 3, bw = 4;
    return 2 * ((size_t)G * xw + bw) * (size_t)Mp;
}

// Bytes of the problems' marks, behind it.
size_t mark_bytes(int64_t B) { return ((size_t)B * sizeof(uint32_t) + 15) / 16 * 16; }

const Tile &tile_of(int k, bool f64) {
    if (f64)
        return kTilesF64[k];
    return k < kNumTilesNarrow ? kTilesNarrow[k] : kTilesWide[k - kNumTilesNarrow];
}

} // namespace

SkResidentPlan sk_resident_plan(int64_t B, int64_t N, int64_t M, bool f64) {
    SkResidentPlan best{-1, 1, 0, 0, 1, 0};
    const char *env = getenv("TORCHMATCH_AMD_SINKHORN_RESIDENT");
    if (env != nullptr && strcmp(env, "0") == 0)
        return best;
    if (B < 1 || N < 1 || M < 1 || M > 4096 || N > (1 << 24))
        return best;
    const int n_tiles = f64 ? kNumTilesF64 : kNumTilesNarrow + kNumTilesWide;
    double best_t = 0.0;
    for (int k = 0; k < n_tiles; ++k) {
        const Tile &tl = tile_of(k, f64);
        const int64_t cw = tl.LC * tl.WC * tl.TC;
        const int64_t R = (tl.NW / tl.WC) * tl.TR * (tl.LC == 64 ? 1 : 4);
        const int64_t nt = 64 * tl.NW;  // columns a workgroup can own when it shares a problem
        if (M > cw)
            continue;
        int64_t G = (N + R - 1) / R;
        if (G > kCus)
            continue;
        if (G == 1 && (tl.WC > 2 || M > 4 * nt))
            G = N > 1 ? 2 : 0;  // (those tiles have no kernel for one workgroup)
        if (G == 0)
            continue;
        const int64_t rows = (N + G - 1) / G;
        G = (N + rows - 1) / rows;
        const int64_t cnp = (M + 63) / 64 * 64;
        const bool direct = G == 1 || (M <= nt && G * cnp <= 6144);
        if (!direct && ((M + G - 1) / G + 15) / 16 * 16 > nt)
            continue;
        const int64_t clusters = G == 1 ? B : (kCus / G < B ? kCus / G : B);
        // (workgroups of four waves fit a CU twice)
        const int64_t fit = tl.NW == 4 ? 2 * kCus : kCus;
        const int64_t rounds = G == 1 ? (B + fit - 1) / fit : (B + clusters - 1) / clusters;
        // us per step of one round, fitted to cycle counts of single phases at
        // (64, 64, 80), (8, 256, 256), (8, 500, 333), (1, 1024, 1024),
        // (16, 2048, 2048) and (1, 4096, 4096): the products and reductions of
        // a wave, then the column update (one workgroup), one exchange hop, or
        // two hops plus the partials' way to memory
        const double e = tl.TC * tl.TR * (f64 ? 2.0 : 1.0);
        const double mb = 8e-6 * (f64 ? 2.0 : 1.0) * (double)(clusters * G * M);
        const double step = (tl.NW == 4 ? 0.58 + 0.0060 * e : 0.83 + 0.0074 * e) +
                            (tl.WC > 1 ? 0.5 : 0.0) +
                            (G == 1 ? 0.5 : direct ? 2.0 + 0.1 * (double)G : 3.2 + 0.7 * mb);
        const double cost = step * (double)rounds;
        if (best.cfg < 0 || cost < best_t) {
            best_t = cost;
            best.cfg = k;
            best.G = (int)G;
            best.clusters = (int)(clusters < 0x7fffffff ? clusters : 0x7fffffff);
            best.rows = (int)rows;
            best.direct = direct ? 1 : 0;
            const int64_t Mp = (M + 15) / 16 * 16;
            best.xch_bytes =
                G == 1 ? 0
                       : sizeof(uint64_t) * xch_words((int)G, Mp, f64) * (size_t)clusters +
                             mark_bytes(B);
        }
    }
    // the streaming step: launches and merge, then 8.5 MB of the matrix a us
    // (fitted up to the Infinity Cache's size, which serves part of it; HBM alone
    // gives 6 to 7), read twice by the two-sweep form (float64, odd and short rows)
    const bool two = f64 || M % 4 != 0 || M < 128;
    const double mib = (f64 ? 8e-6 : 4e-6) * (double)(B * N * M);
    if (best.cfg >= 0 && best_t > 8.0 + mib / 8.5 * (two ? 2.0 : 1.0))
        best.cfg = -1;
    return best;
}

namespace {
__global__ void __launch_bounds__(256) sk_clear(uint4 *__restrict__ p, size_t n) {
    for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (size_t)gridDim.x * 256)
        p[k] = make_uint4(0, 0, 0, 0);
}
} // namespace

int sk_resident_launch(const SkResidentPlan &plan, const SkResidentIo &io, int64_t B, int64_t N,
                       int64_t M, const double *eps_sched, int32_t n_iter, double rho, bool f64,
                       hipStream_t stream) {
    if (plan.cfg < 0)
        return TM_ERR_UNSUPPORTED_SHAPE;
    ResArgs A;
    A.nseg = 0;
    for (int32_t s = 0; s < n_iter; ++s) {
        if (s == 0 || eps_sched[s] != eps_sched[s - 1]) {
            if (A.nseg == kSkMaxSegments)
                return TM_ERR_UNSUPPORTED_SHAPE;
            A.eps[A.nseg++] = eps_sched[s];
        }
        A.seg_end[A.nseg - 1] = s + 1;
    }
    const Tile &tl = tile_of(plan.cfg, f64);
    A.cost = io.cost;
    A.keep = io.keep;
    A.lmu = io.lmu;
    A.lnu = io.lnu;
    A.log_u = io.log_u;
    A.log_v = io.log_v;
    A.lu64 = io.lu64;
    A.lv64 = io.lv64;
    A.xch = static_cast<uint64_t *>(io.xch);
    A.B = B;
    A.N = (int)N;
    A.M = (int)M;
    A.Mp = (int)((M + 15) / 16 * 16);
    A.G = plan.G;
    A.clusters = plan.clusters;
    A.rows = plan.rows;
    A.direct = plan.direct;
    // column owners' ranges: whole 128-byte lines of words
    A.cpo = plan.direct ? (int)M : (int)(((M + plan.G - 1) / plan.G + 15) / 16 * 16);
    A.n_iter = n_iter;
    A.rho = rho;
    // "exact": every step from the cost (how the tests reach that path)
    const char *env = getenv("TORCHMATCH_AMD_SINKHORN_RESIDENT");
    A.exact_only = env != nullptr && strcmp(env, "exact") == 0;
    // "late": no wait at all, every shared problem is given up
    A.max_polls = env != nullptr && strcmp(env, "late") == 0 ? 0 : kMaxPolls;
    A.given_up = nullptr;
    if (plan.G > 1)
        A.given_up = reinterpret_cast<uint32_t *>(static_cast<char *>(io.xch) + plan.xch_bytes -
                                                  mark_bytes(B));
    // exchange numbers stay below 2^31: at most three per step
    const int64_t rounds = (B + plan.clusters - 1) / plan.clusters;
    if (plan.G > 1 && rounds * 3 * ((int64_t)n_iter + 1) >= (1ll << 30))
        return TM_ERR_UNSUPPORTED_SHAPE;
    void *args[] = {&A};
    if (plan.G == 1) {
        const int64_t grid = B < (1 << 20) ? B : (1 << 20);
        A.clusters = (int)grid;
        if (hipLaunchKernel(tl.solo, dim3((unsigned)grid), dim3((unsigned)tl.NW * 64), args, 0, stream) !=
            hipSuccess)
            return TM_ERR_LAUNCH;
        return TM_OK;
    }
    const size_t n16 = plan.xch_bytes / 16;
    hipLaunchKernelGGL(sk_clear, dim3((unsigned)(n16 / 256 + 1 < 2048 ? n16 / 256 + 1 : 2048)),
                       dim3(256), 0, stream, static_cast<uint4 *>(io.xch), n16);
    if (hipGetLastError() != hipSuccess)
        return TM_ERR_LAUNCH;
    if (hipLaunchCooperativeKernel(tl.shared, dim3((unsigned)(plan.clusters * plan.G)),
                                   dim3((unsigned)tl.NW * 64), args, 0, stream) != hipSuccess) {
        (void)hipGetLastError();
        return TM_ERR_UNSUPPORTED_SHAPE;
    }
    return TM_OK;
}

} // namespace tmamd
