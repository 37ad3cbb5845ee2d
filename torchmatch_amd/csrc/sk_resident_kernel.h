// sk_resident_kernel.h -- the whole Sinkhorn iteration in one launch, with the
// matrix held in registers (gfx950).  Included by the sk_tiles_*.hip files, which
// instantiate the tile configurations.
//
// A solve that launches one or two kernels per step is bound by those
// launches (about 5 us each, 10 us per step) whenever the matrix is small, and
// by re-reading the matrix when it is not.  256 CUs hold 128 MiB of VGPRs, so
// here a problem's matrix is loaded once into the registers of G workgroups
// and every step runs from there.
//
// The step.  With reference potentials (rl_i, c_j) the workgroups hold
//     P_ij = e^(K_ij - rl_i - c_j)         K = -C / eps
// and the potentials as multipliers a_i = e^(log_u_i + rl_i), b_j =
// e^(log_v_j + c_j), so that the two half-steps of the log-domain iteration
// are two matrix-vector products and no exponential:
//     LSE_j(K_ij + log_v_j) = rl_i + log S_i     S_i = sum_j P_ij b_j
//     LSE_i(K_ij + log_u_i) = c_j  + log T_j     T_j = sum_i P_ij a_i
// and, balanced, a_i = mu_i / S_i, b_j = nu_j / T_j.  Unbalanced, the potentials
// themselves are kept too (log_u and log_v in float64): they are damped, so a
// multiplier is not near its marginal but as small as the plan's mass, which
// large costs take out of any float's range.  A scale kappa common to the
// problem is therefore taken out there, P = e^(K - rl - c + kappa), a =
// e^(log_u + rl - kappa), b = e^(log_v + c - kappa) (0 for balanced solves): the
// exact step sets it to the largest column's, so that the columns' and rows'
// multipliers lie around 1 whatever the mass.  P is rounded to float32
// once (relative 2^-24 per entry; the K of the streaming step is rounded to
// float32 at |K| ~ 40, about 2^-19), lane sums are float32 of TC or TR terms,
// sums across lanes and waves and the multipliers are float64.  The float32
// copies of a and b that the products read carry their rounding error over
// to the next step's rounding (ea, eb), so that a fixed rounding of a
// converged multiplier does not drive the potentials' neutral mode
// (log_u + c, log_v - c) step after step.
//
// When that is exact enough.  P is denormal below 2^-126, off by at most 2^-150
// an entry; a step is accepted only while every S_i and T_j lies in [2^-60,
// 2^60] and every multiplier its sums use is at most 2^40, so that what is lost
// is below 2^-150 2^40 2^17 (rows a problem may have) 2^60 = 2^-33 of a sum.
// (The first step is a trial from P around the row maxima; its column multipliers
// may go to 2^60, P is rebuilt around them before they are used.)  A step outside
// the window is done exactly from the cost, with the maximum taken out of every
// sum, the reference's logsumexp, and P is rebuilt around the new potentials.
// Multipliers have no lower bound: a tiny one is denormal, off by
// 2^-150, in the float32 copy that the products read, which is at most 2^-150 P of
// a sum.  So a P with an entry above 2^60 is refused (its row and its column both
// carry less than 2^-60 of the mass, or of the largest column's where there is a
// kappa).  A row or column whose LSE is not finite keeps its potential, as the
// reference's isfinite rule has it.  When epsilon changes, P is rebuilt
// from the cost around the current potentials and the step goes on.
//
// Several workgroups per problem.  Each holds `rows` whole rows, so the row
// half-step is local; the column sums are exchanged through global memory in
// 64-bit words that carry 32 bits of payload and the number of the exchange,
// written and polled with relaxed agent-scope atomics.  A word is its own
// flag: no fence and no L2 write-back is needed, and double buffering by the
// exchange's parity keeps a slot until every reader has moved on.  With few
// columns every workgroup merges all of them (one hop, `direct`); else
// workgroup g owns a range of columns, merges it and sends its multipliers to
// the others (two hops).  Such a grid is launched cooperatively, which
// guarantees that all its workgroups become resident; when the last of them does
// is up to whatever else runs on the device.  Every wait is bounded all the
// same, in polls (time in which a wave does not run itself does not count): a
// workgroup whose wait has lasted 4 million of them, some seconds, gives its
// problem up, and whoever is the first to do so marks it for the others and
// solves it alone from the cost (redo_problem).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <utility>

#include "sk_math.h"
#include "sk_resident.h"
#include "wave.h"

namespace tmamd {
namespace {

constexpr double kSumLo = 0x1p-60, kSumHi = 0x1p60, kMulHi = 0x1p40;
// P above this is refused (kPHi<double>: doubles underflow at 2^-1022); a balanced
// entry of P is below 1 / mu of its row, so rows above kMassLo need no look
template <typename T> constexpr T kPHi = (T)0x1p60;
template <> constexpr double kPHi<double> = 0x1p900;
constexpr double kMassLo = 0x1p-40;
// float multipliers below this carry no rounding (their reciprocal overflows)
constexpr float kCarryLo = 0x1p-120f;

// (a - b) - d, d = a - b rounded (NaN or infinity where one of them is).
__device__ __forceinline__ double diff_error(double a, double b, double d) {
    const double bb = a - d;
    return (a - (d + bb)) + (bb - b);
}

// damp * (lm - (ls + r)) with one rounding in place of three (float64 results).
__device__ __forceinline__ double damped_potential(double damp, double lm, double ls, double r) {
    const double t = ls + r, d = lm - t;
    const double e = diff_error(lm, t, d) - diff_error(ls, -r, t);
    return isfinite(e) ? fma(damp, d, damp * e) : damp * d;
}

// The log unit of each type: base 2 on the native v_exp_f32 for float costs,
// natural with the library's exp / log for double costs.
template <typename T> struct Unit;
template <> struct Unit<float> {
    static constexpr int kPartWords = 1;
    double s2;
    __device__ explicit Unit(double eps) : s2(-kLog2eD / (double)(float)eps) {}
    __device__ double kval(float c) const { return (double)c * s2; }
    static __device__ float term(double t) { return __builtin_amdgcn_exp2f((float)t); }
    static __device__ double logm(double s) { return log2(s); }
    static __device__ double expm(double t) { return exp2(t); }
    static __device__ double log_fast(double s) { return log2_of_sum(s); }
    static __device__ double exp_fast(double t) { return (double)pow2_of(t); }
    // 1 / s: one Newton step on the native reciprocal (about 2^-46)
    static __device__ double recip(double s) {
        const double r = __builtin_amdgcn_rcp(s);
        return fma(fma(-s, r, 1.0), r, r);
    }
    static __device__ double of_nat(double x) { return x * kLog2eD; }
    static __device__ double to_nat(double x) { return x * kLn2D; }
    static __device__ double of_exp2(int e) { return (double)e; }
    // P from its exponent K - l - c, |error| about one ulp (NaN stays NaN)
    static __device__ float build(double k, double l, double c) {
        double t = (k - l) - c;
        t = t < -300.0 ? -300.0 : t;
        const double ti = rint(t);
        return ldexpf(__builtin_amdgcn_exp2f((float)(t - ti)), (int)fmin(ti, 300.0));
    }
};
template <> struct Unit<double> {
    static constexpr int kPartWords = 2;
    double eps;
    __device__ explicit Unit(double e) : eps(e) {}
    __device__ double kval(double c) const { return -c / eps; }
    static __device__ double term(double t) { return exp(t); }
    static __device__ double logm(double s) { return log(s); }
    static __device__ double expm(double t) { return exp(t); }
    static __device__ double log_fast(double s) { return log(s); }
    static __device__ double exp_fast(double t) { return exp(t); }
    static __device__ double recip(double s) { return 1.0 / s; }
    static __device__ double of_nat(double x) { return x; }
    static __device__ double to_nat(double x) { return x; }
    static __device__ double of_exp2(int e) { return (double)e * kLn2D; }
    // With what the two differences round off, which at |K| of 40 is up to 16 ulps
    // of P in every step until P is built again.
    static __device__ double build(double k, double l, double c) {
        const double t = k - l, x = t - c;
        const double p = exp(x), e = diff_error(k, l, t) + diff_error(t, c, x);
        return isfinite(e) ? fma(p, e, p) : p;
    }
};

__device__ __forceinline__ double shift_of(double m) { return isinf(m) ? 0.0 : m; }

// Doubles as integers of the same order (for an integer maximum in LDS).
__device__ __forceinline__ uint64_t order_key(double x) {
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    return (u >> 63) != 0 ? ~u : u | (1ull << 63);
}
__device__ __forceinline__ double of_order_key(uint64_t k) {
    return __longlong_as_double((long long)((k >> 63) != 0 ? k & ~(1ull << 63) : ~k));
}

__device__ __forceinline__ double pack_d(uint32_t lo, uint32_t hi) {
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// a + b after exchanging the halves the lane does not keep: lanes of the
// lower half (of 64, or of each 32) hold a's pair sum, the others b's
__device__ __forceinline__ double pair_swap32(double a, double b) {
    const uint64_t ua = (uint64_t)__double_as_longlong(a), ub = (uint64_t)__double_as_longlong(b);
    const u32x2 lo = __builtin_amdgcn_permlane32_swap((uint32_t)ua, (uint32_t)ub, false, false);
    const u32x2 hi = __builtin_amdgcn_permlane32_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32),
                                                      false, false);
    return pack_d(lo[0], hi[0]) + pack_d(lo[1], hi[1]);
}
__device__ __forceinline__ double pair_swap16(double a, double b) {
    const uint64_t ua = (uint64_t)__double_as_longlong(a), ub = (uint64_t)__double_as_longlong(b);
    const u32x2 lo = __builtin_amdgcn_permlane16_swap((uint32_t)ua, (uint32_t)ub, false, false);
    const u32x2 hi = __builtin_amdgcn_permlane16_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32),
                                                      false, false);
    return pack_d(lo[0], hi[0]) + pack_d(lo[1], hi[1]);
}
__device__ __forceinline__ float pair_swap32(float a, float b) {
    const u32x2 x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                     false);
    return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}
__device__ __forceinline__ float pair_swap16(float a, float b) {
    const u32x2 x = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                     false);
    return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}
template <int CTRL> __device__ __forceinline__ float dpp_t(float x) { return dpp_full_f<CTRL>(x); }
template <int CTRL> __device__ __forceinline__ double dpp_t(double x) { return dpp_full_d<CTRL>(x); }

constexpr int kDppRowRor4 = 0x124, kDppRowRor8 = 0x128;  // rotate within 16 lanes
constexpr int kDppRowNewBcast0 = 0x150;                  // lane n of each 16 to all of them

// Sums of four values over each 16 lanes: lanes with lane % 4 == i get value
// i's.  Two halving steps in the value's type (each lane keeps half of the
// values and sends the other half), the last two in float64.
template <typename T>
__device__ __forceinline__ double row16_sum4(const T (&s)[4], bool odd, bool odd2) {
    const T y0 = (odd ? s[1] : s[0]) + dpp_t<kDppQuadXor1>(odd ? s[0] : s[1]);
    const T y1 = (odd ? s[3] : s[2]) + dpp_t<kDppQuadXor1>(odd ? s[2] : s[3]);
    const T z = (odd2 ? y1 : y0) + dpp_t<kDppQuadXor2>(odd2 ? y0 : y1);
    double d = (double)z;
    d += dpp_full_d<kDppRowRor8>(d);
    d += dpp_full_d<kDppRowRor4>(d);
    return d;
}

// f(0), f(1), ... f(N - 1) with the index as a constant expression
template <typename Fn, int... I>
__device__ __forceinline__ void unroll_seq(Fn &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename Fn> __device__ __forceinline__ void unroll(Fn &&f) {
    unroll_seq(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ float max_t(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double max_t(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ float readlane_t(float x, int lane) { return readlane_f(x, lane); }
__device__ __forceinline__ double readlane_t(double x, int lane) { return readlane_d(x, lane); }

__device__ __forceinline__ void put_word(uint64_t *p, uint32_t payload, uint32_t tag) {
    __hip_atomic_store(p, ((uint64_t)tag << 32) | payload, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get_word(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A bounded wait for workgroups of the same problem: false once it has lasted
// ResArgs::max_polls (asked every 1024 polls), or one of them has given the
// problem up.  `args` fetches the arguments there and then: a polling loop keeps
// the count alone (limit, clock and mark in its registers cost 0.1 us a step of
// (1, 1024, 1024)).
struct Waiter {
    uint32_t polls;
    __device__ explicit Waiter(uint32_t first) : polls(first) {}
    template <typename Args> __device__ bool more(Args &&args, int64_t prob) {
        if ((++polls & 1023u) != 0)
            return true;
        const ResArgs *A = args();
        return polls < A->max_polls && __hip_atomic_load(A->given_up + prob, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT) == 0;
    }
};
// The first count: with a limit of 0 the first poll is the last.
__device__ __forceinline__ uint32_t first_poll(uint32_t max_polls) {
    return max_polls == 0 ? 1023u : 0u;
}
// The kernel's arguments where they are (in the kernel itself only).
__device__ __forceinline__ const ResArgs *res_args() {
    const ResArgs *A = (const ResArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(A));  // not read ahead of need
    return A;
}

// Payloads of the words p(0) ... p(N - 1) once all carry `tag`, all in flight
// at a time.
template <int N, typename P>
__device__ __forceinline__ void wait_words(const ResArgs *A, int64_t prob, P &&p, uint32_t tag,
                                           uint32_t (&x)[N], int &late) {
    uint64_t w[N];
    Waiter wt(first_poll(A->max_polls));
    for (;;) {
        uint32_t diff = 0;
#pragma unroll
        for (int i = 0; i < N; ++i)
            w[i] = get_word(p(i));
#pragma unroll
        for (int i = 0; i < N; ++i)
            diff |= (uint32_t)(w[i] >> 32) ^ tag;
        if (diff == 0)
            break;
        if (late != 0 || !wt.more([A] { return A; }, prob)) {
            late = 1;
            break;
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
        x[i] = (uint32_t)w[i];
}

// One workgroup's share of a problem, R rows of up to CW columns, in one of
// two layouts of a wave (wr, wc) (WC waves side by side share RW rows):
//   LC = 64  the lanes span the columns: lane l holds columns
//            (k*WC + wc)*64 + l, k < TC, of RW = TR rows; for wide matrices
//   LC = 16  four groups of 16 lanes: lane (h, c) holds columns
//            (k*WC + wc)*16 + c of the rows 4*r + h, r < TR, so RW = 4*TR; for
//            up to 256 columns per wave, where the other layout would spend
//            more on reducing a row over 64 lanes than on its products
template <typename T, int NW_, int LC_, int WC_, int TC_, int TR_, bool SOLO_> struct Cfg {
    using Type = T;
    static constexpr int NW = NW_, LC = LC_, WC = WC_, TC = TC_, TR = TR_;
    static constexpr bool SOLO = SOLO_;                    // one workgroup per problem
    static constexpr int NT = NW * 64;                     // threads
    static constexpr int WR = NW / WC;
    static constexpr int RW = LC == 64 ? TR : 4 * TR;      // rows of a wave
    static constexpr int NV = RW / 4;                      // row sums per lane, see lane_row
    static constexpr int R = WR * RW;
    static constexpr int ETC = (LC * TC + 63) / 64;        // columns per lane, exact step
    static constexpr int CW = WC * 64 * ETC;
    static constexpr int NK = (CW + NT - 1) / NT;          // columns per thread
    static constexpr int KC = SOLO ? NK : 1;               // owned columns per thread
    static constexpr int PW = Unit<T>::kPartWords;  // words of a column partial
    static constexpr int XW = PW + 2;               // words of an exact partial (max, sum)
    static constexpr int BW = 4;                    // words of an exact broadcast (c, log_v)
    static_assert(RW <= 64 && RW % 4 == 0, "one row per lane");
    static __device__ __forceinline__ int col(int k, int wc, int lane) {
        return (k * WC + wc) * LC + (lane & (LC - 1));
    }
};

template <typename F> struct Shared {
    using T = typename F::Type;
    double c[F::CW];               // column references, all columns
    double rs[F::WC * F::R];       // row sums of each column wave
    double rl[F::R];               // row references (exact step: log_u)
    double xs[F::NT];              // split column sums
    double xm[F::SOLO ? 1 : F::NT];  // exact step: split column maxima
    double bd[F::KC * F::NT];        // owned columns: multiplier and marginal
    double nu[F::KC * F::NT];        // (unbalanced: log_v and log marginal)
    double kappa;                  // the scale taken out (unbalanced)
    double rm[F::WC * F::R];       // exact step: row maxima
    union {                        // exact step:
        double lv[F::CW];          // log_v of all columns, which it starts from
        uint64_t cm[F::CW];        // then the column maxima (order_key)
    };
    T b[F::CW];
    T cp[F::WR * F::CW];           // column sums of each row wave
    float eb[F::KC * F::NT];
    uint8_t dead[F::KC * F::NT];
    int flag_row[2], flag_all[2], abort;
    int look;  // P's largest entry is looked at (kPHi)
};
#define TM_LDS __attribute__((address_space(3)))
template <typename F> using SharedP = TM_LDS Shared<F> *;

// The row a lane keeps, of its wave's RW: where the reductions leave the row
// sums (lanes past RW keep none).
__device__ __forceinline__ int lane_row(int lane) { return 4 * (lane & 15) + (lane >> 4); }

struct Row {
    double lmu, mu;   // marginal: log units, linear
    double rl, a;     // reference, multiplier of the last accepted step
    double lu;        // log_u where it is explicit (see `derived`)
    float ea;         // rounding carried by the float32 copy of a
    bool dead;        // the LSE is not finite: the potential keeps its value
    bool derived;     // balanced: log_u is log(a) - rl
};

// What a workgroup works on: one problem's rows and exchange buffers.
struct Job {
    const void *C;
    const uint8_t *keep;
    const double *lnu;
    uint64_t *part, *cast;
    const ResArgs *args;
    int64_t prob;
    int M, Mp, G, g, nrow, j0, cn, cnp, direct, unbal;
};

template <typename F, typename T>
__device__ __forceinline__ void load_rows(const Job &J, int row, int wc, int lane,
                                          T (&c)[F::ETC]) {
    const T *C = static_cast<const T *>(J.C);
    const int64_t base = (int64_t)min(row, J.nrow - 1) * J.M;
    // every load goes out unconditionally (in bounds), then what is not there
    // becomes +inf: behind a condition each load is waited for
    uint8_t kp[F::ETC];
#pragma unroll
    for (int k = 0; k < F::ETC; ++k)
        c[k] = C[base + min((k * F::WC + wc) * 64 + lane, J.M - 1)];
    if (J.keep != nullptr) {
#pragma unroll
        for (int k = 0; k < F::ETC; ++k)
            kp[k] = J.keep[base + min((k * F::WC + wc) * 64 + lane, J.M - 1)];
    } else {
#pragma unroll
        for (int k = 0; k < F::ETC; ++k)
            kp[k] = 1;
    }
#pragma unroll
    for (int k = 0; k < F::ETC; ++k) {
        const int j = (k * F::WC + wc) * 64 + lane;
        const bool ok = (row < J.nrow) & (j < J.M) & (kp[k] != 0);
        c[k] = ok ? c[k] : (T)INFINITY;
    }
}

// One step from the cost, the maximum taken out of every sum (the reference's
// logsumexp and its rules); sets the references and multipliers around the
// new potentials.  Not inlined: it runs once per problem (and after a refused
// step) and would cost the step loop its registers.
template <typename F>
__device__ __noinline__ void exact_step(SharedP<F> S, const Job &J, Row &W, double eps, double damp,
                                        uint32_t seq) {
    using T = typename F::Type;
    using U = Unit<T>;
    constexpr int WC = F::WC, WR = F::WR, TC = F::ETC, TR = F::RW, R = F::R, CW = F::CW;
    constexpr int XW = F::XW, PW = F::PW, BW = F::BW;
    constexpr int RG = TC <= 4 ? 4 : 2;  // rows in flight
    const int t = (int)threadIdx.x, lane = lane_id();
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wr = wid / WC, wc = wid % WC;
    const int M = J.M, Mp = J.Mp, G = J.G;
    const U u(eps);
    {
        double lvk[TC];
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            const int j = (k * WC + wc) * 64 + lane;
            lvk[k] = S->lv[j];
        }
#pragma unroll 1
        for (int r0 = 0; r0 < TR; r0 += RG) {
            T c[RG][TC];
#pragma unroll
            for (int r = 0; r < RG; ++r)
                load_rows<F>(J, wr * TR + r0 + r, wc, lane, c[r]);
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                double x[TC];
                double m = -INFINITY;
#pragma unroll
                for (int k = 0; k < TC; ++k) {
                    x[k] = u.kval(c[r][k]) + lvk[k];
                    m = fmax(m, x[k]);
                }
                m = wave_max_all_d(m);
                const double sh = shift_of(m);
                double s = 0.0;
#pragma unroll
                for (int k = 0; k < TC; ++k)
                    s += (double)U::term(x[k] - sh);
                s = wave_sum_all_d(s);
                if (lane == 0) {
                    S->rm[wc * R + wr * TR + r0 + r] = m;
                    S->rs[wc * R + wr * TR + r0 + r] = s;
                }
            }
        }
    }
    __syncthreads();
    for (int j = t; j < CW; j += F::NT)
        S->cm[j] = order_key(-INFINITY);
    double lse = 0.0;
    const int rho = lane_row(lane), row = wr * TR + rho;
    const bool has = rho < TR && row < J.nrow;
    if (has) {
        double m = S->rm[row];
#pragma unroll
        for (int w = 1; w < WC; ++w)
            m = fmax(m, S->rm[w * R + row]);
        const double sh = shift_of(m);
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < WC; ++w) {
            const double sw = S->rs[w * R + row];
            if (sw != 0.0)
                s += WC == 1 ? sw : sw * U::expm(shift_of(S->rm[w * R + row]) - sh);
        }
        lse = U::logm(s) + sh;
        if (W.derived && !W.dead && !J.unbal)
            W.lu = U::logm(W.a) - W.rl;
        W.dead = !isfinite(lse);
        if (!W.dead) {
            const double d = W.lmu - lse;
            W.lu = J.unbal ? damp * d : d;
        }
        W.derived = false;
    }
    if (wc == 0 && rho < TR)
        S->rl[row] = has ? W.lu : -INFINITY;
    __syncthreads();
    {
        double m[TC];
        T s[TC];
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            m[k] = -INFINITY;
            s[k] = (T)0;
        }
#pragma unroll 1
        for (int r0 = 0; r0 < TR; r0 += RG) {
            T c[RG][TC];
#pragma unroll
            for (int r = 0; r < RG; ++r)
                load_rows<F>(J, wr * TR + r0 + r, wc, lane, c[r]);
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                const double l = S->rl[wr * TR + r0 + r];
#pragma unroll
                for (int k = 0; k < TC; ++k)
                    m[k] = fmax(m[k], u.kval(c[r][k]) + l);
            }
        }
        // the workgroup's maximum of every column
#pragma unroll
        for (int k = 0; k < TC; ++k)
            __hip_atomic_fetch_max(&S->cm[(k * WC + wc) * 64 + lane], order_key(m[k]),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TC; ++k)
            m[k] = shift_of(of_order_key(S->cm[(k * WC + wc) * 64 + lane]));
#pragma unroll 1
        for (int r0 = 0; r0 < TR; r0 += RG) {
            T c[RG][TC];
#pragma unroll
            for (int r = 0; r < RG; ++r)
                load_rows<F>(J, wr * TR + r0 + r, wc, lane, c[r]);
#pragma unroll
            for (int r = 0; r < RG; ++r) {
                const double l = S->rl[wr * TR + r0 + r];
#pragma unroll
                for (int k = 0; k < TC; ++k)
                    s[k] += U::term((u.kval(c[r][k]) + l) - m[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < TC; ++k)
            S->cp[wr * CW + (k * WC + wc) * 64 + lane] = s[k];
    }
    __syncthreads();
    const uint32_t tag = seq << 1;
    uint64_t *pw = J.part + (size_t)(seq & 1) * G * XW * Mp;
    uint64_t *cw = J.cast + (size_t)(seq & 1) * BW * Mp;
    int late = 0;
    // this workgroup's (max, sum) of column j
    auto local_pair = [&](int j, double &m, double &s) {
        m = of_order_key(S->cm[j]);
        s = 0.0;
#pragma unroll
        for (int w = 0; w < WR; ++w)
            s += (double)S->cp[w * CW + j];
    };
    if (G > 1) {
        for (int j = t; j < M; j += F::NT) {
            double m, s;
            local_pair(j, m, s);
            uint64_t *p = pw + (size_t)J.g * XW * Mp + j;
            const uint64_t qm = (uint64_t)__double_as_longlong(m);
            put_word(p, (uint32_t)qm, tag);
            put_word(p + Mp, (uint32_t)(qm >> 32), tag);
            if constexpr (PW == 1) {
                put_word(p + 2 * (size_t)Mp, __float_as_uint((float)s), tag);
            } else {
                const uint64_t q = (uint64_t)__double_as_longlong(s);
                put_word(p + 2 * (size_t)Mp, (uint32_t)q, tag);
                put_word(p + 3 * (size_t)Mp, (uint32_t)(q >> 32), tag);
            }
        }
    }
    double gm = -INFINITY, gs = 0.0;  // column t of the owned ones, all workgroups
    if constexpr (!F::SOLO) {
        // thread groups share a column's partials as in the step, each in
        // workgroup order, then the groups' results in theirs: the same in
        // every workgroup that merges this column.  Four partials in flight:
        // one by one, and with load_rows' loads behind conditions, this step
        // took 200 us for four problems of 2048 x 2048 at a time; 50 now, most
        // of it float64 arithmetic (four rows in flight: no faster)
        auto add = [](double &m, double &s, double mq, double sq) {
            const double mn = fmax(m, mq), sh = shift_of(mn);
            s = (s != 0.0 ? s * U::expm(shift_of(m) - sh) : 0.0) +
                (sq != 0.0 ? sq * U::expm(shift_of(mq) - sh) : 0.0);
            m = mn;
        };
        const int split = F::NT / J.cnp, sp = t / J.cnp, jl = t % J.cnp;
        double m = -INFINITY, s = 0.0;
        if (jl < J.cn) {
            const uint64_t *p = pw + J.j0 + jl;
#pragma unroll 1
            for (int q0 = sp; q0 < G; q0 += 4 * split) {
                uint32_t x[4 * XW];
                wait_words<4 * XW>(
                    J.args, J.prob,
                    [&](int i) {
                        const int q = min(q0 + i / XW * split, G - 1);
                        return p + ((size_t)q * XW + i % XW) * Mp;
                    },
                    tag, x, late);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t *xi = x + i * XW;
                    const double sq =
                        PW == 1 ? (double)__uint_as_float(xi[2]) : pack_d(xi[2], xi[XW - 1]);
                    if (q0 + i * split < G)
                        add(m, s, pack_d(xi[0], xi[1]), sq);
                }
            }
        }
        S->xm[t] = m;
        S->xs[t] = s;
        __syncthreads();
        if (t < J.cn) {
            for (int k = 0; k < min(split, G); ++k)
                add(gm, gs, S->xm[k * J.cnp + t], S->xs[k * J.cnp + t]);
        }
    }
#pragma unroll 1
    for (int jl = t; jl < J.cn; jl += F::NT) {
        const int j = J.j0 + jl;
        double m = gm, s = gs;
        if (F::SOLO)
            local_pair(j, m, s);
        const double l = U::logm(s) + shift_of(m);
        double lv = J.unbal ? S->bd[jl] : U::logm(S->bd[jl]) - S->c[j];
        const bool dc = !isfinite(l);
        if (!dc) {
            const double d = U::of_nat(J.lnu[j]) - l;
            lv = J.unbal ? damp * d : d;
        }
        const double cr = !dc ? l : NAN;  // (set below once kappa is known)
        S->eb[jl] = 0.f;
        S->dead[jl] = dc;
        if (G > 1 && !J.direct) {
            const uint64_t q = (uint64_t)__double_as_longlong(cr);
            put_word(cw + j, (uint32_t)q, tag);
            put_word(cw + Mp + j, (uint32_t)(q >> 32), tag);
            const uint64_t ql = (uint64_t)__double_as_longlong(lv);
            put_word(cw + 2 * (size_t)Mp + j, (uint32_t)ql, tag);
            put_word(cw + 3 * (size_t)Mp + j, (uint32_t)(ql >> 32), tag);
        } else {
            S->c[j] = cr;
            S->lv[j] = lv;
        }
    }
    __syncthreads();
    if (G > 1 && !J.direct) {
#pragma unroll 1
        for (int j = t; j < M; j += 2 * F::NT) {
            const int j1 = min(j + F::NT, M - 1);  // (the last column twice at most)
            uint32_t x[8];
            wait_words<8>(
                J.args, J.prob,
                [&](int i) { return cw + (i & 3) * (size_t)Mp + (i < 4 ? j : j1); }, tag, x, late);
            S->c[j] = pack_d(x[0], x[1]);
            S->lv[j] = pack_d(x[2], x[3]);
            if (j + F::NT < M) {
                S->c[j1] = pack_d(x[4], x[5]);
                S->lv[j1] = pack_d(x[6], x[7]);
            }
        }
    }
    // kappa, the same in every workgroup (each has all columns, a thread the
    // columns it stored); then the multipliers around it
    double kap = 0.0;
    if (J.unbal) {
        double m = -INFINITY;
        for (int j = t; j < M; j += F::NT)
            m = fmax(m, S->lv[j] + S->c[j]);  // (NaN, a dead column, drops out)
        m = wave_max_all_d(m);
        if (lane == 0)
            S->xs[wid] = m;
        __syncthreads();
        for (int w = 0; w < F::NW; ++w)
            m = fmax(m, S->xs[w]);
        kap = isfinite(m) ? m : 0.0;
    }
    for (int j = t; j < M; j += F::NT) {
        const double lv = S->lv[j];
        double c = S->c[j];
        if (isnan(c))
            S->c[j] = c = isfinite(lv) ? kap - lv : 0.0;
        S->b[j] = (T)U::expm(lv + c - kap);
    }
    if (t == 0)
        S->kappa = kap;
    if (late)
        S->abort = 1;
    __syncthreads();
    for (int jl = t; jl < J.cn; jl += F::NT) {
        const int j = J.j0 + jl;
        S->bd[jl] = J.unbal ? S->lv[j] : U::expm(S->lv[j] + S->c[j]);
    }
    if (has) {
        W.rl = !W.dead ? lse : isfinite(W.lu) ? kap - W.lu : 0.0;
        W.a = U::expm(W.lu + W.rl - kap);
        W.ea = 0.f;
    }
    __syncthreads();
}

// A step was refused: log_v of the last accepted one, for the exact step.
template <typename F>
__device__ __noinline__ void send_log_v(SharedP<F> S, const Job &J, uint32_t seq) {
    using U = Unit<typename F::Type>;
    const uint32_t tag = seq << 1;
    uint64_t *cw = J.cast + (size_t)(seq & 1) * F::BW * J.Mp;
    for (int jl = (int)threadIdx.x; jl < J.cn; jl += F::NT) {
        const int j = J.j0 + jl;
        const double lv = J.unbal ? S->bd[jl] : U::logm(S->bd[jl]) - S->c[j];
        if (J.direct) {
            S->lv[j] = lv;
        } else {
            const uint64_t q = (uint64_t)__double_as_longlong(lv);
            put_word(cw + j, (uint32_t)q, tag);
            put_word(cw + J.Mp + j, (uint32_t)(q >> 32), tag);
        }
    }
    if (!J.direct) {
        int late = 0;
        for (int j = (int)threadIdx.x; j < J.M; j += F::NT) {
            uint32_t x[2];
            wait_words<2>(
                J.args, J.prob, [&](int i) { return cw + (size_t)i * J.Mp + j; }, tag, x, late);
            S->lv[j] = pack_d(x[0], x[1]);
        }
        if (late)
            S->abort = 1;
    }
    __syncthreads();
}

// Epsilon changed: move the references by powers of two to the current
// potentials (each multiplier back to [1, 2)).
template <typename F>
__device__ __noinline__ void recentre(SharedP<F> S, const Job &J, Row &W) {
    using T = typename F::Type;
    using U = Unit<T>;
    for (int j = (int)threadIdx.x; j < J.M; j += F::NT) {
        const double b = (double)S->b[j];
        int e = 0;
        if (b > 0.0 && isfinite(b))
            e = ilogb(b);
        S->b[j] = (T)ldexp(b, -e);
        S->c[j] -= U::of_exp2(e);
        const int jl = j - J.j0;
        if (jl >= 0 && jl < J.cn && !J.unbal)
            S->bd[jl] = ldexp(S->bd[jl], -e);
    }
    // rows the lane does not have hold a = 0
    if (W.a > 0.0 && isfinite(W.a)) {
        const int e = ilogb(W.a);
        W.a = ldexp(W.a, -e);
        W.rl -= U::of_exp2(e);
    }
}

// Start state of a problem: potentials 0, marginals in log units and linear.
template <typename F>
__device__ __noinline__ void start_problem(SharedP<F> S, const Job &J, Row &W, const double *lmu) {
    using T = typename F::Type;
    using U = Unit<T>;
    const int t = (int)threadIdx.x;
    W = Row{-INFINITY, 0.0, 0.0, 0.0, 0.0, 0.f, false, false};
    if (t == 0)
        S->look = J.unbal;
    __syncthreads();
    const int rho = lane_row(lane_id()), row = (t >> 6) / F::WC * F::RW + rho;
    if (rho < F::RW && row < J.nrow) {
        W.lmu = U::of_nat(lmu[row]);
        W.mu = U::expm(W.lmu);
        W.a = 1.0;
        if (W.mu < kMassLo)
            S->look = 1;
    }
    for (int j = t; j < F::CW; j += F::NT) {
        S->c[j] = j < J.M ? 0.0 : INFINITY;  // columns past M: P = 0, b = 0
        S->b[j] = j < J.M ? (T)1 : (T)0;
        S->lv[j] = 0.0;
    }
    if (t == 0)
        S->kappa = 0.0;
    for (int jl = t; jl < F::KC * F::NT; jl += F::NT) {
        S->bd[jl] = J.unbal ? 0.0 : 1.0;
        S->eb[jl] = 0.f;
        S->dead[jl] = 0;
        const double l = jl < J.cn ? U::of_nat(J.lnu[J.j0 + jl]) : -INFINITY;
        S->nu[jl] = J.unbal ? l : U::expm(l);
    }
    __syncthreads();
}

// A problem that was given up, by one workgroup: every half-step from the cost
// with the maximum taken out, the potentials (in log units until the end) in
// global memory, no other workgroup needed.
template <typename T> __device__ __noinline__ void redo_problem(const ResArgs *A, int64_t p) {
    using U = Unit<T>;
    const int t = (int)threadIdx.x, nt = (int)blockDim.x, lane = lane_id();
    const int N = A->N, M = A->M;
    const T *C = static_cast<const T *>(A->cost) + p * N * (int64_t)M;
    const uint8_t *keep = A->keep != nullptr ? A->keep + p * N * (int64_t)M : nullptr;
    double *lu = (A->lu64 != nullptr ? A->lu64 : static_cast<double *>(A->log_u)) + p * N;
    double *lv = (A->lv64 != nullptr ? A->lv64 : static_cast<double *>(A->log_v)) + p * M;
    for (int i = t; i < N; i += nt)
        lu[i] = 0.0;
    for (int j = t; j < M; j += nt)
        lv[j] = 0.0;
    __syncthreads();
    int seg = 0;
    for (int it = 0; it < A->n_iter; ++it) {
        if (it == A->seg_end[seg])
            ++seg;
        const U u(A->eps[seg]);
        const double damp = A->rho > 0.0 ? 1.0 / (1.0 + A->eps[seg] / A->rho) : 1.0;
        auto value = [&](int64_t o) {
            return u.kval(keep == nullptr || keep[o] != 0 ? C[o] : (T)INFINITY);
        };
        for (int i = t >> 6; i < N; i += nt / 64) {  // a wave per row
            const int64_t o = (int64_t)i * M;
            double m = -INFINITY, s = 0.0;
            for (int j = lane; j < M; j += 64)
                m = fmax(m, value(o + j) + lv[j]);
            m = shift_of(wave_max_all_d(m));
            for (int j = lane; j < M; j += 64)
                s += (double)U::term(value(o + j) + lv[j] - m);
            const double lse = U::logm(wave_sum_all_d(s)) + m;
            if (lane == 0 && isfinite(lse))
                lu[i] = damp * (U::of_nat(A->lmu[p * N + i]) - lse);
        }
        __syncthreads();
        for (int j = t; j < M; j += nt) {  // a thread per column
            double m = -INFINITY, s = 0.0;
            for (int i = 0; i < N; ++i)
                m = fmax(m, value((int64_t)i * M + j) + lu[i]);
            m = shift_of(m);
            for (int i = 0; i < N; ++i)
                s += (double)U::term(value((int64_t)i * M + j) + lu[i] - m);
            const double lse = U::logm(s) + m;
            if (isfinite(lse))
                lv[j] = damp * (U::of_nat(A->lnu[p * M + j]) - lse);
        }
        __syncthreads();
    }
    for (int i = t; i < N; i += nt)
        static_cast<T *>(A->log_u)[p * N + i] = (T)(lu[i] = U::to_nat(lu[i]));
    for (int j = t; j < M; j += nt)
        static_cast<T *>(A->log_v)[p * M + j] = (T)(lv[j] = U::to_nat(lv[j]));
}

// The potentials of a finished problem.  One that this workgroup gave up (and all
// that follow it: its exchanges are no longer those of the others) it solves
// alone, unless another has.  A workgroup that came through the last exchange all
// the same writes its results too, before or after: every value is that of a
// whole solve either way.
template <typename F>
__device__ __noinline__ void finish_problem(SharedP<F> S, const Job &J, Row &W,
                                            typename F::Type *log_u, double *lu64,
                                            typename F::Type *log_v, double *lv64) {
    using T = typename F::Type;
    using U = Unit<T>;
    const int t = (int)threadIdx.x;
    if (S->abort != 0) {
        if constexpr (!F::SOLO) {
            if (t == 0)
                S->flag_row[0] =
                    __hip_atomic_exchange(J.args->given_up + J.prob, 1u, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT) == 0;
            __syncthreads();
            if (S->flag_row[0] != 0)
                redo_problem<T>(J.args, J.prob);
            __syncthreads();
        }
        return;
    }
    const int rho = lane_row(lane_id()), row = (t >> 6) / F::WC * F::RW + rho;
    if ((t >> 6) % F::WC == 0 && rho < F::RW && row < J.nrow) {
        if (W.derived && !W.dead && !J.unbal)
            W.lu = U::logm(W.a) - W.rl;
        const double x = U::to_nat(W.lu);
        log_u[row] = (T)x;
        if (lu64 != nullptr)
            lu64[row] = x;
    }
    if (!J.direct || J.g == 0) {
        for (int jl = t; jl < J.cn; jl += F::NT) {
            const double x =
                U::to_nat(J.unbal ? S->bd[jl] : U::logm(S->bd[jl]) - S->c[J.j0 + jl]);
            log_v[J.j0 + jl] = (T)x;
            if (lv64 != nullptr)
                lv64[J.j0 + jl] = x;
        }
    }
    __syncthreads();  // the next problem rewrites the shared state
}

template <typename F>
__global__ void __launch_bounds__(F::NT)
sk_resident(const ResArgs A) {
    using T = typename F::Type;
    using U = Unit<T>;
    constexpr int LC = F::LC, WC = F::WC, WR = F::WR, TC = F::TC, TR = F::TR, R = F::R;
    constexpr int CW = F::CW, RW = F::RW, NV = F::NV, KC = F::KC, XW = F::XW, PW = F::PW;
    constexpr int BW = F::BW;
    constexpr bool SOLO = F::SOLO;
    __shared__ Shared<F> S;
    const SharedP<F> SP = (SharedP<F>)&S;

    const int t = (int)threadIdx.x;
    const int lane = lane_id();
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wr = wid / WC, wc = wid % WC;
    const int G = SOLO ? 1 : A.G, M = A.M, Mp = A.Mp;
    const bool direct = SOLO || A.direct;
    const int g = SOLO ? 0 : (int)blockIdx.x % G;
    const int cluster = SOLO ? (int)blockIdx.x : (int)blockIdx.x / G;
    const bool unbal = A.rho > 0.0;
    const int i0 = g * A.rows;
    const int nrow = A.N - i0 < A.rows ? A.N - i0 : A.rows;
    const int j0 = direct ? 0 : min(g * A.cpo, M);
    const int cn = direct ? M : min(A.cpo, M - j0);
    // column merge: cnp = 16, 32, ... threads span the owned columns, and when
    // more than one such group fits the workgroup the groups share the G
    // partials of each column (group sp takes q = sp, sp + split, ...), so
    // that no load instruction goes out half empty: each costs about 16
    // cycles of address processing whatever it fetches
    int cnp = 16;
    while (cnp < A.cpo && cnp < F::NT)
        cnp *= 2;
    const int split = SOLO ? 1 : F::NT / cnp;
    const int per = (G + split - 1) / split;  // partials of a column per thread
    uint64_t *part = A.xch + (size_t)cluster * 2 * ((size_t)G * XW + BW) * Mp;
    uint64_t *cast = part + (size_t)2 * G * XW * Mp;
    const int rho = lane_row(lane), lrow = wr * RW + rho;  // the lane's row
    const bool has = rho < RW && lrow < nrow;
    const bool odd = lane & 1, odd2 = lane & 2;
    const uint32_t poll0 = SOLO ? 0 : first_poll(A.max_polls);
    uint32_t seq = 0;
    if (t == 0)
        S.abort = 0;
    __syncthreads();

    for (int64_t prob = cluster; prob < A.B; prob += A.clusters) {
        const int64_t off = (prob * A.N + i0) * (int64_t)M;
        const Job J{static_cast<const T *>(A.cost) + off, A.keep ? A.keep + off : nullptr,
                    A.lnu + prob * M, part, cast, res_args(), prob, M, Mp, G, g, nrow, j0, cn,
                    cnp, direct, unbal};
        Row W;
        start_problem<F>(SP, J, W, A.lmu + prob * A.N + i0);

        // What the next step starts from: `trial`, P around the row maxima and
        // log_v = 0 (the first step; refused where columns underflow);
        // `exact`, the cost; `moved`, P around the current potentials.
        enum { kTrial, kExact, kMoved } start = A.exact_only ? kExact : kTrial;
        int it = 0, seg = 0;
        while (it < A.n_iter && !S.abort) {
            if (start == kExact) {
                const double eps = A.eps[seg];
                exact_step<F>(SP, J, W, eps, unbal ? 1.0 / (1.0 + eps / A.rho) : 1.0, ++seq);
                ++it;
                if (it == A.n_iter)
                    break;
                if (it == A.seg_end[seg])
                    ++seg;
                if (A.exact_only)
                    continue;
            } else if (start == kMoved) {
                recentre<F>(SP, J, W);
            }
            const bool trial = start == kTrial;
            const double mul_hi = trial ? kSumHi : kMulHi;
            const double eps = A.eps[seg];
            const double damp = unbal ? 1.0 / (1.0 + eps / A.rho) : 1.0;

            // ---- P around the references ---------------------------------------
            const double kap = unbal ? readlane_d(S.kappa, 0) : 0.0;
            if (!trial && wc == 0 && rho < RW)
                S.rl[lrow] = has ? W.rl - kap : INFINITY;
            if (t < 2) {
                S.flag_row[t] = 0;
                S.flag_all[t] = 0;
            }
            __syncthreads();
            T v[TR][TC];
            {
                // the cost goes straight to P's registers, every load in
                // flight, and is turned into P in place.  Columns past M and
                // rows past nrow read a neighbour and vanish in the exponent
                // (their references are +inf).  The scheduling barriers keep
                // one row's addresses and temporaries live at a time, and the
                // empty asm keeps the compiler from computing every row's
                // address once, outside the loop over steps.
                const char *C = static_cast<const char *>(J.C);
                const char *keep = reinterpret_cast<const char *>(J.keep);
                int last = nrow - 1, m = M;
                asm volatile("" : "+s"(C), "+s"(keep), "+s"(last), "+s"(m));
                const int h = LC == 64 ? 0 : lane >> 4;
                constexpr int rs = LC == 64 ? 1 : 4;  // wave rows per r
                uint32_t qo[TC];
#pragma unroll
                for (int k = 0; k < TC; ++k)
                    qo[k] = (uint32_t)min(F::col(k, wc, lane), m - 1);
#pragma unroll
                for (int r = 0; r < TR; ++r) {
                    const uint32_t ro = (uint32_t)min(wr * RW + rs * r + h, last) * (uint32_t)m;
#pragma unroll
                    for (int k = 0; k < TC; ++k)
                        v[r][k] = *reinterpret_cast<const T *>(C + (ro + qo[k]) *
                                                                       (uint32_t)sizeof(T));
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (keep != nullptr) {
                    // rows in flight: 16 mask bytes a lane or so (four rows of 16
                    // spilled half of P: the start of (16, 2048, 2048) 512 us
                    // against 640)
                    constexpr int KR = TC >= 12 ? 1 : TC >= 6 ? 2 : TR < 4 ? TR : 4;
#pragma unroll
                    for (int r0 = 0; r0 < TR; r0 += KR) {
                        uint8_t kp[KR][TC];
#pragma unroll
                        for (int r = 0; r < KR && r0 + r < TR; ++r) {
                            const uint32_t ro =
                                (uint32_t)min(wr * RW + rs * (r0 + r) + h, last) * (uint32_t)m;
#pragma unroll
                            for (int k = 0; k < TC; ++k)
                                kp[r][k] = (uint8_t)keep[ro + qo[k]];
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int r = 0; r < KR && r0 + r < TR; ++r)
#pragma unroll
                            for (int k = 0; k < TC; ++k)
                                v[r0 + r][k] = kp[r][k] ? v[r0 + r][k] : (T)INFINITY;
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                const U u(eps);
                if (trial) {
                    // row references: K at the row's smallest cost
                    float mine = INFINITY;
#pragma unroll
                    for (int r = 0; r < TR; ++r) {
                        float x = (float)v[r][0];
#pragma unroll
                        for (int k = 1; k < TC; ++k)
                            x = fminf(x, (float)v[r][k]);
                        x = fminf(x, dpp_full_f<kDppQuadXor1>(x));
                        x = fminf(x, dpp_full_f<kDppQuadXor2>(x));
                        x = fminf(x, dpp_full_f<kDppRowHalfMirror>(x));
                        x = fminf(x, dpp_full_f<kDppRowMirror>(x));
                        if constexpr (LC == 64) {
                            float o;
                            float y = row_swap16_pair(x, o);
                            x = fminf(y, o);
                            y = row_swap32_pair(x, o);
                            x = fminf(y, o);
                            mine = rho == r ? x : mine;
                        } else {
                            mine = (lane & 15) == r ? x : mine;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (rho < RW)
                        S.rm[wc * R + lrow] = mine;
                    __syncthreads();
                    if (has) {
#pragma unroll
                        for (int w = 0; w < WC; ++w)
                            mine = fminf(mine, S.rm[w * R + lrow]);
                        W.rl = __builtin_isfinite(mine) ? u.kval((T)mine) : 0.0;
                    }
                    if (wc == 0 && rho < RW)
                        S.rl[lrow] = has ? W.rl : INFINITY;  // (kappa is 0)
                    __syncthreads();
                }
                double ck[TC];
#pragma unroll
                for (int k = 0; k < TC; ++k)
                    ck[k] = S.c[F::col(k, wc, lane)];
#pragma unroll
                for (int r = 0; r < TR; ++r) {
                    const double l = S.rl[wr * RW + rs * r + h];
#pragma unroll
                    for (int k = 0; k < TC; ++k) {
                        v[r][k] = U::build(u.kval(v[r][k]), l, ck[k]);
                        if (k % 4 == 3)
                            __builtin_amdgcn_sched_barrier(0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (__builtin_expect(__builtin_amdgcn_readfirstlane(S.look) != 0, 0)) {
                    T top = (T)0;
#pragma unroll
                    for (int r = 0; r < TR; ++r)
#pragma unroll
                        for (int k = 0; k < TC; ++k)
                            top = max_t(top, v[r][k]);
                    if (ballot(top > kPHi<T>) != 0 && lane == 0)
                        S.flag_row[0] = 1;  // refuses the first step
                }
            }
            Row L = W;  // W is in memory (it is passed to the calls above)
            // the thread's owned columns t + kc * NT: multiplier (unbalanced:
            // log_v), the rounding its float32 copy carries, the marginal
            // (balanced linear, else in log units), the reference
            double cb[KC], cnu[KC], cref[KC];
            float ceb[KC];
            bool cdead[KC];
#pragma unroll
            for (int kc = 0; kc < KC; ++kc) {
                const int jl = t + kc * F::NT;
                cb[kc] = S.bd[jl];
                ceb[kc] = S.eb[jl];
                cnu[kc] = S.nu[jl];
                cdead[kc] = S.dead[jl] != 0;
                cref[kc] = jl < cn ? S.c[j0 + jl] : 0.0;
            }

            // ---- steps from P until epsilon changes or one is refused ----------
            for (int fp = 0;; fp ^= 1) {
                // the thread's columns, anew each step: kept over the loop, their
                // addresses do not fit the registers beside 128 matrix entries
                // and come back from scratch one by one, each waited for together
                // with the stores before it (us per step with them and without:
                // (16, 2048, 2048) 32.6, 23.6; (1, 4096, 4096) 12.1, 9.6; float64
                // (2, 300, 200) 3.4, 3.1).  A small tile of one workgroup has room
                // for them ((64, 64, 80): 0.89 a step kept, 0.90 not)
                int tj = t;
                if constexpr (!SOLO || TC * TR >= 96)
                    asm volatile("" : "+v"(tj));
                double rsum = 0.0;  // the lane's row
                {
                    T bk[TC];
#pragma unroll
                    for (int k = 0; k < TC; ++k)
                        bk[k] = S.b[F::col(k, wc, lane)];
#pragma unroll
                    for (int q = 0; q < (NV + 3) / 4; ++q) {
                        T z[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if (4 * q + i >= NV) {
                                z[i] = (T)0;
                                continue;
                            }
                            if constexpr (LC == 64) {
                                T s[4];
#pragma unroll
                                for (int x = 0; x < 4; ++x)
                                    s[x] = v[4 * (4 * q + i) + x][0] * bk[0];
#pragma unroll
                                for (int k = 1; k < TC; ++k)
#pragma unroll
                                    for (int x = 0; x < 4; ++x)
                                        s[x] = fma(v[4 * (4 * q + i) + x][k], bk[k], s[x]);
                                z[i] = pair_swap16(pair_swap32(s[0], s[2]),
                                                   pair_swap32(s[1], s[3]));
                            } else {
                                T s = v[4 * q + i][0] * bk[0];
#pragma unroll
                                for (int k = 1; k < TC; ++k)
                                    s = fma(v[4 * q + i][k], bk[k], s);
                                z[i] = s;
                            }
                        }
                        const double x = row16_sum4(z, odd, odd2);
                        rsum = ((lane >> 2) & 3) == q ? x : rsum;
                    }
                }
                if constexpr (WC > 1) {
                    if (rho < RW)
                        S.rs[wc * R + lrow] = rsum;
                    __syncthreads();
                    rsum = 0.0;
                    if (rho < RW) {
#pragma unroll
                        for (int w = 0; w < WC; ++w)
                            rsum += S.rs[w * R + lrow];
                    }
                }
                // the lane's row update, in each of the row's WC waves
                double a_new, lu_new = L.lu;
                float ea_new = 0.f;
                T ah;
                {
                    if (!unbal) {
                        a_new = L.mu * U::recip(rsum);
                    } else {
                        const double ls = U::log_fast(rsum);
                        lu_new = damp * (L.lmu - (ls + L.rl));
                        if constexpr (PW == 1) {
                            a_new = U::exp_fast(lu_new + L.rl - kap);
                        } else {  // (log_u is rounded to its own size, a need not be)
                            a_new = U::exp_fast(damp * (L.lmu - ls) + ((1.0 - damp) * L.rl - kap));
                            if (it + 1 == A.n_iter)
                                lu_new = damped_potential(damp, L.lmu, ls, L.rl);
                        }
                    }
                    const bool ok = L.dead ? rsum == 0.0
                                           : rsum >= kSumLo && rsum <= kSumHi && a_new <= kMulHi;
                    if (L.dead || !has) {
                        a_new = L.a;
                        lu_new = L.lu;
                    }
                    if constexpr (PW == 1) {
                        const double x = fma(a_new, (double)L.ea, a_new);
                        ah = (float)x;
                        if (ah > kCarryLo)
                            ea_new = (float)(x - (double)ah) * __builtin_amdgcn_rcpf(ah);
                    } else {
                        ah = a_new;
                    }
                    if (ballot(has && !ok) != 0 && lane == 0)
                        S.flag_row[fp] = 1;
                }
                {
                    T cs[TC];
#pragma unroll
                    for (int k = 0; k < TC; ++k)
                        cs[k] = (T)0;
                    if constexpr (LC == 64) {
#pragma unroll
                        for (int r = 0; r < TR; ++r) {
                            const T ar = readlane_t(ah, 16 * (r & 3) + (r >> 2));
#pragma unroll
                            for (int k = 0; k < TC; ++k)
                                cs[k] = fma(v[r][k], ar, cs[k]);
                        }
#pragma unroll
                        for (int k = 0; k < TC; ++k)
                            S.cp[wr * CW + F::col(k, wc, lane)] = cs[k];
                    } else {
                        unroll<TR>([&](auto ri) {
                            constexpr int r = decltype(ri)::value;
                            const T ar = dpp_t<kDppRowNewBcast0 + r>(ah);
#pragma unroll
                            for (int k = 0; k < TC; ++k)
                                cs[k] = fma(v[r][k], ar, cs[k]);
                        });
                        // the four groups' sums; each keeps a quarter of the
                        // columns (a column without a partner is kept twice)
                        constexpr int n1 = (TC + 1) / 2, n2 = (n1 + 1) / 2;
                        T y[n1 + 1];
#pragma unroll
                        for (int p = 0; p < n1; ++p)
                            y[p] = pair_swap32(cs[2 * p], cs[min(2 * p + 1, TC - 1)]);
#pragma unroll
                        for (int p = 0; p < n2; ++p) {
                            const T z = pair_swap16(y[2 * p], y[min(2 * p + 1, n1 - 1)]);
                            const int p1 = min(2 * p + ((lane >> 4) & 1), n1 - 1);
                            const int k = min(2 * p1 + (lane >> 5), TC - 1);
                            S.cp[wr * CW + F::col(k, wc, lane)] = z;
                        }
                    }
                }
                __syncthreads();
                if (t == 0) {
                    S.flag_row[fp ^ 1] = 0;
                    S.flag_all[fp ^ 1] = 0;
                }
                uint32_t bad = (uint32_t)S.flag_row[fp];
                int late = 0;
                auto local_sum = [&](int j) {
                    double s[WR];
#pragma unroll
                    for (int w = 0; w < WR; ++w)
                        s[w] = (double)S.cp[w * CW + j];
#pragma unroll
                    for (int h = 1; h < WR; h *= 2)
#pragma unroll
                        for (int w = 0; w + h < WR; w += 2 * h)
                            s[w] += s[w + h];
                    return s[0];
                };
                uint32_t tag = 0;
                // this exchange's slots; a word's byte offset in them fits 32
                // bits (at most 256 workgroups x 4 words x 4096 columns x 8)
                const char *pw = nullptr;
                char *cw = nullptr;
                const uint32_t prow = (uint32_t)(XW * Mp) * 8u;  // one workgroup's partials
                // Sum of column j's partials of workgroups q0, q0 + step, ...
                // (`per` of them, the last perhaps past G), in that order, N
                // in flight at a time.  N is a constant and every load goes out
                // unconditionally: behind branches they would be waited for
                // one by one (about 1100 cycles each).
                auto gather_n = [&](int j, int q0, int step, auto nc) {
                    constexpr int N = decltype(nc)::value;
                    const uint32_t o0 = (uint32_t)q0 * prow + (uint32_t)j * 8u;
                    const uint32_t so = (uint32_t)step * prow;
                    const int mine = q0 + (per - 1) * step < G ? per : per - 1;
                    double acc = 0.0;
                    for (int u0 = 0; u0 < per; u0 += N) {
                        uint64_t w[N][PW];
                        Waiter wt(poll0);
                        for (;;) {
                            uint32_t diff = 0;
#pragma unroll
                            for (int i = 0; i < N; ++i) {
                                const uint32_t o =
                                    u0 + i < mine ? o0 + (uint32_t)(u0 + i) * so : o0;
#pragma unroll
                                for (int p = 0; p < PW; ++p)
                                    w[i][p] = get_word(reinterpret_cast<const uint64_t *>(
                                        pw + (o + (uint32_t)(p * Mp) * 8u)));
                            }
#pragma unroll
                            for (int i = 0; i < N; ++i)
#pragma unroll
                                for (int p = 0; p < PW; ++p)
                                    diff |= (uint32_t)(w[i][p] >> 32) ^ tag;
                            if (diff <= 1u) {
                                bad |= diff;
                                break;
                            }
                            if (!wt.more(res_args, prob)) {
                                late = 1;
                                break;
                            }
                        }
#pragma unroll
                        for (int i = 0; i < N; ++i) {
                            if constexpr (PW == 1)
                                acc += (double)(u0 + i < mine
                                                    ? __uint_as_float((uint32_t)w[i][0])
                                                    : 0.f);
                            else
                                acc += u0 + i < mine
                                           ? pack_d((uint32_t)w[i][0], (uint32_t)w[i][PW - 1])
                                           : 0.0;
                        }
                    }
                    return acc;
                };
                auto gather = [&](int j, int q0, int step) {
                    if (per <= 2)
                        return gather_n(j, q0, step, std::integral_constant<int, 2>{});
                    if (per <= 4)
                        return gather_n(j, q0, step, std::integral_constant<int, 4>{});
                    return gather_n(j, q0, step, std::integral_constant<int, 8>{});
                };
                if constexpr (!SOLO) {
                    ++seq;
                    tag = seq << 1;
                    pw = reinterpret_cast<const char *>(part + (size_t)(seq & 1) * G * XW * Mp);
                    cw = reinterpret_cast<char *>(cast + (size_t)(seq & 1) * BW * Mp);
                    char *mine = const_cast<char *>(pw) + (uint32_t)g * prow;
#pragma unroll
                    for (int kc = 0; kc < F::NK; ++kc) {
                        const int j = tj + kc * F::NT;
                        if (j < M) {
                            const double s = local_sum(j);
                            uint64_t *p = reinterpret_cast<uint64_t *>(mine + (uint32_t)j * 8u);
                            if constexpr (PW == 1) {
                                put_word(p, __float_as_uint((float)s), tag | bad);
                            } else {
                                const uint64_t x = (uint64_t)__double_as_longlong(s);
                                put_word(p, (uint32_t)x, tag | bad);
                                put_word(p + Mp, (uint32_t)(x >> 32), tag | bad);
                            }
                        }
                    }
                    if (split > 1) {
                        const int sp = t / cnp, jl = t % cnp;
                        // (fewer workgroups than groups: the rest have no partial)
                        double acc = jl < cn && sp < G ? gather(j0 + jl, sp, split) : 0.0;
                        // groups within a wave add up over the lanes, the rest
                        // in LDS
                        if (cnp == 16)
                            acc = pair_swap16(acc, acc);
                        if (cnp <= 32)
                            acc = pair_swap32(acc, acc);
                        const int sub = cnp >= 64 ? sp : t >> 6;
                        if (cnp >= 64 || lane < cnp)
                            S.xs[sub * cnp + jl] = acc;
                        if (bad & 1u)
                            S.flag_row[fp] = 1;
                        __syncthreads();
                        bad |= (uint32_t)S.flag_row[fp];
                    }
                }
                double b_new[KC];
                float eb_new[KC];
#pragma unroll
                for (int kc = 0; kc < KC; ++kc) {
                    const int jl = tj + kc * F::NT;
                    if (jl >= cn)
                        break;
                    const int j = j0 + jl;
                    double s;
                    if (SOLO) {
                        s = local_sum(j);
                    } else if (split > 1) {
                        s = 0.0;
                        for (int sub = 0; sub < min(split, F::NW); ++sub)
                            s += S.xs[sub * cnp + jl];
                    } else {
                        s = gather(j, 0, 1);
                    }
                    double b;
                    if (!unbal) {
                        b = cdead[kc] ? cb[kc] : cnu[kc] * U::recip(s);
                        b_new[kc] = b;
                    } else {
                        const double c = cref[kc];
                        const double ls = U::log_fast(s);
                        double lv = cdead[kc] ? cb[kc] : damp * (cnu[kc] - (ls + c));
                        if (PW > 1 && it + 1 == A.n_iter && !cdead[kc])
                            lv = damped_potential(damp, cnu[kc], ls, c);
                        if (PW == 1 || cdead[kc])
                            b = U::exp_fast(lv + c - kap);
                        else
                            b = U::exp_fast(damp * (cnu[kc] - ls) + ((1.0 - damp) * c - kap));
                        b_new[kc] = lv;
                    }
                    const bool ok = cdead[kc] ? s == 0.0
                                              : s >= kSumLo && s <= kSumHi && b <= mul_hi;
                    bad |= ok ? 0u : 1u;
                    eb_new[kc] = 0.f;
                    T h;
                    if constexpr (PW == 1) {
                        const double x = fma(b, (double)ceb[kc], b);
                        h = (float)x;
                        if (h > kCarryLo)
                            eb_new[kc] = (float)(x - (double)h) * __builtin_amdgcn_rcpf(h);
                    } else {
                        h = b;
                    }
                    S.b[j] = h;
                    if (SOLO || direct)
                        continue;
                    if constexpr (!SOLO) {
                        uint64_t *p = reinterpret_cast<uint64_t *>(cw + (uint32_t)j * 8u);
                        if constexpr (PW == 1) {
                            put_word(p, __float_as_uint(h), tag | (bad & 1u));
                        } else {
                            const uint64_t x = (uint64_t)__double_as_longlong(h);
                            put_word(p, (uint32_t)x, tag | (bad & 1u));
                            put_word(p + Mp, (uint32_t)(x >> 32), tag | (bad & 1u));
                        }
                    }
                }
                // every column's multiplier from its owner
                auto gather_b = [&]() {
                    constexpr int NK = F::NK;
                    uint64_t w[NK][PW];
                    Waiter wt(poll0);
                    for (;;) {
                        uint32_t diff = 0;
#pragma unroll
                        for (int kc = 0; kc < NK; ++kc)
#pragma unroll
                            for (int p = 0; p < PW; ++p)
                                w[kc][p] = get_word(reinterpret_cast<const uint64_t *>(
                                    cw + (uint32_t)(min(tj + kc * F::NT, M - 1) + p * Mp) * 8u));
#pragma unroll
                        for (int kc = 0; kc < NK; ++kc)
#pragma unroll
                            for (int p = 0; p < PW; ++p)
                                diff |= (uint32_t)(w[kc][p] >> 32) ^ tag;
                        if (diff <= 1u)
                            break;
                        if (!wt.more(res_args, prob)) {
                            late = 1;
                            break;
                        }
                    }
#pragma unroll
                    for (int kc = 0; kc < NK; ++kc) {
                        bad |= (uint32_t)(w[kc][0] >> 32);
                        const int j = tj + kc * F::NT;
                        if (j < M) {
                            if constexpr (PW == 1)
                                S.b[j] = __uint_as_float((uint32_t)w[kc][0]);
                            else
                                S.b[j] = pack_d((uint32_t)w[kc][0], (uint32_t)w[kc][PW - 1]);
                        }
                    }
                };
                if constexpr (!SOLO) {
                    if (!direct)
                        gather_b();
                }
                if (bad & 1u)
                    S.flag_all[fp] = 1;
                if (late)
                    S.abort = 1;
                __syncthreads();
                if (S.flag_all[fp] | S.abort) {
                    start = kExact;
                    break;
                }
#pragma unroll
                for (int kc = 0; kc < KC; ++kc) {
                    if (t + kc * F::NT < cn) {
                        cb[kc] = b_new[kc];
                        ceb[kc] = eb_new[kc];
                    }
                }
                L.a = a_new;
                L.ea = ea_new;
                L.lu = lu_new;
                L.derived = true;
                ++it;
                if (it == A.seg_end[seg] || trial) {
                    if (it == A.seg_end[seg])
                        ++seg;
                    start = kMoved;
                    break;
                }
            }
            W = L;
#pragma unroll
            for (int kc = 0; kc < KC; ++kc) {
                S.bd[t + kc * F::NT] = cb[kc];
                S.eb[t + kc * F::NT] = ceb[kc];
            }
            __syncthreads();
            if (start == kExact && !S.abort) {  // refused
                if (!direct)
                    ++seq;
                send_log_v<F>(SP, J, seq);
            }
        }
        finish_problem<F>(SP, J, W, static_cast<T *>(A.log_u) + prob * A.N + i0,
                          A.lu64 ? A.lu64 + prob * A.N + i0 : nullptr,
                          static_cast<T *>(A.log_v) + prob * M,
                          A.lv64 ? A.lv64 + prob * M : nullptr);
    }
}

// ---- kernel addresses of a tile configuration -----------------------------------

#define TM_KERNEL(T_, NW_, LC_, WC_, TC_, TR_, SOLO_) \
    reinterpret_cast<const void *>(&sk_resident<Cfg<T_, NW_, LC_, WC_, TC_, TR_, SOLO_>>)
#define TM_TILE(T_, NW_, LC_, WC_, TC_, TR_)                  \
    {                                                         \
        NW_, LC_, WC_, TC_, TR_,                              \
            TM_KERNEL(T_, NW_, LC_, (WC_ > 2 ? 1 : WC_), TC_, TR_, true),     \
            TM_KERNEL(T_, NW_, LC_, WC_, TC_, TR_, false)     \
    }

} // namespace
} // namespace tmamd
