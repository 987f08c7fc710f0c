// x pass of the nonlinear step on wavefront FFTs: templates and radix plans
// (xpass.hip and xpass_b.hip .. xpass_e.hip instantiate them over the lengths).
//
// For each line: inverse real FFTs of the full variables (two real lines are
// packed into one complex sequence, f0 + i f1), the quadratic products and
// the CFL maxima in registers, then forward real FFTs of the products (again
// two per complex sequence, separated with Hermitian symmetry) truncated to
// the kept kx.  This is the x-direction part of c2r_transform / r2c_transform
// (slabs.fftw3mpi/transforms.f90:155-301) fused with the products of
// PL_IMEX_timestepping_marching.f90:279-300 and compute_cfl_based_timestep
// (PL_IMEX_timestepping_marching.f90:200-254).
#pragma once

#include "kernels.hpp"
#include "wavefft.hpp"

namespace coral {

using wfft::Dft;
using wfft::group_sync;

// Radix plans.  Inverse: first stage R0 reads the packed spectrum from HBM,
// InvMid runs in LDS, the last stage RL leaves each lane holding the points
// j + r*N/RL of its lines.  Forward: first stage RL starts from those
// registers, FwdRest finishes in LDS in natural order.  LN lanes (one or
// more wavefronts) share LPW lines; where LPW * N / RL is no multiple of LN the
// last lanes of a register stage idle.  W0 / WL: the swizzles (wfft::swz) of
// the first inverse and first forward stages' LDS writes, which their readers
// (InvMid or the last inverse stage, FwdRest) apply; a swizzle permutes inside
// rows of eight, so it needs N a multiple of eight.
template <int... Rs>
struct Rads {};
template <int N_, int LN_, int LPW_, int R0_, int W0_, class Mid, int RL_, int WL_, class Rest>
struct XPlanOf;
template <int N_, int LN_, int LPW_, int R0_, int W0_, int... Ms, int RL_, int WL_, int... Fs>
struct XPlanOf<N_, LN_, LPW_, R0_, W0_, Rads<Ms...>, RL_, WL_, Rads<Fs...>> {
    static constexpr int N = N_, LN = LN_, LPW = LPW_, R0 = R0_, W0 = W0_, RL = RL_, WL = WL_;
    static_assert((R0 * ... * Ms) * RL == N && (RL * ... * Fs) == N, "the radices multiply to the length");
    static_assert((W0 == 0 && WL == 0) || N % 8 == 0, "swizzles need whole rows of eight");
    static constexpr int W0OUT = sizeof...(Ms) ? 0 : W0;   // swizzle the last inverse stage reads through
    template <int S> using InvMid = wfft::GStagesLSW<LN, N, +1, S, N, W0, false, R0, Ms...>;
    template <int S> using FwdRest = wfft::GStagesLSW<LN, N, -1, S, N, WL, false, RL, Fs...>;
};
// The lines per wavefront and the radices are the fastest of those measured
// per length: lanes of the register stages as full as possible, few LDS
// exchanges, at most 9 points of each full variable pair per lane (12 at 144
// points).  us per launch, 4 full and 9 quadratic variables, FP64, 18480 lines:
//   96: 12 x 8 on five lines 46, 4 x 4 x 6 on four 50, 16 x 6 on four 55;
//   144: 12 x 12 on five lines 64, 6 x 4 x 6 on two 70, 4 x 4 x 3 x 3 on four 97;
//   192: 8 x 4 x 6 on two lines 82, 16 x 12 on four 90, 4 x 4 x 4 x 3 on one 92;
//   288: 8 x 6 x 6 on one line 140, 9 x 4 x 8 on two 151, 12 x 4 x 6 on one 181;
// and 432 at 62640 lines: 8 x 6 x 9 657, 9 x 6 x 8 743, 12 x 6 x 6 893 (288 and
// 432 before balancing).  Against the workgroup-level LDS FFT that takes the
// other lengths (one real line per sequence, radices 2 to 4, a barrier per
// stage), ms per launch: 288 points (192^2 x 65) 1.44 -> 0.23, 432 (288^2 x 97)
// 4.67 -> 0.75, 216 (144 x 96 x 65) 0.64 -> 0.09, 108 (72 x 48 x 41) 0.23 -> 0.03.
template <int N>
struct XPlan;
#define XPLAN(n, ...)                                \
    template <>                                      \
    struct XPlan<n> : XPlanOf<n, __VA_ARGS__> {};
//        N  LN  LPW R0 W0  middle       RL WL  rest
XPLAN(24, 64, 10, 6, 0, Rads<>, 4, 0, Rads<6>)
XPLAN(27, 64, 7, 9, 0, Rads<>, 3, 0, Rads<9>)
XPLAN(36, 64, 10, 6, 0, Rads<>, 6, 0, Rads<6>)
XPLAN(48, 64, 8, 8, 4, Rads<>, 6, 0, Rads<8>)
XPLAN(54, 64, 7, 9, 0, Rads<>, 6, 0, Rads<9>)
XPLAN(72, 64, 7, 9, 0, Rads<>, 8, 4, Rads<9>)
XPLAN(81, 64, 7, 9, 0, Rads<>, 9, 0, Rads<9>)
XPLAN(96, 64, 5, 12, 0, Rads<>, 8, 4, Rads<12>)
XPLAN(108, 64, 5, 12, 0, Rads<>, 9, 0, Rads<12>)
XPLAN(144, 64, 5, 12, 0, Rads<>, 12, 0, Rads<12>)
XPLAN(162, 64, 2, 9, 0, Rads<3>, 6, 0, Rads<3, 9>)
XPLAN(192, 64, 2, 8, 4, Rads<4>, 6, 0, Rads<4, 8>)
XPLAN(216, 64, 2, 9, 0, Rads<3>, 8, 4, Rads<3, 9>)
XPLAN(243, 64, 2, 9, 0, Rads<3>, 9, 0, Rads<3, 9>)
XPLAN(288, 64, 1, 8, 4, Rads<6>, 6, 0, Rads<6, 8>)
XPLAN(324, 64, 1, 9, 0, Rads<6>, 6, 0, Rads<6, 9>)
// 384: the stride-8 writes of the first inverse stage put all 8 lanes of a
// row of eight on the same banks: swizzled (0.613 -> 0.599 ms per launch at
// 384^2 x 193); the 2-way conflicts of the first forward stage's stride-6
// writes cost less than their swizzle (0.624 ms with it)
XPLAN(384, 64, 1, 8, 4, Rads<8>, 6, 0, Rads<8, 8>)
XPLAN(432, 64, 1, 8, 4, Rads<6>, 9, 0, Rads<6, 8>)
XPLAN(486, 64, 1, 9, 0, Rads<6>, 9, 0, Rads<6, 9>)
XPLAN(576, 64, 1, 8, 4, Rads<8>, 9, 0, Rads<8, 8>)
// 648, 729, 768: two wavefronts per line: one lane holds 6 or 9 points of each
// full variable pair (at 768 points 96 VGPRs of them per lane in FP64 on one
// wavefront, which left two wavefronts per SIMD)
XPLAN(648, 128, 1, 9, 0, Rads<8>, 9, 0, Rads<8, 9>)
XPLAN(729, 128, 1, 9, 0, Rads<9>, 9, 0, Rads<9, 9>)
XPLAN(768, 128, 1, 8, 0, Rads<4, 4>, 6, 0, Rads<4, 4, 8>)
#undef XPLAN

// The plan of an element type: the FP32 chain, with half the registers and LDS
// per point, takes more points per lane at 192 points (114 -> 68 us per launch
// at 128^2 x 65) and at 384 (605 -> 528 us at 256^2 x 129).
template <int N, class C>
struct XPlanT : XPlan<N> {};
template <>
struct XPlanT<192, float2> : XPlanOf<192, 64, 4, 16, 0, Rads<>, 12, 0, Rads<16>> {};
template <>
struct XPlanT<384, float2> : XPlanOf<384, 64, 1, 6, 0, Rads<8>, 8, 4, Rads<8, 6>> {};

template <class P>
struct XShape {
    static constexpr int N = P::N, LPW = P::LPW, R0 = P::R0, RL = P::RL, LN = P::LN;
    static constexpr int T0 = N / R0, TL = N / RL;
    static constexpr int NT = (LPW * TL + LN - 1) / LN;  // (line, j) tasks per lane at the register stages
    static constexpr bool FULL = (LPW * TL) % LN == 0;   // every lane has all its tasks
    static constexpr int NK = N / 3;                     // kept kx (the 3/2 rule)
};

// value of full variable A (1 for A < 0) at point r of a task
template <int A, int NPI, int RL, class C>
__device__ inline typename CxT<C>::R fget(const C (&f)[NPI][RL], int r) {
    if constexpr (A < 0)
        return 1;
    else
        return (A & 1) ? f[A >> 1][r].y : f[A >> 1][r].x;
}

// o[r] = F_a at the RL points of a task.  a is the same for the whole
// wavefront: a scalar branch picks the copy (the empty asm keeps the branches
// from being turned into per-element selects, one v_cndmask per candidate).
template <int NPI, int RL, int K = 0, class C>
__device__ inline void pick(const C (&f)[NPI][RL], int a, typename CxT<C>::R (&o)[RL]) {
    if constexpr (K < 2 * NPI) {
        if (a == K) {
            asm volatile("");
#pragma unroll
            for (int r = 0; r < RL; ++r) o[r] = fget<K, NPI, RL>(f, r);
            return;
        }
        pick<NPI, RL, K + 1>(f, a, o);
    } else {
#pragma unroll
        for (int r = 0; r < RL; ++r) o[r] = 1;   // a < 0: the constant ONE
    }
}

template <int NPI, int RL, class C>
__device__ inline void product(const C (&f)[NPI][RL], int a, int b, typename CxT<C>::R (&p)[RL]) {
    typename CxT<C>::R fa[RL], fb[RL];
    pick<NPI, RL>(f, a, fa);
    pick<NPI, RL>(f, b, fb);
#pragma unroll
    for (int r = 0; r < RL; ++r) p[r] = fa[r] * fb[r];
}

// Per-line balancing of packed pairs.  Two real lines packed into one complex
// FFT share its rounding: each comes out with an error of about eps times the
// larger of the two, so a line much smaller than its partner (w beside t, a
// temperature product beside a velocity product) would lose most of its
// digits.  Balanced plans scale each line of a pair by the power of two that
// brings its largest component into [0.5, 1) before the FFT, and scale it back
// after it; both scalings are exact.  The maxima are reduced per line through
// LDS, as the high words of the magnitudes (bit patterns of non-negative
// numbers order as unsigned integers).  The FP32 chain balances at every
// length; FP64 plans balance where the alternative, the LDS FFT with one real
// line per sequence, keeps each line's own rounding (the other five lengths
// have always packed their lines as they are).
template <int N, class C>
constexpr bool x_balanced() {
    return sizeof(C) == 8 || !(N == 96 || N == 144 || N == 192 || N == 384 || N == 768);
}
constexpr int XBAL_SLOTS = 20;   // per lane group: 2 lines x lines per group

__device__ inline unsigned absmax_bits(float v) { return __float_as_uint(fabsf(v)); }
__device__ inline unsigned absmax_bits(double v) { return unsigned(__double2hiint(v)) & 0x7fffffffu; }
template <class C>
__device__ inline unsigned absmax_bits(C v) { return max(absmax_bits(v.x), absmax_bits(v.y)); }

// power of two bringing a positive maximum into [0.5, 1) (1 for zero,
// infinities and NaN), and its inverse; exponents are clamped so that both are
// normal numbers
template <class T>
__device__ inline T bal_pow(unsigned mbits, int sign) {
    constexpr bool D = sizeof(T) == 8;
    constexpr int BIAS = D ? 1023 : 127, SHIFT = D ? 20 : 23, TOP = 2 * BIAS - 2;
    int e = int(mbits >> SHIFT);
    if (mbits == 0u || e > 2 * BIAS) return T(1);
    e = (e < 2 ? 2 : (e > TOP ? TOP : e)) - (BIAS - 1);
    const unsigned hi = unsigned(BIAS + sign * e) << SHIFT;
    if constexpr (D)
        return __hiloint2double(int(hi), 0);
    else
        return __uint_as_float(hi);
}
// maximum over the wavefront, the same in every lane
__device__ inline unsigned wave_umax(unsigned m) {
#define DPP_MAX(ctrl) m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, ctrl, 0xf, 0xf, false))
    DPP_MAX(0x111);   // row_shr:1, 2, 4, 8: the maximum of each row of 16 in its last lane
    DPP_MAX(0x112);
    DPP_MAX(0x114);
    DPP_MAX(0x118);
    DPP_MAX(0x142);   // row_bcast:15, 31: rows into the next ones
    DPP_MAX(0x143);
#undef DPP_MAX
    return (unsigned)__builtin_amdgcn_readlane((int)m, 63);
}
// The maxima of a pair's two lines, for the lines of a lane group: one line
// on one wavefront keeps them in registers, the others in LDS slots 2 l, 2 l + 1.
template <class P>
struct PairMax {
    static constexpr bool WAVE = P::LPW == 1 && P::LN == 64;
    unsigned *slots, m0, m1;
    __device__ inline void begin(int lane) {
        m0 = m1 = 0u;
        if constexpr (!WAVE) {
            if (lane < 2 * P::LPW) slots[lane] = 0u;
            group_sync<P::LN>();
        }
    }
    __device__ inline void add(int l, unsigned a, unsigned b) {
        if constexpr (WAVE) {
            m0 = max(m0, a);
            m1 = max(m1, b);
        } else {
            atomicMax(&slots[2 * l], a);
            atomicMax(&slots[2 * l + 1], b);
        }
    }
    __device__ inline void end() {
        if constexpr (WAVE) {
            m0 = wave_umax(m0);
            m1 = wave_umax(m1);
        } else {
            group_sync<P::LN>();
        }
    }
    __device__ inline unsigned first(int l) const { return WAVE ? m0 : slots[2 * l]; }
    __device__ inline unsigned second(int l) const { return WAVE ? m1 : slots[2 * l + 1]; }
};
template <class T>
__device__ inline T bal_scale(unsigned mbits) { return bal_pow<T>(mbits, -1); }
// A line with an infinity or a NaN stays by itself, as where every line has a
// sequence of its own: the packing leaves its values out of the pair (a branch
// that is not taken otherwise; the empty asm keeps it from being turned into a
// select per value), and the scaling back makes every value of the line a NaN.
// Costs 1 % of the pass: us per launch 753 -> 759 at 288^2 x 97, 233 -> 236 at
// 192^2 x 65, 26.5 -> 27.0 at 72 x 48 x 41.  FP64 only: the lines of the FP32
// chain share their transforms at every length, as those of the five FP64
// lengths that do not balance do.
template <class T>
__device__ inline bool bal_bad(unsigned mbits) {
    return sizeof(T) == 8 && mbits >= 0x7ff00000u;
}
template <class T>
__device__ inline T bal_unscale(unsigned mbits) {
    return bal_bad<T>(mbits) ? T(__builtin_nanf("")) : bal_pow<T>(mbits, +1);
}
template <class V, int K>
__device__ inline void leave_out(bool bad, V (&v)[K]) {
    if (bad) {
        asm volatile("");
#pragma unroll
        for (int r = 0; r < K; ++r) {
            if constexpr (std::is_floating_point<V>::value)
                v[r] = 0;
            else
                v[r] = mkc<V>(0, 0);
        }
    }
}

// forward transforms of product pair pq (products 2 pq, 2 pq + 1) of the
// group's lines and the store of the kept kx
template <class P, int NPI, class C>
__device__ inline void xfwd_pair(const XPassArgs &a, const C (&fv)[XShape<P>::NT][NPI][P::RL], C *buf,
                                 const C *__restrict__ tw, int lane, long long line0, long long nlines, int pq,
                                 unsigned *xmax) {
    using X = XShape<P>;
    using T = typename CxT<C>::R;
    C *H = reinterpret_cast<C *>(a.H);
    constexpr int N = X::N, RL = X::RL, TL = X::TL, LPW = X::LPW, LN = X::LN;
    const int q0 = 2 * pq, q1 = q0 + 1;
    const bool has1 = q1 < a.nquad;
    const int a0 = __builtin_amdgcn_readfirstlane(a.qa[q0]), b0 = __builtin_amdgcn_readfirstlane(a.qb[q0]);
    const int a1 = has1 ? __builtin_amdgcn_readfirstlane(a.qa[q1]) : -1;
    const int b1 = has1 ? __builtin_amdgcn_readfirstlane(a.qb[q1]) : -1;
    auto products = [&](int c, T (&p0)[RL], T (&p1)[RL]) {
        product<NPI, RL>(fv[c], a0, b0, p0);
        if (has1)
            product<NPI, RL>(fv[c], a1, b1, p1);
        else
#pragma unroll
            for (int r = 0; r < RL; ++r) p1[r] = 0;
    };
    PairMax<P> pm{xmax};
    if constexpr (x_balanced<N, C>()) {
        static_assert(2 * LPW <= XBAL_SLOTS, "balancing slots");
        // products of every task first, their per-line maxima, then the scaled FFTs
        T p0[X::NT][RL], p1[X::NT][RL];
        pm.begin(lane);
#pragma unroll
        for (int c = 0; c < X::NT; ++c) {
            const int t = lane + LN * c, l = t / TL;
            if (!X::FULL && t >= LPW * TL) break;
            products(c, p0[c], p1[c]);
            unsigned m0 = 0u, m1 = 0u;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                m0 = max(m0, absmax_bits(p0[c][r]));
                m1 = max(m1, absmax_bits(p1[c][r]));
            }
            pm.add(l, m0, m1);
        }
        pm.end();
#pragma unroll
        for (int c = 0; c < X::NT; ++c) {
            const int t = lane + LN * c, l = t / TL, j = t - l * TL;
            if (!X::FULL && t >= LPW * TL) break;
            const T s0 = bal_scale<T>(pm.first(l)), s1 = bal_scale<T>(pm.second(l));
            leave_out(bal_bad<T>(pm.first(l)), p0[c]);
            leave_out(bal_bad<T>(pm.second(l)), p1[c]);
            C y[RL];
#pragma unroll
            for (int r = 0; r < RL; ++r) y[r] = mkc<C>(p0[c][r] * s0, p1[c][r] * s1);
            Dft<RL, -1>::run(y);
#pragma unroll
            for (int r = 0; r < RL; ++r) buf[l * N + wfft::swz<P::WL>(j * RL + r)] = y[r];
        }
    } else {
#pragma unroll
        for (int c = 0; c < X::NT; ++c) {
            const int t = lane + LN * c, l = t / TL, j = t - l * TL;
            if (!X::FULL && t >= LPW * TL) break;
            T p0[RL], p1[RL];
            products(c, p0, p1);
            C y[RL];
#pragma unroll
            for (int r = 0; r < RL; ++r) y[r] = mkc<C>(p0[r], p1[r]);
            Dft<RL, -1>::run(y);
#pragma unroll
            for (int r = 0; r < RL; ++r) buf[l * N + wfft::swz<P::WL>(j * RL + r)] = y[r];
        }
    }
    group_sync<LN>();
    P::template FwdRest<LPW>::run(buf, tw, lane);
    // the kept kx of the group's lines are consecutive in H: one run of LPW * NK
    // values per variable, whole cache lines also where NK is small
    const long long left = nlines - line0;
    const int have = (left < LPW ? (left < 0 ? 0 : int(left)) : LPW) * X::NK;
    C *h0 = H + ((size_t)q0 * nlines + line0) * X::NK;
    C *h1 = H + ((size_t)q1 * nlines + line0) * X::NK;
#pragma unroll
    for (int i = 0; i < (LPW * X::NK + LN - 1) / LN; ++i) {
        const int e = lane + LN * i;
        if (e < have) {
            const int l = e / X::NK, k = e - l * X::NK;
            const C *L = buf + l * N;
            T hf0 = T(0.5), hf1 = T(0.5);
            if constexpr (x_balanced<N, C>()) {
                hf0 *= bal_unscale<T>(pm.first(l));
                hf1 *= bal_unscale<T>(pm.second(l));
            }
            const C y = L[k], yc = cconj(L[k == 0 ? 0 : N - k]);
            // p0 = (Y + conj Y(-k)) / 2,  p1 = -i (Y - conj Y(-k)) / 2
            h0[e] = mkc<C>(hf0 * (y.x + yc.x), hf0 * (y.y + yc.y));
            if (has1) h1[e] = mkc<C>(hf1 * (y.y - yc.y), -hf1 * (y.x - yc.x));
        }
    }
    group_sync<LN>();
}

// C: element type of G, H and the FFTs (double2, or float2 for the FP32 chain)
template <int N_, int NPI, class C>
__global__ __launch_bounds__(256) void k_xpass_wave(XPassArgs a, const C *__restrict__ tw, long long nlines) {
    using P = XPlanT<N_, C>;
    using X = XShape<P>;
    using T = typename CxT<C>::R;
    constexpr int N = X::N, NK = X::NK, R0 = X::R0, RL = X::RL, T0 = X::T0, TL = X::TL, LPW = X::LPW, LN = X::LN;
    extern __shared__ unsigned char lds_raw[];
    C *lds = reinterpret_cast<C *>(lds_raw);
    __shared__ double cfl_part[4][3];
    __shared__ unsigned xmax_all[4][XBAL_SLOTS];   // per-line maxima of packed pairs (balanced plans)
    // lane in the group of LN lanes that shares LPW lines, group in the workgroup
    const int lane = threadIdx.x % LN, grp = threadIdx.x / LN, wid = threadIdx.x >> 6;
    unsigned *xmax = xmax_all[grp];
    C *buf = lds + grp * LPW * N;
    const C *G = reinterpret_cast<const C *>(a.G);
    const long long line0 = ((long long)blockIdx.x * (blockDim.x / LN) + grp) * LPW;

    // ---- inverse transforms, one packed pair of full variables at a time
    // (half the LDS of both pairs at once, which buys a wavefront per SIMD);
    // the last stage leaves fv[task][pair][r] at x = j + r*TL in registers ----
    C fv[X::NT][NPI][RL];
#pragma unroll
    for (int p = 0; p < NPI; ++p) {
        const int f0 = 2 * p, f1 = 2 * p + 1;
        const bool has1 = f1 < a.nfull;
        PairMax<P> pm{xmax};
        if constexpr (x_balanced<N, C>() && PairMax<P>::WAVE) {
            // the line's maxima from a first read of its spectra (kx = 0
            // imaginary parts dropped); the first stage finds them in cache and
            // holds no second copy in registers (288^2 x 97: 916 -> 761 us)
            const bool valid = line0 < nlines;
            const C *g0 = G + ((size_t)f0 * nlines + (valid ? line0 : 0)) * NK;
            const C *g1 = G + ((size_t)(has1 ? f1 : f0) * nlines + (valid ? line0 : 0)) * NK;
            pm.begin(lane);
#pragma unroll
            for (int i = 0; i < (NK + 63) / 64; ++i) {
                const int k = lane + 64 * i;
                if (k < NK) {
                    const C A = g0[k], B = g1[k];
                    pm.add(0, k ? absmax_bits(A) : absmax_bits(A.x), k ? absmax_bits(B) : absmax_bits(B.x));
                }
            }
            pm.end();
        }
        if constexpr (x_balanced<N, C>() && !PairMax<P>::WAVE) {
            static_assert(2 * LPW <= XBAL_SLOTS, "balancing slots");
            constexpr int TOT = LPW * T0, ROUNDS = (TOT + LN - 1) / LN;
            // the two lines' values first (kept slots only, kx = 0 imaginary
            // parts dropped), their per-line maxima, then the scaled packing
            C va[ROUNDS][R0], vb[ROUNDS][R0];
            pm.begin(lane);
#pragma unroll
            for (int c = 0; c < ROUNDS; ++c) {
                const int b = lane + LN * c;
                if (TOT % LN == 0 || b < TOT) {
                    const int l = b / T0, j = b - l * T0;
                    const long long line = line0 + l;
                    const bool valid = line < nlines;
                    const size_t lo = valid ? (size_t)line : 0;
                    const C *g0 = G + ((size_t)f0 * nlines + lo) * NK;
                    const C *g1 = G + ((size_t)(has1 ? f1 : f0) * nlines + lo) * NK;
                    unsigned ma = 0u, mb = 0u;
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int e = j + r * T0;
                        const int lo = r * T0, hi = lo + T0 - 1;
                        const bool all_pos = hi < NK;
                        const bool all_neg = lo > N - NK;
                        const bool all_zero = lo >= NK && hi <= N - NK;
                        if (all_zero) {
                            va[c][r] = vb[c][r] = mkc<C>(0, 0);
                            continue;
                        }
                        const bool pos = all_pos || (!all_neg && e < NK);
                        const bool neg = all_neg || (!all_pos && e > N - NK);
                        const int k = pos ? e : (neg ? N - e : 0);
                        const C A = g0[k], B = g1[k];
                        const bool e0 = r == 0 && j == 0;
                        const bool keep = valid && (all_pos || all_neg || pos || neg);
                        va[c][r] = mkc<C>(keep ? A.x : T(0), (keep && !e0) ? A.y : T(0));
                        vb[c][r] = mkc<C>((keep && has1) ? B.x : T(0), (keep && has1 && !e0) ? B.y : T(0));
                        ma = max(ma, absmax_bits(va[c][r]));
                        mb = max(mb, absmax_bits(vb[c][r]));
                    }
                    pm.add(l, ma, mb);
                }
            }
            pm.end();
#pragma unroll
            for (int c = 0; c < ROUNDS; ++c) {
                const int b = lane + LN * c;
                if (TOT % LN == 0 || b < TOT) {
                    const int l = b / T0, j = b - l * T0;
                    const T sa = bal_scale<T>(pm.first(l)), sb = bal_scale<T>(pm.second(l));
                    leave_out(bal_bad<T>(pm.first(l)), va[c]);
                    leave_out(bal_bad<T>(pm.second(l)), vb[c]);
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int e = j + r * T0;
                        const int lo = r * T0;
                        const bool all_neg = lo > N - NK;
                        const bool all_pos = lo + T0 - 1 < NK;
                        const bool pos = all_pos || (!all_neg && e < NK);
                        const T ax = va[c][r].x * sa, ay = va[c][r].y * sa;
                        const T bx = vb[c][r].x * sb, by = vb[c][r].y * sb;
                        // pos: A + iB;  neg: conj(A) + i conj(B)
                        va[c][r] = mkc<C>(pos ? ax - by : ax + by, pos ? ay + bx : bx - ay);
                    }
                    Dft<R0, +1>::run(va[c]);
#pragma unroll
                    for (int r = 0; r < R0; ++r) buf[l * N + wfft::swz<P::W0>(j * R0 + r)] = va[c][r];
                }
            }
            group_sync<LN>();
        } else {
            // first stage: packed Hermitian spectra straight from HBM
            constexpr int TOT = LPW * T0, ROUNDS = (TOT + LN - 1) / LN;
            C v[ROUNDS][R0];
#pragma unroll
            for (int c = 0; c < ROUNDS; ++c) {
                const int b = lane + LN * c;
                if (TOT % LN == 0 || b < TOT) {
                    const int l = b / T0, j = b - l * T0;
                    const long long line = line0 + l;
                    const bool valid = line < nlines;
                    const size_t lo = valid ? (size_t)line : 0;
                    const C *g0 = G + ((size_t)f0 * nlines + lo) * NK;
                    const C *g1 = G + ((size_t)(has1 ? f1 : f0) * nlines + lo) * NK;
                    T sa = 1, sb = 1;
                    if constexpr (x_balanced<N, C>()) {
                        // a line left out: its partner's values in its place
                        const bool bad0 = bal_bad<T>(pm.first(l)), bad1 = bal_bad<T>(pm.second(l));
                        const unsigned ma = bad0 ? pm.second(l) : pm.first(l), mb = bad1 ? pm.first(l) : pm.second(l);
                        const C *h0 = g0;
                        g0 = bad0 ? g1 : g0;
                        g1 = bad1 ? h0 : g1;
                        sa = bal_scale<T>(ma);
                        sb = bal_scale<T>(mb);
                    }
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int e = j + r * T0;
                        // the slots [r T0, (r+1) T0) that hold only positive,
                        // only negative or only dealiased kx are known once
                        // the loop is unrolled
                        const int lo = r * T0, hi = lo + T0 - 1;
                        const bool all_pos = hi < NK;
                        const bool all_neg = lo > N - NK;
                        const bool all_zero = lo >= NK && hi <= N - NK;
                        if (all_zero) {
                            v[c][r] = mkc<C>(0, 0);
                            continue;
                        }
                        const bool pos = all_pos || (!all_neg && e < NK);
                        const bool neg = all_neg || (!all_pos && e > N - NK);
                        const int k = pos ? e : (neg ? N - e : 0);
                        C A = g0[k], B = g1[k];
                        if constexpr (x_balanced<N, C>()) {
                            A = cscale(A, sa);
                            B = cscale(B, sb);
                        }
                        const bool e0 = r == 0 && j == 0;   // kx = 0: imaginary parts dropped
                        const T bx = has1 ? B.x : T(0), by = (has1 && !e0) ? B.y : T(0);
                        const T ay = !e0 ? A.y : T(0);
                        // pos: A + iB;  neg: conj(A) + i conj(B)
                        T zx = pos ? A.x - by : A.x + by;
                        T zy = pos ? ay + bx : bx - ay;
                        const bool keep = valid && (all_pos || all_neg || pos || neg);
                        v[c][r] = mkc<C>(keep ? zx : T(0), keep ? zy : T(0));
                    }
                    Dft<R0, +1>::run(v[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < ROUNDS; ++c) {
                const int b = lane + LN * c;
                if (TOT % LN == 0 || b < TOT) {
                    const int l = b / T0, j = b - l * T0;
#pragma unroll
                    for (int r = 0; r < R0; ++r) buf[l * N + wfft::swz<P::W0>(j * R0 + r)] = v[c][r];
                }
            }
            group_sync<LN>();
        }
        P::template InvMid<LPW>::run(buf, tw, lane);
        // last stage into registers
#pragma unroll
        for (int c = 0; c < X::NT; ++c) {
            const int t = lane + LN * c, l = t / TL, j = t - l * TL;
            if (!X::FULL && t >= LPW * TL) break;
            const C *L = buf + l * N;
            C wp[RL];
            wfft::twiddle_powers<RL, +1>(tw, j, wp);
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                C x = L[wfft::swz<P::W0OUT>(j + r * TL)];
                if (r > 0) x = cmul(x, wp[r]);
                fv[c][p][r] = x;
            }
            Dft<RL, +1>::run(fv[c][p]);
            if constexpr (x_balanced<N, C>()) {
                const T ua = bal_unscale<T>(pm.first(l)), ub = bal_unscale<T>(pm.second(l));
#pragma unroll
                for (int r = 0; r < RL; ++r) fv[c][p][r] = mkc<C>(fv[c][p][r].x * ua, fv[c][p][r].y * ub);
            }
        }
        group_sync<LN>();
    }

    // ---- CFL maxima over u, v, w / weight_z (full variables 0, 1, 2) ----
    if constexpr (NPI >= 2) {
      if (a.cflmax && a.nfull >= 3) {
        double mu = 0.0, mv = 0.0, mw = 0.0;
#pragma unroll
        for (int c = 0; c < X::NT; ++c) {
            const int t = lane + LN * c, l = t / TL;
            const long long line = line0 + l;
            if (line < nlines && (X::FULL || t < LPW * TL)) {
                // max |w| / zw = (max |w|) / zw: rounded division by a
                // positive number keeps the order, so one division per task
                double wm = 0.0;
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    mu = fmax(mu, fabs(double(fv[c][0][r].x)));
                    mv = fmax(mv, fabs(double(fv[c][0][r].y)));
                    wm = fmax(wm, fabs(double(fv[c][1][r].x)));
                }
                mw = fmax(mw, wm / a.zweight[unsigned(line) / unsigned(a.NYAA)]);
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            mu = fmax(mu, __shfl_xor(mu, off));
            mv = fmax(mv, __shfl_xor(mv, off));
            mw = fmax(mw, __shfl_xor(mw, off));
        }
        if ((threadIdx.x & 63) == 0) {   // per wavefront, not per lane group
            cfl_part[wid][0] = mu;
            cfl_part[wid][1] = mv;
            cfl_part[wid][2] = mw;
        }
        __syncthreads();
        if (threadIdx.x < 3) {
            double m = 0.0;
            for (int w = 0; w < (int)(blockDim.x >> 6); ++w) m = fmax(m, cfl_part[w][threadIdx.x]);
            atomicMax(&a.cflmax[threadIdx.x], (unsigned long long)__double_as_longlong(m));
        }
      }
    }

    // ---- products and forward transforms, one pair of products at a time
    // (the registers of two would cost a wavefront per SIMD) ----
    const int npairs = (a.nquad + 1) / 2;
    for (int pq = 0; pq < npairs; ++pq) xfwd_pair<P, NPI>(a, fv, buf, tw, lane, line0, nlines, pq, xmax);
}

template <int N, int NPI, class C>
static bool launch_wave(hipStream_t st, const C *tw, const XPassArgs &a) {
    using X = XShape<XPlanT<N, C>>;
    constexpr int WPG = X::LN / 64;   // wavefronts per lane group
    static_assert(4 % WPG == 0, "a workgroup holds whole lane groups");
    const long long nlines = (long long)a.NZAA * a.NYAA;
    const size_t per_group = size_t(X::LPW) * N * sizeof(C);
    const int wpb = a.max_wpb >= 1 && a.max_wpb <= 4 ? a.max_wpb : 4;
    int gpb = wpb / WPG > 0 ? wpb / WPG : 1;   // lane groups per workgroup
    while (gpb > 1 && gpb * per_group > 65536) gpb /= 2;
    if (gpb * per_group > 65536) return false;
    const long long per_block = (long long)gpb * X::LPW;
    const unsigned blocks = unsigned((nlines + per_block - 1) / per_block);
    hipLaunchKernelGGL((k_xpass_wave<N, NPI, C>), dim3(blocks), dim3(X::LN * gpb), gpb * per_group, st, a, tw,
                       nlines);
    check_launch("x pass");
    return true;
}

template <int N, class C>
static bool launch_wave_c(hipStream_t st, const C *tw, const XPassArgs &a) {
    if (!tw || 3 * a.nkx != N) return false;
    switch ((a.nfull + 1) / 2) {
    case 1: return launch_wave<N, 1>(st, tw, a);
    case 2: return launch_wave<N, 2>(st, tw, a);
    case 3: return launch_wave<N, 3>(st, tw, a);
    default: return false;
    }
}

// lengths with an FP32 chain
constexpr bool x_has32(int N) { return N == 96 || N == 144 || N == 192 || N == 384 || N == 768; }

template <int N>
bool xpass_len(hipStream_t st, const FFTPlan &px, const XPassArgs &a) {
    if (!a.fp32) return launch_wave_c<N>(st, px.tw, a);
    if constexpr (x_has32(N)) return launch_wave_c<N>(st, px.twf, a);
    return false;
}

// ---- the x transforms alone (FP64) ----
// c2r of nbatch variables, G[b][line][kx] -> phys[b][line][x], and r2c,
// phys -> H[b][line][kx] (kept kx), on the x pass's plans: two variables of a
// line (b = 2p, 2p + 1, blockIdx.y = p) share one complex sequence, the inverse
// from the packed Hermitian spectra as in the x pass, the forward separated
// with Hermitian symmetry as its products are.  The c2r / r2c of
// slabs.fftw3mpi/transforms.f90:155-301 in x, for the transform seam, the
// physical outputs, the side products and the closure's inputs and outputs.
// At the lengths that balance their pairs in the x pass every variable has a
// sequence of its own (x_pack variables per sequence).
template <int N>
constexpr int x_pack() { return x_balanced<N, double2>() ? 1 : 2; }

template <int N>
__global__ __launch_bounds__(256) void k_xbwd_wave(const double2 *__restrict__ G, double *__restrict__ phys,
                                                   const double2 *__restrict__ tw, long long nlines, int nbatch) {
    using P = XPlan<N>;
    using X = XShape<P>;
    using C = double2;
    constexpr int NK = X::NK, R0 = X::R0, RL = X::RL, T0 = X::T0, TL = X::TL, LPW = X::LPW, LN = X::LN;
    extern __shared__ unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw) + (threadIdx.x / LN) * LPW * N;
    const int lane = threadIdx.x % LN;
    const long long line0 = ((long long)blockIdx.x * (blockDim.x / LN) + threadIdx.x / LN) * LPW;

    const int f0 = x_pack<N>() * blockIdx.y, f1 = f0 + 1;
    const bool has1 = x_pack<N>() == 2 && f1 < nbatch;
    {
        constexpr int TOT = LPW * T0, ROUNDS = (TOT + LN - 1) / LN;
        C v[ROUNDS][R0];
#pragma unroll
        for (int c = 0; c < ROUNDS; ++c) {
            const int b = lane + LN * c;
            if (TOT % LN == 0 || b < TOT) {
                const int l = b / T0, j = b - l * T0;
                const long long line = line0 + l;
                const bool valid = line < nlines;
                const size_t lo = valid ? (size_t)line : 0;
                const C *g0 = G + ((size_t)f0 * nlines + lo) * NK;
                const C *g1 = G + ((size_t)(has1 ? f1 : f0) * nlines + lo) * NK;
#pragma unroll
                for (int r = 0; r < R0; ++r) {
                    const int e = j + r * T0;
                    const int lo_e = r * T0, hi_e = lo_e + T0 - 1;
                    const bool all_pos = hi_e < NK;
                    const bool all_neg = lo_e > N - NK;
                    const bool all_zero = lo_e >= NK && hi_e <= N - NK;
                    if (all_zero) {
                        v[c][r] = mkc<C>(0, 0);
                        continue;
                    }
                    const bool pos = all_pos || (!all_neg && e < NK);
                    const bool neg = all_neg || (!all_pos && e > N - NK);
                    const int k = pos ? e : (neg ? N - e : 0);
                    const C A = g0[k], B = g1[k];
                    const bool e0 = r == 0 && j == 0;   // kx = 0: imaginary parts dropped
                    const double bx = has1 ? B.x : 0.0, by = (has1 && !e0) ? B.y : 0.0;
                    const double ay = !e0 ? A.y : 0.0;
                    // pos: A + iB;  neg: conj(A) + i conj(B)
                    const double zx = pos ? A.x - by : A.x + by;
                    const double zy = pos ? ay + bx : bx - ay;
                    const bool keep = valid && (all_pos || all_neg || pos || neg);
                    v[c][r] = mkc<C>(keep ? zx : 0.0, keep ? zy : 0.0);
                }
                Dft<R0, +1>::run(v[c]);
            }
        }
#pragma unroll
        for (int c = 0; c < ROUNDS; ++c) {
            const int b = lane + LN * c;
            if (TOT % LN == 0 || b < TOT) {
                const int l = b / T0, j = b - l * T0;
#pragma unroll
                for (int r = 0; r < R0; ++r) buf[l * N + wfft::swz<P::W0>(j * R0 + r)] = v[c][r];
            }
        }
        group_sync<LN>();
    }
    P::template InvMid<LPW>::run(buf, tw, lane);
    // last stage in registers: x = j + r TL of both lines, stored to consecutive x
#pragma unroll
    for (int c = 0; c < X::NT; ++c) {
        const int t = lane + LN * c, l = t / TL, j = t - l * TL;
        if (!X::FULL && t >= LPW * TL) break;
        const long long line = line0 + l;
        const C *L = buf + l * N;
        C wp[RL], x[RL];
        wfft::twiddle_powers<RL, +1>(tw, j, wp);
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            x[r] = L[wfft::swz<P::W0OUT>(j + r * TL)];
            if (r > 0) x[r] = cmul(x[r], wp[r]);
        }
        Dft<RL, +1>::run(x);
        if (line < nlines) {
            double *o0 = phys + ((size_t)f0 * nlines + line) * N + j;
            double *o1 = phys + ((size_t)f1 * nlines + line) * N + j;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                o0[r * TL] = x[r].x;
                if (has1) o1[r * TL] = x[r].y;
            }
        }
    }
}

template <int N>
__global__ __launch_bounds__(256) void k_xfwd_wave(const double *__restrict__ phys, double2 *__restrict__ H,
                                                   const double2 *__restrict__ tw, long long nlines, int nbatch) {
    using P = XPlan<N>;
    using X = XShape<P>;
    using C = double2;
    constexpr int NK = X::NK, RL = X::RL, TL = X::TL, LPW = X::LPW, LN = X::LN;
    extern __shared__ unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw) + (threadIdx.x / LN) * LPW * N;
    const int lane = threadIdx.x % LN;
    const long long line0 = ((long long)blockIdx.x * (blockDim.x / LN) + threadIdx.x / LN) * LPW;
    const int f0 = x_pack<N>() * blockIdx.y, f1 = f0 + 1;
    const bool has1 = x_pack<N>() == 2 && f1 < nbatch;
    // first forward stage from the two lines' values at x = j + r TL
#pragma unroll
    for (int c = 0; c < X::NT; ++c) {
        const int t = lane + LN * c, l = t / TL, j = t - l * TL;
        if (!X::FULL && t >= LPW * TL) break;
        const long long line = line0 + l;
        const bool valid = line < nlines;
        const double *i0 = phys + ((size_t)f0 * nlines + (valid ? line : 0)) * N + j;
        const double *i1 = phys + ((size_t)(has1 ? f1 : f0) * nlines + (valid ? line : 0)) * N + j;
        C y[RL];
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const double a = i0[r * TL], b = i1[r * TL];
            y[r] = mkc<C>(valid ? a : 0.0, (valid && has1) ? b : 0.0);
        }
        Dft<RL, -1>::run(y);
#pragma unroll
        for (int r = 0; r < RL; ++r) buf[l * N + wfft::swz<P::WL>(j * RL + r)] = y[r];
    }
    group_sync<LN>();
    P::template FwdRest<LPW>::run(buf, tw, lane);
    const long long left = nlines - line0;
    const int have = (left < LPW ? (left < 0 ? 0 : int(left)) : LPW) * NK;
    C *h0 = H + ((size_t)f0 * nlines + line0) * NK;
    C *h1 = H + ((size_t)f1 * nlines + line0) * NK;
#pragma unroll
    for (int i = 0; i < (LPW * NK + LN - 1) / LN; ++i) {
        const int e = lane + LN * i;
        if (e < have) {
            const int l = e / NK, k = e - l * NK;
            const C *L = buf + l * N;
            const C y = L[k], yc = cconj(L[k == 0 ? 0 : N - k]);
            // f0 = (Y + conj Y(-k)) / 2,  f1 = -i (Y - conj Y(-k)) / 2
            h0[e] = mkc<C>(0.5 * (y.x + yc.x), 0.5 * (y.y + yc.y));
            if (has1) h1[e] = mkc<C>(0.5 * (y.y - yc.y), -0.5 * (y.x - yc.x));
        }
    }
}

// grid of the x transforms: lane groups per workgroup within 64 KiB of LDS,
// blockIdx.y over the sequences
template <int N>
static bool xt_shape(long long nlines, int nbatch, dim3 &grid, dim3 &block, size_t &shm) {
    using X = XShape<XPlan<N>>;
    const size_t per_group = size_t(X::LPW) * N * sizeof(double2);
    int gpb = 4 / (X::LN / 64);
    while (gpb > 1 && gpb * per_group > 65536) gpb /= 2;
    if (gpb * per_group > 65536) return false;
    const long long per_block = (long long)gpb * X::LPW;
    grid = dim3(unsigned((nlines + per_block - 1) / per_block), unsigned((nbatch + x_pack<N>() - 1) / x_pack<N>()));
    block = dim3(X::LN * gpb);
    shm = gpb * per_group;
    return true;
}

template <int N>
bool xbwd_n(hipStream_t st, const double2 *tw, const double2 *G, double *phys, int nbatch, long long nlines) {
    dim3 grid, block;
    size_t shm;
    if (!xt_shape<N>(nlines, nbatch, grid, block, shm)) return false;
    hipLaunchKernelGGL((k_xbwd_wave<N>), grid, block, shm, st, G, phys, tw, nlines, nbatch);
    check_launch("x c2r");
    return true;
}

template <int N>
bool xfwd_n(hipStream_t st, const double2 *tw, const double *phys, double2 *H, int nbatch, long long nlines) {
    dim3 grid, block;
    size_t shm;
    if (!xt_shape<N>(nlines, nbatch, grid, block, shm)) return false;
    hipLaunchKernelGGL((k_xfwd_wave<N>), grid, block, shm, st, phys, H, tw, nlines, nbatch);
    check_launch("x r2c");
    return true;
}

// the lengths, and who compiles them
#define XLENGTHS_A(X) X(24) X(27) X(36) X(48) X(54) X(72)
#define XLENGTHS_B(X) X(81) X(96) X(108) X(144)
#define XLENGTHS_C(X) X(162) X(192) X(216) X(243)
#define XLENGTHS_D(X) X(288) X(324) X(384) X(432)
#define XLENGTHS_E(X) X(486) X(576) X(648) X(729) X(768)
#define XLENGTHS(X) XLENGTHS_A(X) XLENGTHS_B(X) XLENGTHS_C(X) XLENGTHS_D(X) XLENGTHS_E(X)
#define XEXTERN(n)                                                                                       \
    extern template bool xpass_len<n>(hipStream_t, const FFTPlan &, const XPassArgs &);                  \
    extern template bool xbwd_n<n>(hipStream_t, const double2 *, const double2 *, double *, int, long long); \
    extern template bool xfwd_n<n>(hipStream_t, const double2 *, const double *, double2 *, int, long long);
#define XINSTANCE(n)                                                                                     \
    template bool xpass_len<n>(hipStream_t, const FFTPlan &, const XPassArgs &);                         \
    template bool xbwd_n<n>(hipStream_t, const double2 *, const double2 *, double *, int, long long);    \
    template bool xfwd_n<n>(hipStream_t, const double2 *, const double *, double2 *, int, long long);

}  // namespace coral
