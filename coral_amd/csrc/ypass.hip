// y passes of the horizontal transforms on wavefront-local FFTs.
//
// A workgroup owns YL consecutive kx columns of one (variable, z) plane, so
// every global access covers YL consecutive kx (YL complex = 128 B, 64 B from
// 486 points) or a whole kept-ky line; each wavefront transforms its own
// lines in LDS without workgroup barriers (YL / ywaves of them).  These are the y-direction parts of c2r_transform
// (backward c2c in y) and r2c_transform (forward c2c in y, truncated to the
// kept ky), slabs.fftw3mpi/transforms.f90:155-301.
#include "kernels.hpp"
#include "wavefft.hpp"

#include <cstdio>

namespace coral {

using wfft::swz;


// Radix plans.  Stages write swizzled where N is a multiple of
// eight; the other lengths start with a stride-9 or stride-6 stage, whose
// writes spread over the banks by themselves.  Against the workgroup-level LDS
// FFT of the other lengths (radices 2 to 4, a barrier per stage), forward and
// inverse ms per launch: 192^2 x 65 (288 points) 0.29 -> 0.13, 0.13 -> 0.06;
// 288^2 x 97 (432) 1.08 -> 0.43, 0.54 -> 0.20.
template <int N>
struct YPlan;
#define YPLAN(n, ...)                                                                                        \
    template <>                                                                                              \
    struct YPlan<n> {                                                                                        \
        template <int SIGN, int S, int LS>                                                                   \
        using Run = wfft::StagesLSW<n, SIGN, S, LS, 0, n % 8 == 0, 1, __VA_ARGS__>;                          \
    };
YPLAN(24, 4, 6)
YPLAN(27, 9, 3)
YPLAN(36, 6, 6)
YPLAN(48, 6, 8)
YPLAN(54, 9, 6)
YPLAN(72, 9, 8)
YPLAN(81, 9, 9)
YPLAN(96, 4, 4, 6)
YPLAN(108, 9, 12)
YPLAN(144, 4, 4, 3, 3)
YPLAN(162, 9, 3, 6)
YPLAN(192, 4, 4, 4, 3)
YPLAN(216, 9, 4, 6)
YPLAN(243, 9, 9, 3)
YPLAN(288, 9, 4, 8)
YPLAN(324, 9, 6, 6)
YPLAN(384, 4, 4, 4, 6)
YPLAN(432, 9, 6, 8)
YPLAN(486, 9, 9, 6)
YPLAN(576, 9, 8, 8)
YPLAN(648, 9, 9, 8)
YPLAN(729, 9, 9, 9)
YPLAN(768, 8, 4, 4, 6)
#undef YPLAN

// kept ky index jy -> slot of the NYAA-long line
__device__ inline int ky_slot(int jy, int NY, int N) { return jy < NY / 2 ? jy : N - (NY - 1) + jy; }

// kx columns per workgroup for element type C: one 128-byte segment, 64
// bytes from 486 points.  At 768 points a 128-byte tile of lines fills 98 KB of
// LDS and leaves one workgroup per CU; the 49 KB tile fits three (512^2 x 257:
// FP64 yfwd 5.34 -> 4.61 ms, ybwd 2.30 -> 2.06 ms per launch).
constexpr int ycol_bytes(int N) { return N >= 486 ? 64 : 128; }
template <int N, class C>
constexpr int ycols() { return int(ycol_bytes(N) / sizeof(C)); }

// wavefronts per workgroup.  Two up to 81 points, where four lines still leave
// lanes idle.  At 768 points (and from 216 in FP64) one line per
// wavefront rather than four wavefronts of two or four lines each: the
// tile's LDS bounds the workgroups per CU, so four wavefronts per workgroup
// left one to three per SIMD, each with two or four lines' butterflies in
// its registers (768 points, 128-byte tiles: FP64 yfwd 5.90 -> 5.34 ms, FP32
// 3.89 -> 3.00 ms per launch).  The FP32 384-point pass measured slower with
// 16 wavefronts and keeps four.
template <int N, class C>
constexpr int ywaves() {
    return N <= 81 ? 2 : N == 768 || (N >= 216 && sizeof(C) == 16) ? ycols<N, C>() : 4;
}

// G[b][z][y][ix] = sum_jy Fz[b][z][ix*nky + jy] exp(+i ky y)
template <int N, class C>
__global__ __launch_bounds__((64 * ywaves<N, C>())) void k_ybwd_w(const C *__restrict__ Fz, C *__restrict__ G,
                                                               const C *__restrict__ tw, int nkx, int nky, int NY) {
    constexpr int YL = ycols<N, C>(), YT = 64 * ywaves<N, C>();
    constexpr int LS = N + 1, LPW = YL / ywaves<N, C>();
    extern __shared__ unsigned char buf_raw[];   // YL * LS elements (beyond 64 KiB for N = 768)
    C *buf = reinterpret_cast<C *>(buf_raw);
    const int ntile = (nkx + YL - 1) / YL;
    const int tile = blockIdx.x % ntile;
    const size_t bz = blockIdx.x / ntile;
    const int ix0 = tile * YL, nl = min(YL, nkx - ix0);
    const int nsys = nkx * nky;
    // dealiased slots are zero
    for (int e = threadIdx.x; e < YL * (N - nky); e += blockDim.x) {
        const int l = e / (N - nky), k = e - l * (N - nky);
        buf[l * LS + NY / 2 + k] = mkc<C>(0, 0);
    }
    // all of a thread's loads are issued before the first LDS store (a loop
    // of load, wait, store would make them one HBM round trip each)
    const C *src = Fz + bz * nsys + (size_t)ix0 * nky;
    {
        constexpr int PER = (YL * N + YT - 1) / YT;   // nky <= N
        const int cnt = nl * nky;
        C v[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            v[i] = e < cnt ? src[e] : mkc<C>(0, 0);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            if (e < YL * nky) {
                const int l = e / nky, jy = e - l * nky;
                buf[l * LS + ky_slot(jy, NY, N)] = v[i];
            }
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    YPlan<N>::template Run<+1, LPW, LS>::run(buf + w * LPW * LS, tw, lane);
    __syncthreads();
    C *dst = G + bz * N * nkx + ix0;
    {
        constexpr int PER = (N * YL + YT - 1) / YT;   // the last round partial when YT does not divide N*YL
        C v[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            const int y = e / YL, l = e - y * YL;
            v[i] = (N * YL % YT == 0 || e < N * YL)
                       ? buf[l * LS + swz<YPlan<N>::template Run<+1, LPW, LS>::OUT_SWZ>(y)]
                       : mkc<C>(0, 0);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            const int y = e / YL, l = e - y * YL;
            if ((N * YL % YT == 0 || e < N * YL) && l < nl) dst[(size_t)y * nkx + l] = v[i];
        }
    }
}

// Hy[b][z][ix*nky + jy] = sum_y H[b][z][y][ix] exp(-i ky y)
template <int N, class C>
__global__ __launch_bounds__((64 * ywaves<N, C>())) void k_yfwd_w(const C *__restrict__ H, C *__restrict__ Hy,
                                                               const C *__restrict__ tw, int nkx, int nky, int NY) {
    constexpr int YL = ycols<N, C>(), YT = 64 * ywaves<N, C>();
    constexpr int LS = N + 1, LPW = YL / ywaves<N, C>();
    extern __shared__ unsigned char buf_raw[];   // YL * LS elements (beyond 64 KiB for N = 768)
    C *buf = reinterpret_cast<C *>(buf_raw);
    const int ntile = (nkx + YL - 1) / YL;
    const int tile = blockIdx.x % ntile;
    const size_t bz = blockIdx.x / ntile;
    const int ix0 = tile * YL, nl = min(YL, nkx - ix0);
    const int nsys = nkx * nky;
    // all of a thread's loads are issued before the first LDS store
    const C *src = H + bz * N * nkx + ix0;
    {
        constexpr int PER = (N * YL + YT - 1) / YT;   // the last round partial when YT does not divide N*YL
        C v[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            const int y = e / YL, l = e - y * YL;
            v[i] = ((N * YL % YT == 0 || e < N * YL) && l < nl) ? src[(size_t)y * nkx + l] : mkc<C>(0, 0);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            const int y = e / YL, l = e - y * YL;
            if (N * YL % YT == 0 || e < N * YL) buf[l * LS + y] = v[i];
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    YPlan<N>::template Run<-1, LPW, LS>::run(buf + w * LPW * LS, tw, lane);
    __syncthreads();
    C *dst = Hy + bz * nsys + (size_t)ix0 * nky;
    {
        constexpr int PER = (YL * N + YT - 1) / YT;   // nky <= N
        const int cnt = nl * nky;
        C v[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            const int l = e / nky, jy = e - l * nky;
            v[i] = e < cnt ? buf[l * LS + swz<YPlan<N>::template Run<-1, LPW, LS>::OUT_SWZ>(ky_slot(jy, NY, N))]
                           : mkc<C>(0, 0);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = threadIdx.x + i * YT;
            if (e < cnt) dst[e] = v[i];
        }
    }
}

// LDS of a workgroup of the wavefront y pass at length N
template <class C>
static size_t ywave_lds(int N) { return size_t(ycol_bytes(N) / sizeof(C)) * (N + 1) * sizeof(C); }

template <int N, class C>
static void go(hipStream_t st, bool fwd, const C *tw, const C *in, C *out, int nbatch, int NZAA, int nkx, int nky,
               int NY) {
    constexpr int YL = ycols<N, C>();
    const int ntile = (nkx + YL - 1) / YL;
    const dim3 grid(ntile * nbatch * NZAA);
    const size_t shm = ywave_lds<C>(N);
    if (fwd) {
        if (shm > 65536) set_dynamic_lds((const void *)k_yfwd_w<N, C>, shm, "y pass (forward)");
        hipLaunchKernelGGL((k_yfwd_w<N, C>), grid, dim3(64 * ywaves<N, C>()), shm, st, in, out, tw, nkx, nky, NY);
    } else {
        if (shm > 65536) set_dynamic_lds((const void *)k_ybwd_w<N, C>, shm, "y pass (inverse)");
        hipLaunchKernelGGL((k_ybwd_w<N, C>), grid, dim3(64 * ywaves<N, C>()), shm, st, in, out, tw, nkx, nky, NY);
    }
    check_launch("y pass");
}

template <class C>
static bool ypass_wave(hipStream_t st, bool fwd, int N, const C *tw, const C *in, C *out, int nbatch, int NZAA,
                       int nkx, int nky, int NY) {
    if (!tw || nky > N || NY / 2 + (N - nky) > N) return false;
    // the tile of a workgroup must fit the device's LDS (98 KB at N = 768);
    // otherwise the workgroup-level LDS FFT takes the lines
    if (ywave_lds<C>(N) > lds_limit_current()) return false;
    switch (N) {
#define YCASE(n) \
    case n: go<n>(st, fwd, tw, in, out, nbatch, NZAA, nkx, nky, NY); return true;
        YCASE(96) YCASE(144) YCASE(192) YCASE(384) YCASE(768)
    default: break;
    }
    if constexpr (std::is_same<C, double2>::value) {   // the FP32 chain keeps to the lengths above
        switch (N) {
            YCASE(24) YCASE(27) YCASE(36) YCASE(48) YCASE(54) YCASE(72) YCASE(81) YCASE(108) YCASE(162)
            YCASE(216) YCASE(243) YCASE(288) YCASE(324) YCASE(432) YCASE(486) YCASE(576) YCASE(648) YCASE(729)
        default: break;
        }
    }
#undef YCASE
    return false;
}

bool launch_ypass_wave(hipStream_t st, bool fwd, const FFTPlan &py, const double2 *in, double2 *out, int nbatch,
                       int NZAA, int nkx, int nky, int NY) {
    return ypass_wave<double2>(st, fwd, py.N, py.tw, in, out, nbatch, NZAA, nkx, nky, NY);
}

void launch_ypass32(hipStream_t st, bool fwd, const FFTPlan &py, const float2 *in, float2 *out, int nbatch, int NZAA,
                    int nkx, int nky, int NY) {
    if (!ypass_wave<float2>(st, fwd, py.N, py.twf, in, out, nbatch, NZAA, nkx, nky, NY))
        throw std::runtime_error("the FP32 y pass needs a wavefront plan (N = 96, 144, 192, 384, 768) that fits LDS");
}

}  // namespace coral
