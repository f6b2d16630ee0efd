// gd_ring_io.hpp -- the boundary ring passes with compiled FFT plans:
// RING_SYNTH (Fourier records -> colatitude-fastest grid values) and
// RING_ANALYSIS (grid values -> weighted Fourier records).  Included by one
// source per element type.
//
// One block takes RG consecutive ring pairs (a northern ring and its southern
// mirror, one complex transform each) of one level and NF fields.  The first
// stage's butterflies load their inputs from global memory and the last
// stage's store their results to it, so a point passes LDS only between
// stages (one exchange for n <= 324, two beyond).  The grid arrays are
// colatitude-fastest: on their side lanes take the rings of one longitude
// first, on the record side consecutive orders.  RG = 4 (32-byte runs of
// colatitudes) where two blocks fit a CU's LDS, else 2.
//
// Against one block FFT of radices 8/6/4/3/2 with every stage, the input and
// the output passing LDS (and runtime index divisions where a length had no
// plan): FP64 scalar, 384 x 768, 97 levels, 381 MB: synthesis 154 -> 104 us
// (3.7 TB/s), analysis 207 -> 170 us; FP64 vector, 162 x 324, 41 levels:
// 103 -> 20 and 93 -> 17 us; FP64 scalar, 48 x 96, 33 levels: 17 -> 4.0 and
// 14 -> 4.5 us.  The analysis is bound by its record stores (16- and 32-byte
// pieces of different lines).
#pragma once
#include "gd_fft.hpp"
#include "gd_sht.hpp"

namespace {
template <typename T, int N, int NF> struct RingIoShape {
    using F = FftLds<T, N>;
    static constexpr size_t row = sizeof(C2<T>) * F::LD;
    static constexpr int RG = row * NF * 4 <= 80 * 1024 ? 4 : 2;
    static constexpr int NT = RG * NF; // transforms of a block
    static constexpr int RMAX = F::f.r[F::f.n - 1];
    static constexpr int want = (NT * (N / RMAX) + 63) / 64 * 64;
    static constexpr int nthr = want > 256 ? 256 : want;
    static constexpr size_t lds = row * NT;
};

// every butterfly of stage s of the block's transforms, in place in LDS
template <typename T, int N, int NF, int S, int DIR>
__device__ __forceinline__ void ring_io_mid(C2<T> *buf, const C2<T> *tws)
{
    using SH = RingIoShape<T, N, NF>;
    constexpr int R = SH::F::f.r[S], nb = N / R, total = SH::NT * nb, IT = (total + SH::nthr - 1) / SH::nthr;
    C2<T> v[IT][R];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = threadIdx.x + it * SH::nthr;
        if (total % SH::nthr == 0 || g < total) fft_lds_stage<T, N, S, DIR>(buf + g / nb * SH::F::LD, tws, g % nb, v[it]);
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = threadIdx.x + it * SH::nthr;
        if (total % SH::nthr == 0 || g < total) {
            C2<T> *x = buf + g / nb * SH::F::LD;
            if constexpr (S == SH::F::f.n - 1) { // results in natural order
#pragma unroll
                for (int r = 0; r < R; ++r) x[g % nb + r * nb] = v[it][r];
            } else {
                fft_lds_put<T, N, S>(x, g % nb, v[it]);
            }
        }
    }
    __syncthreads();
}

template <typename T, int MODE, int N, int NF>
__global__ void __launch_bounds__((RingIoShape<T, N, NF>::nthr)) ring_plan_kernel(RingArgs a)
{
    using SH = RingIoShape<T, N, NF>;
    using F = typename SH::F;
    constexpr int RG = SH::RG, LD = F::LD, nthr = SH::nthr, R0 = F::f.r[0], nb0 = N / R0;
    constexpr int S = F::f.n - 1, RL = F::f.r[S], nbL = N / RL; // the last stage
    extern __shared__ __align__(16) char smem_raw[];
    C2<T> *buf = reinterpret_cast<C2<T> *>(smem_raw); // transform t = q NF + F at t LD
    const C2<T> *tws = static_cast<const C2<T> *>(a.tws);
    const int L = xcd_logical(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int i0 = L % gridDim.x * RG, lev = L / gridDim.x;
    const int nm = a.mmax + 1, nq = min(RG, a.nlat2 - i0), tid = threadIdx.x;
    constexpr int total0 = SH::NT * nb0, IT0 = (total0 + nthr - 1) / nthr;
    if constexpr (MODE == RING_SYNTH) {
        // Hermitian spectra of the north (X) and south (Y) rings packed as Z = X + iY
#pragma unroll
        for (int it = 0; it < IT0; ++it) {
            const int g = tid + it * nthr, t = g / nb0, j = g % nb0;
            if (total0 % nthr != 0 && g >= total0) continue;
            const int q = min(t / NF, nq - 1), f = t % NF;
            const T *rec = static_cast<const T *>(a.fb) + ((size_t)(i0 + q) * a.nr + lev) * nm * a.nslot_f;
            const int on = f ? a.fn_off[1] : a.fn_off[0], os = f ? a.fs_off[1] : a.fs_off[0];
            C2<T> X[R0], Y[R0], v[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) { // unused orders read record 0
                const int k = j + r * nb0, m = k < nm ? k : (N - k < nm ? N - k : 0);
                X[r] = *reinterpret_cast<const C2<T> *>(rec + (size_t)m * a.nslot_f + on);
                Y[r] = *reinterpret_cast<const C2<T> *>(rec + (size_t)m * a.nslot_f + os);
            }
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const int k = j + r * nb0;
                const T xi = k ? X[r].y : T(0), yi = k ? Y[r].y : T(0);
                const T s = k < nm ? T(1) : T(-1);
                const bool on_ = k < nm || N - k < nm;
                v[r].x = on_ ? X[r].x - s * yi : T(0);
                v[r].y = on_ ? s * xi + Y[r].x : T(0);
            }
            dft<R0, 1>(v);
            fft_lds_put<T, N, 0>(buf + t * LD, j, v);
        }
        __syncthreads();
        if constexpr (S == 2) ring_io_mid<T, N, NF, 1, 1>(buf, tws);
        constexpr int total = SH::NT * nbL, IT = (total + nthr - 1) / nthr;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int g = tid + it * nthr;
            if (total % nthr != 0 && g >= total) continue;
            const int q = g % RG, j = g / RG % nbL, f = g / (RG * nbL);
            C2<T> v[RL];
            fft_lds_stage<T, N, S, 1>(buf + (q * NF + f) * LD, tws, j, v);
            if (q < nq) {
                double *o = (f ? a.phys_out[1] : a.phys_out[0]) + ((size_t)lev * N + j) * a.nlat;
                const int i = i0 + q, is = a.nlat - 1 - i;
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    o[(size_t)(r * nbL) * a.nlat + i] = (double)v[r].x;
                    o[(size_t)(r * nbL) * a.nlat + is] = (double)v[r].y;
                }
            }
        }
    } else {
#pragma unroll
        for (int it = 0; it < IT0; ++it) {
            const int g = tid + it * nthr;
            if (total0 % nthr != 0 && g >= total0) continue;
            const int q = g % RG, j = g / RG % nb0, f = g / (RG * nb0);
            const double *p = (f ? a.phys_in[1] : a.phys_in[0]) + ((size_t)lev * N + j) * a.nlat;
            const int i = i0 + min(q, nq - 1), is = a.nlat - 1 - i;
            double x[R0], y[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                x[r] = p[(size_t)(r * nb0) * a.nlat + i];
                y[r] = p[(size_t)(r * nb0) * a.nlat + is];
            }
            C2<T> v[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) v[r] = C2<T>{(T)x[r], (T)y[r]};
            dft<R0, -1>(v);
            fft_lds_put<T, N, 0>(buf + (q * NF + f) * LD, j, v);
        }
        __syncthreads();
        if constexpr (S == 2) ring_io_mid<T, N, NF, 1, -1>(buf, tws);
        ring_io_mid<T, N, NF, S, -1>(buf, tws);
        // split Z into north X and south Y, form G+- = (X +- Y) * 2 pi w_i / n
        struct alignas(16) Rec {
            T v[4];
        };
        for (int e = tid; e < SH::NT * nm; e += nthr) {
            const int f = e % NF, q = e / NF % RG, m = e / SH::NT;
            if (q >= nq) continue;
            const T c = static_cast<const T *>(a.wq)[i0 + q];
            const C2<T> *b = buf + (q * NF + f) * LD;
            const C2<T> Z = b[m], Zc = b[m ? N - m : 0];
            C2<T> X = C2<T>{T(0.5) * (Z.x + Zc.x), T(0.5) * (Z.y - Zc.y)};
            C2<T> Y = C2<T>{T(0.5) * (Z.y + Zc.y), T(0.5) * (Zc.x - Z.x)};
            const size_t rec = ((size_t)m * a.nlat2 + i0 + q) * a.nr + lev;
            *reinterpret_cast<Rec *>(static_cast<T *>(a.gb) + rec * a.nslot_g + 4 * f) =
                Rec{{(X.x + Y.x) * c, (X.y + Y.y) * c, (X.x - Y.x) * c, (X.y - Y.y) * c}};
        }
    }
}

template <typename T, int MODE, int N> bool ring_plan_launch(hipStream_t st, const RingArgs &a, int nf)
{
    if (nf == 1) {
        using SH = RingIoShape<T, N, 1>;
        hipLaunchKernelGGL((ring_plan_kernel<T, MODE, N, 1>), dim3((a.nlat2 + SH::RG - 1) / SH::RG, a.nr), dim3(SH::nthr),
                           SH::lds, st, a);
    } else {
        using SH = RingIoShape<T, N, 2>;
        hipLaunchKernelGGL((ring_plan_kernel<T, MODE, N, 2>), dim3((a.nlat2 + SH::RG - 1) / SH::RG, a.nr), dim3(SH::nthr),
                           SH::lds, st, a);
    }
    return true;
}

template <typename T, int MODE> bool ring_plan_mode(hipStream_t st, const RingArgs &a, int nf)
{
    switch (a.nlon) {
#define GD_RING_LEN(N) case N: return ring_plan_launch<T, MODE, N>(st, a, nf);
        GD_RING_LENGTHS
#undef GD_RING_LEN
    default: return false;
    }
}
} // namespace
