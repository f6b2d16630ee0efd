// gd_ring_io.hpp -- the boundary ring passes with compiled FFT plans:
// RING_SYNTH (Fourier records -> colatitude-fastest grid values) and
// RING_ANALYSIS (grid values -> weighted Fourier records).  Included by one
// source per element type.
//
// One block takes RG consecutive ring pairs (a northern ring and its southern
// mirror, one complex transform each) of one level and NF fields.  The first
// stage's butterflies load their inputs from global memory, and the synthesis'
// last ones store the grid values to it, so a point crosses LDS only between
// stages: once in plans of two stages (n <= 324, except 243), twice in plans of
// three.  The analysis crosses once more: order m's slots need the results at m
// and n - m.  The grid arrays are
// colatitude-fastest: on their side lanes take the rings of one longitude
// first, on the record side consecutive orders.  RG = 4 (32-byte runs of
// colatitudes) where two blocks fit a CU's LDS, else 2.
//
// Against one block FFT of radices 8/6/4/3/2 with every stage, the input and
// the output passing LDS (and runtime index divisions where a length had no
// plan): FP64 scalar, 384 x 768, 97 levels, 381 MB: synthesis 154 -> 104 us
// (3.7 TB/s), analysis 207 -> 137 us (170 with node-major records); FP64 vector, 162 x 324, 41 levels:
// 103 -> 20 and 93 -> 17 us; FP64 scalar, 48 x 96, 33 levels: 17 -> 4.0 and
// 14 -> 4.5 us.  The analysis is bound by its record stores (32- to 128-byte
// pieces of different lines).
#pragma once
#include "gd_fft.hpp"
#include "gd_sht.hpp"

namespace {
template <typename T, int N, int NF> struct RingIoShape {
    using F = FftRow<T, N>;
    static constexpr int LD = F::ld(F::M / 4);
    static constexpr size_t row = sizeof(C2<T>) * LD;
    static constexpr int RG = row * NF * 4 <= 80 * 1024 ? 4 : 2;
    static constexpr int NT = RG * NF; // transforms of a block
    static constexpr FftStages f = fft_stages(N);
    static constexpr int want = (NT * (N / f.r[f.n - 1]) + 63) / 64 * 64; // the largest radix
    static constexpr int nthr = want > 256 ? 256 : want;
    static constexpr size_t lds = row * NT;
};

template <typename T, int MODE, int N, int NF, bool DEAL>
__global__ void __launch_bounds__((RingIoShape<T, N, NF>::nthr)) ring_plan_kernel(RingArgs a)
{
    using SH = RingIoShape<T, N, NF>;
    constexpr int DIR = MODE == RING_SYNTH ? 1 : -1;
    constexpr FftStages f = fft_stages(N, DIR);
    constexpr int RG = SH::RG, LD = SH::LD, nthr = SH::nthr, R0 = f.r[0], nb0 = N / R0;
    constexpr int S = f.n - 1, RL = f.r[S], nbL = N / RL; // the last stage
    extern __shared__ __align__(16) char smem_raw[];
    C2<T> *buf = reinterpret_cast<C2<T> *>(smem_raw); // transform t = q NF + F at t LD
    const C2<T> *tws = static_cast<const C2<T> *>(a.tws);
    const int L = xcd_logical(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int i0 = L % gridDim.x * RG, lev = L / gridDim.x;
    const int nm = a.mmax + 1, nq = min(RG, a.nlat2 - i0), tid = threadIdx.x;
    constexpr int total0 = SH::NT * nb0, IT0 = (total0 + nthr - 1) / nthr;
    if constexpr (MODE == RING_SYNTH) {
#pragma unroll
        for (int it = 0; it < IT0; ++it) {
            // fields, then rings, fastest: their slots of one order are contiguous
            const int g = tid + it * nthr, F = g % NF, q = g / NF % RG, j = g / SH::NT;
            if (total0 % nthr != 0 && g >= total0) continue;
            const T *rec = static_cast<const T *>(a.fb) + (F ? a.foff[1] : a.foff[0]) +
                           (lev * a.dim.l + (i0 + min(q, nq - 1)) * a.dim.i) * (4 * NF);
            C2<T> v[R0];
            fft_pack_stage<T, N, DEAL>(rec, (unsigned)(a.dim.m * (4 * NF)), nm, j, v);
            fft_lds_put<T, N, 0, 1>(buf + (q * NF + F) * LD, j, v);
        }
        if constexpr (S == 2) fft_rows_stage<T, N, 1, 1, SH::NT, nthr, LD, false>(buf, tws);
        constexpr int total = SH::NT * nbL, IT = (total + nthr - 1) / nthr;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int g = tid + it * nthr;
            const int q = g % RG, j = g / RG % nbL, F = g / (RG * nbL);
            C2<T> v[RL], w[RL];
            fft_tw_load<T, N, S, 1>(tws, j, w);
            if (it == 0) __syncthreads();
            if (total % nthr != 0 && g >= total) continue;
            fft_lds_stage<T, N, S, 1>(buf + (q * NF + F) * LD, w, j, v);
            if (q < nq) {
                double *o = (F ? a.phys_out[1] : a.phys_out[0]) + ((size_t)lev * N + j) * a.nlat;
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
            const int q = g % RG, j = g / RG % nb0, F = g / (RG * nb0);
            const double *p = (F ? a.phys_in[1] : a.phys_in[0]) + ((size_t)lev * N + j) * a.nlat;
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
            fft_lds_put<T, N, 0, -1>(buf + (q * NF + F) * LD, j, v);
        }
        if constexpr (S == 2) fft_rows_stage<T, N, 1, -1, SH::NT, nthr, LD, false>(buf, tws);
        fft_rows_stage<T, N, S, -1, SH::NT, nthr, LD, DEAL>(buf, tws);
        __syncthreads();
        for (int e = tid; e < SH::NT * nm; e += nthr) {
            const int F = e % NF, q = e / NF % RG, m = e / SH::NT;
            if (q >= nq) continue;
            T *rec = static_cast<T *>(a.gb) + 4 * F + (lev * a.dim.l + (i0 + q) * a.dim.i) * (4 * NF);
            const C2<T> *x = buf + (q * NF + F) * LD;
            *reinterpret_cast<RingRec<T> *>(rec + (unsigned)m * (unsigned)(a.dim.m * (4 * NF))) =
                fft_split<T>(x[m], x[m ? N - m : 0], m, static_cast<const T *>(a.wq)[i0 + q]);
        }
    }
}

template <typename T, int MODE, int N, int NF> void ring_plan_launch(hipStream_t st, const RingArgs &a)
{
    using SH = RingIoShape<T, N, NF>;
    const dim3 grid((a.nlat2 + SH::RG - 1) / SH::RG, a.nr), block(SH::nthr);
    if (gd_ring_deal(a)) hipLaunchKernelGGL((ring_plan_kernel<T, MODE, N, NF, true>), grid, block, SH::lds, st, a);
    else hipLaunchKernelGGL((ring_plan_kernel<T, MODE, N, NF, false>), grid, block, SH::lds, st, a);
}

template <typename T, int MODE> bool ring_plan_mode(hipStream_t st, const RingArgs &a, int nf)
{
    if (!gd_offsets_fit(a)) return false;
    switch (a.nlon) {
#define GD_RING_LEN(N)                                         \
    case N:                                                    \
        if (nf == 1) ring_plan_launch<T, MODE, N, 1>(st, a);   \
        else ring_plan_launch<T, MODE, N, 2>(st, a);           \
        return true;
        GD_RING_LENGTHS
#undef GD_RING_LEN
    default: return false;
    }
}
} // namespace
