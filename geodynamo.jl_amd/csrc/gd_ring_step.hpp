// gd_ring_step.hpp -- the step modes' ring passes with compiled FFT plans:
// inverse FFTs of a block's fields, the pointwise products, forward FFTs of
// the products.  Included by one source per element type.
//
// One block takes the ring pair of one node and level (a northern ring and its
// southern mirror, one complex transform) with every field of the mode.  The
// inverse transforms' first stage loads the packed Hermitian spectra from
// global memory, the forward transforms' first stage reads the products (the
// tangential modes form them there, from the fields in LDS; the 15-field step
// forms all five of a point in a pass of its own, so that each field value is
// read once), and every butterfly is held in registers: a point crosses LDS
// twice a stage less than in ring_kernel.  Threads: one butterfly of the
// largest radix each where 512 allow it; groups of 2 and 4 nodes a block were
// slower (fewer resident waves).
//
// Measured at nr = 65 against ring_kernel's plan (us): 15 fields FP32 nlon 96 /
// 192 / 288: 12.2 / 31.9 / 79.5 -> 9.4 / 25.4 / 57.4; FP64 192 / 384: 55 / 336 ->
// 44 / 260; against the runtime plan, tangential FP32 216 / 324: 79 / 165 -> 19 /
// 42.  Some lengths keep ring_kernel's plan (gd_ring.hip: ring_short,
// ring_step_own).
#pragma once
#include "gd_fft.hpp"
#include "gd_sht.hpp"

namespace {
// threads for `total` butterflies: as few rounds as `most` threads allow, evenly
constexpr int ring_step_threads(int total, int most)
{
    const int rounds = (total + most - 1) / most;
    return ((total + rounds - 1) / rounds + 63) / 64 * 64;
}

template <typename T, int MODE, int N> struct RingStepShape {
    using M = StepMode<MODE>;
    static constexpr int LD = FftRow<T, N>::ld(1);
    static constexpr size_t lds = sizeof(C2<T>) * LD * M::NF;
    // launched for this length and mode: its rings fit LDS, no plan of ring_kernel
    // is preferred, and the 15 fields are not refused
    static constexpr bool ok = lds <= 160 * 1024 &&
        (MODE == RING_STEP ? ring_fits(M::NF, N) && !ring_step_own<T>(N) : !ring_short(N));
    static constexpr bool deal_only = 3 * ring_most_orders(M::NF) <= N; // no more orders than a dealiased grid's
    static constexpr FftStages f = fft_stages(N);
    static constexpr int nthr = ring_step_threads(M::NF * (N / f.r[f.n - 1]), 512);
};

// product P at longitude j from the fields' values (field F at x[F * FS + j]),
// north in .x and south in .y
template <typename T, int MODE, int FS, class AT>
__device__ __forceinline__ C2<T> ring_product(const AT &a, const C2<T> *x, int P, int i, int j)
{
    const T ro = (T)a.ro;
    auto f = [&](int F) { return x[F * FS + j]; };
    // velocity.jl:494 theta_{min(j,nlat)}, or the point's own colatitude
    auto trig = [&](const void *t) {
        const T *p = static_cast<const T *>(t);
        if (a.coriolis_index) return C2<T>{p[i], p[a.nlat - 1 - i]};
        const T v = p[j < a.nlat - 1 ? j : a.nlat - 1];
        return C2<T>{v, v};
    };
#define GD_BOTH(expr_x, expr_y) C2<T> { expr_x, expr_y }
    if constexpr (MODE == RING_STEP_TANG || MODE == RING_STEP_TANG_C) {
        // the products of RING_STEP with u_r = omega_r = B_r = j_r = 0: the
        // tangential parts of u x omega, j x B and u x B vanish and u_r dT/dr
        // drops out; the Coriolis term and the tangential advection stay
        // fields: 0 u_t 1 u_p 2 gT_t 3 gT_p (4 gC_t 5 gC_p)
        if (P == 0) {
            const C2<T> c = trig(a.costh), up = f(1);
            return GD_BOTH(-ro * (-c.x * up.x), -ro * (-c.y * up.y));
        }
        if (P == 1) {
            const C2<T> c = trig(a.costh), ut = f(0);
            return GD_BOTH(-ro * (c.x * ut.x), -ro * (c.y * ut.y));
        }
        const C2<T> ut = f(0), up = f(1), gt = f(2 * P - 2), gp = f(2 * P - 1);
        return GD_BOTH(-(ut.x * gt.x + up.x * gp.x), -(ut.y * gt.y + up.y * gp.y));
    } else if constexpr (MODE == RING_ADJ_TANG) {
        // transposed Jacobian of those products at (u, grad T):
        //   u_t* = -ro cth a_p* - g_t a_T*,  u_p* = ro cth a_t* - g_p a_T*,
        //   g_t* = -u_t a_T*,                g_p* = -u_p a_T*
        // fields: 0 u_t 1 u_p 2 a_t* 3 a_p* 4 g_t 5 g_p 6 a_T*
        const C2<T> bT = f(6);
        if (P < 2) {
            const C2<T> c = trig(a.costh), b = f(3 - P), g = f(4 + P);
            const T s = P ? ro : -ro;
            return GD_BOTH(s * c.x * b.x - g.x * bT.x, s * c.y * b.y - g.y * bT.y);
        }
        const C2<T> u = f(P - 2);
        return GD_BOTH(-u.x * bT.x, -u.y * bT.y);
    } else {
        // velocity.jl:512-527, 664-670; magnetic.jl:399-401; scalar_field_common.jl:401-407
        // fields: 0 u_t 1 u_p 2 w_t 3 w_p 4 B_t 5 B_p 6 j_t 7 j_p 8 gT_t 9 gT_p
        //         10 u_r 11 w_r 12 B_r 13 j_r 14 dT_r
        const C2<T> ur = f(10);
        if (P == 0) {
            const C2<T> c = trig(a.costh), up = f(1), wp = f(3), Bp = f(5), jp = f(7), wr = f(11), Br = f(12), jr = f(13);
#define GD_AT(h) -ro * (up.h * wr.h - ur.h * wp.h) + (-ro * (-c.h * up.h)) + ro * (jp.h * Br.h - jr.h * Bp.h)
            return GD_BOTH(GD_AT(x), GD_AT(y));
#undef GD_AT
        }
        if (P == 1) {
            const C2<T> c = trig(a.costh), s = trig(a.sinth), ut = f(0), wt = f(2), Bt = f(4), jt = f(6), wr = f(11),
                        Br = f(12), jr = f(13);
#define GD_AP(h) \
    -ro * (ur.h * wt.h - ut.h * wr.h) + (-ro * (c.h * ut.h + s.h * ur.h)) + ro * (jr.h * Bt.h - jt.h * Br.h)
            return GD_BOTH(GD_AP(x), GD_AP(y));
#undef GD_AP
        }
        if (P == 4) {
            const C2<T> gr = f(14), ut = f(0), up = f(1), gt = f(8), gp = f(9);
            return GD_BOTH(-(ur.x * gr.x + ut.x * gt.x + up.x * gp.x), -(ur.y * gr.y + ut.y * gt.y + up.y * gp.y));
        }
        const C2<T> Br = f(12);
        if (P == 2) {
            const C2<T> up = f(1), Bp = f(5);
            return GD_BOTH(up.x * Br.x - ur.x * Bp.x, up.y * Br.y - ur.y * Bp.y);
        }
        const C2<T> ut = f(0), Bt = f(4);
        return GD_BOTH(ur.x * Bt.x - ut.x * Br.x, ur.y * Bt.y - ut.y * Br.y);
    }
#undef GD_BOTH
}

// block L of the pass: node fastest, then level
template <typename T, int MODE, int N, bool DEAL, class AT>
__device__ __forceinline__ void ring_step_body(const AT &a, int L)
{
    using SH = RingStepShape<T, MODE, N>;
    using M = StepMode<MODE>;
    constexpr FftStages fi = fft_stages(N, 1), ff = fft_stages(N, -1);
    constexpr int LD = SH::LD, nthr = SH::nthr, S = fi.n - 1;
    extern __shared__ __align__(16) char smem_raw[];
    C2<T> *buf = reinterpret_cast<C2<T> *>(smem_raw); // field (or product) F at F LD
    const C2<T> *tws = static_cast<const C2<T> *>(a.tws);
    const int i = L % a.nlat2, lev = L / a.nlat2;
    const int nm = a.mmax + 1, tid = threadIdx.x;
    {
        // lanes take the fields of one order first (contiguous slots)
        constexpr int R0 = fi.r[0], nb0 = N / R0, total = M::NF * nb0, IT = (total + nthr - 1) / nthr;
        const T *rec = static_cast<const T *>(a.fb) + ((size_t)i * a.nr + lev) * nm * (4 * M::NF);
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int g = tid + it * nthr, F = g % M::NF, j = g / M::NF;
            if (total % nthr != 0 && g >= total) continue;
            C2<T> v[R0];
            fft_pack_stage<T, N, DEAL>(rec + 4 * F, 4u * M::NF, nm, j, v);
            fft_lds_put<T, N, 0, 1>(buf + F * LD, j, v);
        }
    }
    if constexpr (S == 2) fft_rows_stage<T, N, 1, 1, M::NF, nthr, LD, false>(buf, tws);
    fft_rows_stage<T, N, S, 1, M::NF, nthr, LD, false>(buf, tws);
    __syncthreads();
    if constexpr (MODE == RING_STEP) {
        for (int j = tid; j < N; j += nthr) {
            C2<T> o[M::NP];
#pragma unroll
            for (int P = 0; P < M::NP; ++P) o[P] = ring_product<T, MODE, LD>(a, buf, P, i, j);
#pragma unroll
            for (int P = 0; P < M::NP; ++P) buf[P * LD + j] = o[P];
        }
        __syncthreads();
    }
    {
        constexpr int R0 = ff.r[0], nb0 = N / R0, total = M::NP * nb0, IT = (total + nthr - 1) / nthr;
        C2<T> v[IT][R0];
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int g = tid + it * nthr, j = g % nb0, P = g / nb0;
            if (total % nthr != 0 && g >= total) continue;
#pragma unroll
            for (int r = 0; r < R0; ++r)
                v[it][r] = MODE == RING_STEP ? buf[P * LD + j + r * nb0]
                                             : ring_product<T, MODE, LD>(a, buf, P, i, j + r * nb0);
            dft<R0, -1>(v[it]);
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int g = tid + it * nthr;
            if (total % nthr != 0 && g >= total) continue;
            fft_lds_put<T, N, 0, -1>(buf + g / nb0 * LD, g % nb0, v[it]);
        }
    }
    if constexpr (S == 2) fft_rows_stage<T, N, 1, -1, M::NP, nthr, LD, false>(buf, tws);
    fft_rows_stage<T, N, S, -1, M::NP, nthr, LD, DEAL>(buf, tws);
    __syncthreads();
    const T c = static_cast<const T *>(a.wq)[i];
    T *gb = static_cast<T *>(a.gb);
    const unsigned ms = (unsigned)(a.nlat2 * a.nr);
    const size_t recs = (size_t)nm * ms, rec0 = (size_t)i * a.nr + lev;
    for (int e = tid; e < M::NP * nm; e += nthr) {
        const int P = e % M::NP, m = e / M::NP, str = gd_comp_str(P, M::NPV);
        T *rec = gb + gd_comp_off(P, M::NPV, recs) + rec0 * str;
        *reinterpret_cast<RingRec<T> *>(rec + (unsigned)m * (ms * str)) =
            fft_split<T>(buf[P * LD + m], buf[P * LD + (m ? N - m : 0)], m, c);
    }
}

template <typename T, int MODE, int N, bool DEAL>
__global__ void __launch_bounds__((RingStepShape<T, MODE, N>::nthr)) ring_step_plan_kernel(RingArgs a)
{
    ring_step_body<T, MODE, N, DEAL>(a, ring_step_block(blockIdx.x, gridDim.x, a.nlat2));
}

// one grid over the ring passes of several shells, dealiased ones or any (their
// own launches' instance, so that each shell gets its own bits)
template <typename T, int MODE, int N, bool DEAL>
__global__ void __launch_bounds__((RingStepShape<T, MODE, N>::nthr)) ring_step_batch_kernel(BatchRef<RingArgs> b)
{
    const int sh = b.shell_of_block[blockIdx.x];
    if (sh == BATCH_PAD) return;
    const auto &a = batch_args(b, sh);
    ring_step_body<T, MODE, N, DEAL>(a, ring_step_block(blockIdx.x - b.block_off[sh], b.block_cnt[sh], a.nlat2));
}

template <typename T, int MODE, int N> bool ring_step_launch(hipStream_t st, const RingArgs &a)
{
    using SH = RingStepShape<T, MODE, N>;
    if constexpr (!SH::ok) {
        return false;
    } else {
        const dim3 grid(a.nlat2 * a.nr), block(SH::nthr);
        if (gd_ring_deal(a)) hipLaunchKernelGGL((ring_step_plan_kernel<T, MODE, N, true>), grid, block, SH::lds, st, a);
        else if constexpr (!SH::deal_only) hipLaunchKernelGGL((ring_step_plan_kernel<T, MODE, N, false>), grid, block, SH::lds, st, a);
        else return false;
        return true;
    }
}

template <typename T, int MODE> bool ring_step_mode(hipStream_t st, const RingArgs &a)
{
    if (!gd_step_offsets_fit(a)) return false;
    switch (a.nlon) {
#define GD_RING_LEN(N) case N: return ring_step_launch<T, MODE, N>(st, a);
        GD_RING_LENGTHS
#undef GD_RING_LEN
    default: return false;
    }
}

template <typename T, int N> bool ring_step_batch_launch(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, bool deal)
{
    using SH = RingStepShape<T, RING_STEP_TANG, N>;
    if constexpr (!SH::ok) {
        return false;
    } else {
        const dim3 grid(nblocks), block(SH::nthr);
        if (deal) hipLaunchKernelGGL((ring_step_batch_kernel<T, RING_STEP_TANG, N, true>), grid, block, SH::lds, st, b);
        else hipLaunchKernelGGL((ring_step_batch_kernel<T, RING_STEP_TANG, N, false>), grid, block, SH::lds, st, b);
        return true;
    }
}

template <typename T> bool ring_step_batch(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, bool deal)
{
    switch (nlon) {
#define GD_RING_LEN(N) case N: return ring_step_batch_launch<T, N>(st, b, nblocks, deal);
        GD_RING_LENGTHS
#undef GD_RING_LEN
    default: return false;
    }
}
} // namespace
