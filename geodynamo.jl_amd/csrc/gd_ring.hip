// gd_ring.hip -- longitude FFTs of a northern ring and its southern mirror as
// one complex FFT; the step modes also evaluate the pointwise nonlinear
// products between the inverse and forward FFTs, so physical-space values
// never leave LDS.  The ring lengths with a compiled plan are in
// gd_ring_io.hpp (boundary passes) and gd_ring_step.hpp (step modes); here are
// the dispatch and the runtime plan (Stockham, radices 2,3,4,6,8, in LDS) of
// any other 2^a 3^b, and compiled plans of that form for the tangential modes'
// most used lengths.
#include <cmath>
#include <cstdint>

#include "gd_fft.hpp"
#include "gd_sht.hpp"

namespace {
template <typename T> __device__ __forceinline__ void dft2(C2<T> &a, C2<T> &b)
{
    C2<T> t = a;
    a = cadd(t, b);
    b = csub(t, b);
}
template <typename T> __device__ __forceinline__ void dft3(C2<T> &v0, C2<T> &v1, C2<T> &v2, int dir)
{
    const T s3 = T(0.86602540378443864676);
    C2<T> t1 = cadd(v1, v2);
    C2<T> t2 = {v0.x - T(0.5) * t1.x, v0.y - T(0.5) * t1.y};
    C2<T> d = csub(v1, v2);
    C2<T> t3 = cmuli(C2<T>{s3 * d.x, s3 * d.y}, dir);
    v0 = cadd(v0, t1);
    v1 = cadd(t2, t3);
    v2 = csub(t2, t3);
}
template <typename T> __device__ __forceinline__ void dft4(C2<T> &v0, C2<T> &v1, C2<T> &v2, C2<T> &v3, int dir)
{
    C2<T> a = cadd(v0, v2), b = csub(v0, v2), c = cadd(v1, v3), d = cmuli(csub(v1, v3), dir);
    v0 = cadd(a, c);
    v2 = csub(a, c);
    v1 = cadd(b, d);
    v3 = csub(b, d);
}

template <int R, typename T> __device__ __forceinline__ void dftR(C2<T> *v, int dir)
{
    if constexpr (R == 2) {
        dft2(v[0], v[1]);
    } else if constexpr (R == 3) {
        dft3(v[0], v[1], v[2], dir);
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3], dir);
    } else if constexpr (R == 6) {
        // 6 = 2 x 3: E = DFT3(v0,v2,v4), O = DFT3(v1,v3,v5), X_k = E_k + w6^k O_k
        C2<T> e0 = v[0], e1 = v[2], e2 = v[4], o0 = v[1], o1 = v[3], o2 = v[5];
        dft3(e0, e1, e2, dir);
        dft3(o0, o1, o2, dir);
        const T h = T(0.5), s3 = T(0.86602540378443864676);
        C2<T> w1 = {h, dir > 0 ? s3 : -s3}, w2 = {-h, dir > 0 ? s3 : -s3};
        o1 = cmul(o1, w1);
        o2 = cmul(o2, w2);
        v[0] = cadd(e0, o0);
        v[3] = csub(e0, o0);
        v[1] = cadd(e1, o1);
        v[4] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[5] = csub(e2, o2);
    } else if constexpr (R == 8) {
        C2<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
        dft4(e0, e1, e2, e3, dir);
        dft4(o0, o1, o2, o3, dir);
        const T r2 = T(0.70710678118654752440);
        const T sg = dir > 0 ? T(1) : T(-1);
        o1 = cmul(o1, C2<T>{r2, sg * r2});
        o2 = cmuli(o2, dir);
        o3 = cmul(o3, C2<T>{-r2, sg * r2});
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, o1);
        v[5] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[6] = csub(e2, o2);
        v[3] = cadd(e3, o3);
        v[7] = csub(e3, o3);
    }
}

// LDS index skew: one pad slot per 16 complex values, so the stride-R writes
// of the early Stockham stages (and stride-Ns groups later) spread over banks.
__device__ __forceinline__ int sk(int e) { return e + (e >> 4); }

// One Stockham stage over nfft transforms of length n (stride ld in buf); in
// place, with every butterfly read before any is written.  Runtime radix plan.
template <int R, typename T>
__device__ __noinline__ void fft_stage(C2<T> *buf, const C2<T> *tw, int nfft, int n, int ld, int Ns, int dir)
{
    constexpr int IT = MAXC / R;
    const int nb = n / R, total = nfft * nb;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int twstep = n / (Ns * R);
    C2<T> v[IT][R];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = tid + it * nthr;
        if (g < total) {
            const int f = g / nb, j = g - f * nb;
            const int k = j % Ns;
#pragma unroll
            for (int r = 0; r < R; ++r) v[it][r] = buf[f * ld + sk(j + r * nb)];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                C2<T> w = tw[k * r * twstep];
                if (dir > 0) w.y = -w.y;
                v[it][r] = cmul(v[it][r], w);
            }
            dftR<R, T>(v[it], dir);
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = tid + it * nthr;
        if (g < total) {
            const int f = g / nb, j = g - f * nb;
            const int k = j % Ns;
            const int idxD = (j / Ns) * Ns * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[f * ld + sk(idxD + r * Ns)] = v[it][r];
        }
    }
    __syncthreads();
}

template <typename T>
__device__ void fft_batch(C2<T> *buf, const C2<T> *tw, int nfft, int n, int ld, const int *radix, int nstages, int dir)
{
    int Ns = 1;
    for (int s = 0; s < nstages; ++s) {
        const int R = radix[s];
        switch (R) {
        case 8: fft_stage<8, T>(buf, tw, nfft, n, ld, Ns, dir); break;
        case 6: fft_stage<6, T>(buf, tw, nfft, n, ld, Ns, dir); break;
        case 4: fft_stage<4, T>(buf, tw, nfft, n, ld, Ns, dir); break;
        case 3: fft_stage<3, T>(buf, tw, nfft, n, ld, Ns, dir); break;
        default: fft_stage<2, T>(buf, tw, nfft, n, ld, Ns, dir); break;
        }
        Ns *= R;
    }
}

// The Stockham write of a butterfly goes to idxD + r NS with idxD = q NS R + k,
// k < NS.  sk(idxD + r NS) - sk(idxD) = r NS + [(idxD + r NS) / 16 - idxD / 16]
// is a constant of r when the bracket is the same for every residue idxD mod
// 16 the butterflies can have: then the R addresses are one base and
// constant offsets.
constexpr bool sk_write_const(int NS, int R)
{
    for (int r = 0; r < R; ++r) {
        int val = -1;
        for (int q = 0; q < 16; ++q)
            for (int k = 0; k < NS && k < 16; ++k) {
                const int res = (q * NS * R + k) % 16;
                const int d = (res + r * NS) / 16;
                if (val < 0) val = d;
                else if (d != val) return false;
            }
    }
    return true;
}
// the offset of write r: the bracket at residue 0 (q = k = 0), which every
// residue shares when sk_write_const holds
constexpr int sk_write_off(int NS, int r) { return r * NS + (r * NS) / 16; }

// NFFT > 0: the transform count is a compile-time constant (nfft is ignored)
template <int R, int NS, int N, int DIR, typename T, int NFFT>
__device__ __forceinline__ void fft_stage_ct(C2<T> *buf, const C2<T> *tw, int nfft)
{
    constexpr int nb = N / R, twstep = N / (NS * R), LD = ring_ld(N);
    constexpr int nthr = RING_THREADS;
    constexpr int IT = NFFT > 0 ? (NFFT * nb + nthr - 1) / nthr : MAXC / R;
    const int total = (NFFT > 0 ? NFFT : nfft) * nb;
    const int tid = threadIdx.x;
    // sk(e + r * s) = sk(e) + r * (s + s / 16) when s is a multiple of 16: the
    // R addresses of a butterfly are then one base and constant offsets
    constexpr bool RD16 = nb % 16 == 0, WR16 = sk_write_const(NS, R);
    C2<T> v[IT][R];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = tid + it * nthr;
        if (g < total) {
            const int f = g / nb, j = g - f * nb;
            const int k = j % NS;
            const int rb = f * LD + sk(j);
#pragma unroll
            for (int r = 0; r < R; ++r) v[it][r] = buf[RD16 ? rb + r * (nb + nb / 16) : f * LD + sk(j + r * nb)];
            if (NS > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    C2<T> w = tw[k * r * twstep];
                    if (DIR > 0) w.y = -w.y;
                    v[it][r] = cmul(v[it][r], w);
                }
            }
            dftR<R, T>(v[it], DIR);
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = tid + it * nthr;
        if (g < total) {
            const int f = g / nb, j = g - f * nb;
            const int k = j % NS;
            const int idxD = (j / NS) * NS * R + k;
            const int wb = f * LD + sk(idxD);
#pragma unroll
            for (int r = 0; r < R; ++r) buf[WR16 ? wb + sk_write_off(NS, r) : f * LD + sk(idxD + r * NS)] = v[it][r];
        }
    }
    __syncthreads();
}

template <typename T, int N, int DIR, int NFFT = 0, int S = 0, int NS = 1>
__device__ __forceinline__ void fft_ct(C2<T> *buf, const C2<T> *tw, int nfft)
{
    if constexpr (S < ct_nstages(N)) {
        constexpr int R = ct_radix(N, S);
        fft_stage_ct<R, NS, N, DIR, T, NFFT>(buf, tw, nfft);
        fft_ct<T, N, DIR, NFFT, S + 1, NS * R>(buf, tw, nfft);
    }
}

// A record of the step's FB, which this pass reads once and nothing reads again:
// a non-temporal load, so that FB does not push the products out of the
// last-level cache before the analyses read them.  96 nodes, 65 levels, rings of
// 384, whole step (us): FP64 tangential 259 -> 245, with composition 390 -> 350;
// FP32 with composition 235 -> 226, 15 fields 456 -> 434 (its vector analysis 62
// -> 44).  The register plans, whose lanes read pieces of several
// orders, lose 5 % of a step that way and keep the ordinary load.
template <typename T> __device__ __forceinline__ RingRec<T> fb_load(const T *p)
{
    typedef T V4 __attribute__((ext_vector_type(4)));
    const V4 q = __builtin_nontemporal_load(reinterpret_cast<const V4 *>(p));
    return RingRec<T>{{q[0], q[1], q[2], q[3]}};
}

// One block per (northern node i, level r) (the launch's own grid, or its share
// of a batched launch).  NC > 0: the ring length is the compile-time constant
// NC (nlon); NC = 0 uses the runtime plan.
template <typename T, int MODE, int NC, class AT> __device__ __forceinline__ void ring_body(const AT &a, int i, int r)
{
    extern __shared__ __align__(16) char smem_raw[];
    const int n = NC > 0 ? NC : a.nlon, nm = a.mmax + 1;
    const int ld = ring_ld(n);
    C2<T> *tw = reinterpret_cast<C2<T> *>(smem_raw);
    C2<T> *buf = tw + n;
    __shared__ int srad[12];
    const int tid = threadIdx.x;
    constexpr int nthr = RING_THREADS;
    const int is = a.nlat - 1 - i; // southern mirror
    const C2<T> *twg = static_cast<const C2<T> *>(a.tw);
    for (int k = tid; k < n; k += nthr) tw[k] = twg[k];
    if (tid < 12) srad[tid] = a.radix[tid];
    __syncthreads();
    // fields in / products out: compile-time for the step modes (0: a boundary pass)
    constexpr int NFC = StepMode<MODE>::NF, NPC = StepMode<MODE>::NP, NPV = StepMode<MODE>::NPV;
    const int NF = NFC ? NFC : a.nfield;

    if (MODE != RING_ANALYSIS) {
        // Hermitian spectra of the north (X) and south (Y) rings packed as Z = X + iY
        // fixed trip count, fully unrolled: every thread's loads are in flight
        // together before the LDS stores consume them.  With a compile-time ring
        // length the first MAXU iterations (enough for the nm <= n/3 orders of
        // the dealiased grids) load unconditionally, clamped to the last element:
        // a guarded load becomes a branch whose join waits for it.  Larger nm
        // take the guarded iterations after.
        constexpr int MAXI = 8;
        constexpr int MAXU0 = (NC > 0 && NFC > 0) ? (NFC * (NC / 3) + nthr - 1) / nthr : 0;
        constexpr int MAXU = MAXU0 < MAXI ? MAXU0 : MAXI;
        const int ne = NF * nm;
        // a step mode's slots of one ring are contiguous, orders outermost
        const size_t rec0 = NFC ? ((size_t)i * a.nr + r) * nm : r * a.dim.l + i * a.dim.i;
        const T *src = static_cast<const T *>(a.fb) + rec0 * (4 * NF);
        RingRec<T> z[MAXI];
#pragma unroll
        for (int it = 0; it < MAXI; ++it) {
            const int e0 = tid + it * nthr;
            if (it < MAXU || e0 < ne) {
                const int e = e0 < ne ? e0 : ne - 1;
                const int F = e % NF, m = e / NF;
                if constexpr (NFC > 0) z[it] = fb_load(src + 4 * e);
                else z[it] = *reinterpret_cast<const RingRec<T> *>(src + m * a.dim.m * (4 * NF) + 4 * F);
            }
        }
#pragma unroll
        for (int it = 0; it < MAXI; ++it) {
            const int e = tid + it * nthr;
            if (e < NF * nm) {
                const int F = e % NF, m = e / NF;
                const T *v = z[it].v;
                if (m == 0) {
                    buf[F * ld] = C2<T>{v[0], v[2]};
                } else {
                    buf[F * ld + sk(m)] = C2<T>{v[0] - v[3], v[1] + v[2]};
                    buf[F * ld + sk(n - m)] = C2<T>{v[0] + v[3], v[2] - v[1]};
                }
            }
        }
        // zero the modes nm .. n-nm of every field
        for (int k = nm + tid; k <= n - nm; k += nthr)
            for (int F = 0; F < NF; ++F) buf[F * ld + sk(k)] = C2<T>{T(0), T(0)};
        __syncthreads();
        if constexpr (NC > 0) fft_ct<T, NC, +1, NFC>(buf, tw, NF);
        else fft_batch<T>(buf, tw, NF, n, ld, srad, a.nstages, +1);
    }

    if (MODE == RING_SYNTH) {
        for (int j = tid; j < n; j += nthr)
            for (int F = 0; F < NF; ++F) {
                double *o = F == 0 ? a.phys_out[0] : a.phys_out[1];
                const C2<T> z = buf[F * ld + sk(j)];
                o[((size_t)r * n + j) * a.nlat + i] = (double)z.x;
                o[((size_t)r * n + j) * a.nlat + is] = (double)z.y;
            }
        return;
    }

    int NP;
    if constexpr (MODE == RING_STEP_TANG || MODE == RING_STEP_TANG_C) {
        // the products of RING_STEP with u_r = omega_r = B_r = j_r = 0: the
        // tangential parts of u x omega, j x B and u x B vanish and u_r dT/dr
        // drops out; the Coriolis term and the tangential advection of T stay,
        // evaluated in the same order as there
        // fields: 0 u_t 1 u_p 2 gT_t 3 gT_p (4 gC_t 5 gC_p: -u.grad C as product 3)
        NP = NPC;
        const T ro = (T)a.ro;
        const T *costh = static_cast<const T *>(a.costh);
        for (int j = tid; j < n; j += nthr) {
            C2<T> f[NFC];
#pragma unroll
            for (int F = 0; F < NFC; ++F) f[F] = buf[F * ld + sk(j)];
            C2<T> o[NPC];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int ti = a.coriolis_index ? (h ? is : i) : (j < a.nlat - 1 ? j : a.nlat - 1);
                const T cth = costh[ti];
#define FV(F) (h ? f[F].y : f[F].x)
                const T ut = FV(0), up = FV(1), gt = FV(2), gp = FV(3);
#undef FV
                const T at = -ro * (-cth * up);
                const T ap = -ro * (cth * ut);
                const T aT = -(ut * gt + up * gp);
                if (h) {
                    o[0].y = at;
                    o[1].y = ap;
                    o[2].y = aT;
                } else {
                    o[0].x = at;
                    o[1].x = ap;
                    o[2].x = aT;
                }
                if constexpr (NFC == 6) {
                    const T ct = h ? f[4].y : f[4].x, cp = h ? f[5].y : f[5].x;
                    const T aC = -(ut * ct + up * cp);
                    if (h) o[3].y = aC;
                    else o[3].x = aC;
                }
            }
#pragma unroll
            for (int P = 0; P < NPC; ++P) buf[P * ld + sk(j)] = o[P];
        }
        __syncthreads();
    } else if constexpr (MODE == RING_ADJ_TANG) {
        // transposed Jacobian of the products above at (u, grad T): with
        // a_t = ro cth u_p, a_p = -ro cth u_t, a_T = -(u_t g_t + u_p g_p),
        //   u_t* = -ro cth a_p* - g_t a_T*,  u_p* = ro cth a_t* - g_p a_T*,
        //   g_t* = -u_t a_T*,                g_p* = -u_p a_T*
        // fields: 0 u_t 1 u_p 2 a_t* 3 a_p* 4 g_t 5 g_p 6 a_T*
        NP = NPC;
        const T ro = (T)a.ro;
        const T *costh = static_cast<const T *>(a.costh);
        for (int j = tid; j < n; j += nthr) {
            C2<T> f[NFC];
#pragma unroll
            for (int F = 0; F < NFC; ++F) f[F] = buf[F * ld + sk(j)];
            C2<T> o[NPC];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int ti = a.coriolis_index ? (h ? is : i) : (j < a.nlat - 1 ? j : a.nlat - 1);
                const T rc = ro * costh[ti];
#define FV(F) (h ? f[F].y : f[F].x)
                const T ut = FV(0), up = FV(1), bt = FV(2), bp = FV(3), gt = FV(4), gp = FV(5), bT = FV(6);
#undef FV
                const T vals[NPC] = {-rc * bp - gt * bT, rc * bt - gp * bT, -ut * bT, -up * bT};
#pragma unroll
                for (int P = 0; P < NPC; ++P) {
                    if (h) o[P].y = vals[P];
                    else o[P].x = vals[P];
                }
            }
#pragma unroll
            for (int P = 0; P < NPC; ++P) buf[P * ld + sk(j)] = o[P];
        }
        __syncthreads();
    } else if (MODE == RING_ANALYSIS) {
        NP = NF;
        for (int j = tid; j < n; j += nthr)
            for (int F = 0; F < NF; ++F) {
                const double *p = F == 0 ? a.phys_in[0] : a.phys_in[1];
                buf[F * ld + sk(j)] = C2<T>{(T)p[((size_t)r * n + j) * a.nlat + i], (T)p[((size_t)r * n + j) * a.nlat + is]};
            }
        __syncthreads();
    } else {
        // pointwise nonlinear terms on the north (.x) and south (.y) rings
        // fields: 0 u_t 1 u_p 2 w_t 3 w_p 4 B_t 5 B_p 6 j_t 7 j_p 8 gT_t 9 gT_p
        //         10 u_r 11 w_r 12 B_r 13 j_r 14 dT_r
        NP = 5;
        const T ro = (T)a.ro;
        const T *sinth = static_cast<const T *>(a.sinth), *costh = static_cast<const T *>(a.costh);
        for (int j = tid; j < n; j += nthr) {
            C2<T> f[15];
#pragma unroll
            for (int F = 0; F < 15; ++F) f[F] = buf[F * ld + sk(j)];
            C2<T> o[5];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                int ti;
                T sth, cth;
                if (a.coriolis_index) {
                    ti = h ? is : i;
                } else {
                    ti = j < a.nlat - 1 ? j : a.nlat - 1; // velocity.jl:494 theta_{min(j,nlat)}
                }
                sth = sinth[ti];
                cth = costh[ti];
#define FV(F) (h ? f[F].y : f[F].x)
                const T ut = FV(0), up = FV(1), wt = FV(2), wp = FV(3), Bt = FV(4), Bp = FV(5);
                const T jt = FV(6), jp = FV(7), gt = FV(8), gp = FV(9);
                const T ur = FV(10), wr = FV(11), Br = FV(12), jr = FV(13), gr = FV(14);
#undef FV
                // velocity.jl:512-527, 664-670; magnetic.jl:399-401; scalar_field_common.jl:401-407
                T at = -ro * (up * wr - ur * wp) + (-ro * (-cth * up));
                T ap = -ro * (ur * wt - ut * wr) + (-ro * (cth * ut + sth * ur));
                at += ro * (jp * Br - jr * Bp);
                ap += ro * (jr * Bt - jt * Br);
                const T bt = up * Br - ur * Bp;
                const T bp = ur * Bt - ut * Br;
                const T aT = -(ur * gr + ut * gt + up * gp);
                const T vals[5] = {at, ap, bt, bp, aT};
#pragma unroll
                for (int P = 0; P < 5; ++P) {
                    if (h) o[P].y = vals[P];
                    else o[P].x = vals[P];
                }
            }
#pragma unroll
            for (int P = 0; P < 5; ++P) buf[P * ld + sk(j)] = o[P];
        }
        __syncthreads();
    }

    if constexpr (NC > 0) fft_ct<T, NC, -1, NPC>(buf, tw, NP);
    else fft_batch<T>(buf, tw, NP, n, ld, srad, a.nstages, -1);

    // split Z into north X and south Y, form G+- = (X +- Y) * 2 pi w_i / n
    const T c = static_cast<const T *>(a.wq)[i];
    T *gb = static_cast<T *>(a.gb);
    const int NPn = NPC ? NPC : NP;
    const unsigned ms = (unsigned)(a.nlat2 * a.nr); // a step mode's records of one order
    const size_t rec0 = (size_t)i * a.nr + r;
    for (int e = tid; e < NPn * nm; e += nthr) {
        const int P = e % NPn, m = e / NPn;
        T *d;
        if constexpr (NFC > 0)
            d = gb + gd_comp_off(P, NPV, (size_t)nm * ms) + ((size_t)m * ms + rec0) * gd_comp_str(P, NPV);
        else
            d = gb + (m * a.dim.m + r * a.dim.l + i * a.dim.i) * (4 * NF) + 4 * P;
        *reinterpret_cast<RingRec<T> *>(d) =
            fft_split<T>(buf[P * ld + sk(m)], buf[P * ld + sk(m ? n - m : 0)], m, c);
    }
}

// a boundary pass takes consecutive nodes of one level on one XCD (their grid
// values share cache lines)
template <typename T, int MODE, int NC> __global__ void __launch_bounds__(256) ring_kernel(RingArgs a)
{
    const int b = blockIdx.x + gridDim.x * blockIdx.y, nblk = gridDim.x * gridDim.y;
    const int L = StepMode<MODE>::NF > 0 ? ring_step_block(b, nblk, a.nlat2) : xcd_logical(b, nblk);
    ring_body<T, MODE, NC>(a, L % a.nlat2, L / a.nlat2);
}

// The boundary passes (RING_SYNTH: Fourier -> physical rings, RING_ANALYSIS:
// physical rings -> Fourier) with RG consecutive ring pairs per block.  The
// physical arrays are colatitude-fastest, so one ring's points lie a whole
// row of nlat doubles apart: with one ring pair per block every lane's load or
// store is its own cache line.  Here lanes take (longitude, ring) with the
// ring fastest, so a wave's access covers runs of RG consecutive colatitudes
// (and their southern mirrors); the RG * NF transforms of the block share the
// twiddles and one batched FFT.  Each transform gets the operations of the
// one-ring form.
template <typename T, int MODE, int RG>
__device__ __forceinline__ void ring_io_body(const RingArgs &a, int g, int r)
{
    static_assert(MODE == RING_SYNTH || MODE == RING_ANALYSIS, "boundary passes only");
    extern __shared__ __align__(16) char smem_raw[];
    const int n = a.nlon, nm = a.mmax + 1;
    const int ld = ring_ld(n);
    C2<T> *tw = reinterpret_cast<C2<T> *>(smem_raw);
    C2<T> *buf = tw + n;
    __shared__ int srad[12];
    const int tid = threadIdx.x;
    constexpr int nthr = RING_THREADS;
    const int NF = a.nfield;
    const int i0 = g * RG, nq = min(RG, a.nlat2 - i0); // this block's ring pairs i0 .. i0 + nq - 1
    const int NT = nq * NF;                             // transform t = q * NF + F
    const C2<T> *twg = static_cast<const C2<T> *>(a.tw);
    for (int k = tid; k < n; k += nthr) tw[k] = twg[k];
    if (tid < 12) srad[tid] = a.radix[tid];
    __syncthreads();
    if (MODE == RING_SYNTH) {
        // Hermitian spectra of the north (X) and south (Y) rings packed as Z = X + iY
        for (int e0 = 0; e0 < NT * nm; e0 += 8 * nthr) {
            C2<T> xn[8], xs[8];
            // loads of 8 elements in flight before their stores; unconditional
            // (clamped to the last element): a guarded load becomes a branch
            // whose join waits for it
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int e = min(e0 + tid + it * nthr, NT * nm - 1);
                const int F = e % NF, q = (e / NF) % nq, m = e / NT;
                const C2<T> *p = reinterpret_cast<const C2<T> *>(
                    static_cast<const T *>(a.fb) + 4 * F + (m * a.dim.m + r * a.dim.l + (i0 + q) * a.dim.i) * (4 * NF));
                xn[it] = p[0];
                xs[it] = p[1];
            }
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int e = e0 + tid + it * nthr;
                if (e < NT * nm) {
                    const int F = e % NF, q = (e / NF) % nq, m = e / NT;
                    C2<T> *b = buf + (q * NF + F) * ld;
                    if (m == 0) {
                        b[0] = C2<T>{xn[it].x, xs[it].x};
                    } else {
                        b[sk(m)] = C2<T>{xn[it].x - xs[it].y, xn[it].y + xs[it].x};
                        b[sk(n - m)] = C2<T>{xn[it].x + xs[it].y, xs[it].x - xn[it].y};
                    }
                }
            }
        }
        for (int k = nm + tid; k <= n - nm; k += nthr)
            for (int t = 0; t < NT; ++t) buf[t * ld + sk(k)] = C2<T>{T(0), T(0)};
        __syncthreads();
        fft_batch<T>(buf, tw, NT, n, ld, srad, a.nstages, +1);
        for (int e = tid; e < n * nq; e += nthr) {
            const int q = e % nq, j = e / nq, i = i0 + q, is = a.nlat - 1 - i;
            for (int F = 0; F < NF; ++F) {
                double *o = a.phys_out[F == 0 ? 0 : 1];
                const C2<T> z = buf[(q * NF + F) * ld + sk(j)];
                o[((size_t)r * n + j) * a.nlat + i] = (double)z.x;
                o[((size_t)r * n + j) * a.nlat + is] = (double)z.y;
            }
        }
        return;
    }
    // the rings' points: UR elements per thread and round, all loads issued
    // (clamped to the last element) before any LDS store and conversion, so
    // a round waits once, not once per element
    constexpr int UR = 4;
    for (int e0 = tid; e0 < n * nq; e0 += UR * nthr) {
        double px[UR][2], py[UR][2];
#pragma unroll
        for (int u = 0; u < UR; ++u) {
            const int e = min(e0 + u * nthr, n * nq - 1);
            const int q = e % nq, j = e / nq, i = i0 + q, is = a.nlat - 1 - i;
            const size_t o = ((size_t)r * n + j) * a.nlat;
            px[u][0] = a.phys_in[0][o + i];
            py[u][0] = a.phys_in[0][o + is];
            if (NF > 1) {
                px[u][1] = a.phys_in[1][o + i];
                py[u][1] = a.phys_in[1][o + is];
            }
        }
#pragma unroll
        for (int u = 0; u < UR; ++u) {
            const int e = e0 + u * nthr;
            if (e < n * nq) {
                const int q = e % nq, j = e / nq;
                buf[(q * NF) * ld + sk(j)] = C2<T>{(T)px[u][0], (T)py[u][0]};
                if (NF > 1) buf[(q * NF + 1) * ld + sk(j)] = C2<T>{(T)px[u][1], (T)py[u][1]};
            }
        }
    }
    __syncthreads();
    fft_batch<T>(buf, tw, NT, n, ld, srad, a.nstages, -1);
    // split Z into north X and south Y, form G+- = (X +- Y) * 2 pi w_i / n
    T *gb = static_cast<T *>(a.gb);
    for (int e = tid; e < NT * nm; e += nthr) {
        const int F = e % NF, q = (e / NF) % nq, m = e / NT, i = i0 + q;
        const T c = static_cast<const T *>(a.wq)[i];
        const C2<T> *b = buf + (q * NF + F) * ld;
        const C2<T> Z = b[sk(m)];
        C2<T> X, Y;
        if (m == 0) {
            X = C2<T>{Z.x, T(0)};
            Y = C2<T>{Z.y, T(0)};
        } else {
            const C2<T> Zc = b[sk(n - m)];
            X = C2<T>{T(0.5) * (Z.x + Zc.x), T(0.5) * (Z.y - Zc.y)};
            Y = C2<T>{T(0.5) * (Z.y + Zc.y), T(0.5) * (Zc.x - Z.x)};
        }
        T *d = gb + (m * a.dim.m + r * a.dim.l + i * a.dim.i) * (4 * NF) + 4 * F;
        d[0] = (X.x + Y.x) * c;
        d[1] = (X.y + Y.y) * c;
        d[2] = (X.x - Y.x) * c;
        d[3] = (X.y - Y.y) * c;
    }
}

// blocks (ring group, level) in XCD-aware order, as the one-ring boundary form
template <typename T, int MODE, int RG> __global__ void __launch_bounds__(256) ring_io_kernel(RingArgs a)
{
    const int L = xcd_logical(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    ring_io_body<T, MODE, RG>(a, L % gridDim.x, L / gridDim.x);
}

// one grid over the ring passes of several shells (step modes): a shell's
// blocks are its (node, level) pairs, node fastest
template <typename T, int MODE, int NC> __global__ void __launch_bounds__(256) ring_batch_kernel(BatchRef<RingArgs> b)
{
    const int sh = b.shell_of_block[blockIdx.x];
    if (sh == BATCH_PAD) return;
    const auto &a = batch_args(b, sh);
    const int L = ring_step_block(blockIdx.x - b.block_off[sh], b.block_cnt[sh], a.nlat2);
    ring_body<T, MODE, NC>(a, L % a.nlat2, L / a.nlat2);
}
} // namespace

template <typename T, int MODE, int NC> static void ring_launch(hipStream_t st, dim3 grid, size_t lds, const RingArgs &a)
{
    hipLaunchKernelGGL((ring_kernel<T, MODE, NC>), grid, dim3(RING_THREADS), lds, st, a);
}

template <typename T> static bool ring_step_own_launch(hipStream_t st, dim3 grid, size_t lds, const RingArgs &a)
{
    switch (a.nlon) {
#define GD_RING_LEN(N)                                          \
    case N:                                                     \
        if constexpr (ring_step_own<T>(N)) {                    \
            ring_launch<T, RING_STEP, N>(st, grid, lds, a);     \
            return true;                                        \
        }                                                       \
        return false;
        GD_RING_LENGTHS
#undef GD_RING_LEN
    default: return false;
    }
}

template <typename T, int MODE> static void ring_dispatch(hipStream_t st, dim3 grid, size_t lds, const RingArgs &a)
{
    switch (a.nlon) {
    case 48: ring_launch<T, MODE, 48>(st, grid, lds, a); break;
    case 96: ring_launch<T, MODE, 96>(st, grid, lds, a); break;
    case 144: ring_launch<T, MODE, 144>(st, grid, lds, a); break;
    case 192: ring_launch<T, MODE, 192>(st, grid, lds, a); break;
    case 288: ring_launch<T, MODE, 288>(st, grid, lds, a); break;
    case 384: ring_launch<T, MODE, 384>(st, grid, lds, a); break;
    default: ring_launch<T, MODE, 0>(st, grid, lds, a); break;
    }
}

static int ring_check(int mode, const RingArgs &a, int *nf_out)
{
    const int nthr = RING_THREADS;
    int nf = (mode == RING_STEP) ? 15 : (mode == RING_STEP_TANG) ? 4 : (mode == RING_STEP_TANG_C) ? 6
           : (mode == RING_ADJ_TANG) ? 7 : a.nfield;
    GD_CHECK(nf >= 1 && nf <= 15, GD_ERR_ARG, "ring: nfield=%d", nf);
    GD_CHECK(a.mmax + 1 <= ring_most_orders(nf), GD_ERR_ARG, "ring: %d fields x %d orders exceed one load batch",
             nf, a.mmax + 1);
    for (int s = 0; s < a.nstages; ++s) {
        int R = a.radix[s];
        long per = ((long)nf * (a.nlon / R) + nthr - 1) / nthr;
        GD_CHECK(per * R <= MAXC, GD_ERR_ARG, "ring: nlon=%d too large for %d fields", a.nlon, nf);
    }
    *nf_out = nf;
    return GD_OK;
}

// a shell's tangential ring pass can join a batched launch (its own launch's checks)
int gd_ring_tang_batchable(const RingArgs &a, bool fp64)
{
    int nf;
    GD_TRY(ring_check(RING_STEP_TANG, a, &nf));
    GD_CHECK((fp64 ? 16 : 8) * ((size_t)ring_ld(a.nlon) * nf + a.nlon) <= 160 * 1024, GD_ERR_ARG,
             "ring batch: nlon=%d needs too much LDS", a.nlon);
    return GD_OK;
}

int gd_ring_tang_form(const RingArgs &a)
{
    if (ring_short(a.nlon) || !gd_ring_compiled(a.nlon) || !gd_step_offsets_fit(a)) return 0;
    return gd_ring_deal(a) ? 1 : 2;
}

// ring pairs per block of the boundary passes of lengths without a compiled
// plan: 2 for FP64 rings, 4 for FP32, halved until the block's transforms fit
// the FFT's per-thread registers (RG nfield nlon <= MAXC threads) and 160 KB
// of LDS
template <typename T> static int ring_io_rg(const RingArgs &a, int nf)
{
    int rg = sizeof(T) == 8 ? 2 : 4;
    while (rg > 1 && ((long)rg * nf * a.nlon > (long)MAXC * RING_THREADS ||
                      sizeof(C2<T>) * ((size_t)ring_ld(a.nlon) * nf * rg + a.nlon) > 160 * 1024))
        rg /= 2;
    return rg;
}

bool gd_ring_compiled(int nlon)
{
    switch (nlon) {
#define GD_RING_LEN(N) case N: return true;
        GD_RING_LENGTHS
#undef GD_RING_LEN
    default: return false;
    }
}

void gd_ring_stage_twiddles(int nlon, std::vector<double> &tw)
{
    tw.clear();
    if (!gd_ring_compiled(nlon)) return;
    tw.resize((size_t)2 * (fft_tw_len(fft_stages(nlon, 1)) + fft_tw_len(fft_stages(nlon, -1))));
    for (int dir : {1, -1}) {
        const FftStages f = fft_stages(nlon, dir);
        for (int s = 1, Ns = f.r[0]; s < f.n; Ns *= f.r[s], ++s)
            for (int r = 0; r < f.r[s]; ++r)
                for (int k = 0; k < Ns; ++k) {
                    const double ang = 2.0 * M_PI * (double)(r * k) / (double)(Ns * f.r[s]);
                    double *o = tw.data() + 2 * (size_t)(fft_tw_off(nlon, dir, s) + r * Ns + k);
                    o[0] = std::cos(ang);
                    o[1] = -std::sin(ang);
                }
    }
}

template <typename T> int gd_launch_ring(hipStream_t st, int mode, const RingArgs &a)
{
    int nf;
    GD_TRY(ring_check(mode, a, &nf));
    if (mode == RING_SYNTH || mode == RING_ANALYSIS) {
        // the boundary passes take one scalar or one (theta, phi) pair: phys_in / phys_out [0], [1]
        GD_CHECK(nf <= 2, GD_ERR_ARG, "ring: %d fields in a boundary pass", nf);
        if (gd_launch_ring_plan<T>(st, mode, a)) return gd_check_launch("ring_plan_kernel");
        const int rg = ring_io_rg<T>(a, nf);
        if (rg > 1) {
            const size_t lds = sizeof(C2<T>) * ((size_t)ring_ld(a.nlon) * nf * rg + a.nlon);
            const dim3 grid((a.nlat2 + rg - 1) / rg, a.nr);
#define GD_RIO(MODE)                                                                                                  \
    {                                                                                                                 \
        if (rg == 4) hipLaunchKernelGGL((ring_io_kernel<T, MODE, 4>), grid, dim3(RING_THREADS), lds, st, a);       \
        else hipLaunchKernelGGL((ring_io_kernel<T, MODE, 2>), grid, dim3(RING_THREADS), lds, st, a);               \
    }
            if (mode == RING_SYNTH) GD_RIO(RING_SYNTH) else GD_RIO(RING_ANALYSIS)
#undef GD_RIO
            return gd_check_launch("ring_io_kernel");
        }
    }
    size_t lds = sizeof(C2<T>) * ((size_t)ring_ld(a.nlon) * nf + a.nlon);
    GD_CHECK(lds <= 160 * 1024, GD_ERR_ARG, "ring: LDS %zu too large", lds);
    dim3 grid(a.nlat2, a.nr);
    if (mode == RING_STEP && ring_step_own_launch<T>(st, grid, lds, a)) return gd_check_launch("ring_kernel");
    if ((mode == RING_STEP || !ring_short(a.nlon)) && gd_launch_ring_step_plan<T>(st, mode, a))
        return gd_check_launch("ring_step_plan_kernel");
    switch (mode) {
    case RING_SYNTH: ring_launch<T, RING_SYNTH, 0>(st, grid, lds, a); break;
    case RING_ANALYSIS: ring_launch<T, RING_ANALYSIS, 0>(st, grid, lds, a); break;
    case RING_STEP_TANG: ring_dispatch<T, RING_STEP_TANG>(st, grid, lds, a); break;
    case RING_STEP_TANG_C: ring_dispatch<T, RING_STEP_TANG_C>(st, grid, lds, a); break;
    case RING_ADJ_TANG: ring_dispatch<T, RING_ADJ_TANG>(st, grid, lds, a); break;
    default: ring_launch<T, RING_STEP, 0>(st, grid, lds, a); break;
    }
    return gd_check_launch("ring_kernel");
}

// The tangential step's ring pass in one grid over several shells of one
// ring length and form
template <typename T, int NC>
static void ring_batch_launch(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, size_t lds)
{
    hipLaunchKernelGGL((ring_batch_kernel<T, RING_STEP_TANG, NC>), dim3(nblocks), dim3(RING_THREADS), lds, st, b);
}

template <typename T> int gd_launch_ring_tang_batch(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, int form)
{
    if (nblocks <= 0) return GD_OK;
    if (form) {
        GD_CHECK(gd_launch_ring_tang_batch_plan<T>(st, b, nblocks, nlon, form == 1), GD_ERR_ARG, "ring batch: no plan of nlon=%d", nlon);
        return gd_check_launch("ring_step_batch_kernel");
    }
    const size_t lds = sizeof(C2<T>) * ((size_t)ring_ld(nlon) * 4 + nlon);
    GD_CHECK(lds <= 160 * 1024, GD_ERR_ARG, "ring batch: LDS %zu too large", lds);
    switch (nlon) {
    case 48: ring_batch_launch<T, 48>(st, b, nblocks, lds); break;
    case 96: ring_batch_launch<T, 96>(st, b, nblocks, lds); break;
    case 144: ring_batch_launch<T, 144>(st, b, nblocks, lds); break;
    case 192: ring_batch_launch<T, 192>(st, b, nblocks, lds); break;
    case 288: ring_batch_launch<T, 288>(st, b, nblocks, lds); break;
    case 384: ring_batch_launch<T, 384>(st, b, nblocks, lds); break;
    default: ring_batch_launch<T, 0>(st, b, nblocks, lds); break;
    }
    return gd_check_launch("ring_batch_kernel");
}
template int gd_launch_ring_tang_batch<float>(hipStream_t, const BatchRef<RingArgs> &, int, int, int);
template int gd_launch_ring_tang_batch<double>(hipStream_t, const BatchRef<RingArgs> &, int, int, int);

template int gd_launch_ring<float>(hipStream_t, int, const RingArgs &);
template int gd_launch_ring<double>(hipStream_t, int, const RingArgs &);
