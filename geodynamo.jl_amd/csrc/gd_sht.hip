// gd_sht.hip -- spherical-harmonic transform kernels for gfx950.
//
//  plm_kernel        FP64 orthonormal P_lm, dP_lm/dtheta, m P_lm/sin(theta) by
//                    the three-term recurrence with a carried base-2 exponent
//  synth_kernel      per-m Legendre contraction on MFMA (16x16x4 f32 / f64):
//                    Fourier(i, col) = sum_l Tab(l, i) a(l, col), split into
//                    (l-m) even / odd partial sums over the northern nodes;
//                    the epilogue forms north/south rings and, for vector
//                    fields, v_theta = dP S + i Q T, v_phi = i Q S - dP T
//  lm_tile_kernel    l-major <-> m-major planes
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "gd_sht.hpp"

// ====================================================================== P_lm
__global__ void plm_kernel(const double *__restrict__ x, const int *__restrict__ moff, int lmax, int mmax, int nlat2,
                           int nlm, double *__restrict__ tab64, float *__restrict__ tab32)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int m = blockIdx.y;
    if (i >= nlat2 || m > mmax) return;
    const double xi = x[i], s = sqrt(1.0 - xi * xi);
    double lg = 0.5 * log(1.0 / (4.0 * M_PI)) + 0.5 * log(2.0 * m + 1.0) + m * log(s);
    for (int k = 1; k <= m; ++k) lg += 0.5 * log((2.0 * k - 1.0) / (2.0 * k));
    int e = (int)floor(lg / M_LN2);
    double val = exp(lg - e * M_LN2);
    if (m & 1) val = -val;
    double pm2 = 0.0, pm1 = val, tprev = 0.0;
    const int K = lmax - m + 1, ne = (K + 1) / 2;
    for (int l = m; l <= lmax; ++l) {
        if (l == m + 1) {
            double cur = sqrt(2.0 * m + 3.0) * xi * pm1;
            pm2 = pm1;
            pm1 = cur;
        } else if (l > m + 1) {
            double a = sqrt((4.0 * l * l - 1.0) / ((double)l * l - (double)m * m));
            double b = sqrt((((double)l - 1) * ((double)l - 1) - (double)m * m) /
                            (4.0 * ((double)l - 1) * ((double)l - 1) - 1.0));
            double cur = a * (xi * pm1 - b * pm2);
            pm2 = pm1;
            pm1 = cur;
        }
        if (fabs(pm1) > 0x1p600) {
            pm1 = ldexp(pm1, -600);
            pm2 = ldexp(pm2, -600);
            e += 600;
        }
        const double t = ldexp(pm1, e);
        const double c = (l == m) ? 0.0 : sqrt((2.0 * l + 1.0) * ((double)l * l - (double)m * m) / (2.0 * l - 1.0));
        const double dp = (l * xi * t - c * tprev) / s;
        const double q = m * t / s;
        tprev = t;
        const int d = l - m;
        const int idx = moff[m] + ((d & 1) ? ne + (d - 1) / 2 : d / 2);
        const size_t o = (size_t)idx * nlat2 + i;
        tab64[o] = t;
        tab64[(size_t)nlm * nlat2 + o] = dp;
        tab64[(size_t)2 * nlm * nlat2 + o] = q;
        if (tab32) {
            tab32[o] = (float)t;
            tab32[(size_t)nlm * nlat2 + o] = (float)dp;
            tab32[(size_t)2 * nlm * nlat2 + o] = (float)q;
        }
    }
}

int gd_launch_plm(hipStream_t st, const double *x, const int *moff, int lmax, int mmax, int nlat2, double *tab64,
                  float *tab32, int nlm)
{
    hipLaunchKernelGGL(plm_kernel, dim3((nlat2 + 63) / 64, mmax + 1), dim3(64), 0, st, x, moff, lmax, mmax, nlat2, nlm,
                       tab64, tab32);
    return gd_check_launch("plm_kernel");
}

// ====================================================================== Legendre GEMMs
namespace {
constexpr int TM = 32; // rows per tile (two 16-row MFMA blocks)

template <typename T> using acc_t = typename Acc4<T>::type;

template <typename T> __device__ __forceinline__ T shfl_xor3(T v) { return __shfl_xor(v, 3); }

// 16-byte vector of T (stores of the staged output tiles)
template <typename T> struct Vec16;
template <> struct Vec16<float> { using type = float4; };
template <> struct Vec16<double> { using type = double2; };

// Tile shape of a synthesis block: NF fields, VC virtual columns per level
// (vector: S_re S_im T_re T_im per field, scalar: re im), NW waves of 16
// columns each, NTILE = 16 NW columns = LT levels; PL output planes of PS
// slots per (node, level) record.
// NG gradient fields (vector only: S alone, T = 0) follow the NF full fields
// with 2 columns each: both components come from the S columns, so the zero
// T columns are not contracted.  A full field's 4 columns must start at a
// multiple of 4 (its epilogue exchanges values within a lane quad); when a
// level's column count is not a multiple of 4, two levels form one group:
// their full fields first, then their gradient fields.
template <bool VEC, int NF, int NW, int NG = 0> struct SynthTile {
    static constexpr int VC = VEC ? 4 * NF + 2 * NG : 2 * NF; // columns per level
    static constexpr int PAIR = (VEC && VC % 4 != 0) ? 2 : 1;  // levels per column group
    static constexpr int GC = VC * PAIR;                        // columns per group
    static constexpr int NTILE = 16 * NW;
    static constexpr int LT = NTILE / GC * PAIR;
    static constexpr int PL = NF + NG, PS = VEC ? 8 : 4; // output planes, slots per record
    static constexpr int RS = PL * PS;
    static constexpr int NT = VEC ? 2 : 1; // tables: (dP, mP/sin) or P
    // virtual column -> (level within the tile, column within the level)
    __device__ static void decode(int vcol, int &lv, int &fv)
    {
        const int g = vcol / GC, w = vcol - g * GC;
        if constexpr (PAIR == 1) {
            lv = g;
            fv = w;
        } else if (w < 8 * NF) {
            lv = 2 * g + w / (4 * NF);
            fv = w % (4 * NF);
        } else {
            const int w2 = w - 8 * NF;
            lv = 2 * g + w2 / (2 * NG);
            fv = 4 * NF + w2 % (2 * NG);
        }
    }
};

// Synthesis contraction for one (m, node tile, level tile), both parity
// groups: the K chunks (KC degrees) of the even group, then of the odd group,
// run as one software-pipelined sequence -- chunk c+1 is loaded into
// registers while the MFMAs consume chunk c.
//   A (tables, shared by the NW waves): double-buffered in LDS with a padded
//     row stride TMA = TM + 4 (the 4-row MFMA step then hits disjoint bank
//     halves); loaded as 16-byte vectors through per-thread pointers when
//     VL (nlat/2 and the node tile are multiples of 4), else element-wise.
//   B (spectral columns, one wave's 16 columns): straight into registers in
//     the MFMA operand layout.  Within a 16-degree chunk, lane group g
//     (lane / 16) takes degrees 4g .. 4g+3 over the chunk's 4 MFMA steps (the
//     same permutation indexes A), so each lane reads 4 consecutive degrees.
constexpr int TMA = TM + 4;
template <typename T, bool VEC, int NF, int NW, int KC, bool VL, int NG, int MM, class AT>
__device__ __forceinline__ void synth_pipeline(const AT &a, const T *__restrict__ in, const T *__restrict__ tab0,
                                               const T *__restrict__ tab1, T *sA, const int *scol, int m,
                                               int i0, int r0, acc_t<T> (&accE)[SynthTile<VEC, NF, NW, NG>::NT][2],
                                               acc_t<T> (&accO)[SynthTile<VEC, NF, NW, NG>::NT][2])
{
    using TL = SynthTile<VEC, NF, NW, NG>;
    static_assert(TL::NTILE % TL::GC == 0, "a block tile holds whole column groups");
    static_assert(KC % 16 == 0, "chunks are whole 16-degree MFMA groups");
    constexpr int NT = TL::NT, VC = TL::VC;
    constexpr int nthr = 64 * NW;
    constexpr int sAsz = NT * KC * TMA;
    constexpr int EA = VL ? 16 / (int)sizeof(T) : 1;       // elements per A load
    constexpr int NAE = NT * KC * TM / EA;                 // A loads per chunk
    constexpr int RA = (NAE + nthr - 1) / nthr;            // per thread
    constexpr int RB = KC / 4;                             // B registers per chunk
    using VA = typename std::conditional<VL, typename Vec16<T>::type, T>::type;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int K = a.moff[m + 1] - a.moff[m], ne = a.ne[m];
    const int nE = (ne + KC - 1) / KC, nC = nE + (K - ne + KC - 1) / KC;
    const int kb0 = a.moff[m];

    // per-thread A element: table t, degree row k of the chunk, node offset i
    const T *pa[RA];
    int ka[RA], sa[RA];
    bool va[RA];
#pragma unroll
    for (int q = 0; q < RA; ++q) {
        const int e = tid + q * nthr;
        const int t = e / (KC * TM / EA), rem = e - t * (KC * TM / EA);
        const int k = rem / (TM / EA), i = (rem - k * (TM / EA)) * EA;
        va[q] = e < NAE && i0 + i < a.nlat2;
        pa[q] = (t == 0 || !va[q] ? tab0 : tab1) + i0 + i;
        ka[q] = k;
        sa[q] = (t * KC + k) * TMA + i;
    }
    // this lane's B column
    const int c16 = lane & 15, g = lane >> 4;
    const int vcol = wave * 16 + c16;
    int lv, fv;
    TL::decode(vcol, lv, fv);
    const int col = scol[fv], r = r0 + lv;
    const bool vb = col >= 0 && r < a.nr;
    const T *pb = in + (size_t)(vb ? r * a.cin + col : 0) * a.nlm + kb0;

    VA ra[RA];
    T rb[RB];
    auto chunk = [&](int c, int &kbase, int &k0, int &Kp) {
        const int p = c < nE ? 0 : 1;
        k0 = (p ? c - nE : c) * KC;
        Kp = p ? K - ne : ne;
        kbase = p ? ne : 0; // relative to moff[m]
    };
    auto gload = [&](int c) {
        int kbase, k0, Kp;
        chunk(c, kbase, k0, Kp);
#pragma unroll
        for (int q = 0; q < RA; ++q) {
            VA v;
            T *pv = reinterpret_cast<T *>(&v);
#pragma unroll
            for (int u = 0; u < EA; ++u) pv[u] = T(0);
            if (va[q] && k0 + ka[q] < Kp)
                v = *reinterpret_cast<const VA *>(pa[q] + (size_t)(kb0 + kbase + k0 + ka[q]) * a.nlat2);
            ra[q] = v;
        }
#pragma unroll
        for (int s = 0; s < RB; ++s) {
            // degree of step s: group h = s / 4 of 16, lane group g, step s % 4
            const int k = (s >> 2) * 16 + 4 * g + (s & 3);
            rb[s] = (vb && k0 + k < Kp) ? pb[kbase + k0 + k] : T(0);
        }
    };
    auto sstore = [&](int buf) {
        T *A = sA + buf * sAsz;
#pragma unroll
        for (int q = 0; q < RA; ++q)
            if (tid + q * nthr < NAE) *reinterpret_cast<VA *>(A + sa[q]) = ra[q];
    };
    auto mma = [&](int buf, const T (&bv)[RB], acc_t<T>(&acc)[NT][2]) {
        const T *A = sA + buf * sAsz;
        if constexpr (MM) {
            // BF16x3: the 4 steps of each 16-degree group as one split-precision
            // 16x16x16 BF16 contraction (same k order: lane group g, degrees 4g+j)
#pragma unroll
            for (int h = 0; h < KC / 16; ++h) {
                const Bf16Pair bp = bf16_split4(bv[4 * h], bv[4 * h + 1], bv[4 * h + 2], bv[4 * h + 3]);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int rb_ = 0; rb_ < 2; ++rb_) {
                        const T *Ar = A + (t * KC + h * 16 + 4 * g) * TMA + rb_ * 16 + c16;
                        const Bf16Pair ap = bf16_split4(Ar[0], Ar[TMA], Ar[2 * TMA], Ar[3 * TMA]);
                        acc[t][rb_] = mfma_bf16x3(ap, bp, acc[t][rb_]);
                    }
            }
            return;
        }
#pragma unroll
        for (int s = 0; s < RB; ++s) {
            const int k = (s >> 2) * 16 + 4 * g + (s & 3);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int rb_ = 0; rb_ < 2; ++rb_) {
                    const T av = A[(t * KC + k) * TMA + rb_ * 16 + c16];
                    acc[t][rb_] = mfma16x16x4(av, bv[s], acc[t][rb_]);
                }
        }
    };
    // chunk c: stage it, start loading c + 1, contract it into acc.  The even
    // chunks (c < nE) and the odd ones run as two loops, each with its own
    // accumulator set: a per-chunk choice between the sets made the compiler
    // copy every accumulator register on each iteration.
    auto step = [&](int c, acc_t<T>(&acc)[NT][2]) {
        sstore(c & 1);
        T bcur[RB];
#pragma unroll
        for (int s = 0; s < RB; ++s) bcur[s] = rb[s];
        __syncthreads();
        if (c + 1 < nC) gload(c + 1);
        mma(c & 1, bcur, acc);
    };
    if (nC > 0) gload(0);
    int c = 0;
    for (; c < nE; ++c) step(c, accE);
    for (; c < nC; ++c) step(c, accO);
}

template <typename T, bool VEC, int NF, int NW, int KC, int NG = 0> constexpr size_t synth_lds_bytes()
{
    using TL = SynthTile<VEC, NF, NW, NG>;
    const size_t pipe = 2 * (size_t)TL::NT * KC * TMA, tile = (size_t)TM * TL::LT * TL::RS;
    return 128 + sizeof(T) * (pipe > tile ? pipe : tile);
}

// The block's output tile is staged in LDS in the order of the records it is
// stored to, as 16-byte vectors: the step's, the fields side by side in a record
// (plane = PS), [node][level][slot]; with NODE (one field, nodes the records'
// fastest index) [level][node][slot].  Every divisor of the store is a constant:
// one loop for both orders, with the order read at run time, took 120 us where
// this takes 111 (batched step, six shells of lmax 63, 65 levels, FP64), 71
// against 64 (FP32, tile 1).
// blk, nblk: the block's index and the block count of this synthesis (the
// launch's own, or its share of a batched launch over several shells)
template <typename T, bool VEC, int NF, int NW, int KC, bool VL, int NG, int MM, bool NODE, class AT>
__device__ __forceinline__ void synth_body(const AT &a, int blk, int nblk)
{
    static_assert(!MM || sizeof(T) == 4, "the BF16x3 contraction takes FP32 operands");
    using TL = SynthTile<VEC, NF, NW, NG>;
    static_assert(!NODE || TL::PL == 1, "node-fastest records hold one field");
    constexpr int NT = TL::NT, VC = TL::VC, LT = TL::LT, RS = TL::RS;
    extern __shared__ __align__(16) char smem_raw[];
    int *scol = reinterpret_cast<int *>(smem_raw);
    T *sA = reinterpret_cast<T *>(smem_raw + 128);
    const int gx = (a.nlat2 + TM - 1) / TM, gy = (a.nr + LT - 1) / LT, nm = a.mmax + 1;
    const int L = xcd_logical(blk, nblk);
    const int bx = L % gx, by = (L / gx) % gy;
    const int m = paired_m(L / (gx * gy), nm), i0 = bx * TM, r0 = by * LT;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (tid < 20) scol[tid] = a.colmap[tid];
    __syncthreads();
    const T *in = static_cast<const T *>(a.in);
    const T *tab0 = static_cast<const T *>(a.tab0);
    const T *tab1 = static_cast<const T *>(a.tab1);
    acc_t<T> accE[NT][2], accO[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            accE[t][rb] = acc_t<T>{0, 0, 0, 0};
            accO[t][rb] = acc_t<T>{0, 0, 0, 0};
        }
    synth_pipeline<T, VEC, NF, NW, KC, VL, NG, MM>(a, in, tab0, tab1, sA, scol, m, i0, r0, accE, accO);
    __syncthreads(); // the tile below reuses the pipeline's LDS

    T *tile = sA;
    auto rec = [&](int pl, int il, int lv_) {
        return tile + (NODE ? lv_ * TM + il : il * LT + lv_) * RS + pl * TL::PS;
    };
    const int vcol = wave * 16 + (lane & 15);
    int lv, fv;
    TL::decode(vcol, lv, fv);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int il = rb * 16 + acc_row<T>(lane, v);
            T on, os;
            int pl, srel;
            if constexpr (VEC) {
                // north / south parity combination: dP flips sign once more than P, Q
                const T dPn = accE[0][rb][v] + accO[0][rb][v], dPs = accO[0][rb][v] - accE[0][rb][v];
                const T Qn = accE[1][rb][v] + accO[1][rb][v], Qs = accE[1][rb][v] - accO[1][rb][v];
                const T Qxn = shfl_xor3(Qn), Qxs = shfl_xor3(Qs);
                const int q = lane & 3; // 0 S_re, 1 S_im, 2 T_re, 3 T_im
                if (NG > 0 && fv >= 4 * NF) {
                    // gradient field: theta = dP S, phi = i Q S (Q S_re -> phi_im,
                    // -Q S_im -> phi_re); the values of the full form with T = 0
                    const int gq = fv - 4 * NF, q2 = gq & 1;
                    T *tg = rec(NF + (gq >> 1), il, lv);
                    tg[q2] = dPn;
                    tg[2 + q2] = dPs;
                    tg[q2 ? 4 : 5] = q2 ? -Qn : Qn;
                    tg[q2 ? 6 : 7] = q2 ? -Qs : Qs;
                    continue;
                }
                if (q == 0) {
                    on = dPn - Qxn;
                    os = dPs - Qxs;
                } else if (q == 1) {
                    on = dPn + Qxn;
                    os = dPs + Qxs;
                } else if (q == 2) {
                    on = -Qxn - dPn;
                    os = -Qxs - dPs;
                } else {
                    on = Qxn - dPn;
                    os = Qxs - dPs;
                }
                pl = fv >> 2;
                srel = 4 * (q >> 1) + (q & 1); // + 2 for south
            } else {
                on = accE[0][rb][v] + accO[0][rb][v];
                os = accE[0][rb][v] - accO[0][rb][v];
                pl = fv >> 1;
                srel = fv & 1; // + 2 for south
            }
            T *t = rec(pl, il, lv) + srel;
            t[0] = on;
            t[2] = os;
        }
    }
    __syncthreads();
    using V = typename Vec16<T>::type;
    constexpr int EV = 16 / sizeof(T);
    constexpr int NV = TM * LT * RS / EV;
    T *out = static_cast<T *>(a.out);
    for (int t = tid; t < NV; t += 64 * NW) {
        const int e = t * EV;
        const int q = e / RS, so = e - q * RS;
        const int il = NODE ? q % TM : q / LT, l2 = NODE ? q / TM : q % LT;
        const int i = i0 + il, r = r0 + l2;
        if (i < a.nlat2 && r < a.nr) {
            T *dst = out + (m * a.dim.m + r * a.dim.l + i * (NODE ? 1 : a.dim.i)) * a.rstr + so;
            *reinterpret_cast<V *>(dst) = *reinterpret_cast<const V *>(tile + e);
        }
    }
}

template <typename T, bool VEC, int NF, int NW, int KC, bool VL, int NG, int MM, bool NODE>
__global__ void __launch_bounds__(64 * NW) synth_kernel(SynthArgs a)
{
    synth_body<T, VEC, NF, NW, KC, VL, NG, MM, NODE>(a, blockIdx.x, gridDim.x);
}

// one grid over the syntheses of several shells (a batched step)
template <typename T, bool VEC, int NF, int NW, int KC, bool VL, int NG = 0, int MM = 0>
__global__ void __launch_bounds__(64 * NW) synth_batch_kernel(BatchRef<SynthArgs> b)
{
    const int sh = b.shell_of_block[blockIdx.x];
    if (sh == BATCH_PAD) return;
    synth_body<T, VEC, NF, NW, KC, VL, NG, MM, false>(batch_args(b, sh), blockIdx.x - b.block_off[sh], b.block_cnt[sh]);
}

} // namespace

template <typename T, bool VEC, int NF, int NW, int KC, int NG, int MM, bool NODE = false>
static void launch_synth_mm(hipStream_t st, const SynthArgs &a)
{
    if constexpr (!NODE && NF == 1 && NG == 0)
        if (a.dim.i == 1) {
            launch_synth_mm<T, VEC, NF, NW, KC, NG, MM, true>(st, a);
            return;
        }
    using TL = SynthTile<VEC, NF, NW, NG>;
    dim3 grid(((a.nlat2 + TM - 1) / TM) * ((a.nr + TL::LT - 1) / TL::LT) * (a.mmax + 1));
    constexpr size_t lds = synth_lds_bytes<T, VEC, NF, NW, KC, NG>();
    // 16-byte table loads need every node row and tile start 16-byte aligned
    if (a.nlat2 % 4 == 0 && ((uintptr_t)a.tab0 % 16) == 0 && ((uintptr_t)a.tab1 % 16) == 0)
        hipLaunchKernelGGL((synth_kernel<T, VEC, NF, NW, KC, true, NG, MM, NODE>), grid, dim3(64 * NW), lds, st, a);
    else
        hipLaunchKernelGGL((synth_kernel<T, VEC, NF, NW, KC, false, NG, MM, NODE>), grid, dim3(64 * NW), lds, st, a);
}

// a.mm = 1: the BF16x3 contraction (FP32 operands only)
template <typename T, bool VEC, int NF, int NW, int KC, int NG = 0>
static void launch_synth(hipStream_t st, const SynthArgs &a)
{
    if constexpr (sizeof(T) == 4) {
        if (a.mm) {
            launch_synth_mm<T, VEC, NF, NW, KC, NG, 1>(st, a);
            return;
        }
    }
    launch_synth_mm<T, VEC, NF, NW, KC, NG, 0>(st, a);
}

template <typename T> int gd_launch_synth_vec(hipStream_t st, const SynthArgs &a)
{
    GD_CHECK(!a.mm || sizeof(T) == 4, GD_ERR_ARG, "synth_vec: the BF16x3 contraction takes FP32 operands");
    GD_CHECK((a.ng == 0 && (a.nf == 1 || a.nf == 2 || a.nf == 3 || a.nf == 5)) || (a.nf == 1 && (a.ng == 1 || a.ng == 2)) ||
                 (a.nf == 2 && a.ng == 1),
             GD_ERR_ARG, "synth_vec: nf=%d ng=%d", a.nf, a.ng);
    GD_CHECK(a.nf + a.ng == 1 || a.plane == 8, GD_ERR_ARG, "synth_vec: fields %zu elements apart, not side by side", a.plane);
    if (gd_launch_synth_reg<T>(st, a, true)) return gd_check_launch("synth_reg_kernel<vec>");
    // one full field with 1 or 2 gradient fields: 6 columns per level (two
    // levels per 12-column group, 3 waves = 8 levels) or 8 (4 waves = 8 levels)
    if (a.ng == 1 && a.nf == 1) launch_synth<T, true, 1, 3, 16, 1>(st, a);
    else if (a.ng == 2 && a.nf == 1) launch_synth<T, true, 1, 4, 16, 2>(st, a);
    else if (a.ng == 1 && a.nf == 2) launch_synth<T, true, 2, 5, 16, 1>(st, a); // 10 columns, 5 waves = 8 levels
    else if (a.nf == 5) launch_synth<T, true, 5, 5, 16>(st, a);
    else if (a.nf == 3) launch_synth<T, true, 3, 3, 16>(st, a); // 12 columns per level, 3 waves = 4 levels
    else if (a.nf == 2) launch_synth<T, true, 2, 4, 16>(st, a);
    else launch_synth<T, true, 1, 1, 16>(st, a);
    return gd_check_launch("synth_kernel<vec>");
}

template <typename T> int gd_launch_synth_scal(hipStream_t st, const SynthArgs &a)
{
    GD_CHECK(!a.mm || sizeof(T) == 4, GD_ERR_ARG, "synth_scal: the BF16x3 contraction takes FP32 operands");
    GD_CHECK(a.nf == 1 || (a.nf == 5 && a.plane == 4), GD_ERR_ARG, "synth_scal: nf=%d (1 or 5, side by side)", a.nf);
    if (gd_launch_synth_reg<T>(st, a, false)) return gd_check_launch("synth_reg_kernel<scal>");
    if (a.nf == 5) launch_synth<T, false, 5, 5, 16>(st, a);
    else launch_synth<T, false, 1, 1, 16>(st, a);
    return gd_check_launch("synth_kernel<scal>");
}

// ---------------------------------------------------------------- batched step launches
// The tangential step's synthesis (u as a full field, grad T as a gradient
// field) in one grid over several shells, with a tile chosen per group:
//   tile 0: 3 waves (8 levels), K chunks of 16 degrees (the step's own form)
//   tile 1: 3 waves, K chunks of 32 degrees
//   tile 2: 6 waves (16 levels), K chunks of 16 (FP32 only: the FP64 output
//           tile would exceed 64 KB of LDS)
static int synth_tile_nw(int tile) { return tile == 2 ? 6 : 3; }
static int synth_tile_kc(int tile) { return tile == 1 ? 32 : 16; }

int gd_synth_tang_blocks(const SynthArgs &a, int tile)
{
    const int nw = synth_tile_nw(tile), lt = 16 * nw / 6; // 6 columns per level, two levels per 12-column group
    return ((a.nlat2 + TM - 1) / TM) * ((a.nr + lt - 1) / lt) * (a.mmax + 1);
}

bool gd_synth_tile_ok(int tile, bool fp64) { return tile == 0 || tile == 1 || (tile == 2 && !fp64); }

template <typename T, int NW, int KC, int MM>
static void synth_batch_launch(hipStream_t st, const BatchRef<SynthArgs> &b, int nblocks)
{
    constexpr size_t lds = synth_lds_bytes<T, true, 1, NW, KC, 1>();
    hipLaunchKernelGGL((synth_batch_kernel<T, true, 1, NW, KC, true, 1, MM>), dim3(nblocks), dim3(64 * NW), lds, st, b);
}

template <typename T>
int gd_launch_synth_tang_batch(hipStream_t st, const BatchRef<SynthArgs> &b, int nblocks, int tile, int mm)
{
    GD_CHECK(gd_synth_tile_ok(tile, sizeof(T) == 8), GD_ERR_ARG, "synth batch: tile %d", tile);
    GD_CHECK(!mm || sizeof(T) == 4, GD_ERR_ARG, "synth batch: the BF16x3 contraction takes FP32 operands");
    if (nblocks <= 0) return GD_OK;
#define GD_SB(NW, KC)                                                                   \
    do {                                                                                \
        if constexpr (sizeof(T) == 4) {                                                 \
            if (mm) synth_batch_launch<T, NW, KC, 1>(st, b, nblocks);                   \
            else synth_batch_launch<T, NW, KC, 0>(st, b, nblocks);                      \
        } else {                                                                        \
            synth_batch_launch<T, NW, KC, 0>(st, b, nblocks);                           \
        }                                                                               \
    } while (0)
    if (tile == 0) GD_SB(3, 16);
    else if (tile == 1) GD_SB(3, 32);
    else if constexpr (sizeof(T) == 4) GD_SB(6, 16);
#undef GD_SB
    return gd_check_launch("synth_batch_kernel");
}
template int gd_launch_synth_tang_batch<float>(hipStream_t, const BatchRef<SynthArgs> &, int, int, int);
template int gd_launch_synth_tang_batch<double>(hipStream_t, const BatchRef<SynthArgs> &, int, int, int);

// one shell's synthesis in tile form `tile` (the autotuner times these alone)
template <typename T> int gd_launch_synth_tang_tile(hipStream_t st, const SynthArgs &a, int tile)
{
    GD_CHECK(gd_synth_tile_ok(tile, sizeof(T) == 8), GD_ERR_ARG, "synth: tile %d", tile);
    GD_CHECK(a.nf == 1 && a.ng == 1 && a.plane == 8, GD_ERR_ARG, "synth tile: the tangential form (nf=1, ng=1)");
    if (tile == 0) launch_synth<T, true, 1, 3, 16, 1>(st, a);
    else if (tile == 1) launch_synth<T, true, 1, 3, 32, 1>(st, a);
    else if constexpr (sizeof(T) == 4) launch_synth<T, true, 1, 6, 16, 1>(st, a);
    return gd_check_launch("synth_kernel<tile>");
}
template int gd_launch_synth_tang_tile<float>(hipStream_t, const SynthArgs &, int);
template int gd_launch_synth_tang_tile<double>(hipStream_t, const SynthArgs &, int);

// a shell's tangential synthesis can join a batched launch: the checks of
// its own launch, and the 16-byte table form (VL) that the batched kernel has
int gd_synth_tang_batchable(const SynthArgs &a)
{
    GD_CHECK(a.nf == 1 && a.ng == 1 && a.plane == 8, GD_ERR_ARG, "synth batch: nf=%d ng=%d", a.nf, a.ng);
    GD_CHECK(a.nlat2 % 4 == 0 && (uintptr_t)a.tab0 % 16 == 0 && (uintptr_t)a.tab1 % 16 == 0, GD_ERR_ARG,
             "synth batch: nlat/2=%d needs 16-byte table rows", a.nlat2);
    return GD_OK;
}

// ====================================================================== l-major <-> m-major planes
// One block moves a 32 x 32 (m, l) tile of one (plane, level) through LDS: in
// the l-major layout the tile's rows are runs of 32 consecutive m, in the
// m-major one its columns are runs of 16 consecutive degrees of one parity,
// so both sides are coalesced.  A gather by index map (one thread an element)
// read or wrote a cache line per element on one side, and a call was a launch
// per plane: set_state or get_state of five fields was ten launches.  At
// lmax=127, nr=65 the ten planes (43 MB in, 43 MB out) took 65 us, now 18 us (4.8 TB/s)
namespace {
constexpr int LMT = 32;
constexpr int LM_THREADS = 256;
__device__ __forceinline__ int lm_of(int l, int m, int mmax)
{
    return l <= mmax ? l * (l + 1) / 2 + m : (mmax + 1) * (mmax + 2) / 2 + (l - mmax - 1) * (mmax + 1) + m;
}
// m-major index of (l, m): LmMaps' order (even l - m first, then odd)
__device__ __forceinline__ int idx_of(int l, int m, int lmax)
{
    const int d = l - m, off = m * (lmax + 1) - m * (m - 1) / 2;
    return off + (d & 1 ? (lmax - m) / 2 + 1 : 0) + (d >> 1);
}

// TO_M: l-major FP64 in, m-major T out (level stride dst_ls); else the reverse, FP64
template <typename T, bool TO_M>
__global__ void __launch_bounds__(LM_THREADS) lm_tile_kernel(LmPlanes a, int lmax, int mmax, int nlm, int nr, int ntile,
                                                             size_t dst_ls)
{
    constexpr int PER = LMT * LMT / LM_THREADS;
    __shared__ double tile[LMT * (LMT + 1)]; // [m][l]
    // consecutive logical blocks (one XCD's) are the tiles of one level: the
    // lines that two tiles share stay in one L2
    const int L = xcd_logical(blockIdx.x, gridDim.x);
    int t = L % ntile;
    const int pr = L / ntile, r = pr % nr, pl = pr / nr;
    int mt = 0, nlt = (lmax + LMT) / LMT; // tiles with l >= m: lt = mt .. nlt - 1 for each mt
    while (t >= nlt - mt) {
        t -= nlt - mt;
        ++mt;
    }
    const int m0 = mt * LMT, l0 = (mt + t) * LMT, tid = threadIdx.x;
    const double *src = a.src[pl] + (size_t)r * nlm;
    T *dst = static_cast<T *>(a.dst[pl]) + (size_t)r * dst_ls;
    // element q of this thread on the l-major side: m fastest; on the m-major
    // side: one m, the 16 degrees of one parity fastest
    auto lside = [&](int q, int &l, int &m) {
        const int e = tid + q * LM_THREADS;
        m = m0 + (e & (LMT - 1));
        l = l0 + e / LMT;
    };
    auto mside = [&](int q, int &l, int &m) {
        const int e = tid + q * LM_THREADS, w = e & (LMT - 1), p = w / (LMT / 2);
        m = m0 + e / LMT;
        l = l0 + 2 * (w & (LMT / 2 - 1)) + ((l0 ^ m ^ p) & 1);
    };
    auto ok = [&](int l, int m) { return m <= mmax && l >= m && l <= lmax; };
    double v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        int l, m;
        if (TO_M) lside(q, l, m);
        else mside(q, l, m);
        v[q] = ok(l, m) ? src[TO_M ? lm_of(l, m, mmax) : idx_of(l, m, lmax)] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        int l, m;
        if (TO_M) lside(q, l, m);
        else mside(q, l, m);
        tile[(m - m0) * (LMT + 1) + l - l0] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        int l, m;
        if (TO_M) mside(q, l, m);
        else lside(q, l, m);
        if (ok(l, m)) dst[TO_M ? idx_of(l, m, lmax) : lm_of(l, m, mmax)] = (T)tile[(m - m0) * (LMT + 1) + l - l0];
    }
}

template <typename T, bool TO_M>
int lm_launch(hipStream_t st, int lmax, int mmax, int nr, const LmPlanes &a, size_t dst_ls)
{
    GD_CHECK(a.n >= 1 && a.n <= LM_MAXPLANES, GD_ERR_ARG, "lm planes: n=%d", a.n);
    const int nlt = (lmax + LMT) / LMT;
    int ntile = 0;
    for (int mt = 0; mt * LMT <= mmax; ++mt) ntile += nlt - mt;
    const long nblk = (long)ntile * nr * a.n;
    GD_CHECK(nblk < (1L << 31), GD_ERR_ARG, "lm planes: %ld blocks", nblk);
    hipLaunchKernelGGL((lm_tile_kernel<T, TO_M>), dim3((unsigned)nblk), dim3(LM_THREADS), 0, st, a, lmax, mmax,
                       gd_nlm_of(lmax, mmax), nr, ntile, dst_ls);
    return gd_check_launch("lm_tile_kernel");
}
} // namespace

template <typename T>
int gd_launch_to_m(hipStream_t st, int lmax, int mmax, int nr, const LmPlanes &a, size_t dst_ls)
{
    return lm_launch<T, true>(st, lmax, mmax, nr, a, dst_ls);
}

int gd_launch_from_m(hipStream_t st, int lmax, int mmax, int nr, const LmPlanes &a)
{
    return lm_launch<double, false>(st, lmax, mmax, nr, a, gd_nlm_of(lmax, mmax));
}

// explicit instantiations
template int gd_launch_synth_vec<float>(hipStream_t, const SynthArgs &);
template int gd_launch_synth_vec<double>(hipStream_t, const SynthArgs &);
template int gd_launch_synth_scal<float>(hipStream_t, const SynthArgs &);
template int gd_launch_synth_scal<double>(hipStream_t, const SynthArgs &);
template int gd_launch_to_m<float>(hipStream_t, int, int, int, const LmPlanes &, size_t);
template int gd_launch_to_m<double>(hipStream_t, int, int, int, const LmPlanes &, size_t);
