// gd_ana.hip -- the analysis' Legendre contraction on MFMA (16x16x4 f32 / f64,
// or BF16x3): X_t(l, col) = sum_i Tab_t(l, i) G(i, col) over the northern nodes
// with G+- = Gn +- Gs, even and odd l - m apart; vector fields combine
// S = X_t - i Y_p, T = -i Y_t - X_p.
#include <algorithm>
#include <cstdint>

#include "gd_sht.hpp"

namespace {
template <typename T> using acc_t = typename Acc4<T>::type;

// Four consecutive elements and two doubles at any element-aligned address
template <typename T> struct Quad;
template <> struct Quad<float> { using type = float __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct Quad<double> { using type = double __attribute__((ext_vector_type(4), aligned(8))); };
using Pair64 = double __attribute__((ext_vector_type(2), aligned(8)));

// groups of 16 nodes of operands in flight, and waves per SIMD whose registers
// are asked for (FP64 tables beyond 96 nodes leave room for one)
template <typename T> constexpr int ana_depth(int h) { return (sizeof(T) == 4 && h % 3 == 0 && h < 12) || h % 2 ? 3 : 2; }
template <typename T> constexpr int ana_occ(int kn) { return sizeof(T) == 4 || kn <= 96 ? 2 : 1; }

// A wave owns a row tile of 16 degrees and keeps its table rows -- both tables
// of a vector field's parity, or both parities of a scalar field -- for all KN
// (>= nk, zero-padded) nodes in registers, in the MFMA operand layout; it
// streams level tiles past them.  Lane column c is a record component (vector:
// 8 levels x (theta, phi), scalar: 16 levels): the component's four contiguous
// slots, one 16-byte (FP64: 32-byte) load, are the operands of four MFMAs
// (two tables or parities x re, im), so nothing passes LDS and no wave waits
// for another.  The loads run D groups of 16 nodes ahead, across tiles.
//
// Nodes: in the k-step j of group h, lane group kq takes node 16 h + 4 kq + j,
// or 16 h + 4 j + kq where nodes are the records' fastest index (a load's lanes
// then share 128-byte lines); BF16x3 contracts the four steps of a group at
// once.  Degrees: register v of lane group g holds degree
// 4 g + v of the tile (FP64: by permuting the table rows), so a lane stores
// runs of four consecutive idx.
//
// A block is one wave (row tiles of one order are few and of very different
// number, and blocks of four left SIMDs idle), with a.tw level tiles; the
// blocks of one order are neighbours on one XCD (their records meet in its L2).
//
// Against a block of four waves with the tables in LDS, one slot per lane and
// load, and node chunks of 96 (us): FP64 at lmax 127, 65 levels, vector 74 ->
// 43 (MFMA floor with the tiles' padding 15); FP32 lmax 255, 97 levels, vector
// 388 -> 216, of which 75 are MFMA; FP64 scalar there 236 -> 168 (40 MFMA); FP64
// lmax 107, 41 levels, vector 46 -> 30.  What is left is the lanes' gather from
// L1 (lanes of one level per 16- or 32-byte piece) and the start of a wave.
template <typename T, bool VEC, int KN, int MM, bool ADD, class AT>
__device__ __forceinline__ void ana_body(const AT &a, int blk, int nblk)
{
    static_assert(!MM || sizeof(T) == 4, "the BF16x3 contraction takes FP32 operands");
    constexpr int H = KN / 16, LT = VEC ? 8 : 16, PS = VEC ? 8 : 4;
    constexpr int D = ana_depth<T>(H);
    // FP32 sums run over at most 128 nodes; the halves of 192 meet in FP64
    constexpr int NS = sizeof(T) == 4 && KN > 128 ? 2 : 1;
    static_assert(KN % 16 == 0 && H % D == 0, "whole 16-node groups, whole rounds of the operand ring");
    using Q = typename Quad<T>::type;
    const int nmz = a.mmax + 1, lane = threadIdx.x;
    const int gw = ((a.maxgroup + 15) / 16) * (VEC ? 2 : 1);
    const int nlt = (a.nr + LT - 1) / LT, gy = (nlt + a.tw - 1) / a.tw;
    int L = xcd_logical(blk, nblk);
    const int wt = L % gw;
    L /= gw;
    const int tile0 = L % gy * a.tw, tile1 = min(tile0 + a.tw, nlt);
    L /= gy;
    const int m = paired_m(L % nmz, nmz), f = L / nmz;
    const int par = VEC ? wt & 1 : 0, row0 = (VEC ? wt >> 1 : wt) * 16;
    const int mo = a.moff[m], K = a.moff[m + 1] - mo, ne = a.ne[m];
    // Slot pair u (0: G+, 1: G-) of the records meets table set u: of a scalar
    // field the even (0) and odd (1) degrees, of a vector field's parity the
    // table Q at u = parity and dP, which has southern sign -(-1)^(l+m), at the
    // other.  Rows left of u's group, and their first idx:
    int Kt[2], kb[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int p = VEC ? par : t;
        Kt[t] = (p ? K - ne : ne) - row0;
        kb[t] = mo + (p ? ne : 0) + row0;
    }
    if (Kt[0] <= 0 && Kt[1] <= 0) return;
    const int c = lane & 15, kq = lane >> 4;
    const int k0 = a.k0, nk = a.nk; // this launch's node chunk

    // Operand addresses: a uniform base and a 32-bit byte offset per lane (the
    // launcher's node chunks keep it in range).  Unconditional at clamped
    // indices (a guarded load becomes a branch): a node past the chunk meets
    // table values that are zero, a level past nr (or a tile past the last)
    // belongs to a column that is never stored.
    const char *gm = reinterpret_cast<const char *>(static_cast<const T *>(a.gb) + f * a.plane +
                                                    (m * a.dim.m + k0 * a.dim.i) * PS);
    const unsigned is = (unsigned)(a.dim.i * PS * sizeof(T)), ls = (unsigned)(a.dim.l * PS * sizeof(T));
    const int lv = VEC ? c >> 1 : c;
    const int nq = a.dim.i == 1 ? 1 : 4, nj = 5 - nq;
    auto gload = [&](int tile, int h, Q (&b)[4]) {
        tile = min(tile, nlt - 1);
        const char *g = gm + (size_t)(tile * LT) * ls;
        const unsigned lo = min(lv, a.nr - 1 - tile * LT) * ls + (VEC ? 4 * (int)sizeof(T) * (c & 1) : 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const Q *>(g + (lo + min(16 * h + nq * kq + nj * j, nk - 1) * is));
    };
    Q b[D][4];
#pragma unroll
    for (int h = 0; h < D; ++h) gload(tile0, h, b[h]);

    // table rows
    const int drow = sizeof(T) == 4 ? c : 4 * (c & 3) + (c >> 2);
    Q A[2][H];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const T *tab = static_cast<const T *>(VEC && t == par ? a.tab1 : a.tab0);
        const bool row = drow < Kt[t];
        const T *pt = tab + (Kt[t] > 0 ? (size_t)kb[t] * a.nlat2 : 0) + k0;
        const unsigned pr = row ? drow * a.nlat2 : 0;
        if (nk % 4 == 0 && nj == 1) {
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const int k = 16 * h + 4 * kq;
                A[t][h] = *reinterpret_cast<const Q *>(pt + (pr + (k < nk ? k : 0)));
            }
        } else {
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j) A[t][h][j] = pt[pr + min(16 * h + nq * kq + nj * j, nk - 1)];
        }
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (!row || 16 * h + nq * kq + nj * j >= nk) A[t][h][j] = T(0);
    }
    Bf16Pair ab[MM ? 2 : 1][MM ? H : 1];
    if constexpr (MM)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int h = 0; h < H; ++h) ab[t][h] = bf16_split4(A[t][h][0], A[t][h][1], A[t][h][2], A[t][h][3]);

    // the scale of this lane's rows 4 kq .. 4 kq + 3, and its outputs
    const int sc = VEC ? (f ? (c & 1 ? a.scale[3] : a.scale[2]) : (c & 1 ? a.scale[1] : a.scale[0])) : a.scale[f];
    double *out = VEC ? (f ? (c & 1 ? a.out[3] : a.out[2]) : (c & 1 ? a.out[1] : a.out[0])) : a.out[f];
    constexpr int NR = VEC ? 1 : 2; // row sets
    double scl[NR][4];
#pragma unroll
    for (int t = 0; t < NR; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int l = m + (VEC ? par : t) + 2 * (row0 + 4 * kq + v);
            const double inv = 1.0 / ((double)max(l, 1) * (double)(l + 1));
            scl[t][v] = sc == 0 ? (l > 0 ? inv : 0.0) : sc == 2 ? -1.0 : 1.0;
        }
    const size_t fs = (size_t)a.nr * a.nlm;
    auto store = [&](int t, int r, int reim, const T (&o)[NS][4]) {
        const int n = Kt[t] - 4 * kq;
        if (r >= a.nr || n <= 0) return;
        double w[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
            w[v] = (double)o[0][v] * scl[VEC ? 0 : t][v];
        if constexpr (NS == 2)
#pragma unroll
            for (int v = 0; v < 4; ++v) w[v] += (double)o[1][v] * scl[VEC ? 0 : t][v];
        if (m == 0 && reim) // imag(m=0) := 0 (shtnskit_field_functions.jl:432-435)
#pragma unroll
            for (int v = 0; v < 4; ++v) w[v] = 0.0;
        double *dst = out + reim * fs + (size_t)r * a.nlm + kb[t] + 4 * kq;
        if (n >= 4) {
            Pair64 *d2 = reinterpret_cast<Pair64 *>(dst);
            Pair64 lo = {w[0], w[1]}, hi = {w[2], w[3]};
            if (ADD) {
                lo += d2[0];
                hi += d2[1];
            }
            d2[0] = lo;
            d2[1] = hi;
        } else
#pragma unroll
            for (int v = 0; v < 3; ++v)
                if (v < n) dst[v] = ADD ? dst[v] + w[v] : w[v];
    };
    for (int tile = tile0; tile < tile1; ++tile) {
        acc_t<T> sum[NS][2][2]; // [.][t][re, im]
#pragma unroll
        for (int n = 0; n < NS; ++n)
#pragma unroll
            for (int t = 0; t < 2; ++t) sum[n][t][0] = sum[n][t][1] = acc_t<T>{0, 0, 0, 0};
#pragma unroll
        for (int h = 0; h < H; ++h) {
            Q(&x)[4] = b[h % D];
            acc_t<T>(&acc)[2][2] = sum[h * NS / H];
            if constexpr (MM) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int ri = 0; ri < 2; ++ri) {
                        const int s = 2 * t + ri;
                        acc[t][ri] = mfma_bf16x3(ab[t][h], bf16_split4(x[0][s], x[1][s], x[2][s], x[3][s]), acc[t][ri]);
                    }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        acc[t][0] = mfma16x16x4(A[t][h][j], x[j][2 * t], acc[t][0]);
                        acc[t][1] = mfma16x16x4(A[t][h][j], x[j][2 * t + 1], acc[t][1]);
                    }
            }
            if (h + D < H) gload(tile, h + D, x);
            else gload(tile + 1, h + D - H, x);
            __builtin_amdgcn_sched_barrier(0); // keeps the loads D groups ahead of their use
        }
        const int r = tile * LT + lv;
        if constexpr (VEC) {
            // lane theta of a level stores S, lane phi T, each with the other's Y
            T re[NS][4], im[NS][4];
            const T sg = c & 1 ? T(-1) : T(1);
#pragma unroll
            for (int n = 0; n < NS; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    acc_t<T>(&acc)[2][2] = sum[n];
                    const T Xre = par ? acc[0][0][v] : acc[1][0][v], Xim = par ? acc[0][1][v] : acc[1][1][v];
                    const T Yre = par ? acc[1][0][v] : acc[0][0][v], Yim = par ? acc[1][1][v] : acc[0][1][v];
                    re[n][v] = sg * Xre + __shfl_xor(Yim, 1);
                    im[n][v] = sg * Xim - __shfl_xor(Yre, 1);
                }
            store(0, r, 0, re);
            store(0, r, 1, im);
        } else {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                T re[NS][4], im[NS][4];
#pragma unroll
                for (int n = 0; n < NS; ++n)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        re[n][v] = sum[n][t][0][v];
                        im[n][v] = sum[n][t][1][v];
                    }
                store(t, r, 0, re);
                store(t, r, 1, im);
            }
        }
    }
}

template <typename T, bool VEC, int KN, int MM, bool ADD>
__global__ void __launch_bounds__(64, (ana_occ<T>(KN))) ana_kernel(AnaArgs a)
{
    ana_body<T, VEC, KN, MM, ADD>(a, blockIdx.x, gridDim.x);
}

// one grid over the analyses of several shells (a batched step)
template <typename T, bool VEC, int KN, int MM>
__global__ void __launch_bounds__(64, (ana_occ<T>(KN))) ana_batch_kernel(BatchRef<AnaArgs> b)
{
    const int sh = b.shell_of_block[blockIdx.x];
    if (sh == BATCH_PAD) return;
    ana_body<T, VEC, KN, MM, false>(batch_args(b, sh), blockIdx.x - b.block_off[sh], b.block_cnt[sh]);
}

int row_tiles(const AnaArgs &a, bool vec) { return ((a.maxgroup + 15) / 16) * (vec ? 2 : 1); }
int level_tiles(const AnaArgs &a, bool vec) { return (a.nr + (vec ? 7 : 15)) / (vec ? 8 : 16); }

template <typename T, bool VEC, int KN, bool ADD = false> void launch_kn(hipStream_t st, const AnaArgs &a, int blocks)
{
    if constexpr (sizeof(T) == 4)
        if (a.mm) {
            hipLaunchKernelGGL((ana_kernel<T, VEC, KN, 1, ADD>), dim3(blocks), dim3(64), 0, st, a);
            return;
        }
    hipLaunchKernelGGL((ana_kernel<T, VEC, KN, 0, ADD>), dim3(blocks), dim3(64), 0, st, a);
}
template <typename T, bool VEC, int KN> void launch_batch_kn(hipStream_t st, const BatchRef<AnaArgs> &b, int nblocks, int mm)
{
    if constexpr (sizeof(T) == 4)
        if (mm) {
            hipLaunchKernelGGL((ana_batch_kernel<T, VEC, KN, 1>), dim3(nblocks), dim3(64), 0, st, b);
            return;
        }
    hipLaunchKernelGGL((ana_batch_kernel<T, VEC, KN, 0>), dim3(nblocks), dim3(64), 0, st, b);
}

// nodes of a wave's tables: the smallest instance that holds all of them, or
// chunks of ANA_MAX, the first of which stores and the others add (the sum
// over nodes is linear; the per-row factors, signs and imag(m=0) := 0 apply to
// every partial alike)
constexpr int ANA_MAX = 192;
int node_tile(int nk) { return nk <= 32 ? 32 : nk <= 48 ? 48 : nk <= 64 ? 64 : nk <= 96 ? 96 : nk <= 128 ? 128 : ANA_MAX; }

template <typename T, bool VEC> void launch_ana(hipStream_t st, const AnaArgs &a, int blocks)
{
    if (a.accum) {
        // the last chunk's remainder seldom needs all ANA_MAX nodes.  Both chunks,
        // us, the second with 192 against 96: scalar, 288 nodes, lmax 383, 9 levels
        // FP32 107 - 86, FP64 130 - 101; vector, 33 levels FP32 351 - 288, FP64 554 -
        // 436 (chunks of 96 throughout, with the tables in LDS: 90, 164, 425, 1024)
        if (a.nk <= 96) launch_kn<T, VEC, 96, true>(st, a, blocks);
        else launch_kn<T, VEC, ANA_MAX, true>(st, a, blocks);
        return;
    }
    switch (node_tile(a.nk)) {
    case 32: launch_kn<T, VEC, 32>(st, a, blocks); break;
    case 48: launch_kn<T, VEC, 48>(st, a, blocks); break;
    case 64: launch_kn<T, VEC, 64>(st, a, blocks); break;
    case 96: launch_kn<T, VEC, 96>(st, a, blocks); break;
    case 128: launch_kn<T, VEC, 128>(st, a, blocks); break;
    default: launch_kn<T, VEC, ANA_MAX>(st, a, blocks); break;
    }
}
} // namespace

// Level tiles per wave: the runs that bring the grid nearest to one wave per
// SIMD (nlm / 16 row tiles plus half a tile per order and parity).  A run pays
// for its tables, so more and shorter ones are slower: FP32, lmax = 127, 65
// levels, runs of 9 / 5 / 3 / 2 / 1 of the 9 tiles: a step of 175.1 / 170.6 /
// 175.9 / 177.6 / 179.3 us.
void gd_ana_plan(AnaArgs &a, bool vec, int maxgroup)
{
    a.maxgroup = maxgroup;
    const long rows = std::max(1L, ((long)a.nlm / 16 + a.mmax + 1) * a.nf / (vec ? 1 : 2)), nlt = level_tiles(a, vec);
    const long runs = std::max(1L, std::min(nlt, (1024 + rows / 2) / rows));
    a.tw = (int)((nlt + runs - 1) / runs);
}
int gd_ana_blocks(const AnaArgs &a, bool vec)
{
    return row_tiles(a, vec) * ((level_tiles(a, vec) + a.tw - 1) / a.tw) * (a.mmax + 1) * a.nf;
}

template <typename T> int gd_launch_ana(hipStream_t st, const AnaArgs &a0, bool vec, int maxgroup)
{
    GD_CHECK(!a0.mm || sizeof(T) == 4, GD_ERR_ARG, "ana: the BF16x3 contraction takes FP32 operands");
    GD_CHECK(a0.nf >= 1 && a0.nf <= 2, GD_ERR_ARG, "ana: nf=%d", a0.nf);
    AnaArgs a = a0;
    gd_ana_plan(a, vec, maxgroup);
    const size_t node = a.dim.i * (vec ? 8 : 4) * sizeof(T); // 32-bit operand offsets: 2 GiB of nodes
    const int chunk = (int)std::max<size_t>(16, std::min<size_t>(ANA_MAX, ((size_t)2 << 30) / node / 16 * 16));
    for (a.k0 = 0; a.k0 < a.nlat2; a.k0 += chunk) {
        a.nk = std::min(chunk, a.nlat2 - a.k0);
        a.accum = a.k0 > 0;
        vec ? launch_ana<T, true>(st, a, gd_ana_blocks(a, vec)) : launch_ana<T, false>(st, a, gd_ana_blocks(a, vec));
    }
    return gd_check_launch(vec ? "ana_kernel<vec>" : "ana_kernel<scal>");
}
template int gd_launch_ana<float>(hipStream_t, const AnaArgs &, bool, int);
template int gd_launch_ana<double>(hipStream_t, const AnaArgs &, bool, int);

// node tile of a batched analysis for nlat/2 (0: not batched)
int gd_ana_kn(int nlat2, bool fp64) { return nlat2 <= (fp64 ? 96 : 128) ? node_tile(nlat2) : 0; }

template <typename T>
int gd_launch_ana_batch(hipStream_t st, const BatchRef<AnaArgs> &b, int nblocks, bool vec, int kn, int mm)
{
    GD_CHECK(!mm || sizeof(T) == 4, GD_ERR_ARG, "ana batch: the BF16x3 contraction takes FP32 operands");
    if (nblocks <= 0) return GD_OK;
    switch (kn) {
    case 32: vec ? launch_batch_kn<T, true, 32>(st, b, nblocks, mm) : launch_batch_kn<T, false, 32>(st, b, nblocks, mm); break;
    case 48: vec ? launch_batch_kn<T, true, 48>(st, b, nblocks, mm) : launch_batch_kn<T, false, 48>(st, b, nblocks, mm); break;
    case 64: vec ? launch_batch_kn<T, true, 64>(st, b, nblocks, mm) : launch_batch_kn<T, false, 64>(st, b, nblocks, mm); break;
    case 96: vec ? launch_batch_kn<T, true, 96>(st, b, nblocks, mm) : launch_batch_kn<T, false, 96>(st, b, nblocks, mm); break;
    case 128:
        if constexpr (sizeof(T) == 4) {
            vec ? launch_batch_kn<T, true, 128>(st, b, nblocks, mm) : launch_batch_kn<T, false, 128>(st, b, nblocks, mm);
            break;
        }
        [[fallthrough]];
    default: GD_CHECK(false, GD_ERR_ARG, "ana batch: node tile %d", kn);
    }
    return gd_check_launch("ana_batch_kernel");
}
template int gd_launch_ana_batch<float>(hipStream_t, const BatchRef<AnaArgs> &, int, bool, int, int);
template int gd_launch_ana_batch<double>(hipStream_t, const BatchRef<AnaArgs> &, int, bool, int, int);
