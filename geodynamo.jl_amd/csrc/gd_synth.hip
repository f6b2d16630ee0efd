// gd_synth.hip -- the synthesis' Legendre contraction on MFMA (16x16x4 f32 /
// f64, or BF16x3) with the spectral columns in registers.
#include <algorithm>
#include <cstdint>

#include "gd_sht.hpp"

namespace {
template <typename T> using acc_t = typename Acc4<T>::type;
template <typename T> struct Quad;
template <> struct Quad<float> { using type = float __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct Quad<double> { using type = double __attribute__((ext_vector_type(4), aligned(8))); };

// the value of lane ^ 1
__device__ __forceinline__ float lane_xor1(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ double lane_xor1(double v)
{
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true));
}

// column tiles of one order: 8 levels x (S, T) of each full vector field, then
// 16 levels of each gradient (or scalar) field
__host__ __device__ inline int synth_tiles8(const SynthArgs &a, bool vec) { return vec ? a.nf * ((a.nr + 7) / 8) : 0; }
__host__ __device__ inline int synth_tiles16(const SynthArgs &a, bool vec) { return (vec ? a.ng : a.nf) * ((a.nr + 15) / 16); }

template <typename T, bool VEC, int MM> struct SynthWave {
    using Q = typename Quad<T>::type;
    // one lane's column: re and im sources (column starts in `in`), output record
    const T *src[2];
    bool ok[2], st;
    T *dst;
    bool full; // (S, T) lanes in pairs; else S alone (gradient) or a scalar
    const char *tab[2];
    unsigned tmax[2]; // largest byte offset of a table element from tab
    int mo, K, ne, nlm, kq, c, ndrow;

    // NG groups of 16 degrees per parity; nodes tile0 .. tile1 - 1
    template <int NG> __device__ __forceinline__ void run(const SynthArgs &a, int tile0, int tile1) const
    {
        constexpr int NT = VEC ? 2 : 1, G = 2 * NG, D = 2; // operand groups in flight
        const unsigned row = (unsigned)(a.nlat2 * sizeof(T));
        // table operands of group g (parity g / NG): degrees 4 kq + j, this lane's node
        auto aload = [&](int tile, int g, T (&x)[NT][4]) {
            const int node = min(tile * 16 + ndrow, a.nlat2 - 1), p = g / NG, h = g % NG;
            const unsigned o = ((p ? ne : 0) + 4 * kq) * row + (unsigned)(node * sizeof(T));
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    x[t][j] = *reinterpret_cast<const T *>(tab[t] + min(o + (16 * h + j) * row, tmax[t]));
        };
        T x[D][NT][4];
#pragma unroll
        for (int g = 0; g < D; ++g) aload(tile0, g, x[g]);
        Q B[G][2];
        Bf16Pair bb[MM ? G : 1][2];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int p = g / NG, k = g % NG * 16 + 4 * kq, kg = (p ? ne : 0) + k, Kp = p ? K - ne : ne;
            const int s = min(mo + kg, nlm - 4);
#pragma unroll
            for (int ri = 0; ri < 2; ++ri) B[g][ri] = *reinterpret_cast<const Q *>(src[ri] + s);
            if (mo + K + 16 * NG > nlm) // a quad that would end past the column starts earlier
#pragma unroll
                for (int ri = 0; ri < 2; ++ri) {
                    const Q b = B[g][ri];
                    const int d = mo + kg - s;
                    Q r = b;
                    r[0] = d == 0 ? b[0] : d == 1 ? b[1] : d == 2 ? b[2] : b[3];
                    r[1] = d == 0 ? b[1] : d == 1 ? b[2] : b[3];
                    r[2] = d == 0 ? b[2] : b[3];
                    B[g][ri] = r;
                }
#pragma unroll
            for (int ri = 0; ri < 2; ++ri) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (!ok[ri] || k + j >= Kp) B[g][ri][j] = T(0);
                if constexpr (MM) bb[g][ri] = bf16_split4(B[g][ri][0], B[g][ri][1], B[g][ri][2], B[g][ri][3]);
            }
        }
        for (int tile = tile0; tile < tile1; ++tile) {
            acc_t<T> acc[2][NT][2]; // [parity][table][re, im]
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[p][t][0] = acc[p][t][1] = acc_t<T>{0, 0, 0, 0};
#pragma unroll
            for (int g = 0; g < G; ++g) {
                T(&y)[NT][4] = x[g % D];
                acc_t<T>(&s)[NT][2] = acc[g / NG];
                if constexpr (MM) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const Bf16Pair ap = bf16_split4(y[t][0], y[t][1], y[t][2], y[t][3]);
                        s[t][0] = mfma_bf16x3(ap, bb[g][0], s[t][0]);
                        s[t][1] = mfma_bf16x3(ap, bb[g][1], s[t][1]);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            s[t][0] = mfma16x16x4(y[t][j], B[g][0][j], s[t][0]);
                            s[t][1] = mfma16x16x4(y[t][j], B[g][1][j], s[t][1]);
                        }
                }
                if (g + D < G) aload(tile, g + D, y);
                else aload(tile + 1, g + D - G, y); // past the last tile: clamped
                __builtin_amdgcn_sched_barrier(0);
            }
            const size_t ds = a.dim.i * a.rstr;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = tile * 16 + 4 * kq + v;
                T *o = dst + i * ds;
                const bool w = st && i < a.nlat2;
                RingRec<T> r0, r1;
                if constexpr (VEC) {
                    // north / south parity combination: dP flips sign once more than P, Q
                    T dn[2], dv[2], qn[2], qs[2];
#pragma unroll
                    for (int ri = 0; ri < 2; ++ri) {
                        const T de = acc[0][0][ri][v], dd = acc[1][0][ri][v];
                        const T qe = acc[0][1][ri][v], qo = acc[1][1][ri][v];
                        dn[ri] = de + dd;
                        dv[ri] = dd - de;
                        qn[ri] = qe + qo;
                        qs[ri] = qe - qo;
                    }
                    if (full) {
                        // lane S: theta = dP S + i Q T, lane T: phi = i Q S - dP T
                        const T sg = c & 1 ? T(-1) : T(1);
                        r0.v[0] = sg * dn[0] - lane_xor1(qn[1]);
                        r0.v[1] = sg * dn[1] + lane_xor1(qn[0]);
                        r0.v[2] = sg * dv[0] - lane_xor1(qs[1]);
                        r0.v[3] = sg * dv[1] + lane_xor1(qs[0]);
                    } else {
                        r0.v[0] = dn[0];
                        r0.v[1] = dn[1];
                        r0.v[2] = dv[0];
                        r0.v[3] = dv[1];
                        r1.v[0] = -qn[1];
                        r1.v[1] = qn[0];
                        r1.v[2] = -qs[1];
                        r1.v[3] = qs[0];
                        if (w) reinterpret_cast<RingRec<T> *>(o)[1] = r1;
                    }
                } else {
#pragma unroll
                    for (int ri = 0; ri < 2; ++ri) {
                        r0.v[ri] = acc[0][0][ri][v] + acc[1][0][ri][v];
                        r0.v[2 + ri] = acc[0][0][ri][v] - acc[1][0][ri][v];
                    }
                }
                if (w) *reinterpret_cast<RingRec<T> *>(o) = r0;
            }
        }
    }
};

// A wave owns a column tile of one order -- 8 levels x (S, T) or 16 levels of
// S, re and im -- and keeps its spectral columns, all degrees of both parities
// (up to KG groups of 16 each), in registers in the MFMA operand layout; it
// streams 16-node table tiles past them.  One table value feeds a re and an im
// product.  A lane ends with the four contiguous slots of one component of a
// record (both components of a gradient field) and stores them directly, so
// nothing passes LDS.  Within a group, step j of lane group kq takes degree
// 4 kq + j, and table rows are permuted so that register v of lane group g
// holds node 4 g + v.
//
// Against blocks that stage tables and output tiles in LDS, 16 degrees and a
// barrier at a time (us): the step's u and grad T at lmax 127, 65 levels FP32 45
// -> 41, FP64 78 -> 71 (MFMA 22), lmax 63 16.4 -> 12.6 and 27 -> 19, lmax 15 7.2 ->
// 4.8; u and grad T, C 56 -> 55 and 104 -> 107; all vector fields of the full step
// 119 -> 103 and 244 -> 189; FP32 vector lmax 255, 97 levels 272 -> 167; FP64
// vector lmax 107, 41 levels 37 -> 27.  Bound by the start of a wave and by loads
// that wait behind a tile's stores, which the counter keeps in order.
template <typename T, bool VEC, int KG, int MM>
__global__ void __launch_bounds__(64, (sizeof(T) == 4 || KG <= 4 ? 2 : 1)) synth_reg_kernel(SynthArgs a, int ny, int tw)
{
    const int nm = a.mmax + 1, n8 = synth_tiles8(a, VEC), nt = n8 + synth_tiles16(a, VEC);
    int L = xcd_logical(blockIdx.x, gridDim.x);
    const int ct = L % nt;
    L /= nt;
    const int m = paired_m(L / ny, nm), tile0 = L % ny * tw, tile1 = min(tile0 + tw, (a.nlat2 + 15) / 16);
    SynthWave<T, VEC, MM> w;
    const int lane = threadIdx.x;
    w.c = lane & 15;
    w.kq = lane >> 4;
    w.ndrow = sizeof(T) == 4 ? w.c : 4 * (w.c & 3) + (w.c >> 2);
    w.mo = a.moff[m];
    w.K = a.moff[m + 1] - w.mo;
    w.ne = a.ne[m];
    w.nlm = a.nlm;
    w.full = ct < n8;
    // field, first input column, and this lane's level and component
    const int nl = w.full ? (a.nr + 7) / 8 : (a.nr + 15) / 16, cf = w.full ? ct : ct - n8, g = cf / nl;
    const int f = w.full || !VEC ? g : a.nf + g, col = w.full ? 4 * g : VEC ? 4 * a.nf + 2 * g : 2 * g;
    const int lev = w.full ? cf % nl * 8 + (w.c >> 1) : cf % nl * 16 + w.c, comp = w.full ? w.c & 1 : 0;
    w.st = lev < a.nr;
    const int r = min(lev, a.nr - 1);
    const T *in = static_cast<const T *>(a.in);
#pragma unroll
    for (int ri = 0; ri < 2; ++ri) {
        const int cs = a.colmap[col + ri], cm = comp ? a.colmap[col + (w.full ? 2 : 0) + ri] : cs;
        w.ok[ri] = w.st && cm >= 0;
        w.src[ri] = in + (size_t)(r * a.cin + max(cm, 0)) * a.nlm;
    }
    w.dst = static_cast<T *>(a.out) + f * a.plane + (m * a.dim.m + r * a.dim.l) * a.rstr + 4 * comp;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        w.tab[t] = static_cast<const char *>(t ? a.tab1 : a.tab0) + (size_t)w.mo * a.nlat2 * sizeof(T);
        const size_t last = ((size_t)(a.nlm - w.mo) * a.nlat2 - 1) * sizeof(T);
        w.tmax[t] = (unsigned)min(last, (size_t)0xFFFFFFF0u);
    }
    const int n = (w.ne + 15) / 16;
    if constexpr (KG >= 8) {
        if (n > 7) return w.template run<8>(a, tile0, tile1);
        if (n > 6) return w.template run<7>(a, tile0, tile1);
        if (n > 5) return w.template run<6>(a, tile0, tile1);
        if (n > 4) return w.template run<5>(a, tile0, tile1);
    }
    if constexpr (KG >= 4) {
        if (n > 3) return w.template run<4>(a, tile0, tile1);
        if (n > 2) return w.template run<3>(a, tile0, tile1);
    }
    if (n > 1) return w.template run<2>(a, tile0, tile1);
    w.template run<1>(a, tile0, tile1);
}

template <typename T, bool VEC, int KG> void launch_kg(hipStream_t st, const SynthArgs &a, int blocks, int ny, int tw)
{
    if constexpr (sizeof(T) == 4)
        if (a.mm) {
            hipLaunchKernelGGL((synth_reg_kernel<T, VEC, KG, 1>), dim3(blocks), dim3(64), 0, st, a, ny, tw);
            return;
        }
    hipLaunchKernelGGL((synth_reg_kernel<T, VEC, KG, 0>), dim3(blocks), dim3(64), 0, st, a, ny, tw);
}
} // namespace

template <typename T> bool gd_launch_synth_reg(hipStream_t st, const SynthArgs &a, bool vec)
{
    // Columns of more than 128 degrees per parity (8 groups of re and im) do not
    // fit the registers of two FP32 waves or one FP64 wave per SIMD, a column's
    // last loads need four values, and FP64 scalars of more than 64 degrees per
    // parity are faster in the LDS form (us, against this one: lmax 150, 65 levels
    // 34 - 37; lmax 190, 17 / 33 / 66 levels 24 - 31, 33 - 38, 51 - 61; lmax 222,
    // 34 levels 48 - 56; lmax 255, 33 / 97 levels 58 - 61, 150 - 153; below, lmax
    // 130, 33 levels 20.5 - 20.0).
    // degrees of order 0: nlm = sum over m of (lmax + 1 - m)
    // So are several FP64 scalars side by side in the step's records beyond 16
    // degrees per parity: the LDS form stores their slots as one run, a lane here
    // 32 bytes of it (five fields, 65 levels, lmax 47 / 95 / 127: 15.3 - 16.2, 58 -
    // 60, 92 - 105; lmax 15: 6.0 - 5.2)
    const int nm = a.mmax + 1, k0 = (a.nlm + a.mmax * nm / 2) / nm, ng = ((k0 + 1) / 2 + 15) / 16;
    if (ng > 8 || a.nlm < 4 || (sizeof(T) == 8 && !vec && (ng > 4 || (ng > 1 && a.nf > 1)))) return false;
    // node tiles per wave: the runs that bring the grid nearest to 8192 waves
    // (order 0 has many times the degrees of the last ones, and a CU's first
    // waves wait for their columns).  Against 2048 waves, us: FP32 vector lmax
    // 255, 97 levels 185 -> 166, FP32 step lmax 127 162.0 -> 161.0
    const int nt = synth_tiles8(a, vec) + synth_tiles16(a, vec), nodes = (a.nlat2 + 15) / 16;
    const int runs = std::max(1, std::min(nodes, (8192 + nm * nt / 2) / (nm * nt)));
    const int tw = (nodes + runs - 1) / runs, ny = (nodes + tw - 1) / tw, blocks = nt * ny * nm;
    if (vec) {
        if (ng <= 2) launch_kg<T, true, 2>(st, a, blocks, ny, tw);
        else if (ng <= 4) launch_kg<T, true, 4>(st, a, blocks, ny, tw);
        else launch_kg<T, true, 8>(st, a, blocks, ny, tw);
    } else {
        if (ng <= 2) launch_kg<T, false, 2>(st, a, blocks, ny, tw);
        else if (ng <= 4) launch_kg<T, false, 4>(st, a, blocks, ny, tw);
        else if constexpr (sizeof(T) == 4) launch_kg<T, false, 8>(st, a, blocks, ny, tw);
    }
    return true;
}
template bool gd_launch_synth_reg<float>(hipStream_t, const SynthArgs &, bool);
template bool gd_launch_synth_reg<double>(hipStream_t, const SynthArgs &, bool);
