// gd_fft.hpp -- register FFT butterflies and the compiled ring-FFT plans.
//
// A transform of length n = 2^a 3^b runs as two or three Stockham stages of
// radix up to 18, each butterfly held in registers: stage s reads
// x[j + r n/R], multiplies by the stage's twiddles and writes
// (j / Ns) Ns R + j % Ns + r Ns (Ns: the product of the earlier radices).
#pragma once
#include "gd_internal.hpp"
#include "gd_sht.hpp"

template <typename T> struct alignas(2 * sizeof(T)) C2 {
    T x, y;
};
template <typename T> __device__ __forceinline__ C2<T> cadd(C2<T> a, C2<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T> __device__ __forceinline__ C2<T> csub(C2<T> a, C2<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T> __device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b)
{
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// multiply by i*dir
template <typename T> __device__ __forceinline__ C2<T> cmuli(C2<T> a, int dir)
{
    return dir > 0 ? C2<T>{-a.y, a.x} : C2<T>{a.y, -a.x};
}

// cos(2 pi k / 144) and sin(2 pi k / 144), k = 0 .. 18: every twiddle inside a
// radix that divides 144
__host__ __device__ constexpr double cos144(int k)
{
    constexpr double c[19] = {
        1.0, 0.9990482215818577624037, 0.996194698091745532295, 0.9914448613738104111446, 0.9848077530122080593667,
        0.9762960071199333659709, 0.9659258262890682867497, 0.9537169507482269211438, 0.9396926207859083840541,
        0.9238795325112867561282, 0.9063077870366499632426, 0.8870108331782217010546, 0.8660254037844386467637,
        0.8433914458128857012729, 0.8191520442889917896845, 0.7933533402912351645798, 0.7660444431189780352024,
        0.7372773368101240413843, 0.7071067811865475244008};
    constexpr double s[19] = {
        0.0, 0.0436193873653359997818, 0.0871557427476581735581, 0.1305261922200515915484,
        0.1736481776669303488517, 0.2164396139381028797596, 0.2588190451025207623489, 0.3007057995042731216225,
        0.3420201433256687330441, 0.3826834323650897717285, 0.422618261740699436187, 0.4617486132350339305629, 0.5,
        0.5372996083468238318408, 0.573576436351046096108, 0.6087614290087206394161, 0.6427876096865393263226,
        0.6755902076156602443483, 0.7071067811865475244008};
    k %= 144;
    if (k > 72) k = 144 - k;
    return k > 54 ? -c[72 - k] : k > 36 ? -s[k - 36] : k > 18 ? s[36 - k] : c[k];
}
__host__ __device__ constexpr double sin144(int k) { return cos144(k + 108); }

// a e^(DIR 2 pi i k / 144), k a constant once the caller's loop is unrolled
template <int DIR, typename T> __device__ __forceinline__ C2<T> rot144(C2<T> a, int k)
{
    k %= 144;
    if (k == 0) return a;
    if (k == 36) return cmuli(a, DIR);
    if (k == 72) return C2<T>{-a.x, -a.y};
    if (k == 108) return cmuli(a, -DIR);
    const T c = (T)cos144(k), s = (T)(DIR * sin144(k));
    return C2<T>{a.x * c - a.y * s, a.x * s + a.y * c};
}

// in-register DFT of radix R (a divisor of 144): v[k] <- sum_n v[n] e^(DIR 2 pi i n k / R)
template <int R, int DIR, typename T> __device__ __forceinline__ void dft(C2<T> *v)
{
    if constexpr (R == 2) {
        const C2<T> t = v[0];
        v[0] = cadd(t, v[1]);
        v[1] = csub(t, v[1]);
    } else if constexpr (R == 3) {
        const T s3 = T(0.86602540378443864676);
        const C2<T> t1 = cadd(v[1], v[2]), d = csub(v[1], v[2]);
        const C2<T> t2 = {v[0].x - T(0.5) * t1.x, v[0].y - T(0.5) * t1.y};
        const C2<T> t3 = cmuli(C2<T>{s3 * d.x, s3 * d.y}, DIR);
        v[0] = cadd(v[0], t1);
        v[1] = cadd(t2, t3);
        v[2] = csub(t2, t3);
    } else if constexpr (R == 4) {
        const C2<T> a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]);
        const C2<T> d = cmuli(csub(v[1], v[3]), DIR);
        v[0] = cadd(a, c);
        v[2] = csub(a, c);
        v[1] = cadd(b, d);
        v[3] = csub(b, d);
    } else {
        // R = A B: n = B n1 + n2, k = k1 + A k2
        constexpr int A = R % 4 == 0 ? (R == 8 ? 2 : 4) : (R == 9 ? 3 : 2), B = R / A;
        static_assert(144 % R == 0, "radix");
        C2<T> u[R];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
            C2<T> w[A];
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) w[n1] = v[B * n1 + n2];
            dft<A, DIR>(w);
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1) u[n2 * A + k1] = rot144<DIR>(w[k1], 144 / R * n2 * k1);
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            C2<T> w[B];
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) w[n2] = u[n2 * A + k1];
            dft<B, DIR>(w);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = w[k2];
        }
    }
}

// the step modes' fields, tangential components among them, products,
// tangential among them
template <int MODE> struct StepMode { static constexpr int NF = 0, NFV = 0, NP = 0, NPV = 0; };
template <> struct StepMode<RING_STEP_TANG> { static constexpr int NF = 4, NFV = 4, NP = 3, NPV = 2; };
template <> struct StepMode<RING_STEP_TANG_C> { static constexpr int NF = 6, NFV = 6, NP = 4, NPV = 2; };
template <> struct StepMode<RING_ADJ_TANG> { static constexpr int NF = 7, NFV = 6, NP = 4, NPV = 4; };
template <> struct StepMode<RING_STEP> { static constexpr int NF = 15, NFV = 10, NP = 5, NPV = 4; };

// Block order of a step mode's pass over nodes (fastest) and levels: block b of
// the launch goes to XCD b % 8, and a node's consecutive levels write pieces of
// the same lines of GB.  Where the nodes are a multiple of 8 they meet on one XCD
// in the launch order; else the blocks are renumbered so that each XCD takes a
// contiguous range.  Measured, launch order against renumbered (us): 192 nodes,
// 33 levels, rings of 768, FP32 tangential 87 / 106, with composition 137 / 162;
// 96 nodes, 65 levels, rings of 384 FP32 36.8 / 38.6, 15 fields 119 / 125, FP64
// 70.7 / 71.7; 54 nodes, rings of 216 FP32 20.0 / 19.1; 81 nodes, rings of 324,
// with composition 56.8 / 55.1.
__device__ __forceinline__ int ring_step_block(int b, int nblk, int nlat2) { return nlat2 % 8 ? xcd_logical(b, nblk) : b; }

// ---- compiled plans: two stages where both radices are at most 18 (the least
// largest radix), else three of at most 12
struct FftStages {
    int n = 0, r[3] = {1, 1, 1};
};
constexpr FftStages fft_stages(int n)
{
    constexpr int set[9] = {3, 4, 6, 8, 9, 12, 16, 18, 0};
    FftStages f;
    for (int a = 0; set[a]; ++a)
        for (int b = a; set[b]; ++b)
            if (set[a] * set[b] == n && (f.n == 0 || set[b] < f.r[1])) {
                f.n = 2;
                f.r[0] = set[a];
                f.r[1] = set[b];
            }
    if (f.n) return f;
    for (int a = 0; set[a]; ++a)
        for (int b = a; set[b]; ++b)
            for (int c = b; set[c] && set[c] <= 12; ++c)
                if (set[a] * set[b] * set[c] == n && (f.n == 0 || set[c] < f.r[2])) {
                    f.n = 3;
                    f.r[0] = set[a];
                    f.r[1] = set[b];
                    f.r[2] = set[c];
                }
    return f;
}
// the stage order of a direction: inverse transforms (dir > 0) start with the
// largest radix divisible by 3 and forward ones end with it, so that on a
// dealiased grid (nm <= n / 3) whole inputs of the first, and whole outputs of
// the last, radix fall into the unused middle third of the orders
constexpr FftStages fft_stages(int n, int dir)
{
    FftStages f = fft_stages(n), g = f;
    int t = 0;
    for (int s = 0; s < f.n; ++s)
        if (f.r[s] % 3 == 0 && (f.r[t] % 3 != 0 || f.r[s] > f.r[t])) t = s;
    int k = 0;
    g.r[k++] = f.r[t];
    for (int s = 0; s < f.n; ++s)
        if (s != t) g.r[k++] = f.r[s];
    if (dir < 0)
        for (int s = 0; 2 * s < f.n; ++s) {
            const int x = g.r[s];
            g.r[s] = g.r[f.n - 1 - s];
            g.r[f.n - 1 - s] = x;
        }
    return g;
}

// Elements k = r n / R .. (r + 1) n / R - 1 of a packed Hermitian spectrum:
// used ones are k < nm (order k) and n - k < nm (order n - k), nm <= n / 2, and
// nm <= n / 3 with DEAL
enum { PART_LOW = 0, PART_HIGH = 1, PART_NONE = 2, PART_BOTH = 3 };
constexpr int fft_part(int r, int R, bool deal)
{
    if (deal && 3 * r >= R && 3 * (r + 1) <= 2 * R) return PART_NONE;
    return 2 * (r + 1) <= R ? PART_LOW : 2 * r >= R ? PART_HIGH : PART_BOTH;
}

// Twiddles of the stages after the first, e^(-2 pi i r k / (Ns R)) at
// [offset + r Ns + k] (r < R, k < Ns), so that consecutive k are consecutive:
// stage 1 at offset 0, stage 2 after it, the forward order's after the inverse's.
constexpr int fft_tw_len(FftStages f) { return f.r[0] * f.r[1] + (f.n == 3 ? f.r[0] * f.r[1] * f.r[2] : 0); }
constexpr int fft_tw_off(int n, int dir, int s)
{
    const FftStages f = fft_stages(n, dir);
    return (dir < 0 ? fft_tw_len(fft_stages(n, 1)) : 0) + (s == 2 ? f.r[0] * f.r[1] : 0);
}

// LDS positions of the two exchanges (padded against bank conflicts): after
// the first stage element e sits at e + (e / r0) P1, after the second of three
// at e + (e / (r0 r1)) P2; ld(w) is the stride from one transform to the next,
// congruent to w modulo a bank row of M elements: lanes on 16 (8-byte) or 8
// (16-byte elements) consecutive transforms fall on different banks with
// w = 1, lanes on four of them and neighbouring elements with w = M / 4.
template <typename T, int N, int DIR> struct FftLds {
    static constexpr FftStages f = fft_stages(N, DIR);
    static constexpr int P1 = f.r[0] % 2 == 0 ? 1 : 0;
    static constexpr int P2 = f.n == 3 ? f.r[0] : 0;
    static constexpr int S1 = N + N / f.r[0] * P1, S2 = N + (f.n == 3 ? f.r[2] * P2 : 0);
    static constexpr int S = S1 > S2 ? S1 : S2;
};
template <typename T, int N> struct FftRow { // both directions
    static constexpr int S = FftLds<T, N, 1>::S > FftLds<T, N, -1>::S ? FftLds<T, N, 1>::S : FftLds<T, N, -1>::S;
    static constexpr int M = sizeof(T) == 8 ? 8 : 16;
    static constexpr int ld(int w) { return S + (w - S % M + M) % M; }
};

// twiddles of butterfly j of stage s (1 or 2); loaded before the barrier that
// makes the stage's inputs visible, so that their latency is hidden by it
template <typename T, int N, int S, int DIR>
__device__ __forceinline__ void fft_tw_load(const C2<T> *tws, int j, C2<T> *w)
{
    constexpr FftStages f = fft_stages(N, DIR);
    constexpr int R = f.r[S], Ns = S == 1 ? f.r[0] : f.r[0] * f.r[1], nb = N / R;
    const C2<T> *tw = tws + fft_tw_off(N, DIR, S) + (nb == Ns ? j : j % Ns);
#pragma unroll
    for (int r = 1; r < R; ++r) w[r] = tw[r * Ns];
}

// butterfly j of stage s: its inputs from one transform's LDS row, times the
// twiddles, transformed
template <typename T, int N, int S, int DIR>
__device__ __forceinline__ void fft_lds_stage(const C2<T> *x, const C2<T> *w, int j, C2<T> *v)
{
    using F = FftLds<T, N, DIR>;
    constexpr FftStages f = F::f;
    constexpr int R = f.r[S], nb = N / R;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int p = S == 1 ? j + r * nb + (j / f.r[0] + r * (nb / f.r[0])) * F::P1 : j + r * (nb + F::P2);
        v[r] = x[p];
    }
#pragma unroll
    for (int r = 1; r < R; ++r) {
        const C2<T> t = DIR > 0 ? C2<T>{w[r].x, -w[r].y} : w[r];
        v[r] = cmul(v[r], t);
    }
    dft<R, DIR>(v);
}

// results of butterfly j of stage s into the next exchange
template <typename T, int N, int S, int DIR>
__device__ __forceinline__ void fft_lds_put(C2<T> *x, int j, const C2<T> *v)
{
    using F = FftLds<T, N, DIR>;
    constexpr FftStages f = F::f;
    if constexpr (S == 0) {
#pragma unroll
        for (int r = 0; r < f.r[0]; ++r) x[j * (f.r[0] + F::P1) + r] = v[r];
    } else {
        static_assert(S == 1 && f.n == 3, "the second exchange of three stages");
#pragma unroll
        for (int r = 0; r < f.r[1]; ++r)
            x[j / f.r[0] * (f.r[0] * f.r[1] + F::P2) + j % f.r[0] + r * f.r[0]] = v[r];
    }
}

// every butterfly of stage S (1 or 2) of ROWS transforms, in place in LDS (LD
// elements from row to row), by NTHR threads: waits for the inputs and leaves
// the results to the caller's (or the next stage's) barrier; the last stage
// leaves them in natural order (with DEAL only those of used orders)
template <typename T, int N, int S, int DIR, int ROWS, int NTHR, int LD, bool DEAL>
__device__ __forceinline__ void fft_rows_stage(C2<T> *buf, const C2<T> *tws)
{
    constexpr FftStages f = fft_stages(N, DIR);
    constexpr int R = f.r[S], nb = N / R, total = ROWS * nb, IT = (total + NTHR - 1) / NTHR;
    C2<T> v[IT][R], w[R];
    fft_tw_load<T, N, S, DIR>(tws, (int)threadIdx.x % nb, w);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = threadIdx.x + it * NTHR;
        if (it > 0 && NTHR % nb != 0) fft_tw_load<T, N, S, DIR>(tws, g % nb, w);
        if (total % NTHR == 0 || g < total) fft_lds_stage<T, N, S, DIR>(buf + g / nb * LD, w, g % nb, v[it]);
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = threadIdx.x + it * NTHR;
        if (total % NTHR == 0 || g < total) {
            C2<T> *x = buf + g / nb * LD;
            if constexpr (S == f.n - 1) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (fft_part(r, R, DEAL) != PART_NONE) x[g % nb + r * nb] = v[it][r];
            } else {
                fft_lds_put<T, N, S, DIR>(x, g % nb, v[it]);
            }
        }
    }
}

// First stage of an inverse transform: butterfly j's inputs from the Fourier
// slots of one component, order m's at rec + m * mstr (T elements), packed as
// Z = X + iY of the north (X) and south (Y) rings: X_m + i Y_m at m, and
// conj(X_m) + i conj(Y_m) at n - m.  The imaginary parts of order 0 do not
// enter, whatever they hold (they are selected away, not multiplied by 0).
// Unused orders read order 0.
template <typename T, int N, bool DEAL>
__device__ __forceinline__ void fft_pack_stage(const T *rec, unsigned mstr, int nm, int j, C2<T> *v)
{
    constexpr int R = fft_stages(N, 1).r[0], nb = N / R;
    RingRec<T> z[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int part = fft_part(r, R, DEAL), k = j + r * nb;
        if (part == PART_NONE) continue;
        const int m = part == PART_LOW || (part == PART_BOTH && 2 * k < N) ? k : N - k;
        z[r] = *reinterpret_cast<const RingRec<T> *>(rec + (m < nm ? (unsigned)m : 0u) * mstr);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int part = fft_part(r, R, DEAL), k = j + r * nb;
        v[r] = C2<T>{T(0), T(0)};
        if (part == PART_NONE) continue;
        const bool low = part == PART_LOW || (part == PART_BOTH && 2 * k < N);
        const int m = low ? k : N - k;
        const bool real = r == 0 && j == 0;
        const T s = low ? T(1) : T(-1), xi = real ? T(0) : z[r].v[1], yi = real ? T(0) : z[r].v[3];
        if (m < nm) v[r] = C2<T>{z[r].v[0] - s * yi, s * xi + z[r].v[2]};
    }
    dft<R, 1>(v);
}

// The Fourier slots of order m from a transform's results Z at m and Zc at
// n - m: split into north X and south Y, G+- = (X +- Y) c.  Order 0 of the real
// rings is real: its imaginary parts are 0 also where Z is not finite.
template <typename T> __device__ __forceinline__ RingRec<T> fft_split(C2<T> Z, C2<T> Zc, int m, T c)
{
    C2<T> X = C2<T>{T(0.5) * (Z.x + Zc.x), T(0.5) * (Z.y - Zc.y)};
    C2<T> Y = C2<T>{T(0.5) * (Z.y + Zc.y), T(0.5) * (Zc.x - Z.x)};
    if (m == 0) {
        X = C2<T>{Z.x, T(0)};
        Y = C2<T>{Z.y, T(0)};
    }
    return RingRec<T>{{(X.x + Y.x) * c, (X.y + Y.y) * c, (X.x - Y.x) * c, (X.y - Y.y) * c}};
}

// ---- which plan a step mode's pass runs
constexpr int MAXC = 32; // complex values a thread holds across one stage's barrier
constexpr int RING_THREADS = 256; // ring_kernel block size
__host__ __device__ constexpr int ring_ld(int n) { return n + (n >> 4) + 1; } // per-transform LDS stride

// ---- compile-time plans: every divisor and twiddle stride is a constant
constexpr int ct_next_radix(int n)
{
    return n % 8 == 0 ? 8 : n % 4 == 0 ? 4 : n % 6 == 0 ? 6 : n % 3 == 0 ? 3 : n % 2 == 0 ? 2 : 0;
}
constexpr int ct_nstages(int n)
{
    int s = 0;
    while (n > 1) {
        n /= ct_next_radix(n);
        ++s;
    }
    return s;
}
constexpr int ct_radix(int n, int stage)
{
    for (int s = 0; s < stage; ++s) n /= ct_next_radix(n);
    return ct_next_radix(n);
}

// Lengths whose tangential modes run ring_kernel's own compiled plan, not the
// register plans.  us at 65 levels,
// against the register plan: FP32 rings of 48 / 96 / 144 / 192 / 288 / 384 4.6
// against 6.9, 6.7 - 8.6, 11.3 - 12.9, 14.4 - 17.2, 29.8 - 32.7, 36.8 - 39.0; FP64
// 5.2 against 7.7, 11.0 - 11.6, 16.7 - 17.6, 24.0 - 30.4, 48.6 - 53.8, 70.7 - 69.4.
// Beyond, at 33 levels (renumbered blocks): 432 FP32 33.2 against 31.4, FP64 56 -
// 54, 576 FP32 55.7 - 51.6, FP64 103 - 99.5, 768 FP32 109 - 106, FP64 199 - 195.
constexpr bool ring_short(int nlon) { return nlon % 48 == 0 && nlon <= 384; }

// The 15-field step keeps ring_kernel's plan where the register plan takes three
// stages, ring_kernel no more, and three of its blocks fit a CU's LDS.  us at 65
// levels, against the register plan: FP32 384 119 - 127 (fits); FP64 384 342 - 260
// and, at 33 levels, FP32 512 89 - 72 (do not fit); FP32 243, five stages, 74 - 47
template <typename T> constexpr bool ring_step_own(int n)
{
    const size_t lds = sizeof(C2<T>) * ((size_t)ring_ld(n) * StepMode<RING_STEP>::NF + n);
    return fft_stages(n).n == 3 && ct_nstages(n) <= 3 && 3 * lds <= 160 * 1024;
}

// what ring_check refuses of nf fields of n points, whichever plan would run:
// more butterflies of a stage of ring_kernel's plan than its threads hold, or
// more than ring_most_orders orders
constexpr bool ring_fits(int nf, int n)
{
    for (int s = 0; s < ct_nstages(n); ++s) {
        const int r = ct_radix(n, s);
        if ((nf * (n / r) + RING_THREADS - 1) / RING_THREADS * r > MAXC) return false;
    }
    return true;
}
constexpr int ring_most_orders(int nf) { return 8 * RING_THREADS / nf; }
