// gd_sht.hpp -- SHT device kernels (gd_sht.hip): argument blocks and launchers.
//
// Device spectral layout ("m-major"): index idx in [0, nlm) with, for each m,
// the block [moff[m], moff[m+1]) holding l = m..lmax, first the ne[m] degrees
// with l-m even, then those with l-m odd (LmMaps).  A spectral column set is
// stored [col][idx] with col = level*cin + c.
//
// Legendre tables Tab[t][idx][i], i in [0, nlat/2) the northern Gauss nodes,
// t = 0 P, 1 dP/dtheta, 2 m P / sin(theta).  Southern values follow from the
// parity P(pi-theta) = (-1)^(l+m) P(theta) (dP flips sign once more).
//
// Fourier arrays (complex of the real longitude transform, m = 0..mmax), a
// record per (m, level, node i):
//   FB  synthesis output, north and south rings of node i: a component's four
//       slots are (north re, im, south re, im); a scalar field has one
//       component, a vector field two (theta, phi), 8 contiguous slots
//   GB  analysis input, a component's four slots (G+ re, im, G- re, im) of
//       G+ = Gn + Gs, G- = Gn - Gs, already weighted by 2 pi w_i / nlon
// The record order is the caller's (RecDim).  The stand-alone transforms keep
// one field's records as [m][level][i]: a Legendre block (one m) and the
// boundary ring passes (a few consecutive nodes of one level) both move whole
// pieces of 64 bytes and more.  The step, whose ring pass takes one node and
// level with every field, keeps FB as [i][level][m] with the fields' slots side
// by side (its reads are contiguous) and GB as [m][i][level].
#pragma once
#include "gd_internal.hpp"

// a component's four slots of one record
template <typename T> struct alignas(16) RingRec {
    T v[4];
};
// record (m, lev, i) is at index m * m + lev * l + i * i (strides in records)
struct RecDim {
    size_t m, l, i;
};
// the stand-alone transforms' [m][level][i], strides padded so that a vector
// field's levels and orders are an odd number of 128-byte lines apart, and the
// records it spans
inline RecDim gd_rec_dim(int nr, int nlat2, bool fp64)
{
    const size_t line = fp64 ? 2 : 4; // records of a vector field's line
    size_t l = (nlat2 + line - 1) / line * line;
    if (l / line % 2 == 0) l += line;
    return RecDim{nr * l + (nr % 2 ? 0 : line), l, 1};
}
// the step's record orders, of FB and of GB
inline RecDim gd_step_fb_dim(int nm, int nr) { return RecDim{1, (size_t)nm, (size_t)nm * nr}; }
inline RecDim gd_step_gb_dim(int nlat2, int nr) { return RecDim{(size_t)nlat2 * nr, 1, (size_t)nr}; }
// planes of products: nv tangential components in pairs, one vector array of
// recs records each, then the scalars
__host__ __device__ inline size_t gd_comp_off(int c, int nv, size_t recs)
{
    return c < nv ? 8 * recs * (c / 2) + 4 * (c % 2) : 4 * recs * c;
}
__host__ __device__ inline int gd_comp_str(int c, int nv) { return c < nv ? 8 : 4; }

struct SynthArgs {
    const void *in;       // T*, [col][idx], col = level*cin + c
    int cin;              // input columns per level
    int nf;               // vector: fields (4 virtual cols each); scalar: fields (2 each)
    int colmap[20];       // virtual col within a level -> input col c, -1 = zero
    const void *tab0;     // vector: dP, scalar: P
    const void *tab1;     // vector: Q = m P / sin
    const int *moff, *ne;
    int nlat2, nr, nlm, mmax;
    void *out;            // T*, FB: field f's record at out + f * plane + rstr * index
    size_t plane;         // elements from one field to the next
    int rstr;             // elements from record to record
    RecDim dim;
    int ng;               // vector: gradient fields (S only, T = 0) after the nf full ones; colmap
                          // then lists 4 nf + 2 ng columns (S_re S_im per gradient field)
    int mm;               // 1: BF16x3 split-precision contraction (FP32 operands), 0: native MFMA
};

struct AnaArgs {
    const void *gb;       // T*, GB: field f's record at gb + f * plane + index * (4 or 8)
    size_t plane;         // elements from one field to the next
    RecDim dim;
    int nf;               // vector fields (components 2V, 2V+1) or scalar fields
    const void *tab0, *tab1;
    const int *moff, *ne;
    int nlat2, nr, nlm, mmax;
    int maxgroup;         // largest parity group, ceil((lmax+1)/2); set by gd_ana_plan
    // outputs, FP64 m-major [reim][level][idx]; vector field V: out[2V] gets S, out[2V+1] gets T
    double *out[4];
    int scale[4];         // 0: /l(l+1) (0 at l=0), 1: x1, 2: x(-1)
    int tw;               // level tiles per wave; set by gd_ana_plan
    // node chunk (set by the launcher): nodes k0 .. k0 + nk - 1, accum = 1 adds
    // to out instead of storing
    int k0, nk, accum;
    int mm;               // 1: BF16x3 split-precision contraction (FP32 operands), 0: native MFMA
};

// A real field F's four slots of a record are at fb + 4 nfield index + 4 F.  The
// boundary passes write (RING_ANALYSIS) gb likewise; a step mode's product P is
// at gb + gd_comp_off(P) + gd_comp_str(P) index.  The step modes' records are in
// the orders gd_step_fb_dim and gd_step_gb_dim.
struct RingArgs {
    const void *fb;       // T*
    void *gb;             // T*
    int nfield;           // real fields to synthesise (SYNTH/STEP) or analyse (ANALYSIS)
    RecDim dim;           // record order of a boundary pass
    // 4 F of a boundary synthesis' field F, an argument: with the constant the
    // compiler holds the first stage in fewer registers and then orders the next
    // stage's loads behind its LDS reads (FP32 vector 384 x 768, 97 levels: 160
    // -> 167 us)
    size_t foff[2];
    const double *phys_in[2];
    double *phys_out[2];
    const void *tw;       // T2[nlon], e^{-2 pi i k / nlon}
    const void *tws;      // T2, twiddles of the compiled plan's stages (null where nlon has none)
    const void *sinth, *costh, *wq; // T[nlat] sin, cos of colatitude; T[nlat2] 2 pi w / nlon
    int nlat, nlat2, nlon, nr, mmax;
    int nstages, radix[12];
    double ro;            // Pm / E
    int coriolis_index;
};

// RING_STEP: 15 fields in (u, omega, B, j, grad T tangential; u_r, omega_r,
// B_r, j_r, dT/dr), 5 products out.  RING_STEP_TANG: the step when every
// radial component is zero -- 4 fields in (u_theta, u_phi, (grad T)_theta,
// (grad T)_phi), 3 products out (the force and -u.grad T; u x B vanishes).
// RING_STEP_TANG_C: the same with the composition's gradient as fields 4, 5
// and -u.grad C as a fourth product.
// RING_ADJ_TANG: the transposed Jacobian of RING_STEP_TANG's products at the
// state (u, grad T) applied to the cotangents of its products -- 7 fields in
// (u_theta, u_phi, cotangent force theta / phi, (grad T)_theta, (grad T)_phi,
// cotangent of -u.grad T), 4 out (cotangents of u_theta, u_phi,
// (grad T)_theta, (grad T)_phi).
enum { RING_SYNTH = 0, RING_ANALYSIS = 1, RING_STEP = 2, RING_STEP_TANG = 3, RING_STEP_TANG_C = 4,
       RING_ADJ_TANG = 5 };

// XCD-aware block order.  Workgroup b of a launch goes to XCD b % 8, and each
// XCD has its own L2; the blocks of one order m share their Legendre table
// tile (and their spectral / Fourier inputs), so the logical index is built
// so that consecutive logical blocks run on one XCD: XCD x takes the x-th
// contiguous range of the logical order.  The m dimension is ordered
// 0, mmax, 1, mmax-1, ... so that equal ranges carry equal work (the degree
// count of m falls linearly with m).
__device__ __forceinline__ int paired_m(int k, int nm) { return (k & 1) ? nm - 1 - (k >> 1) : (k >> 1); }

int gd_launch_plm(hipStream_t st, const double *x, const int *moff, int lmax, int mmax, int nlat2, double *tab64,
                  float *tab32, int nlm);
template <typename T> int gd_launch_synth_vec(hipStream_t st, const SynthArgs &a);
template <typename T> int gd_launch_synth_scal(hipStream_t st, const SynthArgs &a);
// either synthesis with the spectral columns in registers; false beyond its degrees
template <typename T> bool gd_launch_synth_reg(hipStream_t st, const SynthArgs &a, bool vec);
template <typename T> int gd_launch_ana(hipStream_t st, const AnaArgs &a, bool vec, int maxgroup);
template <typename T> int gd_launch_ring(hipStream_t st, int mode, const RingArgs &a);
// ring lengths with a compiled FFT plan (gd_fft.hpp): every 2^a 3^b from 48 to 768
#define GD_RING_LENGTHS                                                                                          \
    GD_RING_LEN(48) GD_RING_LEN(54) GD_RING_LEN(64) GD_RING_LEN(72) GD_RING_LEN(81) GD_RING_LEN(96)              \
    GD_RING_LEN(108) GD_RING_LEN(128) GD_RING_LEN(144) GD_RING_LEN(162) GD_RING_LEN(192) GD_RING_LEN(216)        \
    GD_RING_LEN(243) GD_RING_LEN(256) GD_RING_LEN(288) GD_RING_LEN(324) GD_RING_LEN(384) GD_RING_LEN(432)        \
    GD_RING_LEN(486) GD_RING_LEN(512) GD_RING_LEN(576) GD_RING_LEN(648) GD_RING_LEN(729) GD_RING_LEN(768)
bool gd_ring_compiled(int nlon);
// offsets along m fit 32 bits (the compiled plans' addresses): of a boundary
// pass, of a step mode
inline bool gd_offsets_fit(const RingArgs &a) { return (a.mmax + 1) * a.dim.m * 8 < (size_t)1 << 31; }
inline bool gd_step_offsets_fit(const RingArgs &a)
{
    return (a.mmax + 1) * gd_step_gb_dim(a.nlat2, a.nr).m * 8 < (size_t)1 << 31;
}
// a dealiased grid (the middle third of the orders is unused): instances of
// the compiled plans of their own
inline bool gd_ring_deal(const RingArgs &a) { return 3 * (a.mmax + 1) <= a.nlon; }
// stage twiddles of the compiled plan of nlon, e^{-i angle} as (re, im) pairs
void gd_ring_stage_twiddles(int nlon, std::vector<double> &tw);
// a boundary pass (RING_SYNTH, RING_ANALYSIS; 1 or 2 fields) by the compiled
// plan of its ring length; false where there is none
template <typename T> bool gd_launch_ring_plan(hipStream_t st, int mode, const RingArgs &a);
template <> bool gd_launch_ring_plan<float>(hipStream_t st, int mode, const RingArgs &a);
template <> bool gd_launch_ring_plan<double>(hipStream_t st, int mode, const RingArgs &a);
// a step mode by the compiled plan of its ring length, and the tangential
// step's batched launch; false where there is none
template <typename T> bool gd_launch_ring_step_plan(hipStream_t st, int mode, const RingArgs &a);
template <> bool gd_launch_ring_step_plan<float>(hipStream_t st, int mode, const RingArgs &a);
template <> bool gd_launch_ring_step_plan<double>(hipStream_t st, int mode, const RingArgs &a);
template <typename T> bool gd_launch_ring_tang_batch_plan(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, bool deal);
template <> bool gd_launch_ring_tang_batch_plan<float>(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, bool deal);
template <> bool gd_launch_ring_tang_batch_plan<double>(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, bool deal);
// up to LM_MAXPLANES planes between the l-major layout of the interface
// (level stride nlm) and the m-major device layout, one launch for all:
// to_m writes element type T with dst_ls elements from level to level (nlm for
// a plane, cin * nlm for a synthesis column); from_m is plane to plane
constexpr int LM_MAXPLANES = 10;
struct LmPlanes {
    int n = 0;
    const double *src[LM_MAXPLANES];
    void *dst[LM_MAXPLANES];
    void add(const double *s, void *d)
    {
        src[n] = s;
        dst[n++] = d;
    }
};
template <typename T>
int gd_launch_to_m(hipStream_t st, int lmax, int mmax, int nr, const LmPlanes &a, size_t dst_ls);
int gd_launch_from_m(hipStream_t st, int lmax, int mmax, int nr, const LmPlanes &a);

// ---- batched step launches (gd_sht.hip): one grid over several shells'
// launches of the tangential step's kernels, all in one compile-time form.
// Block counts of one shell: gd_synth_tang_blocks (tile 0, 1, or 2 = FP32
// only), nlat/2 * nr for the ring, gd_ana_blocks (args with gd_ana_plan done)
// for the analyses, whose node tile gd_ana_kn gives (0: several node chunks, not
// batched).
int gd_synth_tang_blocks(const SynthArgs &a, int tile);
bool gd_synth_tile_ok(int tile, bool fp64);
template <typename T>
int gd_launch_synth_tang_batch(hipStream_t st, const BatchRef<SynthArgs> &b, int nblocks, int tile, int mm);
template <typename T> int gd_launch_synth_tang_tile(hipStream_t st, const SynthArgs &a, int tile);
template <typename T> int gd_launch_ring_tang_batch(hipStream_t st, const BatchRef<RingArgs> &b, int nblocks, int nlon, int form);
int gd_synth_tang_batchable(const SynthArgs &a);
int gd_ring_tang_batchable(const RingArgs &a, bool fp64);
// the instance of a shell's tangential ring pass, which a batched launch shares:
// 0 ring_kernel's plans, 1 a compiled register plan on a dealiased grid, 2 on any
int gd_ring_tang_form(const RingArgs &a);
int gd_ana_kn(int nlat2, bool fp64);
void gd_ana_plan(AnaArgs &a, bool vec, int maxgroup);
int gd_ana_blocks(const AnaArgs &a, bool vec);
template <typename T>
int gd_launch_ana_batch(hipStream_t st, const BatchRef<AnaArgs> &b, int nblocks, bool vec, int kn, int mm);
