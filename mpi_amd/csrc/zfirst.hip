// zfirst.hip -- the one-element Dirichlet solve with the z
// contractions outside the x-y transforms, in three kernels.
//
// With the even/odd eigenbasis of the interior operator (diag_body.h) the
// solve is, per (kx, ky), u = V diag(1 / (mu - sigma(kx, ky))) V^-1 rhs, and
// the contractions with V and V^-1 act along z only, so they commute with the
// transforms along x and y:
//   1 zf_expand   y = V^-1 (f + face loads) on the physical columns (FP64
//                 matrix cores), then the first stage of the transform along
//                 y (16 points in registers) and the store of its 8 complex
//                 slots (slot 0 packs the real outputs 0 and 8);
//   2 zf_filter   per eigen-index j and slot: the rest of the transform along
//                 y and all of the one along x, the division by
//                 mu_j - sigma(kx, ky), and both transforms back, in one
//                 read and one write;
//   3 zf_collect  the last 16-point stage, u = V z on the matrix cores, the
//                 end values, the store of u.
// Against transform - mode solve - transform this is three reads and writes
// of the field instead of five and no transform of the face data (Dirichlet
// values are added and returned in physical space): 165 -> 135 us a solve at
// 256^2 x 130.  The adjoint stays with transform - mode solve - transform: its
// sum against the solution, dL/dlambda, cancels to a millionth of its terms, and
// the contractions' rounding, which reaches the quiet (kx, ky) here, left that
// sum up to ten times as far off.
//
// With ny = 16 R2, y = n2 + R2 n1 and ky = k1 + 16 k2: kernel 1 owns 4
// columns (x, n2) and all 16 n1 of each.  Rows are dealt to the matrix tiles
// so that a lane holds all n1 of one column and eigen-index: the 16-point
// transform needs no exchange.  The intermediate is [j][slot][x][n2] complex,
// so a (j, slot) is one contiguous block of nx R2 points: what kernel 2 loads
// whole.
//
// The symmetrised operator's eigenvectors V = F^-1 W are corrected to the
// reference's operator (A = As + Ea, M = Winv F Ea F^-1 W, which maps even to
// odd coordinates and back) to first order in the eigenvectors instead of the
// solution, which makes the correction independent of sigma and so lets it
// stay on the z side: V' = V (I + G), G_ij = M_ij / (mu_j - mu_i), and V'^-1 =
// (I - G) K V^-1 with K = (I - G^2)^-1 (block diagonal, folded into the
// operand).  The largest eigenvalues come in nearly equal even/odd pairs, so
// G reaches 3e-6 there (N = 127): its first 16 x 16 block runs in FP64, the
// rest (to 4.5e-11, N = 124) in bf16 with FP32 sums, the values in two parts.
// A plan whose G is larger keeps transform - mode solve - transform.
#include "diag_body.h"
#include "fft_body.h"

#include <type_traits>

namespace hz {
namespace {

constexpr int kRows = 64;  // tile rows: 4 columns (x, n2) x 16 points n1

// exp(+- 2 pi i k / 16), k < 4, as literals
constexpr double kC1 = 0.92387953251128675613, kS1 = 0.38268343236508977173, kH = 0.70710678118654752440;

// 8-point DFT in registers, SIGN = -1 forward, +1 inverse (unnormalised).
template <int SIGN>
__device__ __forceinline__ void dft8(double (&re)[8], double (&im)[8])
{
    auto bf = [](double &ar, double &ai, double &br, double &bi) {
        const double tr = ar - br, ti = ai - bi;
        ar += br;
        ai += bi;
        br = tr;
        bi = ti;
    };
    auto rot = [](double &r, double &i) {  // times SIGN i
        const double t = r;
        r = SIGN > 0 ? -i : i;
        i = SIGN > 0 ? t : -t;
    };
    // decimation in frequency, outputs in bit-reversed order
#pragma unroll
    for (int k = 0; k < 4; ++k) bf(re[k], im[k], re[k + 4], im[k + 4]);
    {
        const double r5 = re[5], i5 = im[5], r7 = re[7], i7 = im[7];
        re[5] = kH * (r5 - SIGN * i5);
        im[5] = kH * (i5 + SIGN * r5);
        rot(re[6], im[6]);
        re[7] = kH * (-r7 - SIGN * i7);
        im[7] = kH * (-i7 + SIGN * r7);
    }
#pragma unroll
    for (int h = 0; h < 8; h += 4) {
        bf(re[h], im[h], re[h + 2], im[h + 2]);
        bf(re[h + 1], im[h + 1], re[h + 3], im[h + 3]);
        rot(re[h + 3], im[h + 3]);
        bf(re[h], im[h], re[h + 1], im[h + 1]);
        bf(re[h + 2], im[h + 2], re[h + 3], im[h + 3]);
    }
    auto swap = [&](int a, int b) {
        double t = re[a];
        re[a] = re[b];
        re[b] = t;
        t = im[a];
        im[a] = im[b];
        im[b] = t;
    };
    swap(1, 4);
    swap(3, 6);
}

// cos, sin of 2 pi k / 16
__device__ __forceinline__ constexpr double cos16(int k)
{
    return k == 0 ? 1.0 : k == 1 ? kC1 : k == 2 ? kH : k == 3 ? kS1 : k == 4 ? 0.0 : -cos16(8 - k);
}
__device__ __forceinline__ constexpr double sin16(int k)
{
    return k == 0 ? 0.0 : k == 1 ? kS1 : k == 2 ? kH : k == 3 ? kC1 : k == 4 ? 1.0 : sin16(8 - k);
}

// Real 16-point DFT of x[16] : put(s, re, im) receives the outputs
// X_s in slots s = 1 .. 7 and the real outputs (X_0, X_8) in slot 0.  (The
// 8-point transform of x[2m] + i x[2m+1], then outputs k and 8 - k together;
// scheduled pair by pair, so that few are live at once.)
template <class Put>
__device__ __forceinline__ void real_dft16(const double (&x)[16], Put put)
{
    double zr[8], zi[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        zr[m] = x[2 * m];
        zi[m] = x[2 * m + 1];
    }
    dft8<-1>(zr, zi);
    put(0, zr[0] + zi[0], zr[0] - zi[0]);
#pragma unroll
    for (int k = 1; k <= 4; ++k) {
        __builtin_amdgcn_sched_barrier(0);
        // X_k = E + W^k O, X_(8-k) = conj(E - W^k O)
        const double er = 0.5 * (zr[k] + zr[8 - k]), ei = 0.5 * (zi[k] - zi[8 - k]);
        const double dr = 0.5 * (zi[k] + zi[8 - k]), di = 0.5 * (zr[8 - k] - zr[k]);
        const double c = cos16(k), s = sin16(k);
        const double tr = c * dr + s * di, ti = c * di - s * dr;
        put(k, er + tr, ei + ti);
        if (k < 4) put(8 - k, er - tr, ti - ei);
    }
}

// The inverse (unnormalised): x[n] = sum over all 16 outputs of X_k exp(+2 pi i n k / 16).
__device__ __forceinline__ void real_idft16(const double (&re)[8], const double (&im)[8], double (&x)[16])
{
    double zr[8], zi[8];
    zr[0] = re[0] + im[0];
    zi[0] = re[0] - im[0];
#pragma unroll
    for (int k = 1; k <= 4; ++k) {
        // Z_k = S + i W^-k D, Z_(8-k) = conj(S - i W^-k D), S|D = X_k +|- conj X_(8-k)
        const double sr = re[k] + re[8 - k], si = im[k] - im[8 - k];
        const double dr = re[k] - re[8 - k], di = im[k] + im[8 - k];
        const double c = cos16(k), s = sin16(k);
        const double tr = c * dr - s * di, ti = c * di + s * dr;
        zr[k] = sr - ti;
        zi[k] = si + tr;
        if (k < 4) {
            zr[8 - k] = sr + ti;
            zi[8 - k] = tr - si;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    dft8<1>(zr, zi);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        x[2 * m] = zr[m];
        x[2 * m + 1] = zi[m];
    }
}

// Column (x, n2) and y of tile row t: the accumulator element r of row block
// rb in lane group lk is row 16 rb + 4 r + lk, so lane group lk holds column
// c0 + lk and point n1 = 4 rb + r.
struct RowAt {
    int x, y;
    __device__ __forceinline__ RowAt(int t, int c0, int lr2)
    {
        const int c = c0 + (t & 3), n1 = 4 * (t >> 4) + ((t >> 2) & 3);
        x = c >> lr2;
        y = (c & ((1 << lr2) - 1)) + (n1 << lr2);
    }
};

// The correction's operands in the LDS of the tile: every value as two bf16
// parts, its rounding and the rounding of the rest (groups of four values: four
// first parts, four second ones; 16 rows x 4 lane groups of 16 bytes spread over
// the banks), and the first 16 of each half in FP64 (row stride 34).  The two
// corrections nearly cancel in the solution, their roundings do not: with one
// part the sum of fbar u was three times as far off.  At NP = 32 the FP64 block
// is all of G.
template <int NJ>
struct CorrLds {
    static constexpr int LDB = 32 * NJ + 8, LDX = 34;
    static constexpr int XOFF = NJ > 2 ? kRows * LDB / 4 : 0;  // doubles
    static constexpr int DOUBLES = XOFF + kRows * LDX > kRows * (16 * NJ + 2) ? XOFF + kRows * LDX
                                                                              : kRows * (16 * NJ + 2);
};

typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// LDS of one tile of an end kernel.
template <int NJ>
struct alignas(16) EndLds {
    double tile[CorrLds<NJ>::DOUBLES];
    double rows[2][kRows];
};

template <int NJ>
__device__ __forceinline__ void to_corr(const d4 (&acc)[4][1], double *tile, int w, int li, int lk)
{
    using S = CorrLds<NJ>;
    if constexpr (NJ > 2) {
        __bf16 *tb = reinterpret_cast<__bf16 *>(tile) + 8 * ((16 * w + li) / 4) + li % 4;
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = (float)acc[rb][0][r];
                const __bf16 hi = (__bf16)v;
                __bf16 *t = tb + (16 * rb + 4 * r + lk) * S::LDB;
                t[0] = hi;
                t[4] = (__bf16)(v - (float)hi);
            }
    }
    if (w % (NJ / 2) == 0) {
        double *tx = tile + S::XOFF + (w ? 16 : 0) + li;
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) tx[(16 * rb + 4 * r + lk) * S::LDX] = acc[rb][0][r];
    }
}

// acc += the correction's two parts, from to_corr's values: this wave's
// eigen-indices take from the other half's.  (Row permutation and operand
// layouts as tile_gemm_bf16_rows.)
template <int NJ>
__device__ __forceinline__ void correct(d4 (&acc)[4][1], const double *tile, const short *C, const double *X, int w,
                                        int li, int lk)
{
    using S = CorrLds<NJ>;
    constexpr int NP = 16 * NJ, H = NP / 2;
    const int ko = 16 * w >= H ? 0 : H;
    f4 cacc[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) cacc[rb] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (NJ > 2) {
        // one 16x16x32 step: 16 values, their two parts against the same operand
        const s4 *bq = reinterpret_cast<const s4 *>(C) + (ko / 4 + lk) * NP + 16 * w + li;
        const short *arow = reinterpret_cast<const short *>(tile) + (4 * (li % 4) + li / 4) * S::LDB + 2 * ko + 8 * lk;
#pragma unroll
        for (int ks = 0; ks < H / 16; ++ks) {
            const s4 b = bq[4 * ks * NP];
            const s8 bv = {b[0], b[1], b[2], b[3], b[0], b[1], b[2], b[3]};
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const s8 av = *reinterpret_cast<const s8 *>(arow + 16 * rb * S::LDB + 32 * ks);
                cacc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, av),
                                                                   __builtin_bit_cast(bf8, bv), cacc[rb], 0, 0, 0);
            }
        }
    }
    if (w % (NJ / 2) == 0)  // the first 16 of each half
        tile_gemm_deep<16, S::LDX, 4, 1, 16, 4>(acc, tile + S::XOFF + (w ? 0 : 16), X + (w ? 256 : 0), 0, 0, li, lk);
    if constexpr (NJ > 2) {
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[rb][0][r] += (double)cacc[rb][r];
    }
}

// acc = A B over the wave's half (operands as pair_gemm), each half of the sum
// on its own.  Here the contractions run in physical space, where their
// rounding reaches every (kx, ky), also the quiet ones, and a sum's rounding
// grows with its partial sums: two shorter ones halve it.
template <int NJ>
__device__ __forceinline__ void contract(d4 (&acc)[4][1], const double *tile, const double *__restrict__ B, int j,
                                         int li, int lk)
{
    constexpr int NP = 16 * NJ, LD = NP + 2, NPR = NP / 16, D = 2;
    const double *bc = B + 2 * lk * NP + j;
    d4 sum[2][4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) sum[0][rb] = sum[1][rb] = d4{0.0, 0.0, 0.0, 0.0};
    double b[D][2];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        b[d][0] = bc[8 * d * NP];
        b[d][1] = bc[(8 * d + 1) * NP];
    }
#pragma unroll
    for (int p = 0; p < NPR; ++p) {
        const double v0 = b[p % D][0], v1 = b[p % D][1];
        if (p + D < NPR) {
            b[p % D][0] = bc[8 * (p + D) * NP];
            b[p % D][1] = bc[(8 * (p + D) + 1) * NP];
        }
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
            const double2 av = *reinterpret_cast<const double2 *>(tile + (16 * rb + li) * LD + 8 * p + 2 * lk);
            d4 &c = sum[2 * p / NPR][rb];
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, v0, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, v1, c, 0, 0, 0);
        }
    }
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) acc[rb][0] = sum[0][rb] + sum[1][rb];
}

template <int NJ>
__device__ __forceinline__ void to_tile(const d4 (&acc)[4][1], double *tile, int w, int li, int lk)
{
    constexpr int LD = 16 * NJ + 2;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) tile[(16 * rb + 4 * r + lk) * LD + 16 * w + li] = acc[rb][0][r];
}

// Compact index of eigen-index j (even ones first), or -1 in the padding.
template <int H>
__device__ __forceinline__ int compact(int j, int he, int ho)
{
    return j < H ? (j < he ? j : -1) : (j - H < ho ? he + j - H : -1);
}

// ---- 1: contraction, correction, 16-point stage along y ------------------------
// One wave per 16 eigen-indices, 64 rows in LDS (66 KB at NP = 128: two
// work-groups per CU).  256^2 x 129: 134 MB and 15 us of matrix instructions
// in 50 us.  The 1,024 work-groups run as two rounds whose loads (16% of a
// work-group's life), contraction (24%, near the matrix rate of the two that
// share a CU), correction (20%) and stores hardly overlap: without the loads
// 41 us, without the contraction 33, without the stores 44.  Measured by the
// counters: 157 MB, matrix cores busy 37% of the SIMD cycles.  Bounded to 128
// registers it keeps 48 bytes a lane in scratch (16 at smaller NJ).
template <int NJ, bool CUB>
__device__ __forceinline__ void expand_tile(const ZfArgs &a, int c0, int tid, EndLds<NJ> &lds)
{
    constexpr int NP = 16 * NJ, LD = NP + 2, H = NP / 2, T = 64 * NJ;
    double *tile = lds.tile, *row_zl = lds.rows[0], *row_zr = lds.rows[1];
    const int lane = tid % 64, w = uniform(tid / 64), li = lane % 16, lk = lane / 16;
    const int n = a.n, ho = n / 2, he = n - ho;
    if (tid < kRows) {
        const RowAt at(tid, c0, a.lr2);
        const int g = at.x * a.ny + at.y;
        row_zl[tid] = a.gl[g] / a.beta_l;
        row_zr[tid] = a.gr[g] / a.beta_r;
    }
    {
        // folded interior: even coordinate i f_i + f_(n-1-i) (the centre of an
        // odd n alone), odd one the difference; both from one pair of loads
        constexpr int NIT = kRows * H / T;
        double x0[NIT], x1[NIT];
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int idx = tid + T * it, row = idx / H, i = idx % H;
            const RowAt at(row, c0, a.lr2);
            const int col = (at.x * a.ny + at.y) * a.K;
            x0[it] = i < he ? a.f[col + 1 + i] : 0.0;
            x1[it] = i < ho ? a.f[col + n - i] : 0.0;
        }
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
#pragma clang fp contract(off)  // the cubic's values rounded before the fold, as hz_cubic_rhs stores them
            const int idx = tid + T * it, row = idx / H, i = idx % H;
            const double v0 = CUB ? cubic_map(x0[it], true, a.c3, a.c1) : x0[it];
            const double v1 = CUB ? cubic_map(x1[it], true, a.c3, a.c1) : x1[it];
            tile[row * LD + i] = v0 + v1;
            tile[row * LD + H + i] = i < ho ? v0 - v1 : 0.0;
        }
    }
    __syncthreads();
    const int kb = 16 * w >= H ? H : 0;  // the wave's half
    d4 acc[4][1];
    contract<NJ>(acc, tile + kb, a.B1 + kb * NP, 16 * w + li, li, lk);
    const double w0 = a.w0[16 * w + li], wN = a.wN[16 * w + li];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * rb + 4 * r + lk;
            acc[rb][0][r] += fma(row_zl[row], w0, row_zr[row] * wN);
        }
    __syncthreads();  // every wave has read the folded tile
    to_corr<NJ>(acc, tile, w, li, lk);
    __syncthreads();
    correct<NJ>(acc, tile, a.C1, a.X1, w, li, lk);
    const int jc = compact<H>(16 * w + li, he, ho);
    if (jc < 0) return;
    double x[16];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[4 * rb + r] = acc[rb][0][r];
    double2 *t = reinterpret_cast<double2 *>(a.T) + jc * 8 * a.ncol + c0 + lk;
    real_dft16(x, [&](int s, double re, double im) { t[s * a.ncol] = make_double2(re, im); });
}

// ---- 3: 16-point stage back, correction, contraction, store --------------------
// zf_expand's mirror image and bounds; 256^2 x 129: 140 MB in 54 us, matrix cores
// busy 34% of the SIMD cycles, 16 bytes a lane in scratch.
template <int NJ>
__device__ __forceinline__ void collect_tile(const ZfArgs &a, int c0, int tid, EndLds<NJ> &lds)
{
    constexpr int NP = 16 * NJ, LD = NP + 2, H = NP / 2, T = 64 * NJ;
    double *tile = lds.tile;
    const int lane = tid % 64, w = uniform(tid / 64), li = lane % 16, lk = lane / 16;
    const int n = a.n, ho = n / 2, he = n - ho;
    const int jc = compact<H>(16 * w + li, he, ho);
    d4 acc[4][1];
    {
        double x[16], re[8], im[8];
        const double2 *t = reinterpret_cast<const double2 *>(a.T) + (jc < 0 ? 0 : jc) * 8 * a.ncol + c0 + lk;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const double2 v = t[s * a.ncol];
            re[s] = jc < 0 ? 0.0 : v.x;
            im[s] = jc < 0 ? 0.0 : v.y;
        }
        real_idft16(re, im, x);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[rb][0][r] = x[4 * rb + r];
    }
    to_corr<NJ>(acc, tile, w, li, lk);
    __syncthreads();
    correct<NJ>(acc, tile, a.C2, a.X2, w, li, lk);
    __syncthreads();  // every wave has read the uncorrected values
    to_tile<NJ>(acc, tile, w, li, lk);
    __syncthreads();
    const int kb = 16 * w >= H ? H : 0;
    contract<NJ>(acc, tile + kb, a.B2 + kb * NP, 16 * w + li, li, lk);
    __syncthreads();
    to_tile<NJ>(acc, tile, w, li, lk);
    __syncthreads();
    // u_i = e_i + o_i, u_(n-1-i) = e_i - o_i, the centre of an odd n e_i; the
    // end values are the faces'
    for (int idx = tid; idx < kRows * NP; idx += T) {
        const int row = idx / NP, k = idx % NP;
        if (k >= n) continue;
        const RowAt at(row, c0, a.lr2);
        const int i = k < n - 1 - k ? k : n - 1 - k;
        const double e = tile[row * LD + i];
        const double o = 2 * k + 1 == n ? 0.0 : tile[row * LD + H + i];
        a.u[(at.x * a.ny + at.y) * a.K + 1 + k] = k <= n - 1 - k ? e + o : e - o;
    }
    if (tid < 2 * kRows) {
        const int row = tid >> 1, side = tid & 1;
        const RowAt at(row, c0, a.lr2);
        const int g = at.x * a.ny + at.y, end = g * a.K + (side ? n + 1 : 0);
        a.u[end] = side ? a.gr[g] / a.beta_r : a.gl[g] / a.beta_l;
    }
}

template <int NJ, bool CUB>
__global__ __launch_bounds__(64 * NJ, 4) void zf_expand(const ZfArgs a)
{
    __shared__ EndLds<NJ> lds;
    expand_tile<NJ, CUB>(a, 4 * xcd_logical(blockIdx.x, gridDim.x), threadIdx.x, lds);
}

template <int NJ>
__global__ __launch_bounds__(64 * NJ, NJ == 6 ? 3 : 4) void zf_collect(const ZfArgs a)
{
    __shared__ EndLds<NJ> lds;
    collect_tile<NJ>(a, 4 * xcd_logical(blockIdx.x, gridDim.x), threadIdx.x, lds);
}

// Many problems: one (problem, tile) entry per work-group (generic loads would
// cost the filter 100 registers).
__device__ __forceinline__ ZfArgs problem_args(const ZfArgs *__restrict__ Z, int p)
{
    ZfArgs a = Z[p];
    a.nx = uniform(a.nx);
    a.ny = uniform(a.ny);
    a.n = uniform(a.n);
    a.K = uniform(a.K);
    a.lr2 = uniform(a.lr2);
    a.ncol = uniform(a.ncol);
    a.f = as_global(a.f);
    a.u = as_global(a.u);
    a.gl = as_global(a.gl);
    a.gr = as_global(a.gr);
    a.T = as_global(a.T);
    a.B1 = as_global(a.B1);
    a.B2 = as_global(a.B2);
    a.C1 = as_global(a.C1);
    a.C2 = as_global(a.C2);
    a.X1 = as_global(a.X1);
    a.X2 = as_global(a.X2);
    a.w0 = as_global(a.w0);
    a.wN = as_global(a.wN);
    a.mu = as_global(a.mu);
    a.sx = as_global(a.sx);
    a.sy = as_global(a.sy);
    a.twx = as_global(a.twx);
    a.twy = as_global(a.twy);
    return a;
}

// Tiles of a work-group of 512 threads: as many as its threads and the LDS of
// one of the widest hold.
__host__ __device__ constexpr int end_tiles(int NJ) { return NJ >= 6 ? 1 : NJ == 4 ? 2 : 3; }

template <int NJ, bool COLLECT>
__device__ __forceinline__ void end_tiles_of(const ZfArgs &a, int task, char *smem)
{
    asm volatile("" ::: "memory");  // nothing of one size's body is formed ahead of the choice
    constexpr int T = 64 * NJ, PER = end_tiles(NJ);
    const int sub = uniform(threadIdx.x / T), t = task * PER + sub;
    if (sub >= PER || 4 * t >= a.ncol) return;  // waves that ended take no part in the barriers
    EndLds<NJ> &lds = reinterpret_cast<EndLds<NJ> *>(smem)[sub];
    if constexpr (COLLECT)
        collect_tile<NJ>(a, 4 * t, threadIdx.x % T, lds);
    else
        expand_tile<NJ, false>(a, 4 * t, threadIdx.x % T, lds);
}

// Every problem of a batch in one launch: its tasks of different sizes fill the
// chip together, where a launch per size leaves most of it idle for the 10 to
// 20 us that one work-group takes (64 problems, 317 MB: expand 130 us against
// 147 in four launches, collect 140 against 169).  32 bytes a lane in scratch.
template <bool COLLECT>
__global__ __launch_bounds__(512, 4) void zf_end_list(const ZfArgs *__restrict__ Z, const int2 *__restrict__ list)
{
    __shared__ alignas(16) char smem[2 * sizeof(EndLds<4>)];
    static_assert(sizeof(smem) >= sizeof(EndLds<8>) && sizeof(smem) >= end_tiles(2) * sizeof(EndLds<2>),
                  "every size fits");
    const int2 e = list[xcd_logical(blockIdx.x, gridDim.x)];
    const ZfArgs a = problem_args(Z, uniform(e.x));
    const int task = uniform(e.y);
    switch ((a.n + 31) / 32) {
    case 1: end_tiles_of<2, COLLECT>(a, task, smem); break;
    case 2: end_tiles_of<4, COLLECT>(a, task, smem); break;
    case 3: end_tiles_of<6, COLLECT>(a, task, smem); break;
    default: end_tiles_of<8, COLLECT>(a, task, smem); break;
    }
}

// ---- 2: the rest of the transforms and the filter ------------------------------
// One (j, k1) block of NX x R2 points per group of threads, 16 points per
// thread in every stage: x in two register stages (NX = RA RB), the remaining
// R2 points along y in a third, exchanged through LDS (real parts, then
// imaginary parts; rows of R2 padded by one so that a thread's read of a row
// is conflict free).  Bound by memory: 256^2 x 129 134 MB in 38 us, the three
// passes that it replaces (two along y with the mode solve's read and write
// between them) moved 270 MB.
template <int NX, int R2>
struct Filter {
    static constexpr int RA = NX >= 128 ? 16 : 8, RB = NX / RA;
    static constexpr int NY = 16 * R2, CH = NX * R2;  // points of a block
    static constexpr int T = CH >= 4096 ? 256 : CH >= 2048 ? 128 : 64;
    static constexpr int NCH = 16 * T / CH;           // blocks per work-group
    static constexpr int LR = R2 + 1;
    // 16-point stages along y in both directions take 162 registers: bounded to
    // 128 they spill 144 bytes a thread (45 us against 38 at 256^2 x 129); the
    // others fit but for 28 bytes of 64 x 128's
    static constexpr int WAVES = R2 == 16 ? 3 : 4;
    static constexpr int LDS = NCH * NX * LR;         // doubles
    static_assert(NCH >= 1, "a block fits a work-group");
};

template <int NX, int R2>
__device__ __forceinline__ void filter_tile(const ZfArgs &a, int wg, double *tile)
{
    using S = Filter<NX, R2>;
    constexpr int RA = S::RA, RB = S::RB, NY = S::NY, CH = S::CH, T = S::T, NCH = S::NCH, LR = S::LR;
    const int tid = threadIdx.x;
    const int tasks = 9 * a.n;
    // item -> its block in the work-group (of IPB items each) and the rest
    auto block_of = [](int it, int ipb) { return NCH == 1 ? 0 : it / ipb; };
    // task -> (j, k1): k1 = 0 and 8 (the halves of slot 0) next to each other
    auto slot_of = [](int sub) { return sub < 2 ? 8 * sub : sub - 1; };
    double re[16], im[16];
    constexpr int LA = 16 / RA, LC = 16 / R2;

    // ---- load, x stage 1: item (block, q, n2), points x = q + RB n1 ----
#pragma unroll
    for (int l = 0; l < LA; ++l) {
        const int it = tid + T * l, ch = block_of(it, RB * R2), rem = it - ch * (RB * R2);
        const int task = wg * NCH + ch, j = task / 9, k1 = slot_of(task % 9);
        const double2 *src = reinterpret_cast<const double2 *>(a.T) + ((long long)j * 8 + (k1 & 7)) * CH + rem;
#pragma unroll
        for (int n1 = 0; n1 < RA; ++n1) {
            double2 v = make_double2(0.0, 0.0);
            if (task < tasks) v = src[n1 * RB * R2];
            re[l * RA + n1] = k1 == 8 ? v.y : v.x;
            im[l * RA + n1] = (k1 & 7) ? v.y : 0.0;
        }
    }
    auto stage = [&](auto rc, auto lc, auto sign, const double2 *tw, auto body) {
        constexpr int R = decltype(rc)::value, L = decltype(lc)::value, SIGN = decltype(sign)::value;
#pragma unroll
        for (int l = 0; l < 16 / R; ++l) {
            double r[R], i[R];
#pragma unroll
            for (int k = 0; k < R; ++k) {
                r[k] = re[l * R + k];
                i[k] = im[l * R + k];
            }
            body(l, r, i, [&] { dft_regs<R, L, SIGN>(r, i, tw); });
#pragma unroll
            for (int k = 0; k < R; ++k) {
                re[l * R + k] = r[k];
                im[l * R + k] = i[k];
            }
        }
    };
    // exchange: element e of item l goes to tile[to(l, e)], then is read from tile[from(l, e)]
    auto exchange = [&](auto to, auto from) {
#pragma unroll
        for (int k = 0; k < 16; ++k) tile[to(k)] = re[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) re[k] = tile[from(k)];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) tile[to(k)] = im[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) im[k] = tile[from(k)];
        __syncthreads();
    };
    typedef std::integral_constant<int, -1> Fwd;
    typedef std::integral_constant<int, 1> Inv;
    typedef std::integral_constant<int, NX> LX;
    // tile position of (stage-1 item element), (stage-2 ..), (kx of a stage-2
    // item element), (stage-3 ..)
    auto posA = [&](int k) {  // item (ch, q, n2), element k1x
        const int it = tid + T * (k / RA), ch = block_of(it, RB * R2), rem = it - ch * (RB * R2);
        return (ch * NX + (k % RA) * RB + rem / R2) * LR + rem % R2;
    };
    auto posB = [&](int k) {  // item (ch, k1x, n2), element q
        const int it = tid + T * (k / RB), ch = block_of(it, RA * R2), rem = it - ch * (RA * R2);
        return (ch * NX + (rem / R2) * RB + k % RB) * LR + rem % R2;
    };
    auto posK = [&](int k) {  // item (ch, k1x, n2), element k2x: kx = k1x + RA k2x
        const int it = tid + T * (k / RB), ch = block_of(it, RA * R2), rem = it - ch * (RA * R2);
        return (ch * NX + rem / R2 + RA * (k % RB)) * LR + rem % R2;
    };
    auto posC = [&](int k) {  // item (ch, kx), element n2
        const int it = tid + T * (k / R2);
        return it * LR + k % R2;
    };

    stage(std::integral_constant<int, RA>{}, LX{}, Fwd{}, a.twx, [&](int l, auto &r, auto &i, auto dft) {
        TwiddlePowers<RA, NX> t;
        t.load(a.twx, (tid + T * l) % (RB * R2) / R2);
        dft();
        t.template apply<-1>(r, i);
    });
    exchange(posA, posB);
    stage(std::integral_constant<int, RB>{}, LX{}, Fwd{}, a.twx, [&](int, auto &, auto &, auto dft) { dft(); });
    exchange(posK, posC);
    // ---- the remaining points along y, the filter, and back ----
#pragma unroll
    for (int l = 0; l < LC; ++l) {
        const int it = tid + T * l, ch = block_of(it, NX), kx = it - ch * NX;
        const int task = min(wg * NCH + ch, tasks - 1), j = task / 9, k1 = slot_of(task % 9);
        double r[R2], i[R2];
#pragma unroll
        for (int k = 0; k < R2; ++k) {
            r[k] = re[l * R2 + k];
            i[k] = im[l * R2 + k];
        }
        TwiddlePowers<R2, NY> t;
        t.load(a.twy, k1);
        t.template apply<-1>(r, i);
        dft_regs<R2, NY, -1>(r, i, a.twy);
        const double mu = a.mu[j], sx = a.sx[kx <= NX / 2 ? kx : NX - kx];
#pragma unroll
        for (int k = 0; k < R2; ++k) {
            const int ky = k1 + 16 * k;
            const double sig = sx + a.sy[ky <= NY / 2 ? ky : NY - ky];
            const double m = (1.0 / ((double)NX * NY)) / (mu - sig);
            r[k] *= m;
            i[k] *= m;
        }
        dft_regs<R2, NY, 1>(r, i, a.twy);
        t.load(a.twy, k1);  // formed again: kept, the powers would cost 32 registers
        t.template apply<1>(r, i);
#pragma unroll
        for (int k = 0; k < R2; ++k) {
            re[l * R2 + k] = r[k];
            im[l * R2 + k] = i[k];
        }
    }
    exchange(posC, posK);
    stage(std::integral_constant<int, RB>{}, LX{}, Inv{}, a.twx, [&](int, auto &, auto &, auto dft) { dft(); });
    exchange(posB, posA);
#pragma unroll
    for (int l = 0; l < LA; ++l) {
        const int it = tid + T * l, ch = block_of(it, RB * R2), rem = it - ch * (RB * R2);
        const int task = wg * NCH + ch, j = task / 9, k1 = slot_of(task % 9);
        double r[RA], i[RA];
#pragma unroll
        for (int k = 0; k < RA; ++k) {
            r[k] = re[l * RA + k];
            i[k] = im[l * RA + k];
        }
        TwiddlePowers<RA, NX> t;
        t.load(a.twx, rem / R2);
        t.template apply<1>(r, i);
        dft_regs<RA, NX, 1>(r, i, a.twx);
        if (task >= tasks) continue;
        double2 *dst = reinterpret_cast<double2 *>(a.T) + ((long long)j * 8 + (k1 & 7)) * CH + rem;
        if (k1 & 7) {
#pragma unroll
            for (int n1 = 0; n1 < RA; ++n1) dst[n1 * RB * R2] = make_double2(r[n1], i[n1]);
        } else {  // a real sequence: its half of the packed slot
            double *d = reinterpret_cast<double *>(dst) + (k1 >> 3);
#pragma unroll
            for (int n1 = 0; n1 < RA; ++n1) d[2 * n1 * RB * R2] = r[n1];
        }
    }
}

template <int NX, int R2>
__global__ __launch_bounds__((Filter<NX, R2>::T), (Filter<NX, R2>::WAVES)) void zf_filter(const ZfArgs a)
{
    __shared__ double tile[Filter<NX, R2>::LDS];
    filter_tile<NX, R2>(a, xcd_logical(blockIdx.x, gridDim.x), tile);
}

template <int NX, int R2>
__device__ __forceinline__ void filter_of(const ZfArgs &a, int task, double *tile)
{
    asm volatile("" ::: "memory");  // nothing of one grid's body is formed ahead of the choice
    filter_tile<NX, R2>(a, task, tile);
}

// The grids of a batch whose work-groups are one wave (R2 < 16), one launch: 73
// us for 64 problems (317 MB) against 157 in nine; bounded to 128 registers it
// spills and takes 117.
constexpr int kFilterLds = 16 * 32 * 3;  // doubles: 32 x 2 pads most
__global__ __launch_bounds__(64, 3) void zf_filter_list64(const ZfArgs *__restrict__ Z, const int2 *__restrict__ list)
{
    __shared__ double tile[kFilterLds];
    const int2 e = list[xcd_logical(blockIdx.x, gridDim.x)];
    const ZfArgs a = problem_args(Z, uniform(e.x));
    const int task = uniform(e.y);
    switch (a.nx * 1024 + a.ny) {
    case 32 * 1024 + 32: filter_of<32, 2>(a, task, tile); break;
    case 32 * 1024 + 64: filter_of<32, 4>(a, task, tile); break;
    case 32 * 1024 + 128: filter_of<32, 8>(a, task, tile); break;
    case 64 * 1024 + 32: filter_of<64, 2>(a, task, tile); break;
    case 64 * 1024 + 64: filter_of<64, 4>(a, task, tile); break;
    case 64 * 1024 + 128: filter_of<64, 8>(a, task, tile); break;
    case 128 * 1024 + 32: filter_of<128, 2>(a, task, tile); break;
    case 128 * 1024 + 64: filter_of<128, 4>(a, task, tile); break;
    case 128 * 1024 + 128: filter_of<128, 8>(a, task, tile); break;
    case 256 * 1024 + 32: filter_of<256, 2>(a, task, tile); break;
    default: filter_of<256, 4>(a, task, tile); break;
    }
}

// A larger grid of a batch (32 x 256 keeps 48 bytes a lane in scratch).
template <int NX, int R2>
__global__ __launch_bounds__((Filter<NX, R2>::T), (Filter<NX, R2>::WAVES)) void zf_filter_list(
    const ZfArgs *__restrict__ Z, const int2 *__restrict__ list)
{
    __shared__ double tile[Filter<NX, R2>::LDS];
    const int2 e = list[xcd_logical(blockIdx.x, gridDim.x)];
    filter_tile<NX, R2>(problem_args(Z, uniform(e.x)), uniform(e.y), tile);
}

template <int NJ>
int launch_ends(const ZfArgs &a, bool collect, hipStream_t s)
{
    const dim3 grid(a.ncol / 4), block(64 * NJ);
    if (collect)
        hipLaunchKernelGGL(zf_collect<NJ>, grid, block, 0, s, a);
    else if (a.cubic)
        hipLaunchKernelGGL((zf_expand<NJ, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((zf_expand<NJ, false>), grid, block, 0, s, a);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

int launch_ends(const ZfArgs &a, bool collect, hipStream_t s)
{
    switch (diag_padded(a.n)) {
    case 32: return launch_ends<2>(a, collect, s);
    case 64: return launch_ends<4>(a, collect, s);
    case 96: return launch_ends<6>(a, collect, s);
    default: return launch_ends<8>(a, collect, s);
    }
}

template <int NX, int R2>
int launch_filter_t(const ZfArgs &a, hipStream_t s)
{
    using S = Filter<NX, R2>;
    hipLaunchKernelGGL((zf_filter<NX, R2>), dim3((9 * a.n + S::NCH - 1) / S::NCH), dim3(S::T), 0, s, a);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

// The grids of zf_holds.
int launch_filter(const ZfArgs &a, hipStream_t s)
{
    switch (a.nx * 1024 + a.ny) {
    case 64 * 1024 + 128: return launch_filter_t<64, 8>(a, s);
    case 64 * 1024 + 256: return launch_filter_t<64, 16>(a, s);
    case 128 * 1024 + 64: return launch_filter_t<128, 4>(a, s);
    case 128 * 1024 + 128: return launch_filter_t<128, 8>(a, s);
    case 128 * 1024 + 256: return launch_filter_t<128, 16>(a, s);
    case 256 * 1024 + 32: return launch_filter_t<256, 2>(a, s);
    case 256 * 1024 + 64: return launch_filter_t<256, 4>(a, s);
    case 256 * 1024 + 128: return launch_filter_t<256, 8>(a, s);
    default: return launch_filter_t<256, 16>(a, s);
    }
}

}  // namespace

// Three launches instead of five, but few work-groups on a small grid: an end
// kernel has nx ny / 64, each 10 to 16 us from its first load to its last store
// (N = 130), against the transform passes' many short ones.  Measured, us a
// solve, here against transform - mode solve - transform: 64 x 64 x 130 38.5 |
// 33.8, 32 x 256 x 130 49.2 | 47.6; 128 x 64 x 18 21.7 | 20.9, x 66 29.8 | 30.7,
// x 130 45.7 | 47.9; 64 x 128 x 66 32.0 | 30.5, x 99 44.2 | 42.6, x 130 47.7 |
// 48.2; 64 x 256 x 18 23.3 | 25.0, x 130 50.7 | 65.0; 256^2 x 3 26.6 | 32.9, x 67
// 112 | 108, x 98 128 | 131, x 130 135 | 164.  N - 2 > 128 would need end kernels
// of 256 eigen-indices and a larger FP64 block of the correction, a 512-point
// axis filter blocks of 1,024 threads and 135 KB of LDS (512 x 32 points).
bool zf_holds(int nx, int ny, int n)
{
    if (nx < 64 || nx > 256 || ny < 32 || ny > 256 || n < 1 || n > 128) return false;
    return nx * ny >= 16384 || (nx * ny >= 8192 && n >= 64);
}

bool zf_fits(int nx, int ny, int n)
{
    return nx >= 32 && nx <= 256 && ny >= 32 && ny <= 256 && n >= 1 && n <= 128;
}

int zf_kind(int nx, int ny, int n, int stage)
{
    const int grid = nx * 1024 + ny;
    return stage != 1 || (nx * ny <= 16384 && ny < 256) ? 0 : grid;
}

int zf_tasks(int nx, int ny, int n, int stage)
{
    if (stage != 1) {
        const int per = end_tiles(diag_padded(n) / 16);
        return (nx * ny / 64 + per - 1) / per;
    }
    const int points = nx * ny / 16, blocks = points >= 1024 ? 1 : 1024 / points;  // Filter::CH, NCH
    return (9 * n + blocks - 1) / blocks;
}

template <int NX, int R2>
static void launch_filter_list(const ZfArgs *Z, const int2 *list, int count, hipStream_t s)
{
    hipLaunchKernelGGL((zf_filter_list<NX, R2>), dim3(count), dim3(Filter<NX, R2>::T), 0, s, Z, list);
}

int launch_zf_list(const ZfArgs *Z, const int2 *list, int count, int stage, int kind, hipStream_t s)
{
    if (stage == 0)
        hipLaunchKernelGGL(zf_end_list<false>, dim3(count), dim3(512), 0, s, Z, list);
    else if (stage == 2)
        hipLaunchKernelGGL(zf_end_list<true>, dim3(count), dim3(512), 0, s, Z, list);
    else
        switch (kind) {
        case 0: hipLaunchKernelGGL(zf_filter_list64, dim3(count), dim3(64), 0, s, Z, list); break;
        case 32 * 1024 + 256: launch_filter_list<32, 16>(Z, list, count, s); break;
        case 64 * 1024 + 256: launch_filter_list<64, 16>(Z, list, count, s); break;
        case 128 * 1024 + 256: launch_filter_list<128, 16>(Z, list, count, s); break;
        case 256 * 1024 + 128: launch_filter_list<256, 8>(Z, list, count, s); break;
        default: launch_filter_list<256, 16>(Z, list, count, s); break;
        }
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

int launch_zf(const ZfArgs &a, int stage, hipStream_t s)
{
    if (!zf_holds(a.nx, a.ny, a.n)) return set_error(HZ_ERR_UNSUPPORTED, "z-first solve: size out of range");
    return stage == 1 ? launch_filter(a, s) : launch_ends(a, stage == 2, s);
}

}  // namespace hz
