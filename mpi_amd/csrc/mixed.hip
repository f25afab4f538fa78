// mixed.hip -- the MIXED form's mode solve: FP32 matrix-core solves in the
// plan's eigenbasis refined with FP64 matrix-core residuals.  Launch
// wrappers around the tile body in mixed_body.h (scheme described there),
// and the plan-time kernel of the FP64 homogeneous solutions.
#include "mixed_body.h"

namespace hz {
namespace {

// Plan time (once per lambda): ul = V (w0 / (mu - sigma)), ur = V (wN / (mu -
// sigma)) of every mode (NonPeriodic3D_MPI.cpp:203-222 through the
// eigendecomposition), interior values, FP64.
__global__ __launch_bounds__(256) void mixed_homogeneous_kernel(const MixedSetupArgs a)
{
    __shared__ double inv[256];
    const int m = blockIdx.x, tid = threadIdx.x;
    const int n = a.n, NP = a.NP;
    const double sig = a.shift[m];
    for (int k = tid; k < NP; k += 256) inv[k] = k < n ? 1.0 / (a.mu[k] - sig) : 0.0;
    __syncthreads();
    for (int i = tid; i < n; i += 256) {
        double ul = 0.0, ur = 0.0;
        for (int k = 0; k < n; ++k) {
            const double v = a.VT[(long long)k * NP + i] * inv[k];
            ul = fma(v, a.w0[k], ul);
            ur = fma(v, a.wN[k], ur);
        }
        a.UL[(long long)m * n + i] = ul;
        a.UR[(long long)m * n + i] = ur;
    }
}

template <int NJ, int RT, bool GENERAL>
__global__ __launch_bounds__(256, 2) void mixed_modes_kernel(const MixedArgs a)
{
    __shared__ MixedShared<NJ, RT, GENERAL> sh;
    mixed_tile<NJ, RT, GENERAL>(a, blockIdx.x, sh);
}

// The mode solve for N - 2 <= 128, one wave per 16 columns of the padded
// interior (mixed_tile: four waves for all of them), 16 RB rows.
//
// A wave holds its columns of both FP32 operands in registers for all sweeps,
// and right-hand side, 1 / (mu - sigma) and row maxima in the accumulators'
// layout: the FP32 products take their rows permuted (lane row i reads tile
// row 4 (i % 4) + i / 4), which makes their result layout the FP64 one.  The
// products' k order is dealt to the lanes so that each reads the operands of
// four (FP64: two) steps in one 16-byte LDS access.  FP32 right-hand sides lie
// in the tile as the fold's two halves (entry i < n / 2 of the front at i, its
// mirror image at H + i), so that the fold is one addition as the first product
// reads them and a sweep has four barriers.  Only Dzz is read again every
// sweep, from L2.
//
// Bound by the matrix cores: 256^2 x 129 (two sweeps) has 104 us of matrix
// instructions and takes 202 (mixed_tile 313); the two work-groups that share a
// CU keep them busy for two thirds of the time, and 2,064 work-groups leave 16
// for a fifth round.

template <int NJ, int RB, bool GENERAL>
__global__ __launch_bounds__(64 * NJ, NJ == 6 && GENERAL ? 3 : 4) void mixed_waves_kernel(const MixedArgs a)
{
    constexpr int NP = 16 * NJ, H = NP / 2, RT = 16 * RB, T = 64 * NJ, KS = H / 4;
    constexpr int LD = NP + 2, LDF = NP + 4;      // conflict-free row strides
    __shared__ alignas(16) double x[RT * LD];     // the iterate
    __shared__ alignas(16) float t[RT * LDF];     // FP32 right-hand sides, then the folded solution
    __shared__ alignas(16) float z[RT * LDF];     // scaled eigen coordinates
    __shared__ double row_sig[RT], row_zl[RT], row_zr[RT];
    __shared__ long long row_col[RT];
    __shared__ float bmax[NJ][RT], rmax[NJ][RT];
    __shared__ double part[GENERAL ? 2 : 1][GENERAL ? NJ : 1][GENERAL ? RT : 1], row_d[GENERAL ? 2 : 1][GENERAL ? RT : 1];
    const int tid = threadIdx.x, lane = tid % WAVE, w = uniform(tid / WAVE), li = lane % 16, lk = lane / 16;
    const int n = a.n, N = a.N, E = a.ne, K = a.K, M = a.M;
    const int rows_per_fc = 2 * E, fc_per_tile = RT / rows_per_fc, fc0 = blockIdx.x * fc_per_tile, nfc = a.nx * M;
    const int j = 16 * w + li;                // the lane's column
    const int kb = 16 * w >= H ? H : 0;       // the wave's half

    for (int row = tid; row < RT; row += T) {  // row = (fc_local * 2 + plane) * E + e
        const int fl = row / rows_per_fc, rem = row % rows_per_fc, plane = rem / E, e = rem % E, fc = fc0 + fl;
        const bool used = fl < fc_per_tile && fc < nfc;
        row_col[row] = used ? (long long)(fc / M) * a.xs + (long long)(fc % M) * K + (long long)e * (N - 1) +
                                  (plane ? a.plane_off : 0)
                            : -1;
    }
    __syncthreads();
    // every load of the tile in flight before any is waited for
    auto row_of = [&](int rb, int r) { return 16 * rb + 4 * r + lk; };
    double b[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long long col = row_col[row_of(rb, r)];
            b[rb][r] = col >= 0 && j < n ? a.spec[col + 1 + j] : 0.0;
        }
    for (int row = tid; row < RT; row += T) {
        const int fc = fc0 + row / rows_per_fc;
        double sig = 0.0, zl = 0.0, zr = 0.0;
        if (row_col[row] >= 0) {
            const int i = fc / M, m = fc % M;
            sig = a.shift[(i <= a.nx / 2 ? i : a.nx - i) * M + m];
            if (!GENERAL) {  // one element, Dirichlet data on both faces
                const double *bsrc = row & 1 ? a.bc_im : a.bc_re;
                zl = bsrc[fc] / a.beta_l;
                zr = bsrc[(long long)nfc + fc] / a.beta_r;
            }
        }
        row_sig[row] = sig;
        row_zl[row] = zl;
        row_zr[row] = zr;
    }
    float b1[KS], b2[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int k = 16 * (ks / 4) + 4 * lk + ks % 4;
        b1[ks] = a.VinvT32[(kb + k) * NP + j];
        b2[ks] = a.VT32[(kb + k) * NP + j];
    }
    double f0 = 0.0, fN = 0.0;
    if (!GENERAL && j < n) {
        f0 = a.Dzz[(long long)(j + 1) * N];
        fN = a.Dzz[(long long)(j + 1) * N + N - 1];
    }
    const bool jv = j < H ? j < n - n / 2 : j - H < n / 2;
    const double mu = jv ? a.mu[j] : 0.0;
    // the lane's place among the fold's halves (columns past n zero the halves' unused ends)
    const int ho = n / 2, he = n - ho, q = j - n;
    const int fj = j < he ? j : j < n ? H + n - 1 - j : q < H - he ? he + q : H + ho + q - (H - he);
    __syncthreads();

    // largest |v| of each row over the wave's columns
    auto row_max = [&](float (&out)[NJ][RT], const float (&v)[RB][4]) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float m = fabsf(v[rb][r]);
                m = fmaxf(m, __int_as_float(dpp_i32<kDppXor1>(__float_as_int(m))));
                m = fmaxf(m, __int_as_float(dpp_i32<kDppXor2>(__float_as_int(m))));
                m = fmaxf(m, __int_as_float(dpp_i32<kDppHalfMirror>(__float_as_int(m))));
                m = fmaxf(m, __int_as_float(dpp_i32<kDppMirror>(__float_as_int(m))));
                if (li == 0) out[w][row_of(rb, r)] = m;
            }
    };
    float iv[RB][4];
    {
        float f[RB][4];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row_of(rb, r);
                if constexpr (!GENERAL) b[rb][r] = b[rb][r] - f0 * row_zl[row] - fN * row_zr[row];
                f[rb][r] = (float)b[rb][r];
                t[row * LDF + fj] = f[rb][r];
                iv[rb][r] = jv ? (float)(1.0 / (mu - row_sig[row])) : 0.0f;
            }
        if (a.hist) row_max(bmax, f);
    }
    __syncthreads();

    // x += (first: =) the FP32 solve of t
    const int prow = 4 * (li % 4) + li / 4;
    auto fp32_solve = [&](bool first) {
        f4 c[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) c[rb] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        const float sg = kb ? -1.0f : 1.0f;
#pragma unroll
        for (int k4 = 0; k4 < KS / 4; ++k4)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const float *tr = t + (16 * rb + prow) * LDF + 16 * k4 + 4 * lk;
                const f4 v = *reinterpret_cast<const f4 *>(tr), m = *reinterpret_cast<const f4 *>(tr + H);
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    c[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fmaf(sg, m[h], v[h]), b1[4 * k4 + h], c[rb], 0, 0, 0);
            }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) z[row_of(rb, r) * LDF + j] = c[rb][r] * iv[rb][r];
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) c[rb] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k4 = 0; k4 < KS / 4; ++k4)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const f4 v = *reinterpret_cast<const f4 *>(z + (16 * rb + prow) * LDF + kb + 16 * k4 + 4 * lk);
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    c[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[h], b2[4 * k4 + h], c[rb], 0, 0, 0);
            }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) t[row_of(rb, r) * LDF + j] = c[rb][r];
        __syncthreads();
        // unfold: x_i = e_i + o_i, x_(n-1-i) = e_i - o_i, the centre of an odd n e_i
        const int i = max(j < n - 1 - j ? j : n - 1 - j, 0);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row_of(rb, r);
                const float e = t[row * LDF + i], o = 2 * j + 1 == n ? 0.0f : t[row * LDF + H + i];
                const double d = j < n ? (double)(j <= n - 1 - j ? e + o : e - o) : 0.0;
                double &xv = x[row * LD + j];
                xv = first ? d : xv + d;
            }
        __syncthreads();
    };
    fp32_solve(true);

    for (int s = 0; s < a.sweeps; ++s) {
        const double *dzz = a.DzzTP;
        asm volatile("" : "+s"(dzz));  // read every sweep: hoisted out of the loop, it would take 64 registers
        d4 acc[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb] = d4{0.0, 0.0, 0.0, 0.0};
        pair_gemm<NP, LD, RB>(acc, x, dzz, j, li, lk);
        float f[RB][4];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row_of(rb, r);
                const double rv = b[rb][r] - acc[rb][r] + row_sig[row] * x[row * LD + j];
                f[rb][r] = j < n ? (float)rv : 0.0f;
                t[row * LDF + fj] = f[rb][r];
            }
        if (a.hist) row_max(rmax, f);
        __syncthreads();
        if (a.hist)
            for (int row = tid; row < RT; row += T) {
                if (row_col[row] < 0) continue;
                float bm = 0.0f, rm = 0.0f;
#pragma unroll
                for (int c = 0; c < NJ; ++c) {
                    bm = fmaxf(bm, bmax[c][row]);
                    rm = fmaxf(rm, rmax[c][row]);
                }
                a.hist[(long long)s * a.hist_rows + (long long)fc0 * rows_per_fc + row] =
                    bm > 0.0f ? (double)rm / (double)bm : 0.0;
            }
        fp32_solve(false);
    }

    if constexpr (GENERAL) {
        // end-point derivatives of the particular solutions (zero end values)
        const double d0 = j < n ? a.Dz[1 + j] : 0.0, dN = j < n ? a.Dz[(long long)(N - 1) * N + 1 + j] : 0.0;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double xv = x[row_of(rb, r) * LD + j];
                double s0 = d0 * xv, sN = dN * xv;
#pragma unroll
                for (int o = 1; o < 16; o <<= 1) {
                    s0 += __shfl_xor(s0, o);
                    sN += __shfl_xor(sN, o);
                }
                if (li == 0) {
                    part[0][w][row_of(rb, r)] = s0;
                    part[1][w][row_of(rb, r)] = sN;
                }
            }
        __syncthreads();
        for (int q = tid; q < 2 * RT; q += T) {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < NJ; ++c) s += part[q / RT][c][q % RT];
            row_d[q / RT][q % RT] = s;
        }
        __syncthreads();
        for (int sc = tid; sc < 2 * fc_per_tile; sc += T) {
            const int plane = sc & 1, fc = fc0 + (sc >> 1);
            if (fc >= nfc) continue;
            const int i = fc / M, m = fc % M, mode = (i <= a.nx / 2 ? i : a.nx - i) * M + m;
            const double d0ul = a.hom[4 * mode + 0], dNul = a.hom[4 * mode + 1];
            const double d0ur = a.hom[4 * mode + 2], dNur = a.hom[4 * mode + 3];
            const int r0w = sc * E;
            if (a.periodic) {
                periodic_sweep(E, d0ul, dNul, d0ur, dNur, row_d[0] + r0w, row_d[1] + r0w, row_zl + r0w,
                               row_zr + r0w, 1, a.closure ? a.closure + (plane ? nfc : 0) + fc : nullptr);
                continue;
            }
            const double *bsrc = plane ? a.bc_im : a.bc_re;
            robin_sweep(E, d0ul, dNul, d0ur, dNur, bsrc[fc], bsrc[(long long)nfc + fc], a.alpha_l, a.beta_l,
                        a.alpha_r, a.beta_r, row_d[0] + r0w, row_d[1] + r0w, row_zl + r0w, row_zr + r0w);
        }
        __syncthreads();
    }

    // u along z: x (+ zl ul + zr ur with several elements or Robin faces)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row_of(rb, r);
            const long long col = row_col[row];
            if (col < 0 || j >= n) continue;
            double v = x[row * LD + j];
            if constexpr (GENERAL) {
                const int fc = fc0 + row / rows_per_fc, i = fc / M, m = fc % M;
                const int mode = (i <= a.nx / 2 ? i : a.nx - i) * M + m;
                v = v + (row_zl[row] * a.UL[(long long)mode * n + j] + row_zr[row] * a.UR[(long long)mode * n + j]);
            }
            a.spec[col + 1 + j] = v;
        }
    for (int row = tid; row < RT; row += T) {
        const long long col = row_col[row];
        if (col >= 0) {
            a.spec[col] = row_zl[row];
            a.spec[col + N - 1] = row_zr[row];
        }
    }
}

bool is_general(const MixedArgs &a)
{
    return a.ne > 1 || a.alpha_l != 0.0 || a.alpha_r != 0.0 || a.periodic;
}

// WAVES: mixed_waves_kernel, else mixed_modes_kernel.
template <int NJ, int RT, bool WAVES>
int launch_t(const MixedArgs &a, hipStream_t s)
{
    const int fc_per_tile = RT / (2 * a.ne);
    if (fc_per_tile < 1) return set_error(HZ_ERR_UNSUPPORTED, "MIXED form: too many elements for one tile");
    const int blocks = (a.nx * a.M + fc_per_tile - 1) / fc_per_tile;
    if constexpr (WAVES) {
        if (is_general(a))
            hipLaunchKernelGGL((mixed_waves_kernel<NJ, RT / 16, true>), dim3(blocks), dim3(64 * NJ), 0, s, a);
        else
            hipLaunchKernelGGL((mixed_waves_kernel<NJ, RT / 16, false>), dim3(blocks), dim3(64 * NJ), 0, s, a);
    } else {
        if (is_general(a))
            hipLaunchKernelGGL((mixed_modes_kernel<NJ, RT, true>), dim3(blocks), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((mixed_modes_kernel<NJ, RT, false>), dim3(blocks), dim3(256), 0, s, a);
    }
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

}  // namespace

int mixed_tile_rows(int NP)
{
    // NP = 32, 96 split the row blocks between wave pairs: an even number of
    // 16-row blocks
    return (NP == 32 || NP == 96) ? 32 : 16;
}

int launch_mixed_setup(const MixedSetupArgs &a, hipStream_t s)
{
    if (a.modes <= 0) return HZ_OK;
    hipLaunchKernelGGL(mixed_homogeneous_kernel, dim3(a.modes), dim3(256), 0, s, a);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

int launch_mixed_modes(const MixedArgs &a, hipStream_t s)
{
    // one wave per 16 columns to N - 2 = 128 (us a solve, against mixed_tile's:
    // 256^2 x 18 68 | 79, x 66 117 | 152, x 130 272 | 374; 128^2, 4 x 33 87 | 95;
    // Robin 128^2 x 129 120 | 157); above, its operands would take 128 registers
    switch (diag_padded(a.n)) {
    case 32: return launch_t<2, 32, true>(a, s);
    case 64: return launch_t<4, 32, true>(a, s);
    case 96: return launch_t<6, 32, true>(a, s);
    case 128: return launch_t<8, 32, true>(a, s);
    case 256: return launch_t<16, 16, false>(a, s);
    default: return set_error(HZ_ERR_UNSUPPORTED, "MIXED form: N-2 must be <= 256");
    }
}

}  // namespace hz
