// diag_waves_body.h -- the tile of diag_waves.hip (scheme there), also run over
// the problems of a batch.
#pragma once

#include "diag_body.h"

namespace hz {
namespace {

__device__ __forceinline__ double row16_sum(double v)
{
    v += dpp_f64<kDppXor1>(v);
    v += dpp_f64<kDppXor2>(v);
    v += dpp_f64<kDppHalfMirror>(v);
    return v + dpp_f64<kDppMirror>(v);
}

// Tile `bx` (16 RB WR rows); 64 NJ WR threads.
template <int NJ, int WR, int RB, bool ADJ>
__device__ __forceinline__ void diag_waves_tile(const DiagArgs &a, int bx)
{
    constexpr int NC = 16 * NJ, RT = 16 * RB * WR, T = 64 * NJ * WR, LD = NC + 2;
    constexpr int SB = NJ == 1 ? 32 : NC;  // the operands' row stride
    __shared__ alignas(16) double tile[RT * LD];
    __shared__ double row_sig[RT], row_zl[RT], row_zr[RT], row_d0[RT], row_dN[RT], part[2][NJ][RT];
    __shared__ double row_u0[ADJ ? RT : 1], row_uN[ADJ ? RT : 1];
    __shared__ long long row_col[RT];
    const int tid = threadIdx.x, lane = tid % WAVE, w = uniform(tid / WAVE), li = lane % 16, lk = lane / 16;
    const int wc = w % NJ, r0 = (w / NJ) * RB;  // the wave's column tile and first row block
    const int n = a.n, N = a.N, E = a.ne, K = a.K, M = a.M;
    const int rows_per_fc = 2 * E, fc_per_tile = RT / rows_per_fc, fc0 = bx * fc_per_tile, nfc = a.nx * M;
    const int j = 16 * wc + li;
    const bool jv = j < n;
    auto row_of = [&](int rb, int r) { return 16 * (r0 + rb) + 4 * r + lk; };
    auto mode_of = [&](int fc) {
        const int i = fc / M;
        return (i <= a.nx / 2 ? i : a.nx - i) * M + fc % M;
    };

    for (int row = tid; row < RT; row += T) {  // row = (fc_local * 2 + plane) * E + e
        const int fl = row / rows_per_fc, rem = row % rows_per_fc, plane = rem / E, e = rem % E, fc = fc0 + fl;
        const bool used = fl < fc_per_tile && fc < nfc;
        row_col[row] = used ? (long long)(fc / M) * a.xs + (long long)(fc % M) * K + (long long)e * (N - 1) +
                                  (plane ? a.plane_off : 0)
                            : -1;
    }
    __syncthreads();
    double v[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long long col = row_col[row_of(rb, r)];
            v[rb][r] = col >= 0 && jv ? a.spec[col + 1 + j] : 0.0;
        }
    // the real column of this thread's interface system
    const int fcs = fc0 + (tid >> 1);
    const bool sweeps = tid < 2 * fc_per_tile && fcs < nfc;
    double L0 = 0.0, LN = 0.0, R0 = 0.0, RN = 0.0, gl = 0.0, gr = 0.0;
    if (sweeps) {
        const double *h = a.hom + 4 * (long long)mode_of(fcs);
        L0 = h[0];
        LN = h[1];
        R0 = h[2];
        RN = h[3];
        if (!ADJ && !a.periodic) {
            const double *bsrc = tid & 1 ? a.bc_im : a.bc_re;
            gl = bsrc[fcs];
            gr = bsrc[(long long)nfc + fcs];
        }
    }
    const double mu = jv ? a.mu[j] : 0.0, w0 = jv ? a.w0[j] : 0.0, wN = jv ? a.wN[j] : 0.0;
    const double e0 = jv ? a.r0[j] : 0.0, eN = jv ? a.rN[j] : 0.0;
    for (int row = tid; row < RT; row += T) {
        const long long col = row_col[row];
        row_sig[row] = col >= 0 ? a.shift[mode_of(fc0 + row / rows_per_fc)] : 0.0;
        if constexpr (ADJ) {
            row_u0[row] = col >= 0 ? a.spec[col] : 0.0;
            row_uN[row] = col >= 0 ? a.spec[col + N - 1] : 0.0;
        }
        row_zl[row] = 0.0;
        row_zr[row] = 0.0;
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) tile[row_of(rb, r) * LD + j] = v[rb][r];
    __syncthreads();

    d4 acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb] = d4{0.0, 0.0, 0.0, 0.0};
    pair_gemm<NC, LD, RB, SB>(acc, tile + 16 * r0 * LD, a.VinvT, j, li, lk);
    // q = y / (mu - sigma) and its dots (end-point derivatives; the adjoint
    // load on the end values)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row_of(rb, r);
            v[rb][r] = jv ? 1.0 / (mu - row_sig[row]) : 0.0;  // now the reciprocals
            const double q = acc[rb][r] * v[rb][r];
            const double s0 = row16_sum((ADJ ? w0 : e0) * q), sN = row16_sum((ADJ ? wN : eN) * q);
            if (li == 0) {
                part[0][wc][row] = s0;
                part[1][wc][row] = sN;
            }
        }
    __syncthreads();
    auto sum_row = [&](int row) {
        double s0 = part[0][0][row], sN = part[1][0][row];
#pragma unroll
        for (int c = 1; c < NJ; ++c) {
            s0 += part[0][c][row];
            sN += part[1][c][row];
        }
        row_d0[row] = s0;
        row_dN[row] = sN;
    };
    if (E == 1) {
        if (sweeps) sum_row(tid);  // the only row of this thread's column
    } else {
        for (int row = tid; row < RT; row += T) sum_row(row);
        __syncthreads();
    }
    if (sweeps) {
        const int rw = tid * E;  // the column's element rows
        double *d0 = row_d0 + rw, *dN = row_dN + rw, *zl = row_zl + rw, *zr = row_zr + rw;
        if constexpr (!ADJ) {
            if (a.periodic)
                periodic_sweep(E, L0, LN, R0, RN, d0, dN, zl, zr, 1,
                               a.closure ? a.closure + (tid & 1 ? nfc : 0) + fcs : nullptr);
            else
                robin_sweep(E, L0, LN, R0, RN, gl, gr, a.alpha_l, a.beta_l, a.alpha_r, a.beta_r, d0, dN, zl, zr);
        } else if (a.periodic && E > 1) {
            periodic_sweep_adjoint(E, L0, LN, R0, RN, row_u0 + rw, row_uN + rw, d0, dN, zl, zr);
        } else if (a.periodic) {
            // u_0 = u_{N-1} = z = (dN - d0) / bp: zbar collects both end values
            // and the load through ul + ur; d0bar = -zbar / bp, dNbar = zbar / bp
            const double bp = (L0 + R0) - (LN + RN);
            const double zb = (row_u0[rw] + row_uN[rw]) + (d0[0] + dN[0]);
            zl[0] = -zb / bp;
            zr[0] = zb / bp;
        } else {
            double *gre = tid & 1 ? a.gbar_im : a.gbar_re;
            double glb, grb;
            if (E == 1) {
                const double b = -a.alpha_l * L0 + a.beta_l, c = -a.alpha_l * R0;
                const double lb = a.alpha_r * LN;
                const double br = a.alpha_r * RN + a.beta_r - (c / b) * lb;
                const double zlb = row_u0[rw] + d0[0];
                const double zrb = row_uN[rw] + dN[0] - (c / b) * zlb;
                grb = zrb / br;
                glb = zlb / b - (lb / b) * grb;
                zl[0] = a.alpha_l * glb;  // the adjoints of the end-point derivatives
                zr[0] = -a.alpha_r * grb;
            } else {
                robin_sweep_adjoint(E, L0, LN, R0, RN, a.alpha_l, a.beta_l, a.alpha_r, a.beta_r, row_u0 + rw,
                                    row_uN + rw, d0, dN, zl, zr, &glb, &grb);
            }
            gre[fcs] = glb;
            gre[(long long)nfc + fcs] = grb;
        }
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row_of(rb, r);
            const double h = fma(row_zl[row], ADJ ? e0 : w0, row_zr[row] * (ADJ ? eN : wN));
            tile[row * LD + j] = (acc[rb][r] + h) * v[rb][r];
        }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb] = d4{0.0, 0.0, 0.0, 0.0};
    pair_gemm<NC, LD, RB, SB>(acc, tile + 16 * r0 * LD, a.VT, j, li, lk);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long long col = row_col[row_of(rb, r)];
            if (col >= 0 && jv) a.spec[col + 1 + j] = acc[rb][r];
        }
    // element end values (the adjoint load has none)
    for (int row = tid; row < RT; row += T) {
        const long long col = row_col[row];
        if (col < 0) continue;
        a.spec[col] = ADJ ? 0.0 : row_zl[row];
        a.spec[col + N - 1] = ADJ ? 0.0 : row_zr[row];
    }
}

}  // namespace
}  // namespace hz
