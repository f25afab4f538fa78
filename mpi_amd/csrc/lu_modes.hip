// lu_modes.hip -- the reference algorithm per (|kx|,|ky|) mode: one
// work-group factors a mode's operator, solves its right-hand sides and
// writes the assembled columns.
//
// For mode (iw, jw) the work-group
//   1. assembles A = Dzz_int - sigma I (or the caller's operator) and the
//      right-hand sides: the two homogeneous ones (-Dzz[1..N-2][0],
//      -Dzz[1..N-2][N-1], NonPeriodic3D_MPI.cpp:211-219) and the interior
//      spectrum of every element for each real column of the mode
//      (:188-201, :248-325);
//   2. eliminates with the reference's pivot rule (LU_Decomposition.cpp:7-72):
//      the candidate at position i is |a_ik| / s_i where s_i is the max-norm
//      of the ORIGINAL row at position i (the scale is never exchanged with
//      the rows), the strictly-greater test makes the first maximum in
//      position order win, and |scaled pivot| <= 1e-12 is singular.
//      Carrying the right-hand sides through the elimination is LUSolve's
//      forward phase (:86-95);
//   3. back-substitutes the right-hand sides (:97-107);
//   4. forms the end-point derivatives Dz[0|N-1].col (GLLQuadrature.cpp:234-245),
//      runs the element-interface sweep with the Robin end rows
//      (NonPeriodic3D_MPI.cpp:327-580) and assembles u = p + zl ul + zr ur
//      (:582-587) straight into the spectrum.
//
// Exchanges are implicit -- rows never move, every row carries its current
// position -- and exact (the reference's a+b-b exchange arithmetic is a
// rounding-level difference; the standalone factor kernels keep it).
//
// Layout (RT row tiles of 16, RT waves): wave w owns the 16 matrix columns of
// panel w as RT 16 x 16 tiles in the accumulator layout of
// v_mfma_f64_16x16x4f64 (D[i][j] in lane j + 16 (i % 4), element i / 4).  The
// right-hand sides stay in LDS.  Panel p's wave brings its tiles up to date,
// turns them into one row per lane through LDS and eliminates the 16 columns
// by itself: no hand-off between waves inside a panel, where a step is a
// search (DPP on 32-bit keys), a division and the update of the columns to
// its right.  It leaves the multipliers in LDS as matrix-core operands, and
// every later wave applies the 16 steps at once: the pivot rows' values of
// its columns (gathered through LDS), a 16-step triangular solve per column,
// and a rank-16 update of its tiles on the matrix cores.  The wave of panel
// p + 1 does so first and goes straight on to its own panel while the others
// update.  Back substitution runs by panels the same way.  Row tiles whose
// rows are all eliminated are skipped.
//
// What bounds it: the chain of pivot steps (each needs the one before), about
// 1,600 cycles a step of 128 rows, not the arithmetic.  Against the kernel
// that hands every pivot from wave to wave (lu.hip; mode kernel, us, on
// 256^2 unless given): N - 2 = 7: 146 -> 103, 15: 260 -> 123, 31: 546 -> 305,
// 48: 1,042 -> 828, 63: 1,339 -> 1,127; 64 x 32 with 25 elements of 10 points
// 78 -> 35, 128^2 with 8 of 17 243 -> 64, 64^2 with 4 of 33 88 -> 42.
// Above 64 rows a work-group needs 8 waves of 179 registers, one per CU, and
// the other kernel is the faster (127 rows: 5.7 ms against 8.2 and more):
// launch_lu_modes sends N - 2 > 64 there, and small operators of few modes
// (stepwise).  The instance of 8 tiles serves a caller who pins the largest
// shape for a small operator.
#include "hz_internal.h"
#include "sweep.h"
#include "wave_ops.h"

namespace hz {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr double kEps = 1.000000000000E-12;  // include/General.h:15

__host__ __device__ __forceinline__ int rhs_per_element(int nx) { return nx >= 4 ? 4 : 2; }

// LDS of one work-group, in doubles from the start of the dynamic block.
template <int RT>
struct Lds {
    static constexpr int ROWS = 16 * RT;
    // column stride of the panel buffers and of the right-hand sides: 2 mod 4
    // doubles, so that the accumulator layout's 16 columns x 2 rows of a
    // half-wave fall on different banks
    static constexpr int LD = ROWS + 2;
    static constexpr int B = 0;                          // [2][16][LD] panel / multipliers / U panel
    static constexpr int L11 = B + 2 * 16 * LD;          // [2][16][16] the pivot rows' multipliers (or U11)
    static constexpr int U = L11 + 2 * 256;              // [RT - 1][16][16] a wave's pivot rows
    static constexpr int SCL = U + (RT > 1 ? RT - 1 : 1) * 256;  // [ROWS] scale of the row's position
    static constexpr int MASK = SCL + ROWS;              // [2][4] u64: pivot rows, rows not yet eliminated
    static constexpr int POS = MASK + 8;                 // [ROWS] short: position of a row
    static constexpr int PHYS = POS + ROWS / 4;          // [ROWS] short: row at a position
    static constexpr int FLAG = PHYS + ROWS / 4;         // int: singular
    static constexpr int Y = FLAG + 2;                   // [nrhs][LD]
    // after the back substitution B is free: the interface system's arrays
    static size_t bytes(int nrhs) { return sizeof(double) * ((size_t)Y + (size_t)nrhs * LD); }
};

// v is computed here and later loads stay below: without it the compiler
// defers a triangular solve's arithmetic to where its result is stored, with
// all 120 operands loaded and live until there.
__device__ __forceinline__ void pin(double &v) { asm volatile("" : "+v"(v)::"memory"); }

// 64-bit value v[p] of a register array at a uniform slot p < RB.
template <int RB>
__device__ __forceinline__ double slot_value(double v0, double v1, int slot)
{
    if constexpr (RB == 1) return v0;
    return slot ? v1 : v0;
}

// Column j of row slot a of a panel wave's registers, once they hold one row
// per lane.
#define HZ_P(a, j) R[4 * (a) + (j) / 4][(j) % 4]

template <int RT>
struct ModeLu {
    static constexpr int ROWS = 16 * RT, LD = Lds<RT>::LD, RB = (ROWS + 63) / 64;
    static constexpr int ND = RT > 4 ? RT : 4;  // d4 registers of a panel: RT tiles, or 16 columns of RB rows

    double *sm;
    int n, np, nrhs, lane, li, lk, w;
    d4 R[ND];  // this wave's panel w: tiles until it is eliminated, then one row per lane

    __device__ __forceinline__ double *buf(int par) const { return sm + Lds<RT>::B + par * 16 * LD; }
    __device__ __forceinline__ double *l11(int par) const { return sm + Lds<RT>::L11 + par * 256; }
    __device__ __forceinline__ double *y(int r) const { return sm + Lds<RT>::Y + r * LD; }
    __device__ __forceinline__ short *pos() const { return reinterpret_cast<short *>(sm + Lds<RT>::POS); }
    __device__ __forceinline__ short *phys() const { return reinterpret_cast<short *>(sm + Lds<RT>::PHYS); }
    __device__ __forceinline__ unsigned long long *mask(int par) const
    {
        return reinterpret_cast<unsigned long long *>(sm + Lds<RT>::MASK) + 4 * par;
    }
    __device__ __forceinline__ int *flag() const { return reinterpret_cast<int *>(sm + Lds<RT>::FLAG); }

    // ---- pivot search -------------------------------------------------------
    // The reference's ratios compared exactly, over the rows `cand`: the
    // maximum, the first position winning a tie.
    __device__ __forceinline__ void search_exact(const double (&col)[RB], const int (&ps)[RB], const double (&scl)[RB],
                                                 const bool (&cand)[RB], int &wl, int &ws, double &g)
    {
        double best = -2.0;
        int bpos = 0x7fffffff, bslot = 0;
#pragma unroll
        for (int a = 0; a < RB; ++a) {
            if (cand[a]) {
                double ratio = fabs(col[a]) / scl[a];
                if (!(ratio >= 0.0)) ratio = -1.0;  // NaN: lowest priority
                if (ratio > best || (ratio == best && ps[a] < bpos)) {
                    best = ratio;
                    bpos = ps[a];
                    bslot = a;
                }
            }
        }
        g = wave_max_f64(best);
        const bool top = best == g;
        const int mp = wave_min_i32(top ? bpos : 0x7fffffff);
        wl = __builtin_ctzll(__ballot(top && bpos == mp));
        ws = __builtin_amdgcn_readlane(bslot, wl);
    }

    // ---- a panel's 16 pivot steps on one row per lane -------------------------
    __device__ __forceinline__ void factor(int p)
    {
        double *lb = buf(p & 1);
        // tiles -> columns in LDS -> one row per lane
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) lb[li * LD + 16 * t + 4 * r + lk] = R[t][r];
        wave_sync();
        const bool lv = RT >= 4 || lane < ROWS;
#pragma unroll
        for (int a = 0; a < RB; ++a)
#pragma unroll
            for (int j = 0; j < 16; ++j) HZ_P(a, j) = lv ? lb[j * LD + lane + 64 * a] : 0.0;
        wave_sync();
        int ps[RB];
        double scl[RB], isc[RB];
        bool plain = true;  // every scale's reciprocal is an ordinary number
        unsigned long long unpiv[2] = {0, 0};
#pragma unroll
        for (int a = 0; a < RB; ++a) {
            const int row = lane + 64 * a;
            ps[a] = lv && row < n ? pos()[row] : -1;
            scl[a] = lv && row < n ? sm[Lds<RT>::SCL + row] : 1.0;
            isc[a] = 1.0 / scl[a];
            plain = plain && scl[a] < 0x1p1000 && scl[a] > 0x1p-1000;
            unpiv[a] = __ballot(ps[a] >= 16 * p);
        }
        const bool exact = __ballot(plain) != ~0ull;
        // Four steps at a time with the pivot column in a fixed register; after
        // them the columns rotate left by four (the finished ones to the end),
        // so the code of a step exists four times, not sixteen.
#pragma nounroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int kk = 4 * g + s, k = 16 * p + kk;
                double l[RB];
#pragma unroll
                for (int a = 0; a < RB; ++a) l[a] = 0.0;
                if (k < n - 1) {
                    double col[RB];
                    bool cand[RB];
                    int key[RB], kl = -1;
#pragma unroll
                    for (int a = 0; a < RB; ++a) {
                        col[a] = HZ_P(a, s);
                        // upper word of |a| (1/s), within one unit of the exact
                        // ratio's; a NaN's is as large as any and is settled below
                        key[a] = ps[a] >= k ? __double2hiint(fabs(col[a]) * isc[a]) & 0x7fffffff : -1;
                        kl = max(kl, key[a]);
                    }
                    const int km = wave_max_i32(kl);
                    int count = 0, wl = 0, ws = 0;
#pragma unroll
                    for (int a = 0; a < RB; ++a) {
                        cand[a] = key[a] >= km - 1;
                        const unsigned long long mk = __ballot(cand[a]);
                        count += __popcll(mk);
                        if (mk) {
                            wl = __builtin_ctzll(mk);
                            ws = a;
                        }
                    }
                    // one candidate, clearly above the singular test's 1e-12 and
                    // finite: the pivot; otherwise the exact ratios decide
                    if (exact || count != 1 || km < 0x3d800000 || km >= 0x7ff00000) {
                        double gm;
#pragma unroll
                        for (int a = 0; a < RB; ++a)
                            cand[a] = ps[a] >= k && (cand[a] || exact || km >= 0x7ff00000);
                        search_exact(col, ps, scl, cand, wl, ws, gm);
                        if (gm <= kEps && lane == 0) *flag() = 1;  // includes a NaN column (-1)
                    }
                    wl = uniform(wl);
                    ws = uniform(ws);
                    const double piv = lane_f64(slot_value<RB>(col[0], col[RB - 1], ws), wl);
                    const int ppos = __builtin_amdgcn_readlane(RB == 1 || !ws ? ps[0] : ps[RB - 1], wl);
                    // the pivot row takes position k, the row it displaces its position and scale
                    const double sp = lane_f64(slot_value<RB>(scl[0], scl[RB - 1], ws), wl);
                    const double ip = lane_f64(slot_value<RB>(isc[0], isc[RB - 1], ws), wl);
#pragma unroll
                    for (int a = 0; a < RB; ++a) {
                        const bool isp = RB == 1 ? lane == wl : lane == wl && ws == a;
                        const bool mv = ps[a] == k;
                        ps[a] = isp ? k : mv ? ppos : ps[a];
                        scl[a] = mv ? sp : scl[a];
                        isc[a] = mv ? ip : isc[a];
                    }
                    divide(col, piv, l);
#pragma unroll
                    for (int a = 0; a < RB; ++a) {
                        const bool act = ps[a] > k;
                        HZ_P(a, s) = act ? l[a] : col[a];
                        l[a] = act ? l[a] : 0.0;
                    }
                    if (RB == 1 || ws == 0)
                        update_columns<0>(l, wl, s, g);
                    else
                        update_columns<RB - 1>(l, wl, s, g);
                }
                if (lv) {
#pragma unroll
                    for (int a = 0; a < RB; ++a) lb[kk * LD + lane + 64 * a] = l[a];
                }
            }
#pragma unroll
            for (int a = 0; a < RB; ++a) {
                const d4 first = R[4 * a];
                R[4 * a] = R[4 * a + 1];
                R[4 * a + 1] = R[4 * a + 2];
                R[4 * a + 2] = R[4 * a + 3];
                R[4 * a + 3] = first;
            }
        }
        // the pivot rows' multipliers, the rows' positions and scales, the masks
        // (the last position of all is the last row's, not tested by the reference)
        fill16(l11(p & 1), 0.0);
        wave_sync();
        unsigned long long pm[2] = {0, 0};
#pragma unroll
        for (int a = 0; a < RB; ++a) {
            const int row = lane + 64 * a, q = ps[a] - 16 * p;
            pm[a] = __ballot(q >= 0 && q < 16);
            if (q >= 0 && q < 16) {
                phys()[ps[a]] = (short)row;
#pragma unroll
                for (int j = 0; j < 16; ++j) l11(p & 1)[q * 16 + j] = HZ_P(a, j);
            }
            if (lv && row < n) {
                pos()[row] = (short)ps[a];
                sm[Lds<RT>::SCL + row] = scl[a];
            }
        }
        if (lane == 0) {
            mask(p & 1)[0] = pm[0];
            mask(p & 1)[1] = pm[1];
            mask(p & 1)[2] = unpiv[0];
            mask(p & 1)[3] = unpiv[1];
        }
    }

    // l = col / piv.  piv is the same in every lane, so its reciprocal is
    // refined once and each quotient gets one residual correction (as the
    // division's own last steps); extreme pivots take the division.
    __device__ __forceinline__ void divide(const double (&col)[RB], double piv, double (&l)[RB]) const
    {
        const double ap = fabs(piv);
        if (ap > 0x1p-500 && ap < 0x1p500) {  // uniform
            double r = __builtin_amdgcn_rcp(piv);
            r = fma(fma(-piv, r, 1.0), r, r);
            r = fma(fma(-piv, r, 1.0), r, r);
#pragma unroll
            for (int a = 0; a < RB; ++a) {
                const double q = col[a] * r;
                l[a] = fma(fma(-q, piv, col[a]), r, q);
            }
        } else {
#pragma unroll
            for (int a = 0; a < RB; ++a) l[a] = col[a] / piv;
        }
    }

    // Columns right of s: minus l times the pivot row's (lane wl of row slot WS).
    template <int WS>
    __device__ __forceinline__ void update_columns(const double (&l)[RB], int wl, int s, int g)
    {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c < 4 - g) {  // uniform: the rest are finished columns
#pragma unroll
                for (int j = 4 * c; j < 4 * c + 4; ++j) {
                    if (j <= s) continue;
                    const double pv = lane_f64(HZ_P(WS, j), wl);
#pragma unroll
                    for (int a = 0; a < RB; ++a) HZ_P(a, j) = fma(-l[a], pv, HZ_P(a, j));
                }
            }
        }
    }

    // u = L11^-1 u for one column of 16 values (a lane's), L11 unit lower
    // (zero rows past the last panel's end)
    __device__ __forceinline__ void lower_solve(double (&u)[16], const double *L) const
    {
#pragma unroll
        for (int q = 1; q < 16; ++q) {
#pragma unroll
            for (int j = 0; j < q; ++j) u[q] = fma(-L[q * 16 + j], u[j], u[q]);
            pin(u[q]);
        }
    }

    // u = U11^-1 u, U11 upper (identity past the last panel's end)
    __device__ __forceinline__ void upper_solve(double (&u)[16], const double *U) const
    {
#pragma unroll
        for (int q = 15; q >= 0; --q) {
            u[q] = u[q] / U[q * 16 + q];
#pragma unroll
            for (int j = 0; j < q; ++j) u[j] = fma(-U[j * 16 + q], u[q], u[j]);
            pin(u[q]);
        }
    }

    // the rows of panel p's 16 positions, for a lane's right-hand side
    __device__ __forceinline__ void panel_values(int p, const double *yc, double (&u)[16]) const
    {
#pragma unroll
        for (int q = 0; q < 16; ++q) u[q] = yc[phys()[16 * p + q]];
    }

    // an all-zero or identity 16 x 16 block
    __device__ __forceinline__ void fill16(double *blk, double diag) const
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) blk[lane + 64 * i] = lane % 16 == (lane + 64 * i) / 16 ? diag : 0.0;
    }

    // -u[4 s + lk]: the matrix-core operand B[k][j] (k = 4 s + lk) of a lane's column
    __device__ __forceinline__ void operand(const double (&u)[16], double (&b)[4]) const
    {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double lo = lk & 1 ? u[4 * s + 1] : u[4 * s], hi = lk & 1 ? u[4 * s + 3] : u[4 * s + 2];
            b[s] = -(lk & 2 ? hi : lo);
        }
    }

    // a 64-bit mask word, uniform
    __device__ __forceinline__ static unsigned long long uword(unsigned long long v)
    {
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
        const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
        return ((unsigned long long)hi << 32) | lo;
    }

    // acc -= L(panel) u over row tile t
    __device__ __forceinline__ d4 rank16(d4 acc, const double *lb, const double (&b)[4], int t) const
    {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(lb[(4 * s + lk) * LD + 16 * t + li], b[s], acc, 0, 0, 0);
        return acc;
    }

    // ---- panel p's steps applied to this wave's tiles (w > p) -----------------
    __device__ __forceinline__ void update_tiles(int p)
    {
        const double *lb = buf(p & 1);
        double *ub = sm + Lds<RT>::U + (w - 1) * 256;
        const unsigned long long pm[2] = {uword(mask(p & 1)[0]), uword(mask(p & 1)[1])};
        const unsigned long long un[2] = {uword(mask(p & 1)[2]), uword(mask(p & 1)[3])};
        // the pivot rows' values of these columns: groups of four rows (one
        // accumulator element) that hold one
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row0 = 16 * t + 4 * r;
                const unsigned nib = (unsigned)(pm[row0 / 64] >> (row0 % 64)) & 15u;
                if (nib) {  // uniform
                    if ((nib >> lk) & 1) {
                        const int q = pos()[row0 + lk] - 16 * p;
                        ub[q * 16 + li] = R[t][r];
                    }
                }
            }
        wave_sync();
        double u[16], b[4];
#pragma unroll
        for (int q = 0; q < 16; ++q) u[q] = ub[q * 16 + li];
        wave_sync();
        lower_solve(u, l11(p & 1));
        operand(u, b);
#pragma unroll
        for (int t = 0; t < RT; ++t)
            if ((un[t / 4] >> (16 * t % 64)) & 0xffff) R[t] = rank16(R[t], lb, b, t);
    }

    // ---- panel p's steps applied to the right-hand sides 64 c .. 64 c + 63 ----
    // One right-hand side per lane for the pivot rows' solve, then the rows
    // still to be eliminated on the matrix cores, 16 right-hand sides at a time.
    __device__ __forceinline__ void update_rhs(int p, int c)
    {
        const double *lb = buf(p & 1);
        {
            const int r0 = 64 * c + lane;
            const bool lv = r0 < nrhs;
            double *yc = y(lv ? r0 : 0);
            double u[16];
            panel_values(p, yc, u);
            lower_solve(u, l11(p & 1));
            if (lv) {
#pragma unroll
                for (int q = 1; q < 16; ++q) yc[phys()[16 * p + q]] = u[q];
            }
        }
        wave_sync();
        const unsigned long long rest[2] = {uword(mask(p & 1)[2] & ~mask(p & 1)[0]),
                                            uword(mask(p & 1)[3] & ~mask(p & 1)[1])};
        if (!(rest[0] | rest[1])) return;
#pragma nounroll
        for (int c4 = 4 * c; c4 < 4 * c + 4 && 16 * c4 < nrhs; ++c4) {
            const int r0 = 16 * c4 + li;
            const bool lv = r0 < nrhs;
            double *yc = y(lv ? r0 : 0);
            double b[4];
            rhs_operand(p, yc, b);
#pragma unroll
            for (int t = 0; t < RT; ++t)
                if ((rest[t / 4] >> (16 * t % 64)) & 0xffff) update_rhs_tile(lb, b, yc, lv, t, 16 * p + 15, n);
        }
        wave_sync();
    }

    // -y of panel p's pivot rows as the matrix-core operand B[k][j]
    __device__ __forceinline__ void rhs_operand(int p, const double *yc, double (&b)[4]) const
    {
#pragma unroll
        for (int s = 0; s < 4; ++s) b[s] = -yc[phys()[16 * p + 4 * s + lk]];
    }

    // Row tile t of the right-hand sides minus lb b, in the rows at positions
    // in (lo, hi) only.
    __device__ __forceinline__ void update_rhs_tile(const double *lb, const double (&b)[4], double *yc, bool lv, int t,
                                                    int lo, int hi)
    {
        d4 acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = yc[16 * t + 4 * r + lk];
        acc = rank16(acc, lb, b, t);
        if (lv) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * t + 4 * r + lk;
                const int ps = row < n ? pos()[row] : hi;
                if (ps > lo && ps < hi) yc[row] = acc[r];
            }
        }
    }

    // ---- elimination of the matrix and the right-hand sides -------------------
    __device__ __forceinline__ void eliminate()
    {
#pragma nounroll
        for (int p = 0; p <= np; ++p) {
            if (p > 0 && w >= p && w < np) update_tiles(p - 1);
            if (w == p && p < np) factor(p);
            if (p > 0) {
#pragma nounroll
                for (int c = w; 64 * c < nrhs; c += RT) update_rhs(p - 1, c);
            }
            __syncthreads();
        }
    }

    // U11 of panel p and its columns above
    __device__ __forceinline__ void store_upper(int p, double *ub, double *U11) const
    {
        fill16(U11, 1.0);
        wave_sync();
#pragma unroll
        for (int a = 0; a < RB; ++a) {
            const int row = lane + 64 * a;
            const int q = (row < n ? pos()[row] : 0x7fff) - 16 * p;
            if (row < ROWS && p > 0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) ub[j * LD + row] = q < 0 ? HZ_P(a, j) : 0.0;
            }
            if (q >= 0 && q < 16) {
#pragma unroll
                for (int j = 0; j < 16; ++j) U11[q * 16 + j] = HZ_P(a, j);
            }
        }
    }

    // ---- back substitution -----------------------------------------------------
    // Panel p from the last: its wave writes U11 (the pivot rows) and the
    // columns above (zero in the other rows); the waves that hold right-hand
    // sides solve with U11, one right-hand side per lane; every wave subtracts
    // its row tile's product.
    __device__ __forceinline__ void back_substitute()
    {
#pragma nounroll
        for (int p = np - 1; p >= 0; --p) {
            double *ub = buf(p & 1), *U11 = l11(p & 1);
            if (w == p) store_upper(p, ub, U11);
            __syncthreads();
#pragma nounroll
            for (int c = w; 64 * c < nrhs; c += RT) {
                const int r0 = 64 * c + lane;
                const bool lv = r0 < nrhs;
                double *yc = y(lv ? r0 : 0);
                double u[16];
                panel_values(p, yc, u);
                upper_solve(u, U11);
                if (lv) {
#pragma unroll
                    for (int q = 0; q < 16; ++q) yc[phys()[16 * p + q]] = u[q];
                }
            }
            __syncthreads();
            if (p > 0) {
                if (w < np) {
#pragma nounroll
                    for (int c = 0; 16 * c < nrhs; ++c) {
                        const int r0 = 16 * c + li;
                        const bool lv = r0 < nrhs;
                        double *yc = y(lv ? r0 : 0);
                        double b[4];
                        rhs_operand(p, yc, b);
                        update_rhs_tile(ub, b, yc, lv, w, -1, 16 * p);
                    }
                }
                __syncthreads();
            }
        }
    }
};

template <int RT>
constexpr int lu_modes_min_waves() { return RT == 8 ? 2 : 3; }

// ---------------------------------------------------------------------------
template <int RT>
__global__ __launch_bounds__(64 * RT, (lu_modes_min_waves<RT>())) void lu_modes_kernel(const LuModeArgs a)
{
    extern __shared__ double sm[];
    using S = Lds<RT>;
    constexpr int ROWS = S::ROWS, T = 64 * RT;
    ModeLu<RT> m;
    m.sm = sm;
    m.lane = threadIdx.x % 64;
    m.w = uniform(threadIdx.x / 64);
    m.li = m.lane % 16;
    m.lk = m.lane / 16;
    m.n = a.n;
    m.np = (a.n + 15) / 16;
    const int w = m.w, n = a.n, N = a.N, E = a.ne, K = a.K, M = a.M;
    const int mode = blockIdx.x;
    const int iw = mode / M, jw = mode % M;
    const int xi0 = iw, xi1 = a.nx - iw, nxi = (iw != 0 && iw != a.nx / 2) ? 2 : 1;
    const int nc = 2 * nxi;
    const int CPE = rhs_per_element(a.nx);  // right-hand sides per element
    const int nrhs = 2 + CPE * E;
    m.nrhs = nrhs;

    // ---- assemble (row i = position i) ----
    const double sig = a.shift ? a.shift[mode] : 0.0;
    {
        // the operator's columns 16 w .. 16 w + 15, a row stride of ld
        const double *op = a.op_full ? a.op_full + (long long)mode * n * n : a.Dzz + N + 1;
        const int ld = a.op_full ? n : N, j = 16 * w + m.li;
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * t + 4 * r + m.lk;
                m.R[t][r] = i < n && j < n ? op[i * ld + j] : 0.0;
            }
        if (!a.op_full) {  // the diagonal: less the shift, or the caller's
            const double d = a.op_diag ? a.op_diag[(long long)mode * n + (j < n ? j : 0)] : 0.0;
#pragma unroll
            for (int t = 0; t < RT; ++t)
                if (t == w) {  // uniform
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (m.li == 4 * r + m.lk && j < n) m.R[t][r] = a.op_diag ? d : m.R[t][r] - sig;
                }
        }
    }
    for (int i = threadIdx.x; i < ROWS; i += T) {
        // s by position (positions start as the rows), LU_Decomposition.cpp:20-29:
        // the operator's off-diagonal maximum is the plan's, only the diagonal is the mode's
        double s = 0.0;
        if (i < n) {
            if (a.op_full) {
                for (int j = 0; j < n; ++j) s = fmax(s, fabs(a.op_full[((long long)mode * n + i) * n + j]));
            } else {
                const double d = a.op_diag ? a.op_diag[(long long)mode * n + i]
                                           : a.Dzz[(long long)(i + 1) * N + i + 1] - sig;
                s = fmax(a.offmax[i], fabs(d));
            }
        }
        sm[S::SCL + i] = s;
        m.pos()[i] = (short)i;
        m.phys()[i] = (short)i;
    }
    if (threadIdx.x == 0) *m.flag() = 0;
    {
        constexpr int UL = 4;  // loads in flight per thread
        const int total = nrhs * ROWS;
#pragma nounroll
        for (int i0 = threadIdx.x; i0 < total; i0 += UL * T) {
            double v[UL];
#pragma unroll
            for (int u = 0; u < UL; ++u) {
                const int idx = i0 + u * T, r = idx / ROWS, i = idx % ROWS;
                v[u] = 0.0;
                if (idx < total && i < n) {
                    const int e = (r - 2) / CPE, cc = (r - 2) % CPE;
                    if (r < 2)
                        v[u] = -a.Dzz[(long long)(i + 1) * N + (r ? N - 1 : 0)];
                    else if (cc < nc)
                        v[u] = ((cc & 1) ? a.spec_im : a.spec_re)[(long long)((cc >> 1) ? xi1 : xi0) * a.xs +
                                                                  (long long)jw * K + (long long)e * (N - 1) + 1 + i];
                }
            }
#pragma unroll
            for (int u = 0; u < UL; ++u) {
                const int idx = i0 + u * T;
                if (idx < total) m.y(idx / ROWS)[idx % ROWS] = v[u];
            }
        }
    }
    __syncthreads();

    m.eliminate();
    m.back_substitute();

    // ---- end-point derivatives of every right-hand side ----
    // (the panel buffers are free: the interface arrays go there)
    double *dots0 = sm, *dotsN = sm + nrhs, *zeta0 = sm + 2 * nrhs, *zeta1 = sm + 3 * nrhs;
    // one right-hand side per lane of a 16-lane row, every fourth node in each
    // of the four rows
#pragma nounroll
    for (int c = w; 16 * c < nrhs; c += RT) {
        const int r = 16 * c + m.li;
        const double *yr = m.y(r < nrhs ? r : 0);
        double d0 = 0.0, dN = 0.0;
#pragma unroll 4
        for (int q = m.lk; q < n; q += 4) {
            const double v = yr[m.phys()[q]];
            d0 = fma(a.Dz[q + 1], v, d0);
            dN = fma(a.Dz[(long long)(N - 1) * N + q + 1], v, dN);
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) {
            d0 += __shfl_xor(d0, o);
            dN += __shfl_xor(dN, o);
        }
        if (r == 0) {  // ul has u(0) = 1
            d0 += a.Dz[0];
            dN += a.Dz[(long long)(N - 1) * N];
        } else if (r == 1) {  // ur has u(N-1) = 1
            d0 += a.Dz[N - 1];
            dN += a.Dz[(long long)(N - 1) * N + N - 1];
        }
        if (m.lk == 0 && r < nrhs) {
            dots0[r] = d0;
            dotsN[r] = dN;
        }
    }
    __syncthreads();

    // ---- element-interface sweep, one thread per real column ----
    if (threadIdx.x < nc && a.periodic) {
        const int cc = threadIdx.x;
        const long long fc = (long long)((cc >> 1) ? xi1 : xi0) * M + jw;
        periodic_sweep(E, dots0[0], dotsN[0], dots0[1], dotsN[1], dots0 + 2 + cc, dotsN + 2 + cc, zeta0 + cc,
                       zeta1 + cc, CPE, a.closure ? a.closure + ((cc & 1) ? (long long)a.nx * M : 0) + fc : nullptr);
    } else if (threadIdx.x < nc) {
        const int cc = threadIdx.x;
        const long long bcol = (long long)((cc >> 1) ? xi1 : xi0) * M + jw;
        const double *bsrc = (cc & 1) ? a.bc_im : a.bc_re;
        const double gl = bsrc[bcol], gr = bsrc[(long long)a.nx * M + bcol];
        const double d0ul = dots0[0], dNul = dotsN[0], d0ur = dots0[1], dNur = dotsN[1];
        // forward elimination over the elements; b and rhs kept in zeta
        double bprev = -a.alpha_l * d0ul + a.beta_l;
        double cprev = -a.alpha_l * d0ur;
        double rprev = gl + a.alpha_l * dots0[2 + cc];
        zeta0[cc] = bprev;
        zeta1[cc] = rprev;
        for (int e = 1; e < E; ++e) {
            const double lb = dNul;
            const double be = dNur - d0ul - (cprev / bprev) * lb;
            const double re = dots0[2 + CPE * e + cc] - dotsN[2 + CPE * (e - 1) + cc] - (rprev / bprev) * lb;
            bprev = be;
            cprev = -d0ur;
            rprev = re;
            zeta0[CPE * e + cc] = be;
            zeta1[CPE * e + cc] = re;
        }
        const double lb = a.alpha_r * dNul;
        const double br = a.alpha_r * dNur + a.beta_r - (cprev / bprev) * lb;
        const double rhsr = gr - a.alpha_r * dotsN[2 + CPE * (E - 1) + cc] - (rprev / bprev) * lb;
        double zr = rhsr / br;
        for (int e = E - 1; e >= 0; --e) {
            const double be = zeta0[CPE * e + cc], re = zeta1[CPE * e + cc];
            const double ce = (e == 0) ? -a.alpha_l * d0ur : -d0ur;
            const double zl = (re - ce * zr) / be;
            zeta0[CPE * e + cc] = zl;
            zeta1[CPE * e + cc] = zr;
            zr = zl;
        }
    }
    __syncthreads();

    // ---- assembly straight into the spectrum ----
    const int stored = (nrhs - 2) * ROWS;
#pragma nounroll
    for (int idx = threadIdx.x; idx < stored; idx += T) {
        const int r = 2 + idx / ROWS, q = idx % ROWS;  // position q: consecutive lanes store consecutive nodes
        const int e = (r - 2) / CPE, cc = (r - 2) % CPE;
        if (cc >= nc || q >= n) continue;
        const double zl = zeta0[CPE * e + cc], zr = zeta1[CPE * e + cc];
        const long long col = (long long)((cc >> 1) ? xi1 : xi0) * a.xs + (long long)jw * K + (long long)e * (N - 1);
        double *dst = (cc & 1) ? a.spec_im : a.spec_re;
        const int row = m.phys()[q];
        dst[col + 1 + q] = m.y(r)[row] + (zl * m.y(0)[row] + zr * m.y(1)[row]);
        if (q == 0) {
            dst[col] = zl;
            dst[col + N - 1] = zr;
        }
    }
    if (threadIdx.x == 0) a.status[mode] = *m.flag() ? HZ_ERR_SINGULAR : 0;
}

template <int RT>
int launch_modes_t(const LuModeArgs &a, int modes, hipStream_t s)
{
    const size_t lds = Lds<RT>::bytes(2 + rhs_per_element(a.nx) * a.ne);
    hipLaunchKernelGGL((lu_modes_kernel<RT>), dim3(modes), dim3(64 * RT), (unsigned)lds, s, a);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

}  // namespace

int lu_modes_prepare()
{
    const int most = 160 * 1024;
    HZ_HIP(hipFuncSetAttribute((const void *)lu_modes_kernel<1>, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    HZ_HIP(hipFuncSetAttribute((const void *)lu_modes_kernel<2>, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    HZ_HIP(hipFuncSetAttribute((const void *)lu_modes_kernel<4>, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    HZ_HIP(hipFuncSetAttribute((const void *)lu_modes_kernel<8>, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return HZ_OK;
}

int lu_modes_check(int nx, int n, int ne)
{
    if (n > 128) return set_error(HZ_ERR_UNSUPPORTED, "PLAIN_LU form: N-2 must be <= 128");
    const int nrhs = 2 + rhs_per_element(nx) * ne;
    if (nrhs > 4 * (n <= 64 ? 64 : 8))  // what the largest instances' LDS holds
        return set_error(HZ_ERR_UNSUPPORTED, "PLAIN_LU form: too many elements (at most 63, or 127 when nx < 4; "
                                             "7, or 15 when nx < 4, for N-2 > 64)");
    return HZ_OK;
}

int lu_modes_shapes(int nx, int n, int ne, int *cols, int max)
{
    // rows and columns of the four instances (1, 2, 4, 8 tiles of 16; the
    // right-hand sides of the largest stop at 32); an instance holds every
    // smaller n (zero padding)
    static const int caps[] = {16, 32, 64, 128};
    const int nr = (2 + rhs_per_element(nx) * ne + 3) / 4;
    int k = 0;
    for (int cap : caps) {
        if (cap < n || nr > (cap == 128 ? 8 : 64)) continue;
        if (k < max) cols[k] = cap;
        ++k;
    }
    return k;
}

// Small operators on few modes: lu.hip's kernel, whose four waves of a mode start
// and end it sooner and pay by the step, where a panel here costs the same for
// any number of columns: N - 2 just above a multiple of 16, or little of either.
// `c` right-hand sides of elements.  The rule follows from the plan's sizes
// alone, so that every instance gives the same bits.  Measured, us a solve,
// stepwise | panels, one element: 256^2 x 3 79 | 99, x 4 93 | 104, x 5 116 | 115;
// 64^2 x 3 20 | 26, x 9 28.6 | 29.4, x 10 29.8 | 29.6, x 19 46 | 43; 1 x 64 x 9
// 15 | 19, x 16 21.3 | 21.8, x 18 22.7 | 21.6, x 19 25 | 29, x 26 30.9 | 32.1,
// x 34 36.9 | 33.9, x 35 39.9 | 41.1.
static bool stepwise(int n, int c, int modes)
{
    // up to n rows: at most c such right-hand sides, and `work` of them over all
    // modes (`work4` where a mode has four or fewer)
    static const struct {
        int n, c;
        long long work, work4;
    } lines[] = {{1, 30, 68000, 1LL << 62}, {2, 30, 24000, 1LL << 62}, {3, 30, 14000, 48000}, {4, 28, 9200, 22000},
                 {5, 28, 6800, 6800},       {6, 24, 4800, 4800},       {7, 20, 4400, 4400},   {8, 16, 2400, 2800},
                 {10, 10, 1200, 1200},      {12, 6, 400, 400},         {14, 4, 140, 140},     {16, 0, 0, 0},
                 {18, 10, 1200, 1200},      {20, 6, 480, 480},         {22, 6, 400, 400},     {26, 4, 140, 140},
                 {32, 0, 0, 0},             {35, 4, 140, 140}};
    for (const auto &l : lines)
        if (n <= l.n) return c <= l.c && (long long)modes * c <= (c <= 4 ? l.work4 : l.work);
    return false;
}

int launch_lu_modes(const LuModeArgs &a, int modes, hipStream_t s)
{
    if (int st = lu_modes_check(a.nx, a.n, a.ne)) return st;
    const int cols = a.cols ? a.cols : a.n <= 16 ? 16 : a.n <= 32 ? 32 : a.n <= 64 ? 64 : 128;
    int c[4];
    const int k = lu_modes_shapes(a.nx, a.n, a.ne, c, 4);
    bool held = false;
    for (int i = 0; i < k && i < 4; ++i) held = held || c[i] == cols;
    if (!held) return set_error(HZ_ERR_ARG, "PLAIN_LU form: the mode-kernel shape does not hold this plan");
    if (a.n > 64 || stepwise(a.n, rhs_per_element(a.nx) * a.ne, modes))
        return launch_lu_modes_stepwise(a, cols, modes, s);
    switch (cols) {
    case 16: return launch_modes_t<1>(a, modes, s);
    case 32: return launch_modes_t<2>(a, modes, s);
    case 64: return launch_modes_t<4>(a, modes, s);
    default: return launch_modes_t<8>(a, modes, s);
    }
}

}  // namespace hz
