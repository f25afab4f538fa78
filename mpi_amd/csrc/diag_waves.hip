// diag_waves.hip -- the z-diagonalised mode solve of several elements, Robin
// faces or periodic z (scheme in diag_body.h) for N - 2 <= 32: one wave per 16
// columns of the padded interior and 16 RB rows, NJ x WR waves per work-group.
//
// Short chains of dependent steps on little data, so latency bounds them.  All
// of a tile's loads, the interface system's coefficients included, are in
// flight before the first is waited for; the right-hand side stays in the
// accumulators' layout from load to store; one 16-byte LDS read feeds two
// matrix steps; rows are reduced in registers.  N - 2 <= 16 runs on 16 columns,
// a quarter of the work of the 32 that the operands are padded to: 50 -> 24 us
// for 8 elements of 17 points on 128^2 (34 MB: 6 us at the copy rate).
#include "diag_waves_body.h"

namespace hz {
namespace {

template <int NJ, int WR, int RB, bool ADJ>
__global__ __launch_bounds__(64 * NJ * WR, 4) void diag_waves_kernel(const DiagArgs a)
{
    diag_waves_tile<NJ, WR, RB, ADJ>(a, blockIdx.x);
}

template <int NJ, int WR, int RB>
int launch_t(const DiagArgs &a, hipStream_t s)
{
    const int fc_per_tile = 16 * RB * WR / (2 * a.ne);
    const dim3 grid((a.nx * a.M + fc_per_tile - 1) / fc_per_tile), block(64 * NJ * WR);
    if (a.adjoint)
        hipLaunchKernelGGL((diag_waves_kernel<NJ, WR, RB, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((diag_waves_kernel<NJ, WR, RB, false>), grid, block, 0, s, a);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

}  // namespace

// Rows of a tile: a column's 2 E rows must fit it.
int diag_waves_rows(int n) { return n <= 16 ? 128 : 64; }

// Measured, us a solve, here against diag_tile's four waves per 32 to 128
// padded rows: 128^2, 13 x 9 periodic 86 | 127, 8 x 17 70 | 90, 16 x 18 92 |
// 127, 4 x 33 66 | 68; 256^2 x 9 Robin 38 | 46.  At N - 2 = 63 both take the
// same (128^2 Robin 50), at 127 the four waves are faster (84 | 79): more waves
// then wait for the same matrix cores.
bool diag_waves_holds(int n, int ne) { return n >= 1 && n <= 32 && 2 * ne <= diag_waves_rows(n); }

int launch_diag_waves(const DiagArgs &a, hipStream_t s)
{
    if (!diag_waves_holds(a.n, a.ne) || a.eo)
        return set_error(HZ_ERR_UNSUPPORTED, "DIAG form: mode solve out of range");
    if (a.n <= 16) return launch_t<1, 4, 2>(a, s);
    return launch_t<2, 2, 2>(a, s);
}

}  // namespace hz
