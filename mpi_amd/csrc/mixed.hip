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

template <int NJ, int RB, bool GENERAL>
__global__ __launch_bounds__(64 * NJ, NJ == 6 && GENERAL ? 3 : 4) void mixed_waves_kernel(const MixedArgs a)
{
    mixed_waves_tile<NJ, RB, GENERAL>(a, blockIdx.x);
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

// N - 2 padded to 96, several elements and more tiles than two per CU: mixed_tile,
// whose work-group takes 40 KB of LDS and four waves (four per CU) where six waves
// with 53 KB are two per CU, and the elements' sweeps, one lane per column, are
// waited for by fewer others.  Measured, us a solve, mixed_tile | one wave per 16
// columns: 128^2, Robin, 4 x 67 278 | 284, 6 x 67 467 | 496, periodic 6 x 67
// 477 | 520; 64^2 periodic 10 x 67 261 | 287, 16 x 67 307 | 347, 16 x 98 339 | 370;
// below two tiles per CU 32^2 periodic 8 x 67 85 | 76.  (The other padded sizes
// had 16 rows in mixed_tile and gain everywhere.)
bool mixed_by_four_waves(int n, int ne, int columns)
{
    return diag_padded(n) == 96 && ne >= 4 && columns / (16 / ne) >= 512;
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
    case 96:
        return mixed_by_four_waves(a.n, a.ne, a.nx * a.M) ? launch_t<6, 32, false>(a, s) : launch_t<6, 32, true>(a, s);
    case 128: return launch_t<8, 32, true>(a, s);
    case 256: return launch_t<16, 16, false>(a, s);
    default: return set_error(HZ_ERR_UNSUPPORTED, "MIXED form: N-2 must be <= 256");
    }
}

}  // namespace hz
