// misc.hip -- element-wise GLL derivatives (FirstDerivativeZ /
// SecondDerivativeZ, NonPeriodic3D_MPI.cpp:632-683).
//
// out[e][i][j][k] = sum_p D[k][p] u[e][i][j][p] for every element column:
// a batch of small dense products.  The sum runs over p = 0..N-1 in order
// with every product rounded before it is added, as in the reference's loop,
// so the result equals the reference's bit for bit.
#include "hz_internal.h"

namespace hz {
namespace {

// Lanes are columns, a wave's registers hold R output rows of 64 columns.  The
// column tile is staged in LDS (a lane's values one column stride apart: the
// stride is odd, so 64 lanes hit different banks) and takes the results for a
// coalesced store; the matrix value of a step is the same in every lane, so it
// comes through the scalar cache from the transposed copy DT[p][k] (KP = R
// times the strips).  One LDS read and R products and sums a step, where a
// thread per output node read a matrix row (uncoalesced) and a column from the
// caches for every pair.  256^2 columns of N = 129: 2,727 -> 110 us (with strips of 16
// rows and every lane storing its own rows 130); the
// rounded products and sums cannot be fused, N^2 of each per column, which is
// 55 us at one 16-lane operation per clock.
//
// R = 17 where it saves a strip (N = 2^m + 1, the usual GLL sizes, would leave
// one row to a strip of 16 that costs as much as the others, and an odd number
// of waves to the four SIMDs).  The output may be the input: a work-group stores
// its columns after it has read them.
constexpr int kDerivCols = 64;

int deriv_rows(int N) { return (N + 16) / 17 < (N + 15) / 16 ? 17 : 16; }

// Few outputs: one thread per output, so that they spread over the chip (a tile
// of 64 columns is one work-group, whose waves run N steps of 17 products each).
// Eight loads of each operand in flight: one at a time, 256 columns of 129 took
// 17 us against 7.5.
__global__ __launch_bounds__(256) void derivative_few_kernel(const double *__restrict__ DT, int N, int KP, int total,
                                                             const double *__restrict__ u, double *__restrict__ out)
{
#pragma clang fp contract(off)
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int k = idx % N;
    const double *uc = u + (idx - k);
    double acc = 0.0;
#pragma unroll 8
    for (int p = 0; p < N; ++p) acc += DT[p * KP + k] * uc[p];
    out[idx] = acc;
}

// Where that is the faster: to four work-groups of outputs per CU.  Measured, us,
// one thread per output | tiles: 1 column of N = 66 7 | 11, of 257 12 | 76; 256
// columns of 129 7.5 | 26.5; 2,048 of 128 23.5 | 37.4, of 129 29.8 | 26.9; 4,096 of
// 64 13 | 20, of 66 16.5 | 14.4; 8,192 of 32 7.7 | 11.7, of 33 9.7 | 8.3.
bool derivative_few(int N, long long ncols) { return ncols * N <= 1 << 18; }

template <int R>
__global__ __launch_bounds__(1024) void derivative_kernel(const double *__restrict__ DT, int N, int KP, long long ncols,
                                                         const double *u, double *out)
{
#pragma clang fp contract(off)
    extern __shared__ double dtile[];
    const int LD = N | 1;  // odd column stride
    const long long col0 = (long long)blockIdx.x * kDerivCols;
    const int nc = (int)(ncols - col0 < kDerivCols ? ncols - col0 : kDerivCols);
    const double *src = u + col0 * N;
    const int total = nc * N, T = blockDim.x;
    if (LD == N) {
        constexpr int U = 8;
        int i = threadIdx.x;
        for (; i + (U - 1) * T < total; i += U * T) {
            double v[U];
#pragma unroll
            for (int j = 0; j < U; ++j) v[j] = src[i + j * T];
#pragma unroll
            for (int j = 0; j < U; ++j) dtile[i + j * T] = v[j];
        }
        for (; i < total; i += T) dtile[i] = src[i];
    } else {
        for (int i = threadIdx.x; i < total; i += T) dtile[i + i / N] = src[i];
    }
    __syncthreads();
    const int lane = threadIdx.x % 64;
    const int k0 = R * __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    double *uc = dtile + (lane < nc ? lane : 0) * LD;
    double acc[R];
#pragma unroll
    for (int j = 0; j < R; ++j) acc[j] = 0.0;
    if (k0 < N) {
        const double *d = DT + k0;
#pragma unroll 2
        for (int p = 0; p < N; ++p) {
            const double x = uc[p];
#pragma unroll
            for (int j = 0; j < R; ++j) acc[j] += d[(long long)p * KP + j] * x;
        }
    }
    __syncthreads();  // every wave has read the tile
    if (lane < nc) {
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (k0 + j < N) uc[k0 + j] = acc[j];
    }
    __syncthreads();
    double *dst = out + col0 * N;
    if (LD == N) {
        for (int i = threadIdx.x; i < total; i += T) dst[i] = dtile[i];
    } else {
        for (int i = threadIdx.x; i < total; i += T) dst[i] = dtile[i + i / N];
    }
}

__global__ __launch_bounds__(256) void dot_partial_kernel(const double *__restrict__ a, const double *__restrict__ b,
                                                          long long n, double *__restrict__ partial)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        acc = fma(a[i], b[i], acc);
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// f = a3 u^3 + a1 u, one element per thread (one read, one write).
__global__ __launch_bounds__(256) void cubic_kernel(const double *__restrict__ u, double *__restrict__ f, long long n,
                                                    double a3, double a1)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double x = u[i];
    f[i] = x * fma(a3 * x, x, a1);
}

// One backward step of the semi-implicit cubic right-hand side f(u) =
// a3 u^3 + a1 u: ubar = fbar f'(u_in) = fbar (3 a3 u_in^2 + a1) (ubar may be
// fbar), and the work-group's partial sum of fbar (b1 (u_out - u_in) +
// b3 (u_in^3 - u_in)) into partial[blockIdx.x] (a fixed grid and order, so
// the sum is the same on every run).
__global__ __launch_bounds__(256) void cubic_adjoint_kernel(const double *fbar, const double *__restrict__ u_in,
                                                            const double *__restrict__ u_out, long long n, double a3,
                                                            double a1, double b1, double b3, double *ubar,
                                                            double *__restrict__ partial)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const double fb = fbar[i], x = u_in[i], x2 = x * x;
        acc = fma(fb, b1 * (u_out[i] - x) + b3 * (x2 * x - x), acc);
        ubar[i] = fb * fma(3.0 * a3, x2, a1);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// *acc += the sum of partial[0 .. np) (one work-group, fixed order).
__global__ __launch_bounds__(256) void accumulate_final_kernel(const double *__restrict__ partial, int np, double *acc)
{
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < np; i += 256) s += partial[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *acc += red[0];
}

__global__ __launch_bounds__(256) void dot_final_kernel(const double *__restrict__ partial, int np, double *out)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (int i = threadIdx.x; i < np; i += 256) acc += partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

// Spectral derivative along one axis of a half spectrum re/im[A][B][lanes]
// (the transformed axis is A when axis_a, else B, of length L): multiplies by
// (2 pi i k / len)^order with k = j for j < L/2 and j - L otherwise, the
// wavenumber convention of Fourier_Quadrature.cpp:1512-1519 / :1739-1745
// (the Nyquist point counts as -L/2).
__global__ __launch_bounds__(256) void spectral_derivative_kernel(double *__restrict__ re, double *__restrict__ im,
                                                                  long long A, long long B, long long lanes,
                                                                  int axis_a, int L, double len, int order)
{
    const long long total = A * B * lanes;
    const double two_pi = 6.283185307179586476925286766559;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (long long)gridDim.x * blockDim.x) {
        const long long ab = t / lanes;
        const int j = (int)(axis_a ? ab / B : ab % B);
        const double k = j < L / 2 ? (double)j : (double)(j - L);
        const double c = two_pi * k / len;
        const double r = re[t], q = im[t];
        if (order == 1) {
            re[t] = -c * q;
            im[t] = c * r;
        } else {
            re[t] = -(c * c) * r;
            im[t] = -(c * c) * q;
        }
    }
}

}  // namespace

int launch_spectral_derivative(double *re, double *im, long long A, long long B, long long lanes, int axis_a, int L,
                               double len, int order, hipStream_t s)
{
    const long long total = A * B * lanes;
    const int blocks = (int)std::min<long long>(4096, (total + 255) / 256);
    if (total > 0)
        hipLaunchKernelGGL(spectral_derivative_kernel, dim3(blocks), dim3(256), 0, s, re, im, A, B, lanes, axis_a, L,
                           len, order);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

int launch_dot(const double *a, const double *b, long long n, double *partial, double *out, hipStream_t s)
{
    const int blocks = (int)std::min<long long>(kDotPartials, std::max<long long>(1, (n + 255) / 256));
    hipLaunchKernelGGL(dot_partial_kernel, dim3(blocks), dim3(256), 0, s, a, b, n, partial);
    hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(256), 0, s, partial, blocks, out);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

int launch_cubic_adjoint(const double *fbar, const double *u_in, const double *u_out, long long n, double a3,
                         double a1, double b1, double b3, double *ubar, double *partial, double *acc, hipStream_t s)
{
    const int blocks = (int)std::min<long long>(kDotPartials, std::max<long long>(1, (n + 255) / 256));
    hipLaunchKernelGGL(cubic_adjoint_kernel, dim3(blocks), dim3(256), 0, s, fbar, u_in, u_out, n, a3, a1, b1, b3, ubar,
                       partial);
    hipLaunchKernelGGL(accumulate_final_kernel, dim3(1), dim3(256), 0, s, partial, blocks, acc);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

std::vector<double> derivative_operand(const std::vector<double> &D, int N)
{
    const int R = deriv_rows(N), KP = (N + R - 1) / R * R;
    std::vector<double> t((size_t)N * KP, 0.0);
    for (int k = 0; k < N; ++k)
        for (int p = 0; p < N; ++p) t[(size_t)p * KP + k] = D[(size_t)k * N + p];
    return t;
}

int derivative_prepare(int N)
{
    const size_t lds = sizeof(double) * kDerivCols * (N | 1);
    const void *f = deriv_rows(N) == 17 ? (const void *)derivative_kernel<17> : (const void *)derivative_kernel<16>;
    if (lds > 64 * 1024) HZ_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    return HZ_OK;
}

int launch_derivative(const double *DT, int N, long long ncols, const double *u, double *out, hipStream_t s)
{
    if (ncols <= 0) return HZ_OK;
    // one strip per wave
    const int R = deriv_rows(N), strips = (N + R - 1) / R, waves = std::max(2, strips);
    const size_t lds = sizeof(double) * kDerivCols * (N | 1);
    const long long blocks = (ncols + kDerivCols - 1) / kDerivCols;
    if (waves > 16 || lds > 160 * 1024 || blocks > 0x7fffffffLL)
        return set_error(HZ_ERR_UNSUPPORTED, "derivative: field too large");
    const dim3 grid((unsigned)blocks), block(64 * waves);
    const long long total = ncols * N;
    // (outputs that overlap the inputs: a tile has read all of its columns before it stores)
    if (derivative_few(N, ncols) && (out + total <= u || u + total <= out)) {
        hipLaunchKernelGGL(derivative_few_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, DT, N,
                           strips * R, (int)total, u, out);
    } else if (R == 17)
        hipLaunchKernelGGL((derivative_kernel<17>), grid, block, (unsigned)lds, s, DT, N, strips * R, ncols, u, out);
    else
        hipLaunchKernelGGL((derivative_kernel<16>), grid, block, (unsigned)lds, s, DT, N, strips * R, ncols, u, out);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

}  // namespace hz

using namespace hz;

extern "C" int hz_cubic_rhs(const double *u, double *f, long long n, double a3, double a1, hz_stream_t stream)
{
    if (n < 0 || (n > 0 && (!u || !f))) return set_error(HZ_ERR_ARG, "null argument or negative size");
    if (n == 0) return HZ_OK;
    const long long grid = (n + 255) / 256;
    if (grid > 0x7fffffffLL) return set_error(HZ_ERR_ARG, "size too large");
    hipLaunchKernelGGL(cubic_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, u, f, n, a3, a1);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

extern "C" int hz_derivative_z(hz_plan *p, int order, const double *u, double *out, hz_stream_t stream)
{
    if (!p || !u || !out || (order != 1 && order != 2)) return set_error(HZ_ERR_ARG, "bad argument");
    const long long ncols = (long long)p->ne * p->nx * p->ny;
    return launch_derivative(p->d_DzT[order - 1], p->N, ncols, u, out, (hipStream_t)stream);
}
