// fderiv.hip -- Fourier derivative along one axis of a real field in one
// pass: the transform, the wavenumber factor and the transform back stay in a
// work-group (registers and one LDS tile), so the field is read once and
// written once.
//
// Bound by memory: 256^2 x 129 along either axis 34 us (134 MB); a real-to-half
// transform, a factor pass and the transform back took 75.
// W neighbouring lanes per work-group of 256 threads (rows
// of W contiguous values per point), L = R1 R2: thread (w, q), q < R2, holds
// the R1 points q + R2 n1 of line w, stage 2 the R2 points of R1 / R2 indices
// k1 = q + R2 l, and the same two stages back; exchanges through LDS, real
// parts, then imaginary parts.  The factor multiplies in stage 2's order, k =
// k1 + R1 k2, from a table of the wavenumbers in LDS (one division per thread).
#include "fft_body.h"

namespace hz {
namespace {

template <int L>
struct Lines {
    static constexpr int R1 = L >= 128 ? 16 : 8, R2 = L / R1, W = 256 / R2;
};

// (out may be u: a work-group stores its lines after it has read them whole)
template <int L, int ORDER>
__global__ __launch_bounds__(256, 4) void derivative_lines(const double *u, double *out, long long nbatch,
                                                           long long lanes, long long bs, long long ps, double len,
                                                           const double2 *__restrict__ tw)
{
    constexpr int R1 = Lines<L>::R1, R2 = Lines<L>::R2, W = Lines<L>::W, NL = R1 / R2;
    __shared__ double tile[L * W];
    __shared__ double wave[L];
    const int w = threadIdx.x % W, q = threadIdx.x / W;
    const unsigned nlb = (unsigned)((lanes + W - 1) / W);
    const unsigned t = xcd_logical(blockIdx.x, gridDim.x);
    const long long lane = (long long)(t % nlb) * W + w, at = (long long)(t / nlb) * bs + lane;
    const bool live = lane < lanes;

    double re[R1], im[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
        re[n1] = live ? u[at + (q + R2 * n1) * ps] : 0.0;
        im[n1] = 0.0;
    }
    for (int j = threadIdx.x; j < L; j += 256) {
        // the reference's wavenumbers: the Nyquist point counts as -L/2
        const double k = j < L / 2 ? (double)j : (double)(j - L);
        wave[j] = 6.283185307179586476925286766559 * k / len;
    }
    auto exchange = [&](auto to, auto from) {
#pragma unroll
        for (int k = 0; k < R1; ++k) tile[to(k)] = re[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R1; ++k) re[k] = tile[from(k)];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R1; ++k) tile[to(k)] = im[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R1; ++k) im[k] = tile[from(k)];
    };
    auto pos1 = [&](int k1) { return (k1 * R2 + q) * W + w; };                               // point (k1, n2 = q)
    auto pos2 = [&](int e) { return ((q + R2 * (e / R2)) * R2 + e % R2) * W + w; };          // (k1 = q + R2 l, n2)
    {
        TwiddlePowers<R1, L> p;
        p.load(tw, q);
        dft_regs<R1, L, -1>(re, im, tw);
        p.template apply<-1>(re, im);
    }
    exchange(pos1, pos2);
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        double r[R2], i[R2];
#pragma unroll
        for (int k = 0; k < R2; ++k) {
            r[k] = re[l * R2 + k];
            i[k] = im[l * R2 + k];
        }
        dft_regs<R2, L, -1>(r, i, tw);
#pragma unroll
        for (int k = 0; k < R2; ++k) {
            const double c = wave[q + R2 * l + R1 * k];
            if constexpr (ORDER == 1) {
                const double x = r[k];
                r[k] = -c * i[k];
                i[k] = c * x;
            } else {
                r[k] = -(c * c) * r[k];
                i[k] = -(c * c) * i[k];
            }
        }
        dft_regs<R2, L, 1>(r, i, tw);
#pragma unroll
        for (int k = 0; k < R2; ++k) {
            re[l * R2 + k] = r[k];
            im[l * R2 + k] = i[k];
        }
    }
    __syncthreads();
    exchange(pos2, pos1);
    {
        TwiddlePowers<R1, L> p;
        p.load(tw, q);
        p.template apply<1>(re, im);
        dft_regs<R1, L, 1>(re, im, tw);
    }
    if (!live) return;
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) out[at + (q + R2 * n1) * ps] = re[n1] * (1.0 / L);
}

template <int L>
int launch_lines(long long nbatch, long long lanes, long long bs, long long ps, const double *u, double *out,
                 double len, int order, const double2 *tw, hipStream_t s)
{
    constexpr int W = Lines<L>::W;
    const dim3 grid((unsigned)(nbatch * ((lanes + W - 1) / W))), block(256);
    if (order == 1)
        hipLaunchKernelGGL((derivative_lines<L, 1>), grid, block, 0, s, u, out, nbatch, lanes, bs, ps, len, tw);
    else
        hipLaunchKernelGGL((derivative_lines<L, 2>), grid, block, 0, s, u, out, nbatch, lanes, bs, ps, len, tw);
    HZ_HIP(hipGetLastError());
    return HZ_OK;
}

}  // namespace

bool derivative_lines_holds(int L, long long nbatch, long long lanes)
{
    return L >= 32 && L <= 256 && lanes <= (1LL << 40) && nbatch * ((lanes + 15) / 16) < (1LL << 31);
}

int launch_derivative_lines(int L, long long nbatch, long long lanes, long long bs, long long ps, const double *u,
                            double *out, double len, int order, const double2 *tw, hipStream_t s)
{
    switch (L) {
    case 32: return launch_lines<32>(nbatch, lanes, bs, ps, u, out, len, order, tw, s);
    case 64: return launch_lines<64>(nbatch, lanes, bs, ps, u, out, len, order, tw, s);
    case 128: return launch_lines<128>(nbatch, lanes, bs, ps, u, out, len, order, tw, s);
    case 256: return launch_lines<256>(nbatch, lanes, bs, ps, u, out, len, order, tw, s);
    default: return set_error(HZ_ERR_UNSUPPORTED, "Fourier derivative: line length out of range");
    }
}

}  // namespace hz
