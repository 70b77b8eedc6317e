// Declustering noise filter of the plasma electrons (plasma3d/noise_filter.py:
// 53-238), gfx950.  The sort's arrays are its (n, n) lattice in row-major
// order, element (i, j) at i n + j.
//
//   k_dc_rows   inhomogeneity of x_offt and y_offt along both lattice
//               directions (noise_filter.py:53-76, 135-136) and its circular
//               Gaussian smoothing along j;
//   k_dc_cols   the same along i, and the chaotic displacement
//               dx_chaotic = inhomogeneity - smoothed (noise_filter.py:147-170);
//   k_dc_kick   restoring kicks of px and py from the forces of the particle
//               and its four lattice neighbours, and the damping
//               (noise_filter.py:176-232).
//
// The reference smooths with ifft2(fourier_gaussian(fft2(a), sigma)).real:
// multiplying the periodic spectrum by exp(-2 pi^2 sigma^2 (k/n)^2) along
// each axis.  That is a circular convolution with the kernel
// g[m] = (1/n) sum_k exp(-2 pi^2 sigma^2 (k/n)^2) cos(2 pi k m / n), applied
// along j and then along i; the host computes g in float64 and keeps the
// taps above 1e-17 of g[0] (the rest change no float64 result).  Every
// output is one thread's fixed-order sum.  The kick arithmetic is evaluated
// operation by operation as the reference's numpy statements (no fused
// multiply-adds), in float64; px, py are read and written in the bulk type.
#include "common.h"
#include "kernels.h"

namespace lc3d {

constexpr int DC_THREADS = 256;

// Inhomogeneity of d at (i, j) along j (`along_j`) or along i
// (calculate_inhomogeneity_numba with axis 0 or 1).
__device__ __forceinline__ double dc_inhom(const double *__restrict__ d, int n, int i, int j,
                                           bool along_j)
{
    const int64_t o = (int64_t)i * n + j;
    const int64_t st = along_j ? 1 : n;
    const int k = along_j ? j : i;
    if (k >= 1 && k <= n - 2) {
        const double c = d[o], l = d[o - st], r = d[o + st];
        return (c != 0 && l != 0 && r != 0) ? c - (l + r) / 2 : 0.0;
    }
    const int64_t s = k == 0 ? st : -st;   // towards the inside
    const double a = d[o], b = d[o + s], c = d[o + 2 * s];
    return (a != 0 && b != 0 && c != 0) ? a - 2 * b + c : 0.0;
}

// Smoothed values at R consecutive places: sum[r] = sum_t taps[t] in[place r - tap0 - t],
// t ascending.  v(k), called for k = 0, 1, .. in turn, is the element k before
// the first one that the last place reads: it is tap k - (R - 1 - r) of place r,
// so every element is read once for the R places.
template <int R, typename V>
__device__ __forceinline__ void dc_smooth(int ntaps, const double *__restrict__ taps, V v,
                                          double (&sum)[R])
{
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = 0;
    if (ntaps < R) {
        for (int k = 0; k < ntaps + R - 1; ++k) {
            const double x = v(k);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int t = k - (R - 1 - r);
                if (t >= 0 && t < ntaps) sum[r] += taps[t] * x;
            }
        }
        return;
    }
    double x[R - 1];   // the elements that not every place reads: the first ones,
#pragma unroll
    for (int k = 0; k < R - 1; ++k) x[k] = v(k);
#pragma unroll
    for (int k = 0; k < R - 1; ++k)
#pragma unroll
        for (int r = R - 1 - k; r < R; ++r) sum[r] += taps[k - (R - 1 - r)] * x[k];
    int k = R - 1;
#pragma unroll 8
    for (; k < ntaps; ++k) {
        const double c = v(k);
#pragma unroll
        for (int r = 0; r < R; ++r) sum[r] += taps[k - (R - 1 - r)] * c;
    }
    const double *last = taps + ntaps - (R - 1);   // and the last ones
#pragma unroll
    for (int e = 0; e < R - 1; ++e) x[e] = v(k + e);
#pragma unroll
    for (int e = 0; e < R - 1; ++e)
#pragma unroll
        for (int r = 0; r < R - 1 - e; ++r) sum[r] += last[e + r] * x[e];
}

// A lattice row's inhomogeneity of x_offt (blockIdx.y 0) or y_offt (1), and its
// circular convolution along j: out[j] = sum_t taps[t] in[(j - tap0 - t) mod n].
// The row is staged in LDS, unrolled to the n + ntaps - 1 elements that the
// outputs read.  A thread sums DC_ROW outputs from registers, so that an
// element is read from LDS once for them; DC_ROW + 1 doubles of LDS per DC_ROW
// elements keep the threads' reads in different banks.
// Measured, side 836, 55 taps, with the inhomogeneity: 34 -> 18 us, of which the
// lattice's 33 MB take 6; the rest is the blocks' chain of load, stage and sum.
constexpr int DC_MAX_SIDE = 4096;
constexpr int DC_ROW = 4;
__host__ __device__ constexpr int dc_place(int e) { return e + e / DC_ROW; }
__global__ __launch_bounds__(DC_THREADS) void k_dc_rows(int n, int ntaps, int tap0,
                                                        const double *__restrict__ taps,
                                                        const double *__restrict__ xo,
                                                        const double *__restrict__ yo,
                                                        double *__restrict__ dxi,
                                                        double *__restrict__ dyi,
                                                        double *__restrict__ tx,
                                                        double *__restrict__ ty)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    double *ext = reinterpret_cast<double *>(lds_raw);   // in[(e - (tap0 + ntaps - 1)) mod n]
    // Blocks go to the XCDs in turn: a band of rows is one XCD's.
    const int i = blockIdx.x % 8 * ((n + 7) / 8) + blockIdx.x / 8;
    if (i >= n) return;
    const int64_t row = (int64_t)i * n;
    const double *__restrict__ d = blockIdx.y == 0 ? xo : yo;
    double *__restrict__ inhom = blockIdx.y == 0 ? dxi : dyi;
    double *__restrict__ out = blockIdx.y == 0 ? tx : ty;
    int shift = (tap0 + ntaps - 1) % n;
    if (shift < 0) shift += n;
    for (int j = threadIdx.x; j < n; j += DC_THREADS) {
        const double v = (dc_inhom(d, n, i, j, true) + dc_inhom(d, n, i, j, false)) / 2;
        inhom[row + j] = v;
        for (int e = j + shift < n ? j + shift : j + shift - n; e < n + ntaps - 1; e += n)
            ext[dc_place(e)] = v;
    }
    __syncthreads();
    for (int j0 = DC_ROW * threadIdx.x; j0 < n; j0 += DC_ROW * DC_THREADS) {
        const double *at = ext + dc_place(j0);   // j0 is a multiple of DC_ROW
        double sum[DC_ROW];
        dc_smooth<DC_ROW>(ntaps, taps,
                          [&](int k) { return at[dc_place(DC_ROW - 1 + ntaps - 1 - k)]; }, sum);
#pragma unroll
        for (int r = 0; r < DC_ROW; ++r)
            if (j0 + r < n) out[row + j0 + r] = sum[r];
    }
}

// The same along i, then dx_chaotic = inhomogeneity - smoothed (blockIdx.y 0: x,
// 1: y).  A thread sums DC_COL lattice rows of its column from registers.
// Measured, side 836, 55 taps: 84 us (each output read its taps' elements) -> 15,
// of which its 34 MB take 7; with 8 rows a thread, the same.
constexpr int DC_COL = 16, DC_COL_THREADS = 64;
__global__ __launch_bounds__(DC_COL_THREADS) void k_dc_cols(
    int n, int ntaps, int tap0, const double *__restrict__ taps, const double *__restrict__ tx,
    const double *__restrict__ ty, const double *__restrict__ dxi, const double *__restrict__ dyi,
    double *__restrict__ dxc, double *__restrict__ dyc)
{
    // Blocks go to the XCDs in turn: a strip of columns is one XCD's, which
    // reads every element from memory once.
    const int down = (n + DC_COL - 1) / DC_COL;
    const int j = (blockIdx.x % 8 + 8 * (blockIdx.x / (8 * down))) * DC_COL_THREADS + threadIdx.x;
    const int i0 = blockIdx.x / 8 % down * DC_COL;
    if (j >= n) return;
    const double *__restrict__ in = (blockIdx.y == 0 ? tx : ty) + j;
    const double *__restrict__ inhom = (blockIdx.y == 0 ? dxi : dyi) + j;
    double *__restrict__ out = (blockIdx.y == 0 ? dxc : dyc) + j;
    int s = (i0 + DC_COL - 1 - tap0) % n;   // the row that the last place reads first
    if (s < 0) s += n;
    double sum[DC_COL];
    dc_smooth<DC_COL>(ntaps, taps,
                      [&](int) {
                          const double x = in[(int64_t)s * n];
                          s = s == 0 ? n - 1 : s - 1;
                          return x;
                      },
                      sum);
#pragma unroll
    for (int r = 0; r < DC_COL; ++r) {
        const int64_t o = (int64_t)(i0 + r) * n;
        if (i0 + r < n) out[o] = inhom[o] - sum[r];
    }
}

struct KickCoef {
    double xi;        // xi_step
    double mforce;    // -declustering-force
    double xidamp;    // xi_step * damping
    double lim2;      // declustering-limit ** 2
};

// d_limit and the force of the particle at o (noise_filter.py:170-179).
__device__ __forceinline__ void dc_force(const KickCoef &k, double cx, double cy, double &fx,
                                         double &fy, double &dl)
{
#pragma clang fp contract(off)
    const double d = cx * cx + cy * cy;
    dl = d < k.lim2 ? 1 - d / k.lim2 : 0.0;
    fx = k.mforce * cx * dl;
    fy = k.mforce * cy * dl;
}

// px of one particle after noise_filter.py:218-224 (likewise py): the seven
// in-place array statements applied to it in their order.
__device__ __forceinline__ double dc_kick(const KickCoef &k, double p, int i, int j, int n,
                                          double f, double f_im, double f_ip, double f_jm,
                                          double f_jp, double dl, double c, double cprev)
{
#pragma clang fp contract(off)
    if (i >= 1 && i <= n - 2) p += k.xi * f / 2;
    if (i >= 2) p -= k.xi * f_im / 4;
    if (i <= n - 3) p -= k.xi * f_ip / 4;
    if (j >= 1 && j <= n - 2) p += k.xi * f / 2;
    if (j >= 2) p -= k.xi * f_jm / 4;
    if (j <= n - 3) p -= k.xi * f_jp / 4;
    p -= k.xidamp * dl * (c - cprev);
    return p;
}

template <typename TP>
__global__ __launch_bounds__(DC_THREADS) void k_dc_kick(int n, KickCoef k,
                                                        const double *__restrict__ dxc,
                                                        const double *__restrict__ dyc,
                                                        const double *__restrict__ dxp,
                                                        const double *__restrict__ dyp,
                                                        TP *__restrict__ px, TP *__restrict__ py)
{
    const int64_t o = blockIdx.x * (int64_t)DC_THREADS + threadIdx.x;
    if (o >= (int64_t)n * n) return;
    const int i = (int)(o / n), j = (int)(o % n);
    double fx, fy, dl;
    dc_force(k, dxc[o], dyc[o], fx, fy, dl);
    // Forces of the four neighbours (0 where a neighbour is off the lattice;
    // those terms are not applied).
    double nx[4] = {0, 0, 0, 0}, ny[4] = {0, 0, 0, 0};
    const int64_t nb[4] = {o - n, o + n, o - 1, o + 1};
    const bool ok[4] = {i >= 1, i <= n - 2, j >= 1, j <= n - 2};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (ok[q]) {
            double d;
            dc_force(k, dxc[nb[q]], dyc[nb[q]], nx[q], ny[q], d);
        }
    }
    px[o] = (TP)dc_kick(k, (double)px[o], i, j, n, fx, nx[0], nx[1], nx[2], nx[3], dl, dxc[o], dxp[o]);
    py[o] = (TP)dc_kick(k, (double)py[o], i, j, n, fy, ny[0], ny[1], ny[2], ny[3], dl, dyc[o], dyp[o]);
}

template <typename TP>
hipError_t launch_noise_filter(const DeclustGeom &g, const double *xo, const double *yo, TP *px,
                               TP *py, const double *dxp, const double *dyp, double *dxc,
                               double *dyc, hipStream_t s)
{
    const int n = g.side;
    if (n < 3 || n > DC_MAX_SIDE || g.ntaps < 1) return hipErrorInvalidValue;
    const int64_t nn = (int64_t)n * n;
    const unsigned blocks = (unsigned)((nn + DC_THREADS - 1) / DC_THREADS);
    double *dxi = g.scratch, *dyi = g.scratch + nn, *tx = g.scratch + 2 * nn, *ty = g.scratch + 3 * nn;
    const KickCoef k{g.xi_step, -g.force, g.xi_step * g.damping, g.limit * g.limit};
    // Elements read for outputs past the row's end are discarded with them.
    const size_t lds = sizeof(double) * (size_t)dc_place(n + g.ntaps - 1 + DC_ROW);
    k_dc_rows<<<dim3((n + 7) / 8 * 8, 2), DC_THREADS, lds, s>>>(n, g.ntaps, g.tap0, g.taps, xo, yo, dxi, dyi, tx,
                                                  ty);
    const int strips = (n + DC_COL_THREADS - 1) / DC_COL_THREADS, down = (n + DC_COL - 1) / DC_COL;
    k_dc_cols<<<dim3((strips + 7) / 8 * 8 * down, 2), DC_COL_THREADS, 0, s>>>(
        n, g.ntaps, g.tap0, g.taps, tx, ty, dxi, dyi, dxc, dyc);
    k_dc_kick<TP><<<blocks, DC_THREADS, 0, s>>>(n, k, dxc, dyc, dxp, dyp, px, py);
    return hipGetLastError();
}

template hipError_t launch_noise_filter<double>(const DeclustGeom &, const double *, const double *,
                                                double *, double *, const double *, const double *,
                                                double *, double *, hipStream_t);
template hipError_t launch_noise_filter<float>(const DeclustGeom &, const double *, const double *,
                                               float *, float *, const double *, const double *,
                                               double *, double *, hipStream_t);

}  // namespace lc3d
