// Plasma particle push for one xi step (gfx950).
//
// One thread per macro-particle over structure-of-arrays buffers.  The push
// follows plasma3d/move.py:52-148: midpoint position (reflected at
// the wall), 5x5 quartic-spline gather of six fields, two fixed-point passes
// of the relativistic momentum update, position update from the half-step
// momentum, wall reflection and absorption.  In the FP32-bulk form the
// momentum arithmetic runs in float while gamma, the 1/(1 - v_z) factor and
// the positions stay double.
#include "common.h"
#include "kernels.h"

#include <cmath>
#include <type_traits>

namespace lc3d {

template <typename TP>
__global__ __launch_bounds__(256) void k_move_wo_fields(int64_t n, double xi_step,
                                                        const TP *__restrict__ m,
                                                        double *__restrict__ xo,
                                                        double *__restrict__ yo,
                                                        const TP *__restrict__ px,
                                                        const TP *__restrict__ py,
                                                        const double *__restrict__ pz)
{
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double mk = m[k];
    if (mk == 0) return;
    const double a = px[k], b = py[k], c = pz[k];
    const double g = sqrt(mk * mk + c * c + a * a + b * b);
    const double d = g - c;
    xo[k] += a / d * xi_step;
    yo[k] += b / d * xi_step;
}

// Reflection of a position at +-b (plasma3d/move.py:28-49).  Returns true
// when any reflection happened (the caller then zeroes the momenta).
__device__ __forceinline__ bool reflect(double x_init, double y_init, double b, double &x,
                                        double &y, double &xo, double &yo)
{
    bool hit = false;
    if (x > b) { x = 2 * b - x; xo = x - x_init; hit = true; }
    if (x < -b) { x = -2 * b - x; xo = x - x_init; hit = true; }
    if (y > b) { y = 2 * b - y; yo = y - y_init; hit = true; }
    if (y < -b) { y = -2 * b - y; yo = y - y_init; hit = true; }
    return hit;
}

// ---- the field window of a block -----------------------------------------------
// Every particle reads 5 x 5 taps of six fields.  Read from memory that is
// 150 loads a particle, and the L1's address path was the push's bound (its
// texture-address unit 90% busy in float64, 84% in float32: 2290 and 1307
// cache accesses a wave).  The particles of a block are neighbours (they are
// visited strip by strip, see cell_key), so their stencils lie in a window
// of a few hundred grid points, which the block reads once, coalesced, into
// LDS, as three pairs of fields (one 16- or 8-byte LDS read gives two
// fields).  Measured at N = 513, 4 ppc (929,296 particles) inside the step:
// 76 -> 48-50 us in float64 and 43 -> 34-36 us in float32 (the first push 56 ->
// 35 us, which also no longer needs a pass that rounds the float64 fields), for
// 207 and 158 MB of HBM traffic a push (counters), 4.2 and 4.5 TB/s; outside it,
// in lattice tiles, 80 -> 47 us for 1.1e6 float64 particles.
// A block whose stencils span more than PUSH_WINDOW points (the turn of a
// strip, a nearly empty region) reads its taps from memory instead.
// PUSH_WINDOW points take 38 KB in float64, 19 in float32: four and five blocks
// a CU, for which the compiler is held to 128 and 96 registers and spills some
// of them in the forms that a step runs (float64 28 bytes a lane in the first
// push and 12 in the others; float32 36 and 12).
// A sort of fewer than PUSH_FEW particles (STAGED false) leaves CUs idle at
// PUSH_THREADS a block: there the time is the chain of one wave, which the
// window only lengthens, so blocks of one wave read their taps from memory.
// Measured, this form against the staged one: 9,409 particles (N = 129, 1 ppc,
// float64) 7.6 against 10.9 us, 51,529 (257, float32) 7.1 against 8.3; 83,521
// (321, float64) 12.0 against 11.8, 104,976 (193, 4 ppc, float64) 12.6 against 10.9.
constexpr int PUSH_FEW = 65536, PUSH_FEW_THREADS = 64;
constexpr int PUSH_THREADS = 256;
constexpr int PUSH_WINDOW = 800;
constexpr int PUSH_TILE = 16;   // side of a block's lattice tile, when there is no order
static_assert(PUSH_TILE * PUSH_TILE == PUSH_THREADS, "one lattice tile per block");

template <typename T> struct alignas(2 * sizeof(T)) FieldPair {
    T a, b;
};

// Bounds of the block's stencil cells: rows r0 .. r1 and columns c0 .. c1
// (r0 > r1: no particle gathers).
struct PushBox {
    int r0, r1, c0, c1;
};

// Minimum of v over the block's lanes for each of four values; every thread
// calls it.  Cell indices are exact in float.
__device__ __forceinline__ PushBox block_box(bool in, int ix, int iy, float (*red)[4])
{
    constexpr float FAR = 1 << 20;
    float v[4] = {in ? (float)ix : FAR, in ? (float)-ix : FAR, in ? (float)iy : FAR,
                  in ? (float)-iy : FAR};
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = fminf(v[k], __shfl_xor(v[k], off));
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) red[threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < PUSH_THREADS / 64; ++w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = fminf(v[k], red[w][k]);
    }
    return PushBox{(int)v[0], -(int)v[1], (int)v[2], -(int)v[3]};
}

// One particle per thread: state read, midpoint and its stencil cell, the
// block's field window, the gather, the momentum and position update, and
// with BIN the particle's deposit record and cell, written at its binning
// position (the thread's place in the visiting order).
//
// With `order` the block takes PUSH_THREADS consecutive particles of it.
// Without (the first push of a run, or one outside a step) it takes a
// PUSH_TILE x PUSH_TILE tile of the side x side lattice, if side > 0, else
// consecutive particles; the binning position is then the particle index.
//
// momenta: store px, py and pz.  The first two pushes of a step need not:
// the next push starts from the previous layer's momenta again and the
// deposit reads its records (24 of the 192 bytes a particle moves in
// float64).  An absorbed particle's are stored always, no later push writes
// them.
template <typename TP, typename TF, bool FIRST, bool BIN, bool STAGED>
__global__ __launch_bounds__(STAGED ? PUSH_THREADS : PUSH_FEW_THREADS,
                             STAGED ? (sizeof(TP) == 4 ? 5 : 4) : 1) void k_push(
    PushGeom g, Fields6<TF> f, SortArrays<TP> a, BinState bs, const int *__restrict__ order,
    int side, bool momenta)
{
    __shared__ FieldPair<TP> s_f[3][STAGED ? PUSH_WINDOW : 1];
    __shared__ float s_red[PUSH_THREADS / 64][4];
    constexpr int THREADS = STAGED ? PUSH_THREADS : PUSH_FEW_THREADS;
    if (BIN) clear_scan(bs);
    // Consecutive blocks of the order go to the same XCD, so each XCD's L2
    // fetches the field rows of its own stretch of cells.
    const int block = xcd_swizzle(blockIdx.x, gridDim.x);
    int64_t j, k;
    bool have;
    if (!STAGED || order != nullptr || side == 0) {
        j = block * (int64_t)THREADS + threadIdx.x;
        have = j < g.n;
        k = have && order ? (int64_t)order[j] : j;   // the particle this thread pushes
    } else {
        const int tiles = (side + PUSH_TILE - 1) / PUSH_TILE;
        const int li = block / tiles * PUSH_TILE + threadIdx.x / PUSH_TILE;
        const int lj = block % tiles * PUSH_TILE + threadIdx.x % PUSH_TILE;
        have = li < side && lj < side;
        j = k = (int64_t)li * side + lj;
    }
    const int N = g.N;
    const double b = g.boundary, dxi = g.xi_step;
    // FP32-bulk (float32 momenta): quotients that share a divisor are taken
    // as products with its reciprocal (one float64 division instead of two
    // or three; the results differ by at most an ulp of float64, far below
    // the float32 momenta).  The float64 form divides as
    // plasma3d/move.py:52-148 does.
    constexpr bool RCP = std::is_same<TP, float>::value;

    double xi0 = 0, yi0 = 0, xop = 0, yop = 0, opz = 0, m = 0, xof = 0, yof = 0;
    TP opx = 0, opy = 0, q = 0;
    if (have) {
        xi0 = a.x_init[k];
        yi0 = a.y_init[k];
        xop = a.xo_prev[k];
        yop = a.yo_prev[k];
        opx = a.px_prev[k];
        opy = a.py_prev[k];
        opz = a.pz_prev[k];
        m = (double)a.m[k];
        if (FIRST) {
            // particles_full = copy(particles_prev) + free-streaming estimate
            q = a.q_prev[k];
            xof = xop;
            yof = yop;
            if (m != 0) {
                const double A = opx, B = opy, C = opz;
                const double gm = sqrt(m * m + C * C + A * A + B * B);
                if constexpr (RCP) {
                    const double r = dxi / (gm - C);
                    xof = xop + A * r;
                    yof = yop + B * r;
                } else {
                    xof = xop + A / (gm - C) * dxi;
                    yof = yop + B / (gm - C) * dxi;
                }
            }
        } else {
            q = a.q[k];
            xof = a.xo[k];
            yof = a.yo[k];
        }
    }
    const bool live = have && q != TP(0);

    // Midpoint between the previous position and the current estimate.
    double x = xi0 + (xop + xof) * 0.5, y = yi0 + (yop + yof) * 0.5;
    TP px = opx, py = opy;
    double pz = opz;
    {
        double xo_tmp = 0, yo_tmp = 0;
        if (live && reflect(xi0, yi0, b, x, y, xo_tmp, yo_tmp)) {
            px = py = TP(0);
            pz = 0;
        }
    }
    int ix = 0, iy = 0;
    double xl = 0, yl = 0;
    bool inside = false;
    if (live) {
        bool finite;
        inside = stencil_cell(x, y, g.h, N, ix, iy, xl, yl, finite);
        // Outside the grid (or not finite): no field is gathered.
        if (!inside) atomicOr(bs.err, finite ? ERR_PARTICLE_OFF_GRID : ERR_NONFINITE);
    }

    // The block's window: the stencils of all its particles.  A stencil cell
    // is at least 2 and at most N - 3, so the window lies in the grid.
    PushBox box{1, 0, 0, 0};
    if constexpr (STAGED) box = block_box(inside, ix, iy, s_red);
    const int width = box.c1 - box.c0 + 5, rows = box.r1 - box.r0 + 5;
    const bool window = STAGED && box.r0 <= box.r1 && width * rows <= PUSH_WINDOW;
    if (window) {
        const float inv = 1.0f / (float)width;
        for (int p = threadIdx.x; p < width * rows; p += PUSH_THREADS) {
            // p / width, exact: (p + 1/2) / width is at least 1/(2 width) from
            // an integer, and p < PUSH_WINDOW.
            const int r = (int)(((float)p + 0.5f) * inv), c = p - r * width;
            const int id = (box.r0 - 2 + r) * N + box.c0 - 2 + c;
            s_f[0][p] = FieldPair<TP>{(TP)f.Ex[id], (TP)f.Bx[id]};
            s_f[1][p] = FieldPair<TP>{(TP)f.Ey[id], (TP)f.By[id]};
            s_f[2][p] = FieldPair<TP>{(TP)f.Ez[id], (TP)f.Bz[id]};
        }
    }
    if constexpr (STAGED) __syncthreads();

    // 5x5 gather of the six fields at the midpoint (move.py:90-107).
    TP Ex = 0, Ey = 0, Ez = 0, Bx = 0, By = 0, Bz = 0;
    if (inside) {
        TP wx[5], wy[5];
        weights4<TP>((TP)xl, wx);
        weights4<TP>((TP)yl, wy);
        if (window) {
            const int base = (ix - box.r0) * width + iy - box.c0;
#pragma unroll
            for (int kx = 0; kx < 5; ++kx) {
                const int row = base + kx * width;
#pragma unroll
                for (int ky = 0; ky < 5; ++ky) {
                    const TP w = wx[kx] * wy[ky];
                    const FieldPair<TP> fx = s_f[0][row + ky], fy = s_f[1][row + ky],
                                        fz = s_f[2][row + ky];
                    Ex += fx.a * w;
                    Bx += fx.b * w;
                    Ey += fy.a * w;
                    By += fy.b * w;
                    Ez += fz.a * w;
                    Bz += fz.b * w;
                }
            }
        } else {
#pragma unroll
            for (int kx = 0; kx < 5; ++kx) {
                const int row = (ix + kx - 2) * N + iy - 2;
#pragma unroll
                for (int ky = 0; ky < 5; ++ky) {
                    const TP w = wx[kx] * wy[ky];
                    const int id = row + ky;
                    Ex += (TP)f.Ex[id] * w;
                    Bx += (TP)f.Bx[id] * w;
                    Ey += (TP)f.Ey[id] * w;
                    By += (TP)f.By[id] * w;
                    Ez += (TP)f.Ez[id] * w;
                    Bz += (TP)f.Bz[id] * w;
                }
            }
        }
    }

    int key = -1;
    if (live) {
        // Two fixed-point passes of the momentum update (move.py:110-125).
        const double qd = (double)q * dxi;
        TP dpx, dpy, dpz;
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            const double P = px, Q = py, R = pz;
            const double gm = sqrt(m * m + R * R + P * P + Q * Q);
            double ux, uy, uz;
            if constexpr (RCP) {
                const double ig = 1 / gm;
                ux = P * ig;
                uy = Q * ig;
                uz = R * ig;
            } else {
                ux = P / gm;
                uy = Q / gm;
                uz = R / gm;
            }
            const TP vx = (TP)ux, vy = (TP)uy, vz = (TP)uz;
            const TP factor = (TP)(qd / (1 - uz));
            dpx = factor * (Ex + vy * Bz - vz * By);
            dpy = factor * (Ey - vx * Bz + vz * Bx);
            dpz = factor * (Ez + vx * By - vy * Bx);
            px = opx + dpx * TP(0.5);
            py = opy + dpy * TP(0.5);
            pz = opz + (double)(dpz * TP(0.5));
        }

        // Position from the half-step momentum, then the full-step momentum.
        double xo, yo;
        {
            const double P = px, Q = py, R = pz;
            const double gm = sqrt(m * m + R * R + P * P + Q * Q);
            const double d = gm - R;
            if constexpr (RCP) {
                const double r = dxi / d;
                xo = xop + P * r;
                yo = yop + Q * r;
            } else {
                xo = xop + P / d * dxi;
                yo = yop + Q / d * dxi;
            }
        }
        px = opx + dpx;
        py = opy + dpy;
        pz = opz + (double)dpz;

        x = xi0 + xo;
        y = yi0 + yo;
        if (reflect(xi0, yi0, b, x, y, xo, yo)) {
            px = py = TP(0);
            pz = 0;
        }
        x = xi0 + xo;
        y = yi0 + yo;
        bool absorbed = false;
        if (x >= b || x <= -b || y >= b || y <= -b) {
            xo = yo = 0;
            px = py = TP(0);
            pz = 0;
            absorbed = true;
        }

        a.xo[k] = xo;
        a.yo[k] = yo;
        if (momenta || absorbed) {
            a.px[k] = px;
            a.py[k] = py;
            a.pz[k] = pz;
        }
        if (FIRST || absorbed) a.q[k] = absorbed ? TP(0) : q;

        if (BIN && !absorbed)
            key = bin_particle<TP>(xi0 + xo, yi0 + yo, g.h, N, (double)px, (double)py, (double)pz,
                                   m, (double)q, static_cast<DepRec<TP> *>(bs.rec), j, bs.err);
    } else if (FIRST && have) {
        a.xo[k] = xof;
        a.yo[k] = yof;
        a.px[k] = opx;
        a.py[k] = opy;
        a.pz[k] = opz;
        a.q[k] = q;
    }
    if (BIN) {
        // Unbinned particles are counted (and ranked) in count[cell_keys(N)].
        // Threads without a particle stay to the count so that whole waves
        // reach it.
        const int r = count_rank(bs.count, have ? (key >= 0 ? key : cell_keys(N)) : -1);
        if (have) {
            bs.key[j] = key;
            bs.pid[j] = (int)k;
            bs.rank[j] = r;
        }
    }
}

template <typename TP>
hipError_t launch_move_wo_fields(int64_t n, double xi_step, const TP *m, double *xo, double *yo,
                                 const TP *px, const TP *py, const double *pz, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int blocks = (int)((n + 255) / 256);
    k_move_wo_fields<TP><<<blocks, 256, 0, s>>>(n, xi_step, m, xo, yo, px, py, pz);
    return hipGetLastError();
}

template <typename TP, typename TF>
hipError_t launch_push(const PushGeom &g, const Fields6<TF> &f, const SortArrays<TP> &a,
                       bool first, bool bin, bool momenta, const BinState &bs, const int *order,
                       hipStream_t s, KernelTimer *timer)
{
    if (g.n <= 0) return hipSuccess;
    hipError_t e;
    if (timer && (e = timer->begin(KC_PUSH, 1, s)) != hipSuccess) return e;
    auto launch = [&](auto first_c, auto bin_c) {
        constexpr bool FIRST = decltype(first_c)::value, BIN = decltype(bin_c)::value;
        if (g.n < PUSH_FEW) {
            const int blocks = (int)((g.n + PUSH_FEW_THREADS - 1) / PUSH_FEW_THREADS);
            k_push<TP, TF, FIRST, BIN, false><<<blocks, PUSH_FEW_THREADS, 0, s>>>(
                g, f, a, bs, order, 0, momenta);
            return;
        }
        // Without an order the blocks take tiles of the particles' square
        // lattice: a run of 256 particles of one lattice row would span a
        // window of a hundred cells.
        int side = order ? 0 : (int)std::lround(std::sqrt((double)g.n));
        if ((int64_t)side * side != g.n) side = 0;
        const int64_t tiles = (side + PUSH_TILE - 1) / PUSH_TILE;
        const int blocks = (int)(side ? tiles * tiles : (g.n + PUSH_THREADS - 1) / PUSH_THREADS);
        k_push<TP, TF, FIRST, BIN, true><<<blocks, PUSH_THREADS, 0, s>>>(g, f, a, bs, order, side,
                                                                         momenta);
    };
    if (first && bin) launch(std::true_type{}, std::true_type{});
    else if (first) launch(std::true_type{}, std::false_type{});
    else if (bin) launch(std::false_type{}, std::true_type{});
    else launch(std::false_type{}, std::false_type{});
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (timer) return timer->end(s);
    return hipSuccess;
}

template hipError_t launch_move_wo_fields<double>(int64_t, double, const double *, double *,
                                                  double *, const double *, const double *,
                                                  const double *, hipStream_t);
template hipError_t launch_move_wo_fields<float>(int64_t, double, const float *, double *,
                                                 double *, const float *, const float *,
                                                 const double *, hipStream_t);
template hipError_t launch_push<double, double>(const PushGeom &, const Fields6<double> &,
                                                const SortArrays<double> &, bool, bool, bool,
                                                const BinState &, const int *, hipStream_t,
                                                KernelTimer *);
template hipError_t launch_push<float, double>(const PushGeom &, const Fields6<double> &,
                                               const SortArrays<float> &, bool, bool, bool,
                                                const BinState &, const int *, hipStream_t,
                                                KernelTimer *);
template hipError_t launch_push<float, float>(const PushGeom &, const Fields6<float> &,
                                              const SortArrays<float> &, bool, bool, bool,
                                                const BinState &, const int *, hipStream_t,
                                                KernelTimer *);

}  // namespace lc3d
