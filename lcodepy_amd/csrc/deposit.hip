// Plasma charge/current deposit (plasma3d/weights.py:35-67, 249-285), gfx950.
//
// The reference scatters 25 taps x 4 grids per particle (serially on the
// CPU, with float64 global atomics on the GPU).  Here the deposit is a
// gather over cell-sorted particles:
//
//   1. bin      cell of every particle (fused into the push when possible),
//               written with its deposit record at its binning position
//               (the binning thread's index, so the writes are contiguous),
//               integer atomic count per cell (one atomic per run of equal
//               cells in a wave), which also gives each particle its rank in
//               its cell;
//   2. scan     exclusive prefix of the counts -> start of each cell's list
//               (the counts are cleared for the next deposit); cells of more
//               than SMALL_CELL particles are queued as dense;
//   3. scatter  binning positions and particle ids into their cell's list at
//               their ranks; the ids are the cell order the next push visits
//               (so binning positions follow the cell order, and a cell's
//               records lie close together);
//   4. dense    per dense cell its list in particle-id order and its 5 x 5 x 4
//               taps, by a wave, four waves or a workgroup with a fixed-order
//               reduction;
//   5. gather   one workgroup per tile of output cells sorts the lists of the
//               source cells around it by particle id, stages their records
//               in LDS and sums them, every output cell in a fixed order.
//
// A cell's particles are always summed in the order of their ids, so that no
// sum depends on atomic arrival order or on the order the particles were
// visited in.
// Every output value is written by exactly one thread: no floating-point
// atomics, and the result is bit-reproducible run to run.  The sums over cells
// are float64 in both forms.
#include "common.h"
#include "kernels.h"

#include <climits>
#include <type_traits>

namespace lc3d {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_PER = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_PER;
static_assert(SCAN_TILE == SCAN_TILE_CELLS, "scan tiles as allocated");
constexpr int SMALL_CELL = 16;          // lists a gather thread sorts; longer ones are dense
constexpr int WAVE_CELL = 64;           // dense lists up to this long are one wave's
constexpr int MAX_SORTED_CELL = 16384;  // lists sorted by a workgroup in LDS

// ---- binning ------------------------------------------------------------------
template <typename TP>
__global__ __launch_bounds__(256) void k_bin(int64_t n, double h, int N,
                                             const double *__restrict__ x_init,
                                             const double *__restrict__ y_init,
                                             const double *__restrict__ xo,
                                             const double *__restrict__ yo,
                                             const TP *__restrict__ px, const TP *__restrict__ py,
                                             const double *__restrict__ pz, const TP *__restrict__ q,
                                             const TP *__restrict__ m, BinState bs)
{
    clear_scan(bs);
    // Threads past the end stay to the count so that whole waves reach it.
    // Particle k is binned at position k.
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    int key = -1;
    if (k < n) {
        if (q[k] != TP(0))
            key = bin_particle<TP>(x_init[k] + xo[k], y_init[k] + yo[k], h, N, (double)px[k],
                                   (double)py[k], (double)pz[k], (double)m[k], (double)q[k],
                                   static_cast<DepRec<TP> *>(bs.rec), k, bs.err);
        bs.key[k] = key;
        bs.pid[k] = (int)k;
    }
    // Unbinned particles are counted (and ranked) in count[cell_keys(N)].
    const int r = count_rank(bs.count, k < n ? (key >= 0 ? key : cell_keys(N)) : -1);
    if (k < n) bs.rank[k] = r;
}

// ---- exclusive scan of the cell counts ---------------------------------------------
// Inclusive scan of v over the wave's lanes in order (__shfl_up steps).
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(v, d);
        if (lane >= d) v += u;
    }
    return v;
}

// Exclusive scan of v over the block's SCAN_THREADS threads (every thread
// calls it); total = the block's sum.  The waves scan themselves, then add
// the totals of the waves before them (sh: SCAN_THREADS / 64 ints).
__device__ __forceinline__ int block_exclusive_scan(int v, int *sh, int &total)
{
    constexpr int W = SCAN_THREADS / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int incl = wave_inclusive_scan(v);
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    int off = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const int t = sh[w];
        off += w < wave ? t : 0;
        sum += t;
    }
    total = sum;
    __syncthreads();   // sh is reused by the next call
    return off + incl - v;
}

// One pass, no block waiting for another.  Each block scans its tile of
// SCAN_TILE cells into lstart (starts within the tile, lstart[ncell] included)
// and clears the counts it read (ready for the next binning pass); then adds
// the tile's total to base[t] of every later tile t by integer atomics, so
// that when the pass has ended base[t] is the sum of the tiles before t,
// whatever order the blocks ran in.  A cell's list starts at
// lstart[c] + base[c / SCAN_TILE] (list_start).  base and the queue of dense
// cells are empty when the pass begins (the binning pass clears them); a dense
// cell takes a slot of the queue (at most n / (SMALL_CELL + 1) < bigcap cells
// can be dense), those of at most WAVE_CELL particles from its front and the
// others from its back, and dslot is written, and read, for dense cells only.
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_cells(int ncell, int ntiles, BinState bs)
{
    __shared__ int sh[SCAN_THREADS / 64];
    int *__restrict__ count = bs.count;
    const int first = blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER;
    // A thread's counts and starts are whole int4s, but at the end of the cells
    // (word by word, each access of a wave touched 16 lines: N = 1025 19.7 -> 15.6
    // us, 513 7.1 -> 5.4, 129 4.9 -> 3.2).  The rest at 1025 is the tiles' atomics;
    // tiles of 4096 cells took 10 us there but 6.0 at 513 and 4.3 at 129.
    const bool whole = first + SCAN_PER <= ncell;
    int4 *__restrict__ count4 = reinterpret_cast<int4 *>(count + first);
    int4 *__restrict__ lstart4 = reinterpret_cast<int4 *>(bs.lstart + first);
    int c[SCAN_PER], start[SCAN_PER];
    int s = 0;
    if (whole) {
#pragma unroll
        for (int i = 0; i < SCAN_PER / 4; ++i) {
            const int4 v = count4[i];
            c[4 * i] = v.x;
            c[4 * i + 1] = v.y;
            c[4 * i + 2] = v.z;
            c[4 * i + 3] = v.w;
            count4[i] = int4{0, 0, 0, 0};
        }
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_PER; ++i) {
            c[i] = first + i < ncell ? count[first + i] : 0;
            if (first + i < ncell) count[first + i] = 0;
        }
    }
#pragma unroll
    for (int i = 0; i < SCAN_PER; ++i) s += c[i];
    int total;
    int run = block_exclusive_scan(s, sh, total);
#pragma unroll
    for (int i = 0; i < SCAN_PER; ++i) {
        start[i] = run;
        run += c[i];
    }
    if (whole) {
#pragma unroll
        for (int i = 0; i < SCAN_PER / 4; ++i)
            lstart4[i] = int4{start[4 * i], start[4 * i + 1], start[4 * i + 2], start[4 * i + 3]};
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_PER; ++i)
            if (first + i <= ncell) bs.lstart[first + i] = start[i];
    }
#pragma unroll
    for (int i = 0; i < SCAN_PER; ++i) {
        if (c[i] > SMALL_CELL) {
            // Two atomics, so that each is at one address and a wave's add as one.
            int slot;
            if (c[i] <= WAVE_CELL) slot = atomicAdd(&bs.nbig[0], 1);
            else slot = bs.bigcap - 1 - atomicAdd(&bs.nbig[1], 1);
            if (slot >= 0 && slot < bs.bigcap) bs.big[slot] = first + i;
            bs.dslot[first + i] = slot;
            if (c[i] > MAX_SORTED_CELL) atomicOr(bs.err, ERR_CELL_OVERFLOW);
        }
    }
    if (total != 0)
        for (int t = blockIdx.x + 1 + threadIdx.x; t < ntiles; t += SCAN_THREADS)
            atomicAdd(&bs.base[t], total);
}

// Start of cell c's list (c <= ncell) after k_scan_cells.
__device__ __forceinline__ int list_start(const BinState &bs, int c)
{
    return bs.lstart[c] + bs.base[c / SCAN_TILE];
}

// ---- scatter positions into the cell lists ---------------------------------------
// Places binning position j, and the particle binned there, at its rank in
// its cell's list; particles that are not binned (q = 0 or off the grid) go
// after all the lists, at their rank among the unbinned ones, so that pos and
// idx are permutations.  count[ncell] counted them and is cleared here.
__global__ __launch_bounds__(256) void k_scatter(int64_t n, int ncell, BinState bs)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (j >= n) return;
    if (j == 0) bs.count[ncell] = 0;
    const int key = bs.key[j];
    const int slot = list_start(bs, key < 0 ? ncell : key) + bs.rank[j];
    bs.pos[slot] = (int)j;
    bs.idx[slot] = bs.pid[j];
}

// ---- dense cells: sort and taps ------------------------------------------------------
// The 5 x 5 taps x 4 currents around each dense cell, out[slot][tap][q], tap =
// 5 a + b for the target cell (ix + a - 2, iy + b - 2), q = ro jx jy jz.  The
// cell's list is sorted by particle id (lists of more than MAX_SORTED_CELL keep
// arrival order); particle i of it is summed by thread i (of DENSE_THREADS,
// each a contiguous segment of a longer list), and the threads' sums are
// combined by a butterfly within each wave and then the four waves in a fixed
// order.  The butterfly hands half of the values that are left to the partner
// lane at every step (a sixth of the shuffles, the same sums).
//
// A list of at most WAVE_CELL particles is one wave's, one of at most
// DENSE_THREADS four waves', which rank it by comparing ids; a longer one is
// sorted in the workgroup's LDS.  One workgroup per list of any length left 4
// waves on a CU (N = 513, 16 ppc, float64: 2424 -> 144 us; lists of about 180,
// N = 417, float32: 30 -> 25 us).
constexpr int DENSE_VALUES = 25 * 4;
constexpr int DENSE_THREADS = 256;   // of a list longer than a wave
constexpr int DENSE_BLOCK = 2 * DENSE_THREADS, DENSE_WAVES = DENSE_BLOCK / 64;

// Two of the four currents of one particle at a time (PAIR_VALUES sums a
// lane: all four would spill in float64): acc[2 (5 a + b) + r] += c_r w_a w_b.
constexpr int PAIR_VALUES = DENSE_VALUES / 2;
template <typename T>
__device__ __forceinline__ void add_pair_taps(const DepRec<T> &d, int pair, T inv_h,
                                              T (&acc)[PAIR_VALUES])
{
    const T c0 = pair ? d.c2 : d.c0, c1 = pair ? d.c3 : d.c1;
    T wx[5], wy[5];
    weights4<T>(d.xl, wx);
    weights4<T>(d.yl, wy);
#pragma unroll
    for (int a = 0; a < 5; ++a) {
#pragma unroll
        for (int b = 0; b < 5; ++b) {
            const T w = (wx[a] * inv_h) * (wy[b] * inv_h);
            acc[2 * (5 * a + b) + 0] += c0 * w;
            acc[2 * (5 * a + b) + 1] += c1 * w;
        }
    }
}

// One step of the halving butterfly: M values at distance off become (M + 1) / 2,
// the sums over the lane pair of the lower half (lanes without bit off) or
// the upper one.
template <int M, typename T, int K>
__device__ __forceinline__ void halve(T (&v)[K], int off, bool upper)
{
    constexpr int H = (M + 1) / 2;
#pragma unroll
    for (int k = 0; k < H; ++k) {
        const T lo = v[k], hi = H + k < M ? v[H + k] : T(0);
        v[k] = (upper ? hi : lo) + __shfl_xor(upper ? lo : hi, off);
    }
}

// The sums of a wave's PAIR_VALUES: lane's is value wave_value(lane), or none (-1).
template <typename T>
__device__ __forceinline__ T wave_sums(T (&v)[PAIR_VALUES], int lane)
{
    halve<50>(v, 32, lane & 32);
    halve<25>(v, 16, lane & 16);
    halve<13>(v, 8, lane & 8);
    halve<7>(v, 4, lane & 4);
    halve<4>(v, 2, lane & 2);
    halve<2>(v, 1, lane & 1);
    return v[0];
}
__device__ __forceinline__ int wave_value(int lane)
{
    constexpr int KEPT[6] = {25, 13, 7, 4, 2, 1};   // by the lower half of each step
    int value = 0, left = PAIR_VALUES;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const bool upper = lane & (32 >> k);
        value += upper ? KEPT[k] : 0;
        left = upper ? left - KEPT[k] : min(left, KEPT[k]);
    }
    return left > 0 ? value : -1;
}

template <typename T>
__global__ __launch_bounds__(DENSE_BLOCK) void k_dense_cells(double h, BinState bs)
{
    __shared__ __align__(16) unsigned long long s[MAX_SORTED_CELL];   // particle id << 32 | position
    __shared__ T red[DENSE_WAVES][PAIR_VALUES];
    const int few = min(bs.nbig[0], bs.bigcap), many = min(bs.nbig[1], bs.bigcap - few);
    const DepRec<T> *__restrict__ rec = static_cast<const DepRec<T> *>(bs.rec);
    T *__restrict__ out = static_cast<T *>(bs.dense);
    const int t = threadIdx.x, lane = t % 64, wave = t / 64;
    const T inv_h = T(1.0 / h);
    const int value = wave_value(lane);

    for (int b = blockIdx.x * DENSE_WAVES + wave; b < few; b += gridDim.x * DENSE_WAVES) {
        const int c = bs.big[b];
        const int st = list_start(bs, c), n = list_start(bs, c + 1) - st;   // n <= WAVE_CELL
        int id = INT_MAX, at = 0;
        if (lane < n) {
            id = bs.idx[st + lane];
            at = bs.pos[st + lane];
        }
        // Lane i takes the particle whose id has i smaller ones before it.
        int place = 0, from = 0;
        for (int j = 0; j < n; ++j) place += __shfl(id, j) < id ? 1 : 0;
        for (int j = 0; j < n; ++j)
            if (__shfl(place, j) == lane) from = j;
        at = __shfl(at, from);
        DepRec<T> d{};
        if (lane < n) d = rec[at];
#pragma unroll 1
        for (int pair = 0; pair < 2; ++pair) {
            T acc[PAIR_VALUES];
#pragma unroll
            for (int k = 0; k < PAIR_VALUES; ++k) acc[k] = T(0);
            if (lane < n) add_pair_taps<T>(d, pair, inv_h, acc);
            const T v = wave_sums(acc, lane);
            if (value >= 0)
                out[(size_t)b * DENSE_VALUES + 4 * (value / 2) + 2 * pair + value % 2] = v;
        }
    }

    // The longer lists, two to a workgroup: half of its waves each.  Every
    // thread reaches the barriers, also without a list.
    const int half = t / DENSE_THREADS, u = t % DENSE_THREADS;
    int *ids = reinterpret_cast<int *>(s) + half * 2 * DENSE_THREADS, *order = ids + DENSE_THREADS;
    for (int b0 = 2 * blockIdx.x; b0 < many; b0 += 2 * gridDim.x) {
        {
            const int b = bs.bigcap - 1 - (b0 + half);
            int st = 0, n = 0;
            if (b0 + half < many) {
                const int c = bs.big[b];
                st = list_start(bs, c);
                n = list_start(bs, c + 1) - st;
                if (n > DENSE_THREADS) n = 0;
            }
            int id = INT_MAX, at = 0;
            if (u < n) {
                id = bs.idx[st + u];
                at = bs.pos[st + u];
            }
            ids[u] = id;
            __syncthreads();
            int rank = 0;
            for (int j = 0; j < n; j += 4) {   // past the list: INT_MAX, not less
                const int4 o = *reinterpret_cast<const int4 *>(ids + j);
                rank += (o.x < id) + (o.y < id) + (o.z < id) + (o.w < id);
            }
            if (u < n) order[rank] = at;
            __syncthreads();
            DepRec<T> d{};
            if (u < n) d = rec[order[u]];
#pragma unroll 1
            for (int pair = 0; pair < 2; ++pair) {
                T acc[PAIR_VALUES];
#pragma unroll
                for (int k = 0; k < PAIR_VALUES; ++k) acc[k] = T(0);
                if (u < n) add_pair_taps<T>(d, pair, inv_h, acc);
                const T v = wave_sums(acc, lane);
                if (value >= 0) red[wave][value] = v;
                __syncthreads();
                if (n > 0 && u < PAIR_VALUES) {
                    const T (*r)[PAIR_VALUES] = red + half * (DENSE_THREADS / 64);
                    out[(size_t)b * DENSE_VALUES + 4 * (u / 2) + 2 * pair + u % 2] =
                        (r[0][u] + r[1][u]) + (r[2][u] + r[3][u]);
                }
                __syncthreads();
            }
        }
        for (int k = b0; k < min(b0 + 2, many); ++k) {   // the whole block
            const int b = bs.bigcap - 1 - k, c = bs.big[b];
            const int st = list_start(bs, c), n = list_start(bs, c + 1) - st;
            if (n <= DENSE_THREADS) continue;
            const bool sorted = n <= MAX_SORTED_CELL;
            if (sorted) {
                int P = 1;
                while (P < n) P <<= 1;
                for (int i = t; i < P; i += DENSE_BLOCK) {
                    unsigned long long v = ~0ull;
                    if (i < n)
                        v = (unsigned long long)(unsigned)bs.idx[st + i] << 32 |
                            (unsigned)bs.pos[st + i];
                    s[i] = v;
                }
                __syncthreads();
                for (int w = 2; w <= P; w <<= 1) {
                    for (int j = w >> 1; j > 0; j >>= 1) {
                        for (int i = t; i < P; i += DENSE_BLOCK) {
                            const int l = i ^ j;
                            if (l > i) {
                                const unsigned long long x = s[i], y = s[l];
                                if ((x > y) == ((i & w) == 0)) {
                                    s[i] = y;
                                    s[l] = x;
                                }
                            }
                        }
                        __syncthreads();
                    }
                }
            }
            // Both halves sum the list, a pair of currents each.
            T acc[PAIR_VALUES];
#pragma unroll
            for (int q = 0; q < PAIR_VALUES; ++q) acc[q] = T(0);
            const int seg = (n + DENSE_THREADS - 1) / DENSE_THREADS;
            const int j0 = min(n, u * seg), j1 = min(n, (u + 1) * seg);
            for (int j = j0; j < j1; ++j)
                add_pair_taps<T>(rec[sorted ? (int)(unsigned)s[j] : bs.pos[st + j]], half, inv_h,
                                 acc);
            const T v = wave_sums(acc, lane);
            if (value >= 0) red[wave][value] = v;
            __syncthreads();
            if (u < PAIR_VALUES) {
                const T (*r)[PAIR_VALUES] = red + half * (DENSE_THREADS / 64);
                out[(size_t)b * DENSE_VALUES + 4 * (u / 2) + 2 * half + u % 2] =
                    (r[0][u] + r[1][u]) + (r[2][u] + r[3][u]);
            }
            __syncthreads();   // s and red are written again
        }
    }
}

// ---- gather deposit -------------------------------------------------------------------
// One block per tile of TX x GATHER_TY output cells; per output row ox of the
// tile and source column cy (GATHER_TY + 4 = 32 of them, half a wave) G
// threads, each for 4 / G of the currents.  A thread adds the particles of the
// five source cells (ox - 2 .. ox + 2, cy), each with its x weight towards row
// ox, into the five y taps of its currents, in registers; the taps meet at the
// end by shuffles along the half wave, where output cell (ox, o) takes tap b of
// column o + 2 - b.
//
// The records of the source cells are staged in LDS, as many whole source
// rows at a time as GatherPlan::cap holds (a row's lists of at most
// SMALL_CELL particles always fit), in the order of their particle ids: a
// thread per cell ranks its list's ids in registers.  Reading them from
// memory, once per x offset, was 23.8e6 cache accesses a deposit in float64,
// two thirds of the time; the taps of every x offset also passed through LDS
// with a barrier each, and 80 KB a block left two blocks to a CU.
// Measured with the list sort it replaces: N = 513, 4 ppc 92 -> 55 us in
// float64 and 48 -> 34 us in float32; 769, 9 ppc, float64 508 -> 238 us; 321, 4
// ppc, float64 48 -> 32 us.  It is bound by the vector units (the waves run as
// long as their fullest cells) and by the blocks' chain of list, record and
// sum.  Staging with a thread per particle instead of a thread per cell took
// 65 us in float32 (its ranks are a serial chain of LDS reads).
// A grid of fewer blocks of TX = 8, G = 1 than GATHER_FEW takes TX = 4, G = 2:
// a CU holds several blocks, and each has more waves for its chain.  The
// second weights cost less than that until the vector units are full.
// Measured, TX = 8, G = 1 against TX = 4, G = 2 (N = 513, 1368 blocks of the
// first: 54.8 us against 56.5 in float64 and 37.2 against 34.3 in float32; 769,
// 2912, float64, 237 against 271; 1025, 5032, float32, 118 against 125), and
// TX = 4, G = 2 against TX = 4, G = 1
// (281, 4 ppc, float32, 20.1 us against 26.0; 321 float64 32.4 against 35.0;
// 129 float64 9.4 against 11.6).
template <typename T> constexpr int GATHER_FEW = sizeof(T) == 4 ? 2048 : 1024;
constexpr int GATHER_TY = 28, GATHER_COLS = GATHER_TY + 4;
static_assert(GATHER_COLS == 32, "a source row is half a wave");
// cap: records staged at a time (31 KB; a block's LDS is 36 to 41 KB in all,
// four blocks a CU).
template <typename T> struct GatherPlan {
    static constexpr int cap = sizeof(T) == 4 ? 1280 : 640;
    static_assert(cap >= GATHER_COLS * SMALL_CELL, "one source row always fits");
};

// The places (ranks by particle id) of a list's n <= W particles, and their
// binning positions into out in that order.  W registers a particle's worth:
// the caller takes the smallest W of 4, 8, 16 that serves its wave.
template <int W>
__device__ __forceinline__ void order_list(const int *__restrict__ idx,
                                           const int *__restrict__ pos, int n, int *out)
{
    int id[W], at[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        id[k] = k < n ? idx[k] : INT_MAX;
        at[k] = k < n ? pos[k] : 0;
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
        int rank = 0;
#pragma unroll
        for (int j = 0; j < W; ++j) rank += id[j] < id[k] ? 1 : 0;
        if (k < n) out[rank] = at[k];
    }
}

// Adds Q of a particle's currents, from the first'th on, to its taps toward x
// offset A (target cells (ix + A - 2, iy + b - 2)): tp[b][q] += c_q (w_A(xl) / h)
// (w_b(yl) / h).  Float32 takes the current times the x weight first, float64
// the weight product first (plasma3d/weights.py:58-67).
template <int A, int Q, typename T>
__device__ __forceinline__ void add_taps(const DepRec<T> &d, int first, T inv_h, T (&tp)[5][Q])
{
    const T *c = &d.c0 + first;
    T wy[5];
    weights4<T>(d.yl, wy);
#pragma unroll
    for (int b = 0; b < 5; ++b) wy[b] *= inv_h;
    const T wx = w4_tap<A, T>(d.xl) * inv_h;
    if constexpr (std::is_same<T, float>::value) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const T cw = c[q] * wx;
#pragma unroll
            for (int b = 0; b < 5; ++b) tp[b][q] += cw * wy[b];
        }
    } else {
#pragma unroll
        for (int b = 0; b < 5; ++b) {
            const T w = wx * wy[b];
#pragma unroll
            for (int q = 0; q < Q; ++q) tp[b][q] += c[q] * w;
        }
    }
}

// Every output value is the sum, in a fixed order, of the taps that reach it:
// per source column the five source cells in order, each cell's particles in
// the order of their ids (float32: a cell's sum in float32, then float64),
// then the five columns in float64; written by one thread.
template <typename TP, typename TG, int TX, int G>
__global__ __launch_bounds__(TX *GATHER_COLS *G) void k_deposit_gather(
    int N, double h, BinState bs, TG *__restrict__ ro, TG *__restrict__ jx, TG *__restrict__ jy,
    TG *__restrict__ jz, const TG *__restrict__ bg_ro, TG *__restrict__ ro1, TG *__restrict__ jx1,
    TG *__restrict__ jy1, TG *__restrict__ jz1)
{
    using T = TP;   // arithmetic type of the taps
    constexpr int Q = 4 / G, THREADS = TX * GATHER_COLS * G, ROWS = TX + 4, CELLS = ROWS * GATHER_COLS;
    constexpr int CAP = GatherPlan<T>::cap, CHUNKS = CELLS / 64, WAVES = THREADS / 64;
    static_assert(CELLS % 64 == 0, "the prefix takes whole waves of cells");
    __shared__ DepRec<T> s_rec[CAP];
    __shared__ int s_pos[CAP];           // binning positions of the staged records
    __shared__ int s_first[CELLS];       // a source cell's list start
    __shared__ int s_dense[CELLS];       // its slot if it is dense, else -1
    __shared__ int s_off[CELLS + 1];     // particles in the cells before it (dense cells none)
    __shared__ int s_sum[CHUNKS];

    // Tile rows are dealt to the XCDs in turn: contiguous bands of the grid
    // left the XCDs of the outer bands idle, where there is little plasma
    // (76 -> 55 us in float64 at N = 513).
    const int tpr = (N + GATHER_TY - 1) / GATHER_TY;
    const int local = blockIdx.x / 8;
    const int X0 = (local / tpr * 8 + blockIdx.x % 8) * TX, Y0 = (local % tpr) * GATHER_TY;
    if (X0 >= N) return;
    const DepRec<T> *__restrict__ rec = static_cast<const DepRec<T> *>(bs.rec);
    const T *__restrict__ dense = static_cast<const T *>(bs.dense);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;

    // Source cell c of the tile: row c / 32, column c % 32 from (X0 - 2, Y0 - 2);
    // none outside the grid.
    for (int c = t; c < CELLS; c += THREADS) {
        const int cx = X0 - 2 + c / GATHER_COLS, cy = Y0 - 2 + c % GATHER_COLS;
        int first = 0, n = 0, slot = -1;
        if (cx >= 0 && cx < N && cy >= 0 && cy < N) {
            const int key = cell_key(cx, cy, N);
            first = list_start(bs, key);
            n = list_start(bs, key + 1) - first;
            if (n > SMALL_CELL) {
                slot = bs.dslot[key];
                n = 0;
            }
        }
        s_first[c] = first;
        s_dense[c] = slot;
        s_off[c + 1] = n;
    }
    __syncthreads();
    for (int k = wave; k < CHUNKS; k += WAVES) {
        const int v = wave_inclusive_scan(s_off[64 * k + lane + 1]);
        s_off[64 * k + lane + 1] = v;
        if (lane == 63) s_sum[k] = v;
    }
    __syncthreads();
    for (int k = wave; k < CHUNKS; k += WAVES) {
        int before = 0;
        for (int q = 0; q < k; ++q) before += s_sum[q];
        s_off[64 * k + lane + 1] += before;
    }
    if (t == 0) s_off[0] = 0;
    __syncthreads();

    const int cy = t % GATHER_COLS, ox = t / GATHER_COLS % TX, g = t / (GATHER_COLS * TX);
    const T inv_h = T(1.0 / h);
    double sum[5][Q];
#pragma unroll
    for (int b = 0; b < 5; ++b)
#pragma unroll
        for (int q = 0; q < Q; ++q) sum[b][q] = 0;

    int r0 = 0;
    while (r0 < ROWS) {   // source rows r0 .. r1 - 1, the same for every thread
        const int base = s_off[GATHER_COLS * r0];
        int r1 = r0 + 1;
        while (r1 < ROWS && s_off[GATHER_COLS * (r1 + 1)] - base <= CAP) ++r1;
        const int total = s_off[GATHER_COLS * r1] - base;
        // Whole waves reach the ballots: the loop's bound is rounded up to them.
        const int cells = GATHER_COLS * (r1 - r0), whole = (cells + 63) & ~63;
        for (int i = t; i < whole; i += THREADS) {
            const int c = GATHER_COLS * r0 + i;
            int n = 0, off = 0, first = 0;
            if (i < cells) {
                off = s_off[c] - base;
                n = s_off[c + 1] - base - off;
                first = s_first[c];
            }
            const int *idx = bs.idx + first, *pos = bs.pos + first;
            if (__ballot(n > 8)) order_list<16>(idx, pos, n, s_pos + off);
            else if (__ballot(n > 4)) order_list<8>(idx, pos, n, s_pos + off);
            else order_list<4>(idx, pos, n, s_pos + off);
        }
        __syncthreads();
        // Two records in flight a thread (57 -> 50 us where a few cells hold most
        // of the plasma; four: slower where the lists are even).
        for (int i = t; i < total; i += 2 * THREADS) {
            const int j = min(i + THREADS, total - 1);
            const DepRec<T> a = rec[s_pos[i]], b = rec[s_pos[j]];
            s_rec[i] = a;
            if (i + THREADS < total) s_rec[j] = b;
        }
        __syncthreads();
        // Source row r reaches output row ox by x offset A = ox + 4 - r.
        auto visit = [&](auto a_const) {
            constexpr int A = decltype(a_const)::value;
            const int r = ox + 4 - A;
            if (r < r0 || r >= r1) return;
            const int c = GATHER_COLS * r + cy, slot = s_dense[c];
            if (slot >= 0) {
                const T *v = dense + (size_t)slot * DENSE_VALUES + 4 * (5 * A) + Q * g;
#pragma unroll
                for (int b = 0; b < 5; ++b)
#pragma unroll
                    for (int q = 0; q < Q; ++q) sum[b][q] += (double)v[4 * b + q];
                return;
            }
            const int e = s_off[c + 1] - base;
            if constexpr (std::is_same<T, float>::value) {
                T tp[5][Q];
#pragma unroll
                for (int b = 0; b < 5; ++b)
#pragma unroll
                    for (int q = 0; q < Q; ++q) tp[b][q] = T(0);
                for (int i = s_off[c] - base; i < e; ++i)
                    add_taps<A, Q, T>(s_rec[i], Q * g, inv_h, tp);
#pragma unroll
                for (int b = 0; b < 5; ++b)
#pragma unroll
                    for (int q = 0; q < Q; ++q) sum[b][q] += (double)tp[b][q];
            } else {
                for (int i = s_off[c] - base; i < e; ++i)
                    add_taps<A, Q, T>(s_rec[i], Q * g, inv_h, sum);
            }
        };
        visit(std::integral_constant<int, 4>{});
        visit(std::integral_constant<int, 3>{});
        visit(std::integral_constant<int, 2>{});
        visit(std::integral_constant<int, 1>{});
        visit(std::integral_constant<int, 0>{});
        __syncthreads();   // s_pos and s_rec are written again
        r0 = r1;
    }

    // Output column o = cy of the tile sums tap b of source column cy + 4 - b.
    double out[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        out[q] = 0;
#pragma unroll
        for (int b = 0; b < 5; ++b) out[q] += b < 4 ? __shfl(sum[b][q], (lane + 4 - b) & 63) : sum[b][q];
    }
    const int gx = X0 + ox, gy = Y0 + cy;
    if (cy < GATHER_TY && gx < N && gy < N) {
        const int o = gx * N + gy;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int c = Q * g + q;
            (c == 0 ? ro : c == 1 ? jx : c == 2 ? jy : jz)[o] = (TG)out[q];
            if (bg_ro != nullptr)
                (c == 0 ? ro1 : c == 1 ? jx1 : c == 2 ? jy1 : jz1)[o] = c == 0 ? bg_ro[o] : TG(0);
        }
    }
}

template <typename TP, typename TG>
hipError_t launch_deposit(const PushGeom &g, const SortArrays<TP> &a, bool use_full, bool binned,
                          const BinState &bs, TG *ro, TG *jx, TG *jy, TG *jz, const TG *bg_ro,
                          TG *ro1, TG *jx1, TG *jy1, TG *jz1, hipStream_t s, KernelTimer *timer)
{
    const int N = g.N;
    const int ncell = cell_keys(N);
    const double *xo = use_full ? a.xo : a.xo_prev;
    const double *yo = use_full ? a.yo : a.yo_prev;
    const TP *px = use_full ? a.px : a.px_prev;
    const TP *py = use_full ? a.py : a.py_prev;
    const double *pz = use_full ? a.pz : a.pz_prev;
    const TP *q = use_full ? a.q : a.q_prev;
    const int pblocks = (int)((g.n + 255) / 256);
    const int ntiles = scan_tiles(ncell);   // cells 0..ncell
    if (ntiles != bs.nbase) return hipErrorInvalidValue;
    hipError_t e;
    if (timer && (e = timer->begin(KC_DEPOSIT, 1, s)) != hipSuccess) return e;
    if (g.n > 0) {
        if (!binned)
            k_bin<TP><<<pblocks, 256, 0, s>>>(g.n, g.h, N, a.x_init, a.y_init, xo, yo, px, py, pz,
                                              q, a.m, bs);
        k_scan_cells<<<ntiles, SCAN_THREADS, 0, s>>>(ncell, ntiles, bs);
        k_scatter<<<pblocks, 256, 0, s>>>(g.n, ncell, bs);
        // One block per CU (a block takes 134 KB of LDS): the queue is striding.
        k_dense_cells<TP><<<256, DENSE_BLOCK, 0, s>>>(g.h, bs);
    } else {
        // Empty sort: every cell list is empty (the binning pass, which has no
        // particle, clears what the scan adds to).
        k_bin<TP><<<1, 256, 0, s>>>(0, g.h, N, a.x_init, a.y_init, xo, yo, px, py, pz, q, a.m, bs);
        k_scan_cells<<<ntiles, SCAN_THREADS, 0, s>>>(ncell, ntiles, bs);
    }
    const int tpr = (N + GATHER_TY - 1) / GATHER_TY;
    // Tile rows rounded up to a multiple of the XCDs.
    const int tiles8 = ((N + 7) / 8 + 7) / 8 * 8 * tpr, tiles4 = ((N + 3) / 4 + 7) / 8 * 8 * tpr;
    if (tiles8 < GATHER_FEW<TP>)
        k_deposit_gather<TP, TG, 4, 2><<<tiles4, 8 * GATHER_COLS, 0, s>>>(
            N, g.h, bs, ro, jx, jy, jz, bg_ro, ro1, jx1, jy1, jz1);
    else
        k_deposit_gather<TP, TG, 8, 1><<<tiles8, 8 * GATHER_COLS, 0, s>>>(
            N, g.h, bs, ro, jx, jy, jz, bg_ro, ro1, jx1, jy1, jz1);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (timer) return timer->end(s);
    return hipSuccess;
}

template hipError_t launch_deposit<double, double>(const PushGeom &, const SortArrays<double> &,
                                                   bool, bool, const BinState &, double *,
                                                   double *, double *, double *, const double *,
                                                   double *, double *, double *, double *,
                                                   hipStream_t, KernelTimer *);
template hipError_t launch_deposit<float, float>(const PushGeom &, const SortArrays<float> &,
                                                 bool, bool, const BinState &, float *, float *,
                                                 float *, float *, const float *, float *,
                                                 float *, float *, float *, hipStream_t, KernelTimer *);

}  // namespace lc3d
