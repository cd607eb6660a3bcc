// FP64 geometric multigrid for the Poisson initialisation (PoissonSolver.cpp:85-201
// replaces Belos block-CG + ML smoothed aggregation by line-relaxation
// multigrid on the same cutoffStencil operator, PoissonSolver.cpp:678-766).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <memory>
#include <type_traits>
#include <vector>

#include "csrst_hip.h"
#include "hip_util.h"
#include "poisson_mg.h"

using hu::DBuf;
using hu::Error;

namespace pmg {

// the levels that k_tail takes, in device memory (a kernel argument indexed by
// a loop would be copied to scratch)
constexpr int kMaxTail = 10;
struct Tail {
    Level fine;                 // the level above (nx = 0: none, the tail starts at level 0)
    Level lv[kMaxTail];
    int n, sweeps;              // levels; sweeps on the last
};

namespace {

constexpr int kBlock = 256;
constexpr int kNu = 2;             // sweeps before and after the coarse correction
constexpr int kCoarseSweeps = 8;   // most sweeps on the coarsest level
constexpr int kMaxTab = 32;        // run starts with a factor table of their own
// Levels of at most this many nodes run in one workgroup (k_tail), where a
// barrier replaces a launch, but one CU's loads have to bring 32 B a node and
// half sweep, and a wave solves several columns in turn.  us per V-cycle with
// 2048, 4096, 8192, 16384 nodes: 512 x 256 243, 207, 212, 281; 1024 x 512 266,
// 264, 264, 327; 2000 x 64 195, 224, 302, 497; 300 x 100 174, 188, 229, 319;
// 100 x 2000 332, 325, 325, 340; 2048 x 1024 405, 411, 404, 438.  Without the
// tail 64 x 48 takes 246 and 2000 x 64 258, with it 131 and 224.
constexpr int kTailNodes = 4096;
// Coarsening ends once a red/black sweep damps the smoothest error by this
// factor: the x coupling is then weak against the line's own smallest
// eigenvalue, and coarser levels would add launches only.
constexpr double kWeak = 0.03;

int nblk(size_t n) { return (int)((n + kBlock - 1) / kBlock); }

// kBlock rows j of a column i per workgroup, in a flat grid as the tiles are
unsigned row_blocks(int nx, int ny) { return (unsigned)nx * (unsigned)nblk(ny); }
__device__ __forceinline__ void row_block(int ny, int &i, int &j)
{
    const unsigned per = (unsigned)(ny + kBlock - 1) / kBlock;
    i = (int)(blockIdx.x / per);
    j = (int)(blockIdx.x % per) * kBlock + (int)threadIdx.x;
}

// ---------------------------------------------------------------------------
// set-up

// Node classes (row-major) into the level-0 unknown mask (column-major).
__global__ void __launch_bounds__(kBlock) k_act(const uint8_t *cls, uint8_t *act, int nx, int ny, int pitch, int M)
{
    __shared__ uint8_t t[kTile][kTile + 4];
    const int a = threadIdx.x % kTile, b = threadIdx.x / kTile;
    int i0, j0;
    tile_origin(nx, i0, j0);
    for (int r = b; r < kTile; r += kBlock / kTile) {
        const int i = i0 + a, j = j0 + r;
        t[r][a] = i < nx && j < ny && cls[(size_t)j * nx + i] == kUnknown ? 1 : 0;
    }
    __syncthreads();
    for (int r = b; r < kTile; r += kBlock / kTile) {
        const int i = i0 + r, j = j0 + a;
        if (i < nx && j < pitch) act[(size_t)i * pitch + row_pos(j, M)] = t[a][r];
    }
}

// The runs of unknowns of each column, one wave per column.
__global__ void __launch_bounds__(kBlock) k_rows(const uint8_t *act, ColRows *rows, int nx, int ny, int pitch, int M)
{
    const int i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= nx) return;
    const uint8_t *a = act + (size_t)i * pitch;
    int lo = ny, hi = 0, runs = 0;
    for (int j = lane; j < ny; j += 64) {
        if (!a[row_pos(j, M)]) continue;
        lo = min(lo, j);
        hi = max(hi, j + 1);
        runs += j == 0 || !a[row_pos(j - 1, M)] ? 1 : 0;
    }
    lo = hu::wave_min(lo);
    hi = hu::wave_max(hi);
    for (int o = 32; o > 0; o >>= 1) runs += __shfl_xor(runs, o, 64);
    if (lane == 0) rows[i] = runs == 0 ? ColRows{0, 0, -1, 0} : ColRows{lo, runs == 1 ? hi : -1, -1, 0};
}

// Thomas elimination of a run's matrix tridiag(-r, 1, -r), r = cy / (2 (cx + cy)):
// its factors depend on the row's place k in the run alone, g_0 = r,
// g_k = r / (1 - r g_{k-1}), in closed form sinh((k+1) theta) / sinh((k+2) theta)
// with cosh theta = 1 / (2 r) = 1 + cx / cy.  One table per level serves every
// column, so that a line solve has no division.
__device__ __forceinline__ double factor(int k, double theta)
{
    const double a = 2.0 * theta * (k + 1), b = 2.0 * theta * (k + 2);
    return b > 1e-290 ? exp(-theta) * (expm1(-a) / expm1(-b)) : (k + 1.0) / (k + 2.0);
}
__global__ void k_factors(double *g, int n, double theta)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) g[k] = factor(k, theta);
}

// The factors in column order for runs that start at row start[blockIdx.y]
// (zero above it): the lanes of a line solve read them as they read a column.
__global__ void k_tables(double *gt, const int *start, int ny, int pitch, int M, double theta)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x, lo = start[blockIdx.y];
    if (j < pitch) gt[(size_t)blockIdx.y * pitch + row_pos(j, M)] = j >= lo && j < ny ? factor(j - lo, theta) : 0.0;
}

// ---------------------------------------------------------------------------
// line solves: one wave per column, lane l holds rows l M .. l M + M - 1

template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_or(double identity, double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v), d = __builtin_bit_cast(unsigned long long, identity);
    const int lo = __builtin_amdgcn_update_dpp((int)(d & 0xffffffffu), (int)(u & 0xffffffffu), CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(d >> 32), (int)(u >> 32), CTRL, ROWMASK, 0xf, false);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

template <int CTRL, int ROWMASK>
__device__ __forceinline__ void scan_step(double &G, double &Y)
{
    const double g = dpp_or<CTRL, ROWMASK>(1.0, G), y = dpp_or<CTRL, ROWMASK>(0.0, Y);
    Y = fma(G, y, Y);
    G *= g;
}

// Scan of the lanes' affine maps y -> G y + Y, lane 0 first: on return Y is
// the map's value of zero through this lane, G the product of the factors.
__device__ __forceinline__ void affine_scan(double &G, double &Y)
{
    scan_step<0x111, 0xf>(G, Y);   // row_shr:1
    scan_step<0x112, 0xf>(G, Y);   // row_shr:2
    scan_step<0x114, 0xf>(G, Y);   // row_shr:4
    scan_step<0x118, 0xf>(G, Y);   // row_shr:8
    scan_step<0x142, 0xa>(G, Y);   // row_bcast:15
    scan_step<0x143, 0xc>(G, Y);   // row_bcast:31
}

// the value of the lane before (lane 0: first) and after (lane 63: last)
__device__ __forceinline__ double from_prev(double v, double first) { return dpp_or<0x138, 0xf>(first, v); }   // wave_shr:1
__device__ __forceinline__ double from_next(double v, double last) { return dpp_or<0x130, 0xf>(last, v); }     // wave_shl:1

// Thomas with the elimination factors g (0 at a row that is no unknown, which
// separates the runs): forward y_j = g_j (e_j + y_{j-1}), backward
// x_j = y_j + g_j x_{j+1}, with e = rhs / cy.  Both are affine recurrences:
// each lane composes its M rows' maps, a wave scan gives the value that enters
// the lane, a second pass applies it.  v: e in, x out; yin and xin enter
// before row 0 and after the last lane's last row; yout is what leaves it.
template <int M>
__device__ __forceinline__ double forward_rows(double (&v)[M], const double (&g)[M], double yin)
{
    double G = 1.0, Y = 0.0;
#pragma unroll
    for (int t = 0; t < M; ++t) {
        v[t] *= g[t];
        Y = fma(g[t], Y, v[t]);
        G *= g[t];
    }
    affine_scan(G, Y);
    const double all = fma(G, yin, Y);               // y after this lane
    double y = from_prev(all, yin);
#pragma unroll
    for (int t = 0; t < M; ++t) {
        y = fma(g[t], y, v[t]);
        v[t] = y;
    }
    return all;                                      // lane 63: y after the chunk
}

template <int M>
__device__ __forceinline__ void backward_rows(double (&v)[M], const double (&g)[M], double xin)
{
    double G = 1.0, X = 0.0;
#pragma unroll
    for (int t = M - 1; t >= 0; --t) {
        X = fma(g[t], X, v[t]);
        G *= g[t];
    }
    // the scan runs from the last lane to the first: on mirrored lanes
    const int mirror = 63 - (int)(threadIdx.x & 63);
    G = __shfl(G, mirror, 64);
    X = __shfl(X, mirror, 64);
    affine_scan(G, X);
    const double in = from_prev(fma(G, xin, X), xin);
    double x = __shfl(in, mirror, 64);
#pragma unroll
    for (int t = M - 1; t >= 0; --t) {
        x = fma(g[t], x, v[t]);
        v[t] = x;
    }
}

// this lane's rows of a column (or of the chunk of a long one)
template <int M>
__device__ __forceinline__ void load_rows(const double *col, double (&v)[M])
{
    const double2 *p = reinterpret_cast<const double2 *>(col) + (threadIdx.x & 63);
#pragma unroll
    for (int t = 0; t < M; t += 2) {
        const double2 d = p[32 * t];
        v[t] = d.x;
        v[t + 1] = d.y;
    }
}
template <int M>
__device__ __forceinline__ void store_rows(double *col, const double (&v)[M])
{
    double2 *p = reinterpret_cast<double2 *>(col) + (threadIdx.x & 63);
#pragma unroll
    for (int t = 0; t < M; t += 2) p[32 * t] = make_double2(v[t], v[t + 1]);
}

// 1 where row j0 + t of level-0 column c is an unknown, as a bit mask; chunk:
// the first row of the wave's chunk, j0 = chunk + lane M
template <int M>
__device__ __forceinline__ uint32_t unknown_bits(const Level &L, int c, int chunk)
{
    const ColRows r = L.rows[c];
    const int lane = threadIdx.x & 63;
    uint32_t m = 0;
    if (r.hi >= 0) {
        const int j0 = chunk + lane * M, a = max(r.lo - j0, 0), b = min(r.hi - j0, M);
        if (b > a) m = (b - a >= 32 ? 0xffffffffu : ((1u << (b - a)) - 1u)) << a;
    } else {
        const uint8_t *act = L.act + (size_t)c * L.pitch + chunk + 2 * lane;
#pragma unroll
        for (int t = 0; t < M; ++t)
            if (act[(t >> 1) * 128 + (t & 1)]) m |= 1u << t;
    }
    return m;
}

// Elimination factors of this lane's rows of level-0 column c.  cnt: unknowns
// that end the rows before the chunk's first row, in and out (only columns of
// several runs use it).  Called by whole waves.
template <int M>
__device__ __forceinline__ void factors(const Level &L, int c, int chunk, double (&g)[M], int &cnt)
{
    const ColRows r = L.rows[c];
    const int lane = threadIdx.x & 63, j0 = chunk + lane * M;
    if (r.hi >= 0 && r.tab >= 0) {
        load_rows<M>(L.gt + (size_t)r.tab * L.pitch + chunk, g);
#pragma unroll
        for (int t = 0; t < M; ++t) g[t] = j0 + t < r.hi ? g[t] : 0.0;
        return;
    }
    if (r.hi >= 0) {
#pragma unroll
        for (int t = 0; t < M; ++t) {
            const int j = j0 + t;
            g[t] = j >= r.lo && j < r.hi ? L.g[j - r.lo] : 0.0;
        }
        return;
    }
    // place in the run: trailing unknowns of the lanes before, by a scan of
    // (all rows unknown, trailing unknowns)
    const uint32_t m = unknown_bits<M>(L, c, chunk);
    const uint32_t full = M == 32 ? 0xffffffffu : (1u << (M & 31)) - 1u;
    int all = m == full ? 1 : 0;
    int tr = all ? M : __clz((int)~(m << (32 - M)));
    for (int o = 1; o < 64; o <<= 1) {
        const int pa = __shfl_up(all, o, 64), pt = __shfl_up(tr, o, 64);
        if (lane >= o) {
            tr += all ? pt : 0;
            all &= pa;
        }
    }
    tr += all ? cnt : 0;
    int k = __shfl_up(tr, 1, 64);
    if (lane == 0) k = cnt;
    cnt = __shfl(tr, 63, 64);
#pragma unroll
    for (int t = 0; t < M; ++t) {
        const bool on = (m >> t) & 1u;
        g[t] = on ? L.g[k] : 0.0;
        k = on ? k + 1 : 0;
    }
}

enum Guess { kPlain, kZero, kProlong };

// e = (rhs + cx (phi_{i-1} + phi_{i+1})) / cy of a column's rows.  kZero: the
// iterate is zero.  kProlong: the coarse correction is added to the neighbours
// as they are read; i is even, so they are the odd columns, which take half of
// each coarse neighbour.  The corrected iterate is not stored: the line solve
// replaces the even columns and the next half sweep the odd ones.
template <int M, int GUESS>
__device__ __forceinline__ void line_rhs(const Level &L, const Level &C, int i, int chunk, double (&e)[M])
{
    load_rows<M>(L.rhs + (size_t)i * L.pitch + chunk, e);
    if (GUESS != kZero) {
        double mid[M];
        if (GUESS == kProlong) load_rows<M>(C.phi + (size_t)(i >> 1) * C.pitch + chunk, mid);
#pragma unroll
        for (int side = -1; side <= 1; side += 2) {
            const int n = i + side;
            if (n < 0 || n >= L.nx) continue;
            double v[M];
            load_rows<M>(L.phi + (size_t)n * L.pitch + chunk, v);
            if (GUESS == kProlong) {
                const int I = (i >> 1) + side;
                double far[M];
#pragma unroll
                for (int t = 0; t < M; ++t) far[t] = 0.0;
                if (I >= 0 && I < C.nx) load_rows<M>(C.phi + (size_t)I * C.pitch + chunk, far);
                const uint32_t on = unknown_bits<M>(L, n << L.shift, chunk);
#pragma unroll
                for (int t = 0; t < M; ++t)
                    if ((on >> t) & 1u) v[t] += 0.5 * (mid[t] + far[t]);
            }
#pragma unroll
            for (int t = 0; t < M; ++t) e[t] = fma(L.cx, v[t], e[t]);
        }
    }
    const double icy = 1.0 / L.cy;
#pragma unroll
    for (int t = 0; t < M; ++t) e[t] *= icy;
}

// exact line solve of column i (a column with no unknowns keeps its zeros)
template <int M, int GUESS>
__device__ __forceinline__ void smooth_column(const Level &L, const Level &C, int i)
{
    const ColRows r = L.rows[(size_t)i << L.shift];
    if (r.lo == r.hi) return;
    constexpr int chunk = 0;
    double e[M], g[M];
    int cnt = 0;
    line_rhs<M, GUESS>(L, C, i, chunk, e);
    factors<M>(L, i << L.shift, chunk, g, cnt);
    forward_rows<M>(e, g, 0.0);
    backward_rows<M>(e, g, 0.0);
    store_rows<M>(L.phi + (size_t)i * L.pitch + chunk, e);
}

// Coarse right-hand side of column I: full weighting in x of the fine residual
// at columns 2 I - 1 .. 2 I + 1.  The odd columns' residual is round-off (the
// last half sweep solved them), but it is what cancels their round-off in the
// even column's: without it the coarse levels amplify that to an error of
// 8e-12 of phi on a 2048 x 1024 grid, against 5e-14.  solve: the first half
// sweep of the coarse level (even columns, from a zero iterate) on the rows at
// hand.
template <int M>
__device__ __forceinline__ void restrict_column(const Level &F, const Level &C, int I, bool solve)
{
    const ColRows r = F.rows[(size_t)I << C.shift];
    if (r.lo == r.hi) return;
    constexpr int chunk = 0;
    double left[M], mid[M], right[M], v[M];
    auto column = [&](int i, double (&d)[M]) {
        if (i >= 0 && i < F.nx) {
            load_rows<M>(F.phi + (size_t)i * F.pitch + chunk, d);
        } else {
#pragma unroll
            for (int t = 0; t < M; ++t) d[t] = 0.0;
        }
    };
    column(2 * I - 2, left);
    column(2 * I - 1, mid);
#pragma unroll
    for (int t = 0; t < M; ++t) v[t] = 0.0;
    const double diag = 2.0 * (F.cx + F.cy);
#pragma unroll
    for (int side = -1; side <= 1; ++side) {
        const int i = 2 * I + side;
        column(i + 1, right);
        if (i >= 0 && i < F.nx) {
            double q[M];
            load_rows<M>(F.rhs + (size_t)i * F.pitch + chunk, q);
            const uint32_t on = unknown_bits<M>(F, i << F.shift, chunk);
            const double below = from_prev(mid[M - 1], 0.0), above = from_next(mid[0], 0.0);
            const double w = side == 0 ? 0.5 : 0.25;
#pragma unroll
            for (int t = 0; t < M; ++t) {
                const double a = t > 0 ? mid[t - 1] : below, b = t + 1 < M ? mid[t + 1] : above;
                const double s = fma(F.cx, left[t] + right[t], q[t]);
                v[t] += (on >> t) & 1u ? w * fma(F.cy, a + b, fma(-diag, mid[t], s)) : 0.0;
            }
        }
#pragma unroll
        for (int t = 0; t < M; ++t) {
            left[t] = mid[t];
            mid[t] = right[t];
        }
    }
    const uint32_t on = unknown_bits<M>(F, I << C.shift, chunk);
#pragma unroll
    for (int t = 0; t < M; ++t) v[t] = (on >> t) & 1u ? v[t] : 0.0;
    store_rows<M>(C.rhs + (size_t)I * C.pitch + chunk, v);
    if (!solve) return;
    double g[M];
    int cnt = 0;
    factors<M>(C, I << C.shift, chunk, g, cnt);
    const double icy = 1.0 / C.cy;
#pragma unroll
    for (int t = 0; t < M; ++t) v[t] *= icy;
    forward_rows<M>(v, g, 0.0);
    backward_rows<M>(v, g, 0.0);
    store_rows<M>(C.phi + (size_t)I * C.pitch + chunk, v);
}

// Consecutive workgroup ids run on the 8 XCDs in turn: each XCD takes a
// contiguous range of columns, so that a column read as a neighbour of two
// solved ones comes through one L2.
__device__ __forceinline__ int xcd_block()
{
    const int b = blockIdx.x, n = gridDim.x & ~7;
    return b < n ? (b & 7) * (n >> 3) + (b >> 3) : b;
}

constexpr int kWaves = kBlock / 64;   // columns per workgroup

// this wave's place in its workgroup, as a scalar
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Half sweep of the columns 2 k + color.  Bound by the latency of its loads and
// the launch: 3.1 us at 512 x 256, where a workgroup per column with cyclic
// reduction in LDS took 5.2 us; 32 B and 8 operations a row.
template <int M, int GUESS>
__global__ void __launch_bounds__(kBlock) k_smooth(Level L, Level C, int color)
{
    const int i = 2 * (xcd_block() * kWaves + wave_id()) + color;
    if (i < L.nx) smooth_column<M, GUESS>(L, C, i);
}

template <int M>
__global__ void __launch_bounds__(kBlock) k_restrict(Level F, Level C)
{
    const int I = xcd_block() * kWaves + wave_id();
    if (I < C.nx) restrict_column<M>(F, C, I, (I & 1) == 0);
}

// The V-cycle's coarse levels in one workgroup.  Data stays in global memory (one CU's caches); a barrier
// orders the half sweeps.  Wave w takes columns w, w + waves, ... of a colour.
template <int M, int GUESS>
__device__ __forceinline__ void tail_sweep(const Level &L, const Level &C, int color, int wave, int waves)
{
    for (int i = 2 * wave + color; i < L.nx; i += 2 * waves) smooth_column<M, GUESS>(L, C, i);
    __syncthreads();
}

template <int M, int NT>
__global__ void __launch_bounds__(NT) k_tail(const Tail *tail)
{
    const Tail &T = *tail;
    const int wave = wave_id(), waves = NT / 64;
    for (int l = 0; l < T.n; ++l) {
        const Level &L = T.lv[l];
        const bool top = l == 0 && T.fine.nx == 0;
        if (top) {
            tail_sweep<M, kPlain>(L, L, 0, wave, waves);
        } else {
            const Level &F = l == 0 ? T.fine : T.lv[l - 1];
            for (int I = wave; I < L.nx; I += waves) restrict_column<M>(F, L, I, (I & 1) == 0);
            __syncthreads();
        }
        tail_sweep<M, kPlain>(L, L, 1, wave, waves);
        const int sweeps = l + 1 == T.n ? T.sweeps : kNu;
        for (int k = 1; k < sweeps; ++k) {
            tail_sweep<M, kPlain>(L, L, 0, wave, waves);
            tail_sweep<M, kPlain>(L, L, 1, wave, waves);
        }
    }
    for (int l = T.n - 2; l >= 0; --l) {
        const Level &L = T.lv[l];
        tail_sweep<M, kProlong>(L, T.lv[l + 1], 0, wave, waves);
        tail_sweep<M, kPlain>(L, L, 1, wave, waves);
        for (int k = 1; k < kNu; ++k) {
            tail_sweep<M, kPlain>(L, L, 0, wave, waves);
            tail_sweep<M, kPlain>(L, L, 1, wave, waves);
        }
    }
}

// Lines of more than 64 kMaxLane rows: the same solve in chunks, y kept in phi
// between the passes.
template <int GUESS>
__global__ void __launch_bounds__(kBlock) k_smooth_long(Level L, Level C, int color)
{
    constexpr int M = kLongLane, N = 64 * M;
    const int i = 2 * (xcd_block() * kWaves + wave_id()) + color, lane = threadIdx.x & 63;
    if (i >= L.nx) return;
    const ColRows r = L.rows[(size_t)i << L.shift];
    if (r.lo == r.hi) return;
    double *phi = L.phi + (size_t)i * L.pitch;
    const int chunks = (L.ny + N - 1) / N;
    double v[M], g[M], y = 0.0, x = 0.0;
    int cnt = 0, before = 0;             // lane c keeps the count before chunk c < 64; later chunks count again
    for (int c = 0; c < chunks; ++c) {
        before = c < 64 && lane == c ? cnt : before;
        line_rhs<M, GUESS>(L, C, i, c * N, v);
        factors<M>(L, i << L.shift, c * N, g, cnt);
        y = __shfl(forward_rows<M>(v, g, y), 63, 64);
        store_rows<M>(phi + c * N, v);
    }
    for (int c = chunks - 1; c >= 0; --c) {
        cnt = __shfl(before, c & 63, 64);
        if (r.hi < 0 && c >= 64) {
            cnt = 0;
            const uint8_t *act = L.act + ((size_t)i << L.shift) * L.pitch;
            while (cnt < c * N && act[row_pos(c * N - 1 - cnt, M)]) ++cnt;
        }
        load_rows<M>(phi + c * N, v);
        factors<M>(L, i << L.shift, c * N, g, cnt);
        backward_rows<M>(v, g, x);
        x = __shfl(v[0], 0, 64);
        store_rows<M>(phi + c * N, v);
    }
}

// residual at row j of column i (an unknown)
__device__ __forceinline__ double residual_at(const Level &L, int i, int j)
{
    const size_t k = L.at(i, j);
    const double l = i > 0 ? L.phi[k - L.pitch] : 0.0, r = i + 1 < L.nx ? L.phi[k + L.pitch] : 0.0;
    const double d = j > 0 ? L.phi[L.at(i, j - 1)] : 0.0, u = j + 1 < L.ny ? L.phi[L.at(i, j + 1)] : 0.0;
    return L.rhs[k] - (2.0 * (L.cx + L.cy) * L.phi[k] - L.cx * (l + r) - L.cy * (d + u));
}

// restriction for long lines, a thread per coarse node
__global__ void __launch_bounds__(kBlock) k_restrict_long(Level F, Level C)
{
    int I, j;
    row_block(C.ny, I, j);
    if (j >= C.ny) return;
    const int p = row_pos(j, F.lane);
    double v = 0.0;
    if (F.act[((size_t)I << C.shift) * F.pitch + p])
        for (int side = -1; side <= 1; ++side) {
            const int i = 2 * I + side;
            if (i < 0 || i >= F.nx || !F.act[((size_t)i << F.shift) * F.pitch + p]) continue;
            v += (side == 0 ? 0.5 : 0.25) * residual_at(F, i, j);
        }
    C.rhs[(size_t)I * C.pitch + p] = v;
}

// ---------------------------------------------------------------------------
// norms, in a fixed order: block partials, then one block

__device__ __forceinline__ double block_sum(double s)
{
    __shared__ double sh[kBlock];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    return sh[0];
}

// level-0 residual and its sum of squares, one wave per column
template <int M>
__global__ void __launch_bounds__(kBlock) k_residual(Level L, double *partial)
{
    const int i = xcd_block() * kWaves + wave_id();
    double s = 0.0;
    if (i < L.nx) {
        const ColRows r = L.rows[i];
        if (r.lo != r.hi) {
            double p[M], q[M], v[M];
            load_rows<M>(L.phi + (size_t)i * L.pitch, p);
            load_rows<M>(L.rhs + (size_t)i * L.pitch, q);
#pragma unroll
            for (int side = -1; side <= 1; side += 2) {
                if (i + side < 0 || i + side >= L.nx) continue;
                load_rows<M>(L.phi + (size_t)(i + side) * L.pitch, v);
#pragma unroll
                for (int t = 0; t < M; ++t) q[t] = fma(L.cx, v[t], q[t]);
            }
            const uint32_t on = unknown_bits<M>(L, i, 0);
            const double below = from_prev(p[M - 1], 0.0), above = from_next(p[0], 0.0);
            const double diag = 2.0 * (L.cx + L.cy);
#pragma unroll
            for (int t = 0; t < M; ++t) {
                const double a = t > 0 ? p[t - 1] : below, b = t + 1 < M ? p[t + 1] : above;
                v[t] = (on >> t) & 1u ? fma(L.cy, a + b, fma(-diag, p[t], q[t])) : 0.0;
                s = fma(v[t], v[t], s);
            }
            store_rows<M>(L.res + (size_t)i * L.pitch, v);
        }
    }
    s = block_sum(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}
__global__ void __launch_bounds__(kBlock) k_residual_long(Level L, double *partial)
{
    int i, j;
    row_block(L.ny, i, j);
    double s = 0.0;
    if (j < L.ny) {
        const size_t k = L.at(i, j);
        s = L.act[k] ? residual_at(L, i, j) : 0.0;
        L.res[k] = s;
    }
    s = block_sum(s * s);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kBlock) k_sum_final(const double *partial, int nb, double *out)
{
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBlock) s += partial[b];
    s = block_sum(s);
    if (threadIdx.x == 0) *out = s;
}

// The caller's row-major right-hand side and guess into level 0, a tile per
// workgroup.  Right-hand side of the unknown rows: b plus the known
// neighbours' values (cutoffStencil keeps the coupling to a flagged neighbour
// that is itself an identity row, PoissonSolver.cpp:700-741); its sum of
// squares goes to the partials.
__global__ void __launch_bounds__(kBlock) k_load(const uint8_t *cls, const double *b, const double *phi, Level L,
                                                 double *partial)
{
    __shared__ double tr[kTile][kTile + 1], tp[kTile][kTile + 1];
    const int a = threadIdx.x % kTile, row = threadIdx.x / kTile;
    int i0, j0;
    tile_origin(L.nx, i0, j0);
    double s = 0.0;
    for (int r = row; r < kTile; r += kBlock / kTile) {
        const int i = i0 + a, j = j0 + r;
        double v = 0.0, p = 0.0;
        if (i < L.nx && j < L.ny) {
            const size_t k = (size_t)j * L.nx + i;
            if (cls[k] == kUnknown) {
                v = b[k];
                if (i > 0 && cls[k - 1] == kKnown) v += L.cx * b[k - 1];
                if (i + 1 < L.nx && cls[k + 1] == kKnown) v += L.cx * b[k + 1];
                if (j > 0 && cls[k - L.nx] == kKnown) v += L.cy * b[k - L.nx];
                if (j + 1 < L.ny && cls[k + L.nx] == kKnown) v += L.cy * b[k + L.nx];
                p = phi[k];
            }
        }
        tr[r][a] = v;
        tp[r][a] = p;
        s += v * v;
    }
    __syncthreads();
    for (int r = row; r < kTile; r += kBlock / kTile) {
        const int i = i0 + r, j = j0 + a;
        if (i < L.nx && j < L.pitch) {
            const size_t k = L.at(i, j);
            L.rhs[k] = tr[a][r];
            L.phi[k] = tp[a][r];
        }
    }
    s = block_sum(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// Solution out: unknowns from the level, identity rows phi = b.
__global__ void __launch_bounds__(kBlock) k_store(const uint8_t *cls, const double *b, Level L, double *phi)
{
    __shared__ double t[kTile][kTile + 1];
    const int a = threadIdx.x % kTile, row = threadIdx.x / kTile;
    int i0, j0;
    tile_origin(L.nx, i0, j0);
    for (int r = row; r < kTile; r += kBlock / kTile) {
        const int i = i0 + r, j = j0 + a;
        t[r][a] = i < L.nx && j < L.ny ? L.phi[L.at(i, j)] : 0.0;
    }
    __syncthreads();
    for (int r = row; r < kTile; r += kBlock / kTile) {
        const int i = i0 + a, j = j0 + r;
        if (i >= L.nx || j >= L.ny) continue;
        const size_t k = (size_t)j * L.nx + i;
        phi[k] = cls[k] == kUnknown ? t[a][r] : b[k];
    }
}

// ---------------------------------------------------------------------------
// rows per lane: the smallest of these M with 64 M >= ny
int rows_per_lane(int ny)
{
    for (int m : {2, 4, 6, 8, 10, 12, 16, 24})
        if (64 * m >= ny) return m;
    return ny <= 64 * kMaxLane ? kMaxLane : kLongLane;
}

template <class F>
void with_rows(const Level &L, F f)
{
    switch (L.lane) {
    case 2: f(std::integral_constant<int, 2>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 6: f(std::integral_constant<int, 6>()); break;
    case 8: f(std::integral_constant<int, 8>()); break;
    case 10: f(std::integral_constant<int, 10>()); break;
    case 12: f(std::integral_constant<int, 12>()); break;
    case 16: f(std::integral_constant<int, 16>()); break;
    case 24: f(std::integral_constant<int, 24>()); break;
    default: f(std::integral_constant<int, kMaxLane>()); break;
    }
}

bool is_long(const Level &L) { return L.ny > 64 * kMaxLane; }

template <int GUESS>
void half_sweep(const Level &L, const Level &C, int color, hipStream_t s)
{
    const int cols = (L.nx + 1 - color) / 2;
    if (cols <= 0) return;
    const int nb = (cols + kWaves - 1) / kWaves;
    if (is_long(L)) k_smooth_long<GUESS><<<nb, kBlock, 0, s>>>(L, C, color);
    else with_rows(L, [&](auto m) { k_smooth<decltype(m)::value, GUESS><<<nb, kBlock, 0, s>>>(L, C, color); });
}

void restrict_to(const Level &F, const Level &C, hipStream_t s)
{
    if (is_long(F)) {
        k_restrict_long<<<row_blocks(C.nx, C.ny), kBlock, 0, s>>>(F, C);
        k_smooth_long<kZero><<<((C.nx + 1) / 2 + kWaves - 1) / kWaves, kBlock, 0, s>>>(C, C, 0);
    } else {
        const int nb = (C.nx + kWaves - 1) / kWaves;
        with_rows(F, [&](auto m) { k_restrict<decltype(m)::value><<<nb, kBlock, 0, s>>>(F, C); });
    }
}

// waves as the registers of M rows allow
void run_tail(const Tail *tail, const Level &L, hipStream_t s)
{
    with_rows(L, [&](auto m) {
        constexpr int M = decltype(m)::value, NT = M <= 8 ? 1024 : M <= 16 ? 512 : 256;
        k_tail<M, NT><<<1, NT, 0, s>>>(tail);
    });
}

}  // namespace

Solver::~Solver()
{
    if (hnorm_) (void)hipHostFree(hnorm_);
}

void Solver::setup(int nx, int ny, double hx, double hy, const uint8_t *cls, hipStream_t s)
{
    if (nx < 1 || ny < 1) throw Error(CSRST_EINVAL, "empty Poisson grid");
    if (!(hx > 0) || !(hy > 0)) throw Error(CSRST_EINVAL, "Poisson spacings must be positive");
    nx_ = nx; ny_ = ny; s_ = s; cls_ = cls;
    lv_.clear();
    const int M = rows_per_lane(ny), pitch = (ny + 64 * M - 1) / (64 * M) * (64 * M);
    int n = nx;
    double cx = 1.0 / (hx * hx);
    const double cy = 1.0 / (hy * hy);
    // damping of a line's smoothest error by a red/black sweep
    const double sn = std::sin(0.5 * M_PI / (ny + 1)), lam = 4 * cy * sn * sn;
    double damp = 0;
    while (true) {
        Level L;
        L.nx = n; L.ny = ny; L.pitch = pitch; L.lane = M; L.shift = (int)lv_.size(); L.cx = cx; L.cy = cy;
        lv_.push_back(L);
        damp = std::pow(2 * cx / (2 * cx + lam), 2);
        if (n <= 2 || damp <= kWeak) break;
        n = (n + 1) / 2;
        cx *= 0.25;
    }
    const int nl = (int)lv_.size();
    coarse_ = kCoarseSweeps;
    for (int k = kCoarseSweeps - 1; k >= 2 * kNu && std::pow(damp, k) <= 1e-5; --k) coarse_ = k;
    const size_t m0 = (size_t)nx * pitch;
    auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
    cols_.alloc(align(m0) + nx * sizeof(ColRows));
    uint8_t *act = cols_.p;
    ColRows *rows = reinterpret_cast<ColRows *>(cols_.p + align(m0));
    k_act<<<num_tiles(nx, pitch), kBlock, 0, s_>>>(cls, act, nx, ny, pitch, M);
    k_rows<<<(nx + kWaves - 1) / kWaves, kBlock, 0, s_>>>(act, rows, nx, ny, pitch, M);
    HU_LAUNCH_CHECK();
    // the first kMaxTab run starts get tables (a straight chamber has one)
    std::vector<ColRows> hrows(nx);
    HU_CHECK(hipMemcpyAsync(hrows.data(), rows, nx * sizeof(ColRows), hipMemcpyDeviceToHost, s_));
    HU_CHECK(hipStreamSynchronize(s_));
    std::vector<int> start, tab(ny, -1);
    for (ColRows &r : hrows) {
        if (r.hi <= r.lo) continue;
        if (tab[r.lo] < 0 && (int)start.size() < kMaxTab) {
            tab[r.lo] = (int)start.size();
            start.push_back(r.lo);
        }
        r.tab = tab[r.lo];
    }
    const int nt = (int)start.size();
    // one block of device memory: factors, partials, then the levels' phi
    // (cleared: columns without unknowns are never written), rhs and the
    // level-0 residual
    size_t off = 0, cells = 0;
    auto take = [&](size_t b) { const size_t o = off; off += align(b); return o; };
    const size_t parts = std::max(num_tiles(nx, pitch), row_blocks(nx, ny));
    const size_t oStart = take((size_t)nt * sizeof(int)), oTail = take(sizeof(Tail)), oPart = take(parts * sizeof(double));
    const size_t oG = take((size_t)nl * ny * sizeof(double)), oGt = take((size_t)nl * nt * pitch * sizeof(double));
    for (const Level &L : lv_) cells += (size_t)L.nx * pitch;
    const size_t oPhi = take(cells * sizeof(double)), oRhs = take(cells * sizeof(double));
    const size_t oRes = take(m0 * sizeof(double));
    mem_.alloc(off);
    auto reals = [&](size_t o) { return reinterpret_cast<double *>(mem_.p + o); };
    int *dstart = reinterpret_cast<int *>(mem_.p + oStart);
    partial_ = reals(oPart);
    size_t at = 0;
    for (Level &L : lv_) {
        L.act = act;
        L.rows = rows;
        L.g = reals(oG) + (size_t)L.shift * ny;
        L.gt = reals(oGt) + (size_t)L.shift * nt * pitch;
        L.phi = reals(oPhi) + at;
        L.rhs = reals(oRhs) + at;
        at += (size_t)L.nx * pitch;
    }
    lv_[0].res = reals(oRes);
    Tail T;
    t0_ = nl;
    if (!is_long(lv_[0]))
        while (t0_ > 0 && nl - t0_ < kMaxTail && (size_t)lv_[t0_ - 1].nx * ny <= kTailNodes) --t0_;
    T.n = nl - t0_;
    T.sweeps = coarse_;
    if (t0_ > 0) T.fine = lv_[t0_ - 1];
    for (int l = t0_; l < nl; ++l) T.lv[l - t0_] = lv_[l];
    tail_ = reinterpret_cast<Tail *>(mem_.p + oTail);
    if (!hnorm_ && hipHostMalloc(&hnorm_, sizeof(double), hipHostMallocDefault) != hipSuccess) {
        hnorm_ = nullptr;
        throw Error(CSRST_ENOMEM, "hipHostMalloc failed");
    }
    HU_CHECK(hipMemcpyAsync(rows, hrows.data(), nx * sizeof(ColRows), hipMemcpyHostToDevice, s_));
    if (nt) HU_CHECK(hipMemcpyAsync(dstart, start.data(), (size_t)nt * sizeof(int), hipMemcpyHostToDevice, s_));
    HU_CHECK(hipMemcpyAsync(tail_, &T, sizeof(T), hipMemcpyHostToDevice, s_));
    HU_CHECK(hipMemsetAsync(mem_.p + oPhi, 0, off - oPhi, s_));
    for (const Level &L : lv_) {
        const double theta = 2.0 * std::asinh(std::sqrt(0.5 * (L.cx / L.cy)));
        k_factors<<<nblk(ny), kBlock, 0, s_>>>(const_cast<double *>(L.g), ny, theta);
        if (nt) k_tables<<<dim3(nblk(pitch), nt), kBlock, 0, s_>>>(const_cast<double *>(L.gt), dstart, ny, pitch, M, theta);
    }
    HU_LAUNCH_CHECK();
    HU_CHECK(hipStreamSynchronize(s_));              // the copies' sources end here
}

void Solver::cycle()
{
    const int n = (int)lv_.size();
    const int t0 = t0_;
    for (int l = 0; l < t0; ++l) {
        const Level &L = lv_[l];
        if (l == 0) half_sweep<kPlain>(L, L, 0, s_);
        else restrict_to(lv_[l - 1], L, s_);
        half_sweep<kPlain>(L, L, 1, s_);
        const int sweeps = l + 1 == n ? coarse_ : kNu;
        for (int k = 1; k < sweeps; ++k) {
            half_sweep<kPlain>(L, L, 0, s_);
            half_sweep<kPlain>(L, L, 1, s_);
        }
    }
    if (t0 < n) run_tail(tail_, lv_[t0], s_);
    for (int l = std::min(t0, n - 1) - 1; l >= 0; --l) {
        const Level &L = lv_[l];
        half_sweep<kProlong>(L, lv_[l + 1], 0, s_);
        half_sweep<kPlain>(L, L, 1, s_);
        for (int k = 1; k < kNu; ++k) {
            half_sweep<kPlain>(L, L, 0, s_);
            half_sweep<kPlain>(L, L, 1, s_);
        }
    }
    HU_LAUNCH_CHECK();
}

double Solver::read_norm()
{
    k_sum_final<<<1, kBlock, 0, s_>>>(partial_, npart_, hnorm_);
    HU_LAUNCH_CHECK();
    HU_CHECK(hipStreamSynchronize(s_));
    return std::sqrt(*static_cast<volatile double *>(hnorm_));
}

double Solver::resnorm()
{
    const Level &L = lv_[0];
    if (is_long(L)) {
        npart_ = (int)row_blocks(L.nx, L.ny);
        k_residual_long<<<npart_, kBlock, 0, s_>>>(L, partial_);
    } else {
        npart_ = (L.nx + kWaves - 1) / kWaves;
        with_rows(L, [&](auto m) { k_residual<decltype(m)::value><<<npart_, kBlock, 0, s_>>>(L, partial_); });
    }
    return read_norm();
}

double Solver::begin(const double *b, const double *phi0)
{
    const Level &L = lv_[0];
    npart_ = (int)num_tiles(L.nx, L.pitch);
    k_load<<<npart_, kBlock, 0, s_>>>(cls_, b, phi0, L, partial_);
    return read_norm();
}

double Solver::residual(const double *b, const double *phi)
{
    begin(b, phi);
    return resnorm();
}

void Solver::store(const double *b, double *phi)
{
    const Level &L = lv_[0];
    k_store<<<num_tiles(L.nx, L.ny), kBlock, 0, s_>>>(cls_, b, L, phi);
    HU_LAUNCH_CHECK();
}

Stats Solver::solve(const double *b, double *phi, double tol, int maxit)
{
    Stats st;
    st.bnorm = begin(b, phi);
    double r = resnorm();
    st.resid0 = r;
    const double target = tol * (st.bnorm > 0 ? st.bnorm : 1.0);
    int flat = 0;   // cycles in a row that gained less than 5%: the round-off floor
    while (r > target && st.cycles < maxit && flat < 3) {
        cycle();
        ++st.cycles;
        const double rn = resnorm();
        if (!std::isfinite(rn)) throw Error(CSRST_EHIP, "multigrid diverged");
        flat = rn > 0.95 * r ? flat + 1 : 0;
        r = rn;
    }
    st.resid = r;
    store(b, phi);
    return st;
}

}  // namespace pmg

// ---------------------------------------------------------------------------
// Standalone solve on host arrays.

extern "C" int csrst_poisson_solve(int nx, int ny, double hx, double hy, const uint8_t *cls, const double *b,
                                   double *phi, double tol, int maxit, int *cycles, double *resid)
{
    hipStream_t s = nullptr;
    try {
        if (!cls || !b || !phi || nx < 1 || ny < 1 || maxit < 0 || !(tol >= 0))
            throw Error(CSRST_EINVAL, "bad Poisson arguments");
        const size_t m = (size_t)nx * ny;
        for (size_t k = 0; k < m; ++k)
            if (cls[k] > pmg::kKnown) throw Error(CSRST_EINVAL, hu::fmt("node class %d at %zu", cls[k], k));
        HU_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        DBuf<uint8_t> dcls;
        DBuf<double> db, dphi;
        dcls.alloc(m); db.alloc(m); dphi.alloc(m);
        HU_CHECK(hipMemcpyAsync(dcls.p, cls, m, hipMemcpyHostToDevice, s));
        hu::Stage stage;
        stage.in(db.p, b, m * sizeof(double), s);
        stage.in(dphi.p, phi, m * sizeof(double), s);
        pmg::Solver sol;
        sol.setup(nx, ny, hx, hy, dcls.p, s);
        const pmg::Stats st = sol.solve(db.p, dphi.p, tol, maxit);
        stage.out(phi, dphi.p, m * sizeof(double), s);
        HU_CHECK(hipStreamDestroy(s));
        s = nullptr;
        if (cycles) *cycles = st.cycles;
        if (resid) *resid = st.bnorm > 0 ? st.resid / st.bnorm : st.resid;
        return CSRST_OK;
    } catch (const std::exception &e) {
        if (s) { (void)hipStreamSynchronize(s); (void)hipStreamDestroy(s); }
        const Error *he = dynamic_cast<const Error *>(&e);
        hu::global_error() = e.what();
        return he ? he->code : CSRST_EINVAL;
    }
}
