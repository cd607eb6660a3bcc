// csrst_sf.hip -- the reference's ShapeFunction and ScatterGatherImpl
// interfaces as stateless kernels on caller memory, FP64.
//
//   csrst_sg_gather / csrst_sg_scatter       ScatterGatherImpl<IntOp,double>
//                                            ::gather / ::scatter
//                                            (ScatterGatherImpl.hh:27-641)
//   csrst_sf_current_density                 ShapeFunction<IntOp>::
//                                            getCurrentDensity{X,Y}
//   csrst_sf_charge_density                  ShapeFunction<IntOp>::getChargeDensity
//   csrst_sf_charge_density_diff             ShapeFunction<IntOp>::getChargeDensityDiff
//                                            (ShapeFunction.hh:30-508)
//
// Fields are dense patches of nodes [ny][nx] (x fastest) of a mesh with the
// given origin and spacing; particle positions are (x, y) pairs, the layout
// of the reference's Vektor<double,2> attributes.  Every array argument is a
// device pointer; work is queued on the caller's stream and the call
// returns when it has finished.
//
// Arithmetic follows the reference order and this file is compiled without
// FMA contraction.  Sums over particles are made deterministic the way the
// reference orders them, so that the per-node sums equal a CPU loop over the
// particles bit for bit.  A particle makes one or more items: a stencil of
// weights with its first node.  Small deposits (node_scan_fits) let a wave per
// node walk the items in order; large ones write every contribution in
// (particle, item, statement) order, sort them stably by node, and add each
// node's run sequentially from 0.0.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <climits>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "csrst_hip.h"
#include "hip_util.h"
#include "pic_math.h"

using hu::Error;
using pm::vec2;

namespace {

constexpr int kB = 256;
constexpr unsigned kEmpty = 0xffffffffu;
constexpr int kMaxSeg = 4;       // segments of one trajectory (c dt <= h: at most 3)

struct Patch {
    int i0, j0, nx, ny;          // absolute index of node (0, 0) and extent
    double o[2], h[2];           // mesh origin (absolute node 0) and spacing
};

int blocks(size_t n) { return (int)((n + kB - 1) / kB); }

// contributions per particle of the fixed-slot layout (an unused slot is kEmpty)
int slots_current(int order) { return kMaxSeg * (order == 0 ? 2 : order == 1 ? 6 : 12); }

// ---------------------------------------------------------------------------
// What a particle deposits.  An Op has NX x NY nodes per item, at most ITEMS
// items per particle, begin(k, state) -> the number of items (-1: a trajectory
// that crosses more lines than one push can), and item(state, g, I, J, w): the
// first node (relative to the patch) and the weights of item g, x fastest.

// first node I of a stencil relative to the patch's i0, or kOff if all its (at
// most 4) nodes lie outside a patch of nx nodes.  Patches may have up to 2^31 - 1
// nodes a side, so node indices past the first are formed as unsigned.
constexpr int kOff = -8;
__device__ __forceinline__ int rel(long long I, int i0, int nx)
{
    const long long d = I - i0;
    return d < kOff || d >= nx ? kOff : (int)d;
}

// getCurrentDensityBase{X,Y} + getCurrentDensity{X,Y}: the trajectory oldR -> R
// split at the (dual) cell lines, each segment's current on its stencil
// (ZerothOrderShapeFunction.cpp:202-294, FirstOrderShapeFunction.cpp:226-329,
// 540-683, SecondOrderShapeFunction.cpp:222-345, 583-826).
template <int ORDER, int COMP>
struct CurrentOp {
    static constexpr int NX = ORDER == 0 ? (COMP == 0 ? 1 : 2) : ORDER == 1 ? (COMP == 0 ? 2 : 3) : (COMP == 0 ? 3 : 4);
    static constexpr int NY = ORDER == 0 ? (COMP == 0 ? 2 : 1) : ORDER == 1 ? (COMP == 0 ? 3 : 2) : (COMP == 0 ? 4 : 3);
    static constexpr int NN = NX * NY, ITEMS = kMaxSeg;
    Patch p;
    double dt;
    const double *oldR, *R, *Q;
    struct State {
        pm::Crossings<double> c;
        vec2<double> od, odt, delta;
        double covered, q;
    };
    __device__ __forceinline__ int begin(int k, State &s) const
    {
        const vec2<double> org = pm::mk(p.o[0], p.o[1]);
        const vec2<double> dx = pm::mk(p.h[0], p.h[1]);
        const double ox = oldR[2 * k], oy = oldR[2 * k + 1], rx = R[2 * k], ry = R[2 * k + 1];
        const vec2<double> o = pm::mk(ox - org.x, oy - org.y);
        const vec2<double> e = pm::mk(rx - org.x, ry - org.y);
        s.od = pm::mk(1.0 / dx.x, 1.0 / dx.y);
        if (ORDER == 0) s.odt = pm::mk(1.0 / (dx.y * dt), 1.0 / (dx.x * dt));
        else s.odt = pm::mk(s.od.x / dt, s.od.y / dt);
        const vec2<double> D = pm::mk(rx - ox, ry - oy);
        s.delta = pm::mk(D.x * s.od.x, D.y * s.od.y);
        s.covered = sqrt(D.x * D.x + D.y * D.y);
        s.q = Q[k];
        if (!pm::crossings(s.c, o, e, dx, ORDER == 1) || s.c.n - 1 > kMaxSeg) return -1;
        return s.c.n - 1;
    }
    __device__ __forceinline__ void item(const State &s, int g, int &I, int &J, double (&w)[NN]) const
    {
        const vec2<double> a = s.c.s[g], b = s.c.s[g + 1];
        const vec2<double> xi = pm::mk(a.x * s.od.x, a.y * s.od.y);
        const vec2<double> xf = pm::mk(b.x * s.od.x, b.y * s.od.y);
        const vec2<double> seg = pm::mk(b.x - a.x, b.y - a.y);
        pm::SegCurrent<double> sc;
        pm::segment_current(sc, ORDER, COMP, xi, xf, seg, s.covered, s.q, s.odt, s.delta);
        I = rel(sc.I0, p.i0, p.nx);
        J = rel(sc.J0, p.j0, p.ny);
#pragma unroll
        for (int t = 0; t < NN; ++t) w[t] = sc.w[t];
    }
};

// getChargeDensityImpl (ZerothOrderShapeFunction.cpp:296-383,
// FirstOrderShapeFunction.cpp:331-430, SecondOrderShapeFunction.cpp:347-450);
// DIFF: then the stencil at oldR with the opposite sign, the second half of
// getChargeDensityDiffImpl.
template <int ORDER, bool DIFF>
struct ChargeOp {
    static constexpr int NX = ORDER + 2, NY = ORDER + 2, NN = NX * NY, ITEMS = DIFF ? 2 : 1;
    Patch p;
    const double *R, *oldR, *Q;
    struct State {
        int k;
    };
    __device__ __forceinline__ int begin(int k, State &s) const
    {
        s.k = k;
        return ITEMS;
    }
    __device__ __forceinline__ void item(const State &s, int g, int &I, int &J, double (&w)[NN]) const
    {
        const double *r = (g == 0 ? R : oldR) + 2 * s.k;
        const double q = Q[s.k];
        double wx[NX], wy[NY];
        int I0, J0;
        pm::charge_weights<ORDER>(pm::mk((r[0] - p.o[0]) / p.h[0], (r[1] - p.o[1]) / p.h[1]), q, wx, wy, I0, J0);
#pragma unroll
        for (int b = 0; b < NY; ++b)
#pragma unroll
            for (int a = 0; a < NX; ++a) {
                const double v = pm::charge_w<ORDER>(q, wx[a], wy[b]);
                w[b * NX + a] = g == 0 ? v : -v;
            }
        I = rel(I0, p.i0, p.nx);
        J = rel(J0, p.j0, p.ny);
    }
};

// ScatterGatherImpl::scatter of one value (ScatterGatherImpl.hh:136-194,
// 303-392, 529-641): edge component lc (0 Ex, 1 Ey) or the cell field (lc 2).
template <int ORDER>
struct ScatterOp {
    static constexpr int NX = ORDER + 2, NY = ORDER + 2, NN = NX * NY, ITEMS = 1;
    Patch p;
    int lc;
    const double *R, *val;
    struct State {
        int k;
    };
    __device__ __forceinline__ int begin(int k, State &s) const
    {
        s.k = k;
        return 1;
    }
    __device__ __forceinline__ void item(const State &s, int, int &I, int &J, double (&w)[NN]) const
    {
        const vec2<double> od = pm::mk(1.0 / p.h[0], 1.0 / p.h[1]);
        const vec2<double> pp = pm::mk((R[2 * s.k] - p.o[0]) * od.x, (R[2 * s.k + 1] - p.o[1]) * od.y);
        const double v = val[s.k];
        pm::Stencil<double> st = lc < 2 ? pm::edge_stencil(ORDER, lc, pp) : pm::cell_stencil(ORDER, pp);
        if (lc == 2 && ORDER == 1) {
            // the S1 cell scatter forms its outer weights directly (ScatterGatherImpl.hh:372-380)
            const double dx = pp.x - ((double)(st.I0 + 1) + 0.5), dy = pp.y - ((double)(st.J0 + 1) + 0.5);
            st.wx[0] = 0.5 * (0.5 - dx) * (0.5 - dx);
            st.wy[0] = 0.5 * (0.5 - dy) * (0.5 - dy);
        }
#pragma unroll
        for (int b = 0; b < NY; ++b)
#pragma unroll
            for (int a = 0; a < NX; ++a) w[b * NX + a] = pm::scatter_w(st, a, b, v);
        I = rel(st.I0, 0, p.nx);      // the stencil is relative to the patch's node (0, 0)
        J = rel(st.J0, 0, p.ny);
    }
};

// error flags of a call, plain stores of 1: [0] a stencil left the patch (its
// nodes outside are dropped), [1] too many crossings
template <class Op>
__device__ __forceinline__ bool inside(const Op &op, int I, int J)
{
    return I >= 0 && J >= 0 && I <= op.p.nx - Op::NX && J <= op.p.ny - Op::NY;
}

// ---------------------------------------------------------------------------
// Small deposits: items in order, then a wave per node.  Nothing is sorted.

constexpr int kNone = INT_MIN;     // I of an unused item

// one thread per (particle, item): short chains, many waves
template <class Op>
__global__ void __launch_bounds__(64) k_items(Op op, int n, int2 *at, double *w, int *flags)
{
    const int it = blockIdx.x * 64 + threadIdx.x, k = it / Op::ITEMS, g = it % Op::ITEMS;
    if (k >= n) return;
    typename Op::State s;
    const int items = op.begin(k, s);
    if (items < 0) flags[1] = 1;
    if (g >= items) {
        at[it] = make_int2(kNone, 0);
        return;
    }
    int I, J;
    double v[Op::NN];
    op.item(s, g, I, J, v);
    if (!inside(op, I, J)) flags[0] = 1;
    at[it] = make_int2(I, J);
#pragma unroll
    for (int t = 0; t < Op::NN; ++t) w[(size_t)it * Op::NN + t] = v[t];
}

__device__ __forceinline__ double lane_value(double v, int lane)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(u & 0xffffffffu), lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(u >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// A wave per node: 64 items at a time, the lanes whose stencil holds the node
// load its weight and append it, in item order, to the wave's list in LDS; every
// 64 entries are added in that order by readlane, without a branch per entry (a
// scalar loop over the hits took 100 cycles each).  mode as in k_runs.  Bound by
// the walk over the items, which are read from L2.  2000 S2 particles on 64 x
// 48 nodes take 33 us here, against 115 us for sorting their 96000
// slots and adding the runs.
template <int NX, int NY>
__global__ void __launch_bounds__(kB) k_node_scan(const int2 *at, const double *w, int items, int nx, int ny, double *f,
                                                  double div, int mode)
{
    constexpr int U = 4;             // groups of 64 items whose loads are in flight together
    __shared__ double list[kB / 64][64 * (U + 1)];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int node = blockIdx.x * (kB / 64) + wave;
    if (node >= nx * ny) return;
    const int i = node % nx, j = node / nx;
    double *buf = list[wave];
    double s = 0.0;
    int have = 0;                    // entries in the list, the same in every lane
    bool any = false;
    int2 a[U], nxt[U];
    auto fetch = [&](int base, int2 (&d)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int it = base + 64 * u + lane;
            d[u] = it < items ? at[it] : make_int2(kNone, 0);
        }
    };
    // adds the first `many` entries of the list in order
    auto add = [&](int from, int many) {
        const double v = buf[from + lane];
        if (many == 64) {
#pragma unroll
            for (int q = 0; q < 64; ++q) s += lane_value(v, q);
        } else {
            for (int q = 0; q < many; ++q) s += lane_value(v, q);
        }
    };
    fetch(0, a);
    for (int base = 0; base < items; base += 64 * U) {
        double v[U];
        bool h[U];
        fetch(base + 64 * U, nxt);   // beyond the items: no load
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int it = base + 64 * u + lane;
            const unsigned di = (unsigned)i - (unsigned)a[u].x, dj = (unsigned)j - (unsigned)a[u].y;
            h[u] = di < (unsigned)NX && dj < (unsigned)NY;
            v[u] = 0.0;
            if (h[u]) v[u] = w[(size_t)it * (NX * NY) + dj * NX + di];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned long long m = __ballot(h[u]);
            if (h[u])
                buf[have + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = v[u];
            have += __popcll(m);
            a[u] = nxt[u];
        }
        if (have >= 64) {
            any = true;
            __builtin_amdgcn_wave_barrier();
            int done = 0;
            for (; have - done >= 64; done += 64) add(done, 64);
            // the rest moves to the front (fewer than 64 entries)
            const double r = buf[done + lane];
            have -= done;
            __builtin_amdgcn_wave_barrier();
            if (lane < have) buf[lane] = r;
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (have) {
        any = true;
        __builtin_amdgcn_wave_barrier();
        add(0, have);
    }
    if (lane == 0) {
        if (mode == 0) f[node] = any ? 0.0 + s / div : 0.0;
        else if (any) f[node] += s;
    }
}

// The node scan's time is a wave per node (0.17 ns a node, as long as 400 items
// take) and every item once per node (0.3 to 0.6 ps each), and at least one
// wave's walk over the items (0.7 us per 256).  us, scan / sort, S2 currents (4
// items a particle) | S0 charges:
//   32 x 32 nodes    n 128 23/69 | 17/27    n 8192 121/131 | 40/66     n 32768 376/319 | 101/86
//   128 x 128        n 1   20/45 | 19/25    n 1024  62/93  | 27/41     n 8192  308/126 | 88/64
//   512 x 512        n 1   66/47 | 59/27    n 128  102/74  | 60/29
//   4096 x 4096      n 1 3100/69 | 2750/45
// (the line lies where they cross, with the node's own cost taken high: a charge
// of few particles on 300 x 300 nodes takes about as long either way).
bool node_scan_fits(size_t items, size_t nodes) { return items > 0 && items <= 32768 && nodes <= 90000000u / (items + 1000); }

// ---------------------------------------------------------------------------
// Large deposits: contributions in order, sorted by node.

// number of items of each particle, and their sum per wave
template <class Op>
__global__ void __launch_bounds__(64) k_count(Op op, int n, uint8_t *cnt, int *sum, int *flags)
{
    const int k = blockIdx.x * 64 + threadIdx.x;
    int c = 0;
    if (k < n) {
        typename Op::State s;
        c = op.begin(k, s);
        if (c < 0) flags[1] = 1;
        c = max(c, 0);
        cnt[k] = (uint8_t)c;
    }
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if (threadIdx.x == 0) sum[blockIdx.x] = c;
}

// exclusive sums of sum[0 .. m), in place; the total to *total (host memory)
__global__ void __launch_bounds__(1024) k_scan(int *sum, int m, int *total)
{
    __shared__ int sh[16];
    __shared__ int carry;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < m; base += 1024) {
        const int v = base + tid < m ? sum[base + tid] : 0;
        int x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) sh[wave] = x;
        __syncthreads();
        int before = carry;
        for (int q = 0; q < wave; ++q) before += sh[q];
        if (base + tid < m) sum[base + tid] = before + x - v;
        __syncthreads();
        if (tid == 1023) carry = before + x;
        __syncthreads();
    }
    if (tid == 0) *total = carry;
}

// Contributions of 64 particles per workgroup: key = the node's index in the
// patch (kEmpty outside it), value = its weight.  cnt != null: packed, cnt[k]
// items of particle k, sum[b] before workgroup b's; else ITEMS fixed items per
// particle, unused ones kEmpty.  The rows of an item pass through LDS, so that
// the workgroup writes them along memory (a thread writing its own rows takes a
// cache line each).
template <class Op>
__global__ void __launch_bounds__(64) k_emit(Op op, int n, const uint8_t *cnt, const int *sum, unsigned *key, double *val,
                                             int *flags)
{
    constexpr int NN = Op::NN;
    __shared__ double sv[64 * NN];
    __shared__ unsigned sk[64 * NN];
    __shared__ int first[64];          // the particle's first item (packed: within the launch)
    __shared__ int many[64];
    const int tid = threadIdx.x, k = blockIdx.x * 64 + tid;
    typename Op::State s;
    int items = 0, most;
    if (k < n) items = op.begin(k, s);
    if (items < 0) flags[1] = 1;
    items = max(items, 0);
    if (cnt) {
        // the places are those counted, whatever the caller's arrays hold by now
        const int places = k < n ? cnt[k] : 0;
        int x = places;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (tid >= o) x += y;
        }
        first[tid] = sum[blockIdx.x] + x - places;
        many[tid] = places;
        most = places;
        for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
    } else {
        first[tid] = k * Op::ITEMS;
        many[tid] = k < n ? Op::ITEMS : 0;
        most = Op::ITEMS;
    }
    for (int g = 0; g < most; ++g) {
        int I = 0, J = 0;
        double w[NN];
        const bool on = g < items;
        if (on) {
            op.item(s, g, I, J, w);
            if (!inside(op, I, J)) flags[0] = 1;
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NN; ++t) {
            const unsigned i = (unsigned)I + t % Op::NX, j = (unsigned)J + t / Op::NX;
            const bool in = on && i < (unsigned)op.p.nx && j < (unsigned)op.p.ny;
            sk[tid * NN + t] = in ? j * (unsigned)op.p.nx + i : kEmpty;
            sv[tid * NN + t] = in ? w[t] : 0.0;
        }
        __syncthreads();
        for (int e = tid; e < 64 * NN; e += 64) {
            const int q = e / NN, t = e - q * NN;
            if (g >= many[q]) continue;
            const size_t d = ((size_t)first[q] + g) * NN + t;
            key[d] = sk[e];
            val[d] = sv[e];
        }
    }
}

// ScatterGatherImpl::gather (ScatterGatherImpl.hh:70-134, 202-301, 407-527)
template <int ORDER>
__global__ void __launch_bounds__(kB) k_gather(Patch p, int lc, int s2bug, const double *f, const double *R, int n, double *out,
                         int *err)
{
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;   // n may be 2^31 - 1
    if (k >= (size_t)n) return;
    const vec2<double> od = pm::mk(1.0 / p.h[0], 1.0 / p.h[1]);
    const vec2<double> pp = pm::mk((R[2 * k] - p.o[0]) * od.x, (R[2 * k + 1] - p.o[1]) * od.y);
    bool bad = false;
    auto fetch = [&](long long I, long long J) {
        if (I < 0 || J < 0 || I >= p.nx || J >= p.ny) { bad = true; return 0.0; }
        return f[(size_t)J * p.nx + (size_t)I];
    };
    const pm::Stencil<double> st = lc < 2 ? pm::edge_stencil(ORDER, lc, pp) : pm::cell_stencil(ORDER, pp);
    auto at = [&](long long a, long long b) { return fetch(st.I0 + a, st.J0 + b); };
    out[k] = pm::gather_n<ORDER + 2>(st, s2bug != 0, at);
    if (bad) *err = 1;
}

// Sum of each node's run, in slot order, from 0.0.  mode 0: f[node] = 0.0 +
// sum / div (the ShapeFunction results, written over a cleared patch; div is
// hx hy for a density, 1 for a current); mode 1: f[node] += sum (scatter
// adds into the caller's field).
// A workgroup takes the runs that begin in its kWin entries: it brings them and
// the kExt that follow into LDS, and each thread adds a run, eight loads at a
// time, so a wave adds 64 runs at once.  A run that goes on past both continues
// from memory, 16 entries in flight.  For 5 M entries in runs of 37 on average,
// up to 400: 76 us, bound by the LDS latency of the longest runs (93 us with a
// wave per run and a readlane per entry; one thread per run with a dependent
// load per addition took 467 us on the 9.6 M slots it had).
constexpr int kWin = 2048, kExt = 512;
__global__ void __launch_bounds__(kB) k_runs(const unsigned *key, const double *val, size_t cnt, double *f, double div,
                                             int mode)
{
    __shared__ double sv[kWin + kExt];
    __shared__ unsigned sk[kWin + kExt + 1];   // sk[q + 1]: entry q; sk[0]: the entry before the window
    __shared__ short heads[kWin];
    __shared__ int wsum[kB / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t t0 = (size_t)blockIdx.x * kWin;
    for (int q = tid; q < kWin + kExt; q += kB) {
        const bool in = t0 + q < cnt;
        sk[q + 1] = in ? key[t0 + q] : kEmpty;
        sv[q] = in ? val[t0 + q] : 0.0;
    }
    if (tid == 0) sk[0] = t0 > 0 ? key[t0 - 1] : kEmpty;
    __syncthreads();
    // the heads in order: thread tid looks at entries 8 tid .. 8 tid + 7
    constexpr int PER = kWin / kB;
    int mine = 0;
    unsigned bits = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int q = tid * PER + u;
        if (sk[q + 1] != kEmpty && sk[q + 1] != sk[q]) {
            bits |= 1u << u;
            ++mine;
        }
    }
    int x = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int at = x - mine, total = 0;
    for (int q = 0; q < kB / 64; ++q) {
        at += q < wave ? wsum[q] : 0;
        total += wsum[q];
    }
    for (; bits; bits &= bits - 1) heads[at++] = (short)(tid * PER + __ffs((int)bits) - 1);
    __syncthreads();
    for (int h = tid; h < total; h += kB) {
        int q = heads[h];
        const unsigned node = sk[q + 1];
        double s = 0.0;
        // whole groups of eight: the last of them still this node
        while (q + 8 <= kWin + kExt && sk[q + 8] == node) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = sv[q + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
            q += 8;
        }
        for (; q < kWin + kExt && sk[q + 1] == node; ++q) s += sv[q];
        if (q == kWin + kExt) {
            constexpr int G = 16;
            bool more = true;
            for (size_t u = t0 + kWin + kExt; more; u += G) {
                unsigned kv[G];
                double vv[G];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const bool in = u + g < cnt;
                    kv[g] = in ? key[u + g] : kEmpty;
                    vv[g] = in ? val[u + g] : 0.0;
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    more = more && kv[g] == node;
                    if (more) s += vv[g];
                }
            }
        }
        if (mode == 0) f[node] = 0.0 + s / div;
        else f[node] += s;
    }
}

// the patch cleared (fill kernel: nothing here is a memset node)
__global__ void k_fill(double *f, size_t n, double v)
{
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) f[t] = v;
}
__global__ void k_zero_flags(int *p) { p[0] = 0; p[1] = 0; }

// ---------------------------------------------------------------------------
// Scratch: keys and values twice (sort input and output), the radix sort's
// temporary storage and an error word, carved out of one block.
struct Scratch {
    unsigned *k0, *k1;
    double *v0, *v1;
    void *tmp;
    size_t tmpBytes;
    int *err;
};

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

int key_bits(size_t nodes)
{
    int b = 1;
    while ((1ull << b) < (unsigned long long)nodes + 1) ++b;
    return b;
}

size_t sort_tmp_bytes(size_t cnt)
{
    size_t bytes = 0;
    HU_CHECK(hipcub::DeviceRadixSort::SortPairs((void *)nullptr, bytes, (unsigned *)nullptr, (unsigned *)nullptr,
                                                (double *)nullptr, (double *)nullptr, (int)cnt, 0, 32));
    return bytes;
}

size_t scratch_bytes(size_t cnt, size_t tmp)
{
    return 2 * align256(cnt * sizeof(unsigned)) + 2 * align256(cnt * sizeof(double)) + align256(tmp) + 256;
}

Scratch carve(unsigned char *base, size_t cnt, size_t tmp)
{
    Scratch s;
    size_t off = 0;
    auto take = [&](size_t b) { unsigned char *p = base + off; off += align256(b); return p; };
    s.k0 = (unsigned *)take(cnt * sizeof(unsigned));
    s.k1 = (unsigned *)take(cnt * sizeof(unsigned));
    s.v0 = (double *)take(cnt * sizeof(double));
    s.v1 = (double *)take(cnt * sizeof(double));
    s.tmp = take(tmp);
    s.tmpBytes = tmp;
    s.err = (int *)take(2 * sizeof(int));
    return s;
}

// Stable sort of the slots by node, then the run sums into f.
void reduce(const Scratch &s, size_t cnt, size_t nodes, double *f, double div, int mode, hipStream_t st)
{
    size_t tb = s.tmpBytes;
    HU_CHECK(hipcub::DeviceRadixSort::SortPairs(s.tmp, tb, s.k0, s.k1, s.v0, s.v1, (int)cnt, 0, key_bits(nodes), st));
    k_runs<<<(int)((cnt + kWin - 1) / kWin), kB, 0, st>>>(s.k1, s.v1, cnt, f, div, mode);
    HU_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Workspaces of the calls.  hipMalloc and hipFree of a deposit's 200 MB took
// 4 to 9 ms of a call whose kernels take 1 ms, so blocks are kept between
// calls: a call leases one to itself and returns it after its stream has
// finished.  A request takes a block of at most four times its size (and a few
// MiB), so that a deposit's particle counts don't occupy its sort's workspace.
// Idle blocks are bounded to kKeep bytes per device: a block larger than that is
// freed at its return and leaves the others alone.  A block no call has taken
// for kAge leases is freed, and all of them are freed before any allocation of
// this library is reported as failed.  Each has two words of pinned host memory
// for the error flags (kernels store there, the host reads after the wait) and
// one for a count.
class Lease {
public:
    Lease(size_t bytes, hipStream_t st) : st_(st)
    {
        HU_CHECK(hipGetDevice(&dev_));
        if (!take(bytes)) {
            b_.bytes = (bytes + (1 << 20) - 1) >> 20 << 20;
            hu::give_back().store(&Lease::drop_idle);
            if (hu::device_alloc((void **)&b_.p, b_.bytes) != hipSuccess)
                throw Error(CSRST_ENOMEM, hu::fmt("hipMalloc of %zu bytes failed", b_.bytes));
            b_.dev = dev_;
            if (hipHostMalloc(&b_.host, 64, hipHostMallocDefault) != hipSuccess) {
                (void)hipGetLastError();
                (void)hipFree(b_.p);
                throw Error(CSRST_ENOMEM, "hipHostMalloc failed");
            }
        }
        b_.age = 0;
        for (int q = 0; q < 3; ++q) b_.host[q] = 0;
    }
    Lease(const Lease &) = delete;
    Lease &operator=(const Lease &) = delete;
    ~Lease()
    {
        (void)hipStreamSynchronize(st_);       // an error path may leave kernels in flight
        std::lock_guard<std::mutex> lock(mu());
        auto &v = idle();
        size_t kept = b_.bytes;
        if (kept > kKeep) {
            drop(b_);
            return;
        }
        try {
            v.push_back(b_);
        } catch (const std::exception &) {     // no host memory to note it
            drop(b_);
            return;
        }
        // newest first: what is beyond the bound or too long unused goes
        for (int q = (int)v.size() - 2; q >= 0; --q) {
            if (v[q].dev != dev_) continue;
            kept += v[q].bytes;
            if (++v[q].age > kAge || kept > kKeep) {
                kept -= v[q].bytes;
                drop(v[q]);
                v.erase(v.begin() + q);
            }
        }
    }
    unsigned char *base() const { return b_.p; }
    int *flags() const { return b_.host; }
    int *total() const { return b_.host + 2; }
    // the call's work is done: its error bits (1 left the patch, 2 crossings)
    int wait() const
    {
        HU_CHECK(hipStreamSynchronize(st_));
        const volatile int *h = b_.host;
        return (h[0] ? 1 : 0) | (h[1] ? 2 : 0);
    }

private:
    struct Block {
        unsigned char *p = nullptr;
        size_t bytes = 0;
        int *host = nullptr;
        int dev = 0, age = 0;
    };
    static constexpr size_t kKeep = (size_t)512 << 20, kSmall = (size_t)4 << 20;
    static constexpr int kAge = 64;
    static std::mutex &mu()
    {
        static std::mutex *m = new std::mutex;     // never destroyed: callers may outlive static destruction
        return *m;
    }
    static std::vector<Block> &idle()
    {
        static std::vector<Block> *v = new std::vector<Block>;
        return *v;
    }
    // the smallest idle block that serves `bytes`, if any
    bool take(size_t bytes)
    {
        std::lock_guard<std::mutex> lock(mu());
        auto &v = idle();
        int best = -1;
        for (size_t q = 0; q < v.size(); ++q)
            if (v[q].dev == dev_ && v[q].bytes >= bytes && v[q].bytes <= 4 * bytes + kSmall &&
                (best < 0 || v[q].bytes < v[best].bytes))
                best = (int)q;
        if (best < 0) return false;
        b_ = v[best];
        v.erase(v.begin() + best);
        return true;
    }
    static void drop(Block &x)
    {
        (void)hipFree(x.p);
        (void)hipHostFree(x.host);
    }
    static void drop_idle()
    {
        std::lock_guard<std::mutex> lock(mu());
        for (Block &x : idle()) drop(x);
        idle().clear();
    }
    Block b_;
    hipStream_t st_;
    int dev_ = 0;
};

// Items and contributions are numbered, and sorted, in 32 bits: more than that
// is refused, before any array is touched where the particle count shows it.
void check_count(size_t count, int n)
{
    if (count > (size_t)INT_MAX)
        throw Error(CSRST_EINVAL, hu::fmt("%d particles make %zu contributions; one call takes up to %d (deposit them in "
                                          "several calls)", n, count, INT_MAX));
}

// A deposit: small ones by the node scan, large ones by the sort.  mode 0
// writes the whole patch, mode 1 adds.  Returns the error bits.
template <class Op>
int deposit(const Op &op, int n, double *f, double div, int mode, hipStream_t st)
{
    constexpr bool kPack = Op::ITEMS == kMaxSeg;
    const size_t nodes = (size_t)op.p.nx * op.p.ny, items = (size_t)n * Op::ITEMS;
    check_count(kPack ? items : items * Op::NN, n);
    if (node_scan_fits(items, nodes)) {
        const size_t wo = align256(items * sizeof(int2));
        const Lease ws(wo + items * Op::NN * sizeof(double), st);
        int2 *at = (int2 *)ws.base();
        double *w = (double *)(ws.base() + wo);
        k_items<Op><<<(int)((items + 63) / 64), 64, 0, st>>>(op, n, at, w, ws.flags());
        k_node_scan<Op::NX, Op::NY><<<(int)((nodes + kB / 64 - 1) / (kB / 64)), kB, 0, st>>>(
            at, w, (int)items, op.p.nx, op.p.ny, f, div, mode);
        HU_LAUNCH_CHECK();
        return ws.wait();
    }
    const int nb = (n + 63) / 64;
    size_t cnt = items * Op::NN;
    int e = 0;
    if (mode == 0) k_fill<<<blocks(nodes), kB, 0, st>>>(f, nodes, 0.0);
    if (n == 0) {
        HU_LAUNCH_CHECK();
        HU_CHECK(hipStreamSynchronize(st));
        return 0;
    }
    // currents use two of their four segments on average: count first, so that
    // only what there is is sorted
    const size_t so = align256(n);
    const Lease small(kPack ? so + (size_t)nb * sizeof(int) : 256, st);
    uint8_t *num = kPack ? (uint8_t *)small.base() : nullptr;
    int *sum = (int *)(small.base() + so);
    if constexpr (kPack) {
        k_count<Op><<<nb, 64, 0, st>>>(op, n, num, sum, small.flags());
        k_scan<<<1, 1024, 0, st>>>(sum, nb, small.total());
        HU_LAUNCH_CHECK();
        e = small.wait();
        cnt = (size_t)*(const volatile int *)small.total() * Op::NN;
        if (cnt == 0) return e;
        check_count(cnt, n);
    }
    const size_t tmp = sort_tmp_bytes(cnt);
    const Lease ws(scratch_bytes(cnt, tmp), st);
    const Scratch s = carve(ws.base(), cnt, tmp);
    k_emit<Op><<<nb, 64, 0, st>>>(op, n, num, sum, s.k0, s.v0, ws.flags());
    HU_LAUNCH_CHECK();
    reduce(s, cnt, nodes, f, div, mode, st);
    return e | ws.wait();
}

void check_patch(const Patch &p)
{
    if (p.nx <= 0 || p.ny <= 0) throw Error(CSRST_EINVAL, "empty patch");
    if ((unsigned long long)p.nx * (unsigned long long)p.ny >= 0xffffffffull)
        throw Error(CSRST_EINVAL, "patch has more than 2^32 - 1 nodes");
    if (!(p.h[0] > 0) || !(p.h[1] > 0)) throw Error(CSRST_EINVAL, "spacing must be positive");
}

Patch make_patch(int i0, int j0, int nx, int ny, const double origin[2], const double dx[2])
{
    if (!origin || !dx) throw Error(CSRST_EINVAL, "null origin or spacing");
    Patch p{i0, j0, nx, ny, {origin[0], origin[1]}, {dx[0], dx[1]}};
    check_patch(p);
    return p;
}

int sf_fail(const std::exception &e)
{
    const Error *he = dynamic_cast<const Error *>(&e);
    hu::global_error() = e.what();
    return he ? he->code : CSRST_EINVAL;
}

template <int COMP, class F>
void with_current(const Patch &p, int order, double dt, const double *oldR, const double *R, const double *Q, F go)
{
    if (order == 0) go(CurrentOp<0, COMP>{p, dt, oldR, R, Q});
    else if (order == 1) go(CurrentOp<1, COMP>{p, dt, oldR, R, Q});
    else go(CurrentOp<2, COMP>{p, dt, oldR, R, Q});
}

void current_errors(int e)
{
    if (e & 2) throw Error(CSRST_EINVAL, "a trajectory crossed more cell lines than one push can");
    if (e & 1) throw Error(CSRST_EWINDOW, "a current stencil left the patch (its contribution was dropped)");
}

void check_current_args(int order, int comp, double dt, const double *J, const double *oldR, const double *R,
                        const double *Q, int n)
{
    if (order < 0 || order > 2) throw Error(CSRST_EINVAL, "order must be 0..2");
    if (comp != 0 && comp != 1) throw Error(CSRST_EINVAL, "comp must be 0 or 1");
    if (!(dt > 0)) throw Error(CSRST_EINVAL, "dt must be positive");
    if (n < 0 || !J || (n > 0 && (!oldR || !R || !Q))) throw Error(CSRST_EINVAL, "bad particle arguments");
}

// ---------------------------------------------------------------------------
// Scratch of csrst_sf_current_density_noalloc: one block per device in
// static device memory, held until the process ends.  In host code `scratch`
// only names the symbol; its device address comes from hipGetSymbolAddress,
// once per device with that device current, and is kept per device.
constexpr size_t kScratchBytes = (size_t)32 << 20;   // 32 MiB
constexpr int kMaxDevices = 64;

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

std::mutex g_scratch_mu;
unsigned char *g_scratch[kMaxDevices] = {};

unsigned char *device_scratch()
{
    int dev = 0;
    HU_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) throw Error(CSRST_EINVAL, hu::fmt("device %d beyond the scratch table", dev));
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        HU_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch[dev] = (unsigned char *)p;
    }
    return g_scratch[dev];
}

template <bool DIFF>
int charge(int order, double *rho, int i0, int j0, int nx, int ny, const double origin[2], const double dx[2],
                  const double *R, const double *oldR, const double *Q, int n, void *stream)
{
    try {
        if (order < 0 || order > 2) throw Error(CSRST_EINVAL, "order must be 0..2");
        if (n < 0 || !rho || (n > 0 && (!R || !Q))) throw Error(CSRST_EINVAL, "bad arguments");
        const Patch p = make_patch(i0, j0, nx, ny, origin, dx);
        const hipStream_t st = (hipStream_t)stream;
        const double area = dx[0] * dx[1];
        int e;
        if (order == 0) e = deposit(ChargeOp<0, DIFF>{p, R, oldR, Q}, n, rho, area, 0, st);
        else if (order == 1) e = deposit(ChargeOp<1, DIFF>{p, R, oldR, Q}, n, rho, area, 0, st);
        else e = deposit(ChargeOp<2, DIFF>{p, R, oldR, Q}, n, rho, area, 0, st);
        if (e & 1) throw Error(CSRST_EWINDOW, "a charge stencil left the patch (dropped)");
        return CSRST_OK;
    } catch (const std::exception &e) {
        return sf_fail(e);
    }
}

}  // namespace

extern "C" {

int csrst_sg_gather(int order, int s2bug, int kind, const double *field, int nx, int ny, const double origin[2],
                    const double dx[2], const double *R, int n, double *out, void *stream)
{
    try {
        if (order < 0 || order > 2 || kind < 0 || kind > 2) throw Error(CSRST_EINVAL, "order 0..2, kind 0..2");
        if (n < 0 || (n > 0 && (!field || !R || !out))) throw Error(CSRST_EINVAL, "bad arguments");
        const Patch p = make_patch(0, 0, nx, ny, origin, dx);
        const hipStream_t st = (hipStream_t)stream;
        const Lease ws(256, st);
        auto go = [&](auto kern) { kern<<<blocks(n), kB, 0, st>>>(p, kind, s2bug, field, R, n, out, ws.flags()); };
        if (n > 0) {
            if (order == 0) go(k_gather<0>);
            else if (order == 1) go(k_gather<1>);
            else go(k_gather<2>);
        }
        HU_LAUNCH_CHECK();
        if (ws.wait()) throw Error(CSRST_EWINDOW, "a gather stencil left the patch (its nodes read as 0)");
        return CSRST_OK;
    } catch (const std::exception &e) {
        return sf_fail(e);
    }
}

int csrst_sg_scatter(int order, int kind, double *field, int nx, int ny, const double origin[2], const double dx[2],
                     const double *R, const double *val, int n, void *stream)
{
    try {
        if (order < 0 || order > 2 || kind < 0 || kind > 2) throw Error(CSRST_EINVAL, "order 0..2, kind 0..2");
        if (n < 0 || !field || (n > 0 && (!R || !val))) throw Error(CSRST_EINVAL, "bad arguments");
        const Patch p = make_patch(0, 0, nx, ny, origin, dx);
        if (n == 0) return CSRST_OK;
        const hipStream_t st = (hipStream_t)stream;
        int e;
        if (order == 0) e = deposit(ScatterOp<0>{p, kind, R, val}, n, field, 1.0, 1, st);
        else if (order == 1) e = deposit(ScatterOp<1>{p, kind, R, val}, n, field, 1.0, 1, st);
        else e = deposit(ScatterOp<2>{p, kind, R, val}, n, field, 1.0, 1, st);
        if (e & 1) throw Error(CSRST_EWINDOW, "a scatter stencil left the patch (dropped)");
        return CSRST_OK;
    } catch (const std::exception &e) {
        return sf_fail(e);
    }
}

int csrst_sf_current_density(int order, int comp, double *J, int i0, int j0, int nx, int ny, const double origin[2],
                             const double dx[2], double dt, const double *oldR, const double *R, const double *Q,
                             int n, void *stream)
{
    try {
        check_current_args(order, comp, dt, J, oldR, R, Q, n);
        const Patch p = make_patch(i0, j0, nx, ny, origin, dx);
        int e = 0;
        auto go = [&](auto op) { e = deposit(op, n, J, 1.0, 0, (hipStream_t)stream); };
        if (comp == 0) with_current<0>(p, order, dt, oldR, R, Q, go);
        else with_current<1>(p, order, dt, oldR, R, Q, go);
        current_errors(e);
        return CSRST_OK;
    } catch (const std::exception &e) {
        return sf_fail(e);
    }
}

int csrst_sf_current_density_noalloc(int order, int comp, double *J, int i0, int j0, int nx, int ny,
                                     const double origin[2], const double dx[2], double dt, const double *oldR,
                                     const double *R, const double *Q, int n, void *stream)
{
    try {
        check_current_args(order, comp, dt, J, oldR, R, Q, n);
        const Patch p = make_patch(i0, j0, nx, ny, origin, dx);
        const size_t cnt = (size_t)n * slots_current(order), nodes = (size_t)nx * ny;
        check_count(cnt, n);
        const size_t tmp = sort_tmp_bytes(cnt);      // a size query: nothing is allocated
        const size_t need = scratch_bytes(cnt, tmp);
        if (need > kScratchBytes)
            throw Error(CSRST_EINVAL, hu::fmt("%d particles of order %d need %zu bytes of scratch; the no-allocation "
                                              "entry holds %zu (use csrst_sf_current_density)",
                                              n, order, need, kScratchBytes));
        const Scratch s = carve(device_scratch(), cnt, tmp);
        const hipStream_t st = (hipStream_t)stream;
        k_zero_flags<<<1, 1, 0, st>>>(s.err);
        k_fill<<<blocks(nodes), kB, 0, st>>>(J, nodes, 0.0);
        if (n > 0) {
            auto go = [&](auto op) {
                k_emit<decltype(op)><<<(n + 63) / 64, 64, 0, st>>>(op, n, nullptr, nullptr, s.k0, s.v0, s.err);
            };
            if (comp == 0) with_current<0>(p, order, dt, oldR, R, Q, go);
            else with_current<1>(p, order, dt, oldR, R, Q, go);
            HU_LAUNCH_CHECK();
            reduce(s, cnt, nodes, J, 1.0, 0, st);
        }
        int f[2] = {0, 0};
        HU_CHECK(hipMemcpyAsync(f, s.err, sizeof(f), hipMemcpyDeviceToHost, st));
        HU_CHECK(hipStreamSynchronize(st));
        current_errors((f[0] ? 1 : 0) | (f[1] ? 2 : 0));
        return CSRST_OK;
    } catch (const std::exception &e) {
        return sf_fail(e);
    }
}

int csrst_sf_charge_density(int order, double *rho, int i0, int j0, int nx, int ny, const double origin[2],
                            const double dx[2], const double *R, const double *Q, int n, void *stream)
{
    return charge<false>(order, rho, i0, j0, nx, ny, origin, dx, R, nullptr, Q, n, stream);
}

int csrst_sf_charge_density_diff(int order, double *rho, int i0, int j0, int nx, int ny, const double origin[2],
                                 const double dx[2], const double *R, const double *oldR, const double *Q, int n,
                                 void *stream)
{
    if (n > 0 && !oldR) {
        hu::global_error() = "null oldR";
        return CSRST_EINVAL;
    }
    return charge<true>(order, rho, i0, j0, nx, ny, origin, dx, R, oldR, Q, n, stream);
}

}  // extern "C"
