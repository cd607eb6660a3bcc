// Learned warm start for the Poisson multigrid: a 4-level convolutional
// U-Net (32 base channels) mapping a charge density to a potential, with
// BF16 weights and activations and FP32 accumulation on the MFMA units.
//
// No counterpart in the reference (its Poisson start is Belos CG + ML AMG,
// PoissonSolver.cpp:85-201); the network only supplies the initial guess and
// the multigrid still iterates to its tolerance.
//
// Layout: activations NHWC (channels fastest), weights [Cout][3][3][Cin].
// The 3x3 convolutions (stride 1, zero padding 1) with 32 or more channels on
// both sides are a persistent implicit GEMM on v_mfma_f32_16x16x32_bf16 with
// LDS-staged input tiles and weights (k_conv32p); K runs over (tap, input
// channel).  The same kernel, with transposed weights and mirrored taps, gives
// the input gradient.  The one-channel input layer runs on the vector units, the
// output layer (load-bound) on the MFMA.  The weight gradient is a GEMM over pixels
// on the same MFMA, split across workgroups with FP32 atomics (k_wgrad32,
// k_wgrad_one).  k_conv and k_conv_wgrad (16x16x16) remain for channel counts
// the 32-channel kernels do not take.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <memory>
#include <string>
#include <vector>

#include "csrst_hip.h"
#include "hip_util.h"
#include "poisson_mg.h"

using hu::DBuf;
using hu::Error;

namespace unet {

typedef short sh4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

constexpr int kB = 256;

__device__ __forceinline__ float bf2f(bf16 v) { return __uint_as_float((uint32_t)v << 16); }
// round to nearest even
__host__ __device__ __forceinline__ bf16 f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (bf16)(u >> 16);
}

// MFMA 16x16x16 (BF16 in, FP32 accumulate).  Lane l holds A[l%16][4(l/16)..+3],
// B[4(l/16)..+3][l%16] and D[4(l/16)..+3][l%16].
__device__ __forceinline__ f4 mfma(sh4 a, sh4 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }

__device__ __forceinline__ sh4 load4(const bf16 *p)
{
    const uint2 v = *reinterpret_cast<const uint2 *>(p);
    sh4 r;
    r[0] = (short)(v.x & 0xFFFF); r[1] = (short)(v.x >> 16);
    r[2] = (short)(v.y & 0xFFFF); r[3] = (short)(v.y >> 16);
    return r;
}

// eight bf16 values as floats (one 16-byte load or store)
struct V8 { float v[8]; };

__device__ __forceinline__ V8 ld8(const bf16 *p)
{
    const uint4 u = *reinterpret_cast<const uint4 *>(p);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
    V8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r.v[2 * i] = __uint_as_float(w[i] << 16);
        r.v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
    return r;
}

__device__ __forceinline__ void st8(bf16 *p, const V8 &r)
{
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f2bf(r.v[2 * i]) | ((uint32_t)f2bf(r.v[2 * i + 1]) << 16);
    *reinterpret_cast<uint4 *>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

struct ConvArgs {
    const bf16 *x;       // [P][Cin]
    const bf16 *w;       // [CoutP][9][Cin] (rows past Cout are zero)
    const float *bias;   // [Cout] or null
    bf16 *y;             // [P][Cout] (bf16 out) or null
    float *yf;           // [P][Cout] (fp32 out) or null
    int B, H, W, Cin, Cout, CoutP;
    int flip;            // 1: taps mirrored (input gradient)
    int relu;
    const bf16 *mask;    // [P][Cout] or null: y is zero where this is not positive (the ReLU's gradient)
};

__device__ __forceinline__ bool pos(uint32_t bits) { return __uint_as_float(bits << 16) > 0.f; }

// Implicit-GEMM 3x3 convolution.  grid = (ceil(P / 256), CoutP / (16 MT));
// each of the 4 waves covers 64 consecutive pixels of the block's 256 and MT
// tiles of 16 output channels, so each input load feeds MT MFMAs.
template <int MT>
__global__ void __launch_bounds__(kB) k_conv(ConvArgs a)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int P = a.B * a.H * a.W;
    const int co0 = blockIdx.y * 16 * MT;
    const int pw = blockIdx.x * 256 + wave * 64;
    if (pw >= P) return;
    const int li = lane & 15, kg = lane >> 4;
    f4 acc[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
    // pixel coordinates of this lane's B columns
    int pb[4], py[4], px[4];
    bool pv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int p = pw + 16 * t + li;
        pv[t] = p < P;
        const int pp = pv[t] ? p : 0;
        px[t] = pp % a.W;
        py[t] = (pp / a.W) % a.H;
        pb[t] = pp / (a.W * a.H);
    }
    const int Cin = a.Cin;
    if ((Cin & 15) == 0) {
        for (int tap = 0; tap < 9; ++tap) {
            const int dy = (a.flip ? 1 - tap / 3 : tap / 3 - 1), dx = (a.flip ? 1 - tap % 3 : tap % 3 - 1);
            int off[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int ys = py[t] + dy, xs = px[t] + dx;
                const bool ok = pv[t] && ys >= 0 && ys < a.H && xs >= 0 && xs < a.W;
                off[t] = ok ? ((pb[t] * a.H + ys) * a.W + xs) * Cin : -1;
            }
            const bf16 *wr = a.w + ((size_t)(co0 + li) * 9 + tap) * Cin;
            const size_t mstride = (size_t)16 * 9 * Cin;   // next 16 output channels
            for (int c0 = 0; c0 < Cin; c0 += 16) {
                sh4 av[MT], bv[4];
#pragma unroll
                for (int m = 0; m < MT; ++m) av[m] = load4(wr + m * mstride + c0 + 4 * kg);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    bv[t] = sh4{0, 0, 0, 0};
                    if (off[t] >= 0) bv[t] = load4(a.x + off[t] + c0 + 4 * kg);
                }
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[m][t] = mfma(av[m], bv[t], acc[m][t]);
            }
        }
    } else if (MT == 1) {
        // small Cin: K = 9 Cin flattened as k = tap * Cin + ci, padded to 16
        const int K = 9 * Cin;
        for (int k0 = 0; k0 < K; k0 += 16) {
            sh4 av;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = k0 + 4 * kg + r;
                av[r] = k < K ? (short)a.w[(size_t)(co0 + li) * 9 * Cin + k] : (short)0;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                sh4 bv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int k = k0 + 4 * kg + r;
                    short v = 0;
                    if (k < K && pv[t]) {
                        const int tap = k / Cin, ci = k % Cin;
                        const int dy = (a.flip ? 1 - tap / 3 : tap / 3 - 1), dx = (a.flip ? 1 - tap % 3 : tap % 3 - 1);
                        const int ys = py[t] + dy, xs = px[t] + dx;
                        if (ys >= 0 && ys < a.H && xs >= 0 && xs < a.W)
                            v = (short)a.x[((size_t)(pb[t] * a.H + ys) * a.W + xs) * Cin + ci];
                    }
                    bv[r] = v;
                }
                acc[0][t] = mfma(av, bv, acc[0][t]);
            }
        }
    }
    // epilogue: rows co0 + 16 m + 4 kg + r, column = pixel
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (!pv[t]) continue;
            const size_t p = (size_t)pw + 16 * t + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = co0 + 16 * m + 4 * kg + r;
                if (co >= a.Cout) continue;
                float v = acc[m][t][r] + (a.bias ? a.bias[co] : 0.f);
                if (a.relu) v = v > 0.f ? v : 0.f;
                if (a.mask && !pos(a.mask[p * a.Cout + co])) v = 0.f;
                if (a.y) a.y[p * a.Cout + co] = f2bf(v);
                if (a.yf) a.yf[p * a.Cout + co] = v;
            }
        }
}

// ---------------------------------------------------------------------------
// The 3x3 convolution for Cin a multiple of 32 and Cout of 16 MF on the
// gfx950 v_mfma_f32_16x16x32_bf16 (K = 32 input channels of one tap per MFMA),
// persistent: a workgroup of 8 waves keeps one block of 16 MF output channels
// and walks its work items (a 16 x 32 pixel tile, a chunk of 32 input
// channels) tile by tile.  Per item the (16+2) x (32+2) input pixels with their
// halo and the 16 MF x 9 x 32 weights sit in LDS and each wave runs 9 taps x
// MF x 4 MFMAs on tile rows 2w and 2w+1.  The global loads of the next DEPTH
// items are in flight in registers while the current one computes (DEPTH 2
// where one item's matrix work is too short to cover the memory latency);
// with Cin = 32 the weights are staged once for all tiles.  An LDS pixel (or
// weight row) holds 32 channels in 64 B padded to 80 B, so the 16-byte reads
// of eight consecutive lanes fall on distinct banks.  Lane l holds
// A[l%16][8(l/16)..+7] and B[8(l/16)..+7][l%16] (one 16-byte LDS read each)
// and D[4(l/16)..+3][l%16].
constexpr int kTW = 32;                       // output tile: pixels per row
constexpr int kIW = kTW + 2;                  // input tile row with the halo
constexpr int kPS = 40;                       // LDS stride of 32 channels, in bf16
constexpr int kPH = 16;                       // output rows per tile
constexpr int kPIH = kPH + 2;                 // input rows with the halo
constexpr int kPB = 512;                      // threads: 8 waves
constexpr int kXSeg = kPIH * kIW * 4;         // 16-byte segments of one input tile chunk
constexpr int kXPer = (kXSeg + kPB - 1) / kPB;

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f4 mfma32(bf8 a, bf8 b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

inline int conv32p_tiles(const ConvArgs &a)
{
    return a.B * ((a.H + kPH - 1) / kPH) * ((a.W + kTW - 1) / kTW);
}

// MASK: the epilogue applies a.mask (the input gradients); without it the
// mask's registers would cost the forward layers 2 %.
template <int MF, int DEPTH, bool MASK>
__global__ void __launch_bounds__(kPB, 1) k_conv32p(ConvArgs a)
{
    constexpr int kWSeg = 9 * 16 * MF * 4;    // 16-byte segments of one weight chunk
    constexpr int kWPer = (kWSeg + kPB - 1) / kPB;
    __shared__ __attribute__((aligned(16))) bf16 sX[kPIH * kIW * kPS];
    __shared__ __attribute__((aligned(16))) bf16 sW[9 * 16 * MF * kPS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, kg = lane >> 4;
    const int nCo = a.CoutP / (16 * MF);
    const int tilesX = (a.W + kTW - 1) / kTW, tilesY = (a.H + kPH - 1) / kPH;
    const int nTiles = a.B * tilesX * tilesY;
    const int cb = blockIdx.x % nCo, g = blockIdx.x / nCo, G = gridDim.x / nCo;
    const int co0 = cb * 16 * MF;
    const int Cin = a.Cin, nChunks = Cin / 32;
    if (g >= nTiles) return;
    const int nItems = ((nTiles - g + G - 1) / G) * nChunks;   // tiles g, g + G, ... times chunks
    const bool wOnce = nChunks == 1;
    uint4 rxA[kXPer], rwA[kWPer], rxB[DEPTH == 2 ? kXPer : 1], rwB[DEPTH == 2 ? kWPer : 1];
    f4 acc[MF][4];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
    // this lane's biases in registers: a global load in the epilogue would
    // make its wait also wait for the prefetch in flight
    float bias[MF][4];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[m][r] = a.bias ? a.bias[co0 + 16 * m + 4 * kg + r] : 0.f;
    // item -> (image, tile origin, first input channel)
#define CONV32P_ORIGIN(item)                                       \
    const int tile_ = g + ((item) / nChunks) * G;                  \
    const int c0 = ((item) % nChunks) * 32;                        \
    const int x0 = (tile_ % tilesX) * kTW;                         \
    const int y0 = ((tile_ / tilesX) % tilesY) * kPH;              \
    const int bimg = (tile_ / tilesX) / tilesY;
    // global loads of an item into rx (and rw)
#define CONV32P_FETCH(item, withW, rx, rw)                                                                           \
    {                                                                                                                \
        CONV32P_ORIGIN(item)                                                                                         \
        _Pragma("unroll") for (int j = 0; j < kXPer; ++j)                                                            \
        {                                                                                                            \
            const int s = tid + kPB * j;                                                                             \
            const int pix = s >> 2, seg = s & 3;                                                                     \
            const int iy = pix / kIW, ix = pix - iy * kIW;                                                           \
            const int ys = y0 + iy - 1, xs = x0 + ix - 1;                                                            \
            const bool in = s < kXSeg && ys >= 0 && ys < a.H && xs >= 0 && xs < a.W;                                 \
            rx[j] = in ? *reinterpret_cast<const uint4 *>(a.x + ((size_t)(bimg * a.H + ys) * a.W + xs) * Cin + c0 +  \
                                                          8 * seg)                                                   \
                       : make_uint4(0u, 0u, 0u, 0u);                                                                 \
        }                                                                                                            \
        if (withW) {                                                                                                 \
            _Pragma("unroll") for (int j = 0; j < kWPer; ++j)                                                        \
            {                                                                                                        \
                const int s = tid + kPB * j;                                                                         \
                const int seg = s & 3, r = s >> 2;              /* LDS row r = tap * 16 MF + col */                \
                const int tap = r / (16 * MF), col = r - tap * (16 * MF);                                            \
                rw[j] = s < kWSeg ? *reinterpret_cast<const uint4 *>(a.w + ((size_t)(co0 + col) * 9 + tap) * Cin +  \
                                                                     c0 + 8 * seg)                                   \
                                  : make_uint4(0u, 0u, 0u, 0u);                                                      \
            }                                                                                                        \
        }                                                                                                            \
    }
    // one item: its registers into LDS, the loads of item + DEPTH issued, the
    // MFMAs, and after the tile's last chunk bias, ReLU, bf16 store
#define CONV32P_STEP(item, rx, rw)                                                                                   \
    {                                                                                                                \
        const bool loadW = !wOnce || (item) == 0;                                                                    \
        __syncthreads();                                                                                             \
        _Pragma("unroll") for (int j = 0; j < kXPer; ++j)                                                            \
        {                                                                                                            \
            const int s = tid + kPB * j;                                                                             \
            if (s < kXSeg) *reinterpret_cast<uint4 *>(&sX[(s >> 2) * kPS + 8 * (s & 3)]) = rx[j];                    \
        }                                                                                                            \
        if (loadW)                                                                                                   \
            _Pragma("unroll") for (int j = 0; j < kWPer; ++j)                                                        \
            {                                                                                                        \
                const int s = tid + kPB * j;                                                                         \
                const int seg = s & 3;                                                                               \
                if (s < kWSeg) *reinterpret_cast<uint4 *>(&sW[(s >> 2) * kPS + 8 * seg]) = rw[j];                     \
            }                                                                                                        \
        __syncthreads();                                                                                             \
        const bool lastChunk = (item) % nChunks == nChunks - 1;                                                      \
        uint2 mk[MASK ? MF : 1][4];                                                                                  \
        if (MASK && lastChunk) {           /* before the prefetch, so that their wait does not include it */         \
            CONV32P_ORIGIN(item)                                                                                     \
            (void)c0;                                                                                                \
            _Pragma("unroll") for (int t = 0; t < 4; ++t)                                                            \
            {                                                                                                        \
                const int yy = y0 + 2 * wave + (t >> 1), xx = x0 + 16 * (t & 1) + li;                               \
                const bool ok = yy < a.H && xx < a.W;                                                                \
                const size_t p = ok ? ((size_t)bimg * a.H + yy) * a.W + xx : 0;                                      \
                _Pragma("unroll") for (int m = 0; m < (MASK ? MF : 1); ++m) mk[m][t] =                               \
                    *reinterpret_cast<const uint2 *>(a.mask + p * a.Cout + co0 + 16 * m + 4 * kg);                   \
            }                                                                                                        \
        }                                                                                                            \
        if ((item) + DEPTH < nItems) CONV32P_FETCH((item) + DEPTH, !wOnce, rx, rw)                                   \
        _Pragma("unroll") for (int tap = 0; tap < 9; ++tap)                                                          \
        {                                                                                                            \
            const int dy = a.flip ? 1 - tap / 3 : tap / 3 - 1, dx = a.flip ? 1 - tap % 3 : tap % 3 - 1;              \
            bf8 av[MF], bv[4];                                                                                       \
            _Pragma("unroll") for (int m = 0; m < MF; ++m) av[m] =                                                   \
                *reinterpret_cast<const bf8 *>(&sW[(tap * 16 * MF + 16 * m + li) * kPS + 8 * kg]);                   \
            _Pragma("unroll") for (int t = 0; t < 4; ++t)                                                            \
            {                                                                                                        \
                const int ry = 2 * wave + (t >> 1) + 1 + dy, rxx = 16 * (t & 1) + li + 1 + dx;                      \
                bv[t] = *reinterpret_cast<const bf8 *>(&sX[(ry * kIW + rxx) * kPS + 8 * kg]);                        \
            }                                                                                                        \
            _Pragma("unroll") for (int m = 0; m < MF; ++m)                                                           \
                _Pragma("unroll") for (int t = 0; t < 4; ++t) acc[m][t] = mfma32(av[m], bv[t], acc[m][t]);           \
        }                                                                                                            \
        if (lastChunk) {                                                                                             \
            CONV32P_ORIGIN(item)                                                                                     \
            (void)c0;                                                                                                \
            _Pragma("unroll") for (int t = 0; t < 4; ++t)                                                            \
            {                                                                                                        \
                const int yy = y0 + 2 * wave + (t >> 1), xx = x0 + 16 * (t & 1) + li;                               \
                const bool ok = yy < a.H && xx < a.W;                                                                \
                const size_t p = ((size_t)bimg * a.H + yy) * a.W + xx;                                               \
                _Pragma("unroll") for (int m = 0; m < MF; ++m)                                                       \
                {                                                                                                    \
                    const int co = co0 + 16 * m + 4 * kg;                                                            \
                    float v[4];                                                                                      \
                    _Pragma("unroll") for (int r = 0; r < 4; ++r)                                                    \
                    {                                                                                                \
                        v[r] = acc[m][t][r] + bias[m][r];                                                            \
                        if (a.relu) v[r] = v[r] > 0.f ? v[r] : 0.f;                                                  \
                    }                                                                                                \
                    acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};                                                              \
                    if (MASK) {                                                                                      \
                        const uint2 k = mk[MASK ? m : 0][t];                                                                    \
                        v[0] = pos(k.x & 0xFFFFu) ? v[0] : 0.f;                                                      \
                        v[1] = pos(k.x >> 16) ? v[1] : 0.f;                                                          \
                        v[2] = pos(k.y & 0xFFFFu) ? v[2] : 0.f;                                                      \
                        v[3] = pos(k.y >> 16) ? v[3] : 0.f;                                                          \
                    }                                                                                                \
                    if (ok && a.y) {                                                                                 \
                        uint2 o;                                                                                     \
                        o.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);                                   \
                        o.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);                                   \
                        *reinterpret_cast<uint2 *>(a.y + p * a.Cout + co) = o;                                       \
                    }                                                                                                \
                    if (ok && a.yf)                                                                                  \
                        _Pragma("unroll") for (int r = 0; r < 4; ++r) a.yf[p * a.Cout + co + r] = v[r];              \
                }                                                                                                    \
            }                                                                                                        \
        }                                                                                                            \
    }
    CONV32P_FETCH(0, true, rxA, rwA)
    if (DEPTH == 2 && nItems > 1) CONV32P_FETCH(1, !wOnce, rxB, rwB)
    for (int item = 0; item < nItems; item += DEPTH) {
        CONV32P_STEP(item, rxA, rwA)
        if (DEPTH == 2 && item + 1 < nItems) CONV32P_STEP(item + 1, rxB, rwB)
    }
#undef CONV32P_STEP
#undef CONV32P_FETCH
#undef CONV32P_ORIGIN
}

// 3x3 convolution from one input channel to Cout (a multiple of 8, at most
// 256) channels: one thread per pixel; the weights as floats in LDS, [tap][co],
// read by every lane at one address.  2 B in and 2 Cout B out per pixel, 2.4 TB/s
// (2048 x 1024 x 4 pixels to 32 channels 224 us): the 9 Cout products, their LDS
// reads and the strided stores bound it alike.  A thread per pixel and 8 channels,
// whose stores are contiguous, repeats the input's loads and takes 330 us.
__global__ void __launch_bounds__(kB) k_conv_c1(ConvArgs a)
{
    __shared__ float sw[9 * 256];
    for (int k = threadIdx.x; k < a.Cout * 9; k += kB) {
        const int tap = k / a.Cout, co = k - tap * a.Cout;
        sw[k] = bf2f(a.w[co * 9 + tap]);
    }
    __syncthreads();
    const int p = blockIdx.x * kB + threadIdx.x;        // pixels < 2^31 (checked by the caller)
    if (p >= a.B * a.H * a.W) return;
    const int xx = p % a.W, yy = (p / a.W) % a.H, b = p / (a.W * a.H);
    float xin[9];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        const int dy = a.flip ? 1 - tap / 3 : tap / 3 - 1, dx = a.flip ? 1 - tap % 3 : tap % 3 - 1;
        const int ys = yy + dy, xs = xx + dx;
        xin[tap] = (ys >= 0 && ys < a.H && xs >= 0 && xs < a.W) ? bf2f(a.x[((size_t)b * a.H + ys) * a.W + xs]) : 0.f;
    }
    for (int g = 0; g < a.Cout / 8; ++g) {
        V8 o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o.v[i] = a.bias ? a.bias[8 * g + i] : 0.f;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const float4 w0 = *reinterpret_cast<const float4 *>(&sw[tap * a.Cout + 8 * g]);
            const float4 w1 = *reinterpret_cast<const float4 *>(&sw[tap * a.Cout + 8 * g + 4]);
            o.v[0] += w0.x * xin[tap]; o.v[1] += w0.y * xin[tap]; o.v[2] += w0.z * xin[tap]; o.v[3] += w0.w * xin[tap];
            o.v[4] += w1.x * xin[tap]; o.v[5] += w1.y * xin[tap]; o.v[6] += w1.z * xin[tap]; o.v[7] += w1.w * xin[tap];
        }
        if (a.relu)
#pragma unroll
            for (int i = 0; i < 8; ++i) o.v[i] = o.v[i] < 0.f ? 0.f : o.v[i];
        if (a.mask) {
            const V8 k = ld8(a.mask + (size_t)p * a.Cout + 8 * g);
#pragma unroll
            for (int i = 0; i < 8; ++i) o.v[i] = k.v[i] > 0.f ? o.v[i] : 0.f;
        }
        st8(a.y + (size_t)p * a.Cout + 8 * g, o);
    }
}

// 3x3 convolution from Cin (a multiple of 32) channels to one, as nine dot
// products per input pixel: an MFMA with the taps as its rows (9 of 16) and 16
// consecutive pixels as its columns, whose operand is the kilobyte those pixels
// occupy, straight from memory.  The products of a 16 x 32 pixel tile and its
// halo go to LDS, [tap][pixel], and each output adds its nine.  Load-bound: 2
// Cin B in (1.2 times with the halo) and 2 (+4) B out per pixel.  With the
// products on the vector units from an LDS copy of the input 2048 x 1024 x 4
// pixels of 32 channels took 258 us; 124 us now.
constexpr int kOH = 16, kOW = 32, kOBatch = 5;   // output tile, operands in flight of a wave
constexpr int kOIW = kOW + 2, kOIH = kOH + 2, kOPix = kOIW * kOIH, kOGroups = (kOPix + 15) / 16;
__global__ void __launch_bounds__(kB) k_conv_to1(ConvArgs a)
{
    __shared__ float sP[9][kOGroups * 16];
    const int tilesX = (a.W + kOW - 1) / kOW, tilesY = (a.H + kOH - 1) / kOH;
    int tile = blockIdx.x;
    const int tx = tile % tilesX;
    tile /= tilesX;
    const int ty = tile % tilesY, bimg = tile / tilesY;
    const int x0 = tx * kOW, y0 = ty * kOH, Cin = a.Cin;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, kg = lane >> 4;
    const bf8 zero = __builtin_bit_cast(bf8, make_uint4(0u, 0u, 0u, 0u));
    for (int g0 = wave; g0 < kOGroups; g0 += kOBatch * (kB / 64)) {
        const bf16 *src[kOBatch];
        bool in[kOBatch];
        f4 acc[kOBatch];
#pragma unroll
        for (int k = 0; k < kOBatch; ++k) {
            const int pix = 16 * (g0 + k * (kB / 64)) + li, ys = y0 + pix / kOIW - 1, xs = x0 + pix % kOIW - 1;
            in[k] = pix < kOPix && ys >= 0 && ys < a.H && xs >= 0 && xs < a.W;
            src[k] = a.x + (((size_t)bimg * a.H + ys) * a.W + xs) * Cin + 8 * kg;
            acc[k] = f4{0.f, 0.f, 0.f, 0.f};
        }
        for (int c0 = 0; c0 < Cin; c0 += 32) {
            // the row of the operand is the tap; rows 9 .. 15 are zero
            const bf8 av = li < 9 ? *reinterpret_cast<const bf8 *>(a.w + li * Cin + c0 + 8 * kg) : zero;
            bf8 bv[kOBatch];
#pragma unroll
            for (int k = 0; k < kOBatch; ++k) bv[k] = in[k] ? *reinterpret_cast<const bf8 *>(src[k] + c0) : zero;
#pragma unroll
            for (int k = 0; k < kOBatch; ++k) acc[k] = mfma32(av, bv[k], acc[k]);
        }
#pragma unroll
        for (int k = 0; k < kOBatch; ++k) {
            const int pix = 16 * (g0 + k * (kB / 64)) + li;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * kg + r < 9 && pix < kOGroups * 16) sP[4 * kg + r][pix] = acc[k][r];
        }
    }
    __syncthreads();
    const float bias = a.bias ? a.bias[0] : 0.f;
    for (int q = threadIdx.x; q < kOH * kOW; q += kB) {
        const int ry = q / kOW, rx = q % kOW, yy = y0 + ry, xx = x0 + rx;
        if (yy >= a.H || xx >= a.W) continue;
        float v = 0.f;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int dy = a.flip ? 1 - tap / 3 : tap / 3 - 1, dx = a.flip ? 1 - tap % 3 : tap % 3 - 1;
            v += sP[tap][(ry + 1 + dy) * kOIW + rx + 1 + dx];
        }
        v += bias;
        if (a.relu && v < 0.f) v = 0.f;
        const size_t p = ((size_t)bimg * a.H + yy) * a.W + xx;
        if (a.mask && !pos(a.mask[p])) v = 0.f;
        if (a.y) a.y[p] = f2bf(v);
        if (a.yf) a.yf[p] = v;
    }
}

// k_conv32p where the channels allow it (Cin a multiple of 32, Cout of 32);
// the one-channel input and output layers on their load-bound kernels;
// otherwise k_conv with the widest channel blocking that divides CoutP
// (small Cin takes the flattened path, one tile)
void launch_conv(const ConvArgs &a, hipStream_t s)
{
    if (a.Cin % 32 == 0 && a.Cout % 32 == 0 && a.CoutP == a.Cout) {
        // one persistent workgroup per CU and occupancy slot
        static int slots4 = 0, slots2 = 0;
        if (!slots4) {
            int dev = 0, cus = 0, o4 = 0, o2 = 0;
            HU_CHECK(hipGetDevice(&dev));
            HU_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
            HU_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&o4, k_conv32p<4, 1, false>, kPB, 0));
            HU_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&o2, k_conv32p<2, 2, false>, kPB, 0));
            slots2 = cus * std::max(o2, 1);
            slots4 = cus * std::max(o4, 1);
        }
        const int mf = a.Cout % 64 == 0 ? 4 : 2, nCo = a.Cout / (16 * mf);
        const int G = std::max(1, std::min(conv32p_tiles(a), (mf == 4 ? slots4 : slots2) / nCo));
        if (mf == 4 && a.mask) k_conv32p<4, 1, true><<<G * nCo, kPB, 0, s>>>(a);
        else if (mf == 4) k_conv32p<4, 1, false><<<G * nCo, kPB, 0, s>>>(a);
        else if (a.mask) k_conv32p<2, 2, true><<<G * nCo, kPB, 0, s>>>(a);
        else k_conv32p<2, 2, false><<<G * nCo, kPB, 0, s>>>(a);
        return;
    }
    if (a.Cin == 1 && a.Cout % 8 == 0 && a.Cout <= 256 && a.y && (double)a.B * a.H * a.W < 2e9) {
        const int n = a.B * a.H * a.W;
        k_conv_c1<<<(n + kB - 1) / kB, kB, 0, s>>>(a);
        return;
    }
    if (a.Cout == 1 && a.Cin % 32 == 0) {
        k_conv_to1<<<a.B * ((a.H + kOH - 1) / kOH) * ((a.W + kOW - 1) / kOW), kB, 0, s>>>(a);
        return;
    }
    const int P = a.B * a.H * a.W;
    const int mt = (a.Cin & 15) ? 1 : (a.CoutP % 64 == 0) ? 4 : (a.CoutP % 32 == 0) ? 2 : 1;
    const dim3 grid((P + 255) / 256, a.CoutP / (16 * mt));
    if (mt == 4) k_conv<4><<<grid, kB, 0, s>>>(a);
    else if (mt == 2) k_conv<2><<<grid, kB, 0, s>>>(a);
    else k_conv<1><<<grid, kB, 0, s>>>(a);
}

// Gradients are added with the hardware's FP32 atomic (atomicAdd compiles to a
// compare-and-swap loop).
// Weight gradient dW[co][tap][ci] += sum_p dY[p][co] X[p + s(tap)][ci]:
// M = Cout, N = 9 Cin (n = tap * Cin + ci), K = pixels, split over blockIdx.z.
// grid = (ceil(9 Cin / 64), CoutP / 16, splits); 64 threads per block.
__global__ void __launch_bounds__(64) k_conv_wgrad(const bf16 *dy, const bf16 *x, float *dw, int B, int H, int W,
                                                  int Cin, int Cout, int chunk)
{
    const int lane = threadIdx.x, li = lane & 15, kg = lane >> 4;
    const int P = B * H * W, N = 9 * Cin;
    const int co0 = blockIdx.y * 16;
    const int n0 = blockIdx.x * 64;
    const int k0 = blockIdx.z * chunk, k1 = min(P, k0 + chunk);
    f4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    int tapn[4], cin[4];
    bool nv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int n = n0 + 16 * t + li;
        nv[t] = n < N;
        tapn[t] = nv[t] ? n / Cin : 0;
        cin[t] = nv[t] ? n % Cin : 0;
    }
    const int co = co0 + li;
    for (int kb = k0; kb < k1; kb += 16) {
        sh4 av;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = kb + 4 * kg + r;
            av[r] = (p < k1 && co < Cout) ? (short)dy[(size_t)p * Cout + co] : (short)0;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            sh4 bv;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = kb + 4 * kg + r;
                short v = 0;
                if (p < k1 && nv[t]) {
                    const int xx = p % W, yy = (p / W) % H, bb = p / (W * H);
                    const int ys = yy + tapn[t] / 3 - 1, xs = xx + tapn[t] % 3 - 1;
                    if (ys >= 0 && ys < H && xs >= 0 && xs < W)
                        v = (short)x[((size_t)(bb * H + ys) * W + xs) * Cin + cin[t]];
                }
                bv[r] = v;
            }
            acc[t] = mfma(av, bv, acc[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (!nv[t]) continue;
        const int n = n0 + 16 * t + li;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = co0 + 4 * kg + r;
            if (c < Cout) unsafeAtomicAdd(&dw[(size_t)c * N + n], acc[t][r]);
        }
    }
}

// Weight gradient for Cin and Cout multiples of 32 on v_mfma_f32_16x16x32_bf16:
// dW[co][tap][ci] = sum_p dY[p][co] X[p + s(tap)][ci], K = pixels.  A
// workgroup (4 waves) owns a block of 16 CF WCO output channels x 64 / WCO
// input channels, all 9 taps, and sums over the 8 x 32 pixel tiles
// blockIdx / nBlk, + ksplit, ...; wave w takes output-channel fragments
// (w % WCO) CF .. + CF - 1 and input-channel fragment w / WCO.  Per tile dY
// and the input with its halo are staged in LDS transposed (pixels fastest,
// 4 pixels per 8-byte write), so a lane's 8 consecutive pixels of a row are
// one 16-byte read.  Per K step (one tile row) and tap row dy, two aligned
// reads of the input row give the three dx shifts by funnel shifts of the
// lane's registers.  Row pitches are padded so that 16 lanes' 16-byte reads
// fall on distinct banks.  One atomic per weight and workgroup at the end.
// Two workgroups fit a CU, so 512 fill the chip; each more only adds its
// 18 000 atomics: 64 to 64 channels over 256 x 256 x 4 pixels take 102 us with
// 1024 workgroups, 77 with 512, 92 with 256.
constexpr int kWgBlocks = 512;
constexpr int kWgTH = 8, kWgTW = 32;          // pixel tile
constexpr int kDyPitch = kWgTH * kWgTW + 8;   // bf16 per output channel in LDS
constexpr int kXCols = 40;                    // input columns x0 - 1 .. x0 + 38
constexpr int kXPitch = (kWgTH + 2) * kXCols + 8;   // bf16 per input channel in LDS

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf8 as_bf8(u4v v) { return __builtin_bit_cast(bf8, v); }

template <int CF, int WCO>
__global__ void __launch_bounds__(kB, 2) k_wgrad32(const bf16 *dy, const bf16 *x, float *dw, float *db, int B, int H,
                                                   int W, int Cin, int Cout, int ksplit)
{
    constexpr int CO_BLK = 16 * CF * WCO, CI_BLK = 16 * (4 / WCO);
    __shared__ __attribute__((aligned(16))) bf16 sD[CO_BLK * kDyPitch];
    __shared__ __attribute__((aligned(16))) bf16 sXt[CI_BLK * kXPitch];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, kg = lane >> 4;
    const int nCoB = Cout / CO_BLK, nCiB = Cin / CI_BLK, nBlk = nCoB * nCiB;
    const int blk = blockIdx.x % nBlk, kz = blockIdx.x / nBlk;
    const int co0 = (blk % nCoB) * CO_BLK, ci0 = (blk / nCoB) * CI_BLK;
    const int cf0 = (wave % WCO) * CF, nf = wave / WCO;
    const int tilesX = (W + kWgTW - 1) / kWgTW, tilesY = (H + kWgTH - 1) / kWgTH, nTiles = B * tilesX * tilesY;
    f4 acc[CF][9];
#pragma unroll
    for (int m = 0; m < CF; ++m)
#pragma unroll
        for (int t = 0; t < 9; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
    // the bias gradient, from the dY that is staged anyway (one block of input
    // channels does it): this thread always stages channels co0 + 8 (tid % (CO_BLK / 8))
    const bool bias = ci0 == 0;
    float bs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int tile = kz; tile < nTiles; tile += ksplit) {
        const int tx = tile % tilesX, rest = tile / tilesX;
        const int x0 = tx * kWgTW, y0 = (rest % tilesY) * kWgTH, bimg = rest / tilesY;
        __syncthreads();
        // dY: units (row, 4-pixel group, 8-channel group)
        for (int u = tid; u < kWgTH * (kWgTW / 4) * (CO_BLK / 8); u += kB) {
            const int cg = u % (CO_BLK / 8), r2 = u / (CO_BLK / 8);
            const int x4 = r2 % (kWgTW / 4), r = r2 / (kWgTW / 4);
            const int yy = y0 + r;
            uint4 v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int xx = x0 + 4 * x4 + q;
                v[q] = (yy < H && xx < W)
                           ? *reinterpret_cast<const uint4 *>(dy + (((size_t)bimg * H + yy) * W + xx) * Cout + co0 + 8 * cg)
                           : make_uint4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                auto h = [&](const uint4 &w) -> uint32_t {
                    const uint32_t d = e < 2 ? w.x : e < 4 ? w.y : e < 6 ? w.z : w.w;
                    return (e & 1) ? (d >> 16) : (d & 0xFFFFu);
                };
                const uint2 o = make_uint2(h(v[0]) | (h(v[1]) << 16), h(v[2]) | (h(v[3]) << 16));
                *reinterpret_cast<uint2 *>(&sD[(8 * cg + e) * kDyPitch + r * kWgTW + 4 * x4]) = o;
                if (bias) bs[e] += (bf2f(h(v[0])) + bf2f(h(v[1]))) + (bf2f(h(v[2])) + bf2f(h(v[3])));
            }
        }
        // input with its halo: units (row, 4-column group, 8-channel group)
        for (int u = tid; u < (kWgTH + 2) * (kXCols / 4) * (CI_BLK / 8); u += kB) {
            const int ig = u % (CI_BLK / 8), r2 = u / (CI_BLK / 8);
            const int c4 = r2 % (kXCols / 4), r = r2 / (kXCols / 4);
            const int ys = y0 + r - 1;
            uint4 v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int xs = x0 - 1 + 4 * c4 + q;
                v[q] = (ys >= 0 && ys < H && xs >= 0 && xs < W)
                           ? *reinterpret_cast<const uint4 *>(x + (((size_t)bimg * H + ys) * W + xs) * Cin + ci0 + 8 * ig)
                           : make_uint4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                auto h = [&](const uint4 &w) -> uint32_t {
                    const uint32_t d = e < 2 ? w.x : e < 4 ? w.y : e < 6 ? w.z : w.w;
                    return (e & 1) ? (d >> 16) : (d & 0xFFFFu);
                };
                const uint2 o = make_uint2(h(v[0]) | (h(v[1]) << 16), h(v[2]) | (h(v[3]) << 16));
                *reinterpret_cast<uint2 *>(&sXt[(8 * ig + e) * kXPitch + r * kXCols + 4 * c4]) = o;
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int r = 0; r < kWgTH; ++r) {
            bf8 av[CF];
#pragma unroll
            for (int m = 0; m < CF; ++m)
                av[m] = *reinterpret_cast<const bf8 *>(&sD[(16 * (cf0 + m) + li) * kDyPitch + r * kWgTW + 8 * kg]);
#pragma unroll
            for (int dyi = 0; dyi < 3; ++dyi) {
                const bf16 *row = &sXt[(16 * nf + li) * kXPitch + (r + dyi) * kXCols + 8 * kg];
                const u4v f0 = *reinterpret_cast<const u4v *>(row), f1 = *reinterpret_cast<const u4v *>(row + 8);
                u4v s1, s2;   // shifted by one and by two columns
                s1[0] = __builtin_amdgcn_alignbit(f0[1], f0[0], 16);
                s1[1] = __builtin_amdgcn_alignbit(f0[2], f0[1], 16);
                s1[2] = __builtin_amdgcn_alignbit(f0[3], f0[2], 16);
                s1[3] = __builtin_amdgcn_alignbit(f1[0], f0[3], 16);
                s2[0] = f0[1]; s2[1] = f0[2]; s2[2] = f0[3]; s2[3] = f1[0];
                const bf8 bv[3] = {as_bf8(f0), as_bf8(s1), as_bf8(s2)};
#pragma unroll
                for (int dxi = 0; dxi < 3; ++dxi)
#pragma unroll
                    for (int m = 0; m < CF; ++m)
                        acc[m][3 * dyi + dxi] = mfma32(av[m], bv[dxi], acc[m][3 * dyi + dxi]);
            }
        }
    }
    if (bias) {
        __syncthreads();
        float *sb = reinterpret_cast<float *>(sD);     // [256][8]
#pragma unroll
        for (int e = 0; e < 8; ++e) sb[tid * 8 + e] = bs[e];
        __syncthreads();
        if (tid < CO_BLK) {
            const int g = tid / 8, e = tid % 8;
            float t = 0.f;
            for (int q = g; q < kB; q += CO_BLK / 8) t += sb[q * 8 + e];
            unsafeAtomicAdd(&db[co0 + tid], t);
        }
    }
    // D[4 kg + rr][li]: output channel co0 + 16 (cf0 + m) + 4 kg + rr, input channel ci0 + 16 nf + li
    const int ci = ci0 + 16 * nf + li;
#pragma unroll
    for (int m = 0; m < CF; ++m)
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const int co = co0 + 16 * (cf0 + m) + 4 * kg + rr;
                unsafeAtomicAdd(&dw[((size_t)co * 9 + t) * Cin + ci], acc[m][t][rr]);
            }
}

// Weight gradient of the one-channel layers on the same MFMA path: OUT1 is the
// output layer (Cin = 32, Cout = 1), otherwise the input layer (Cin = 1,
// Cout = 32).  The one channel fills row (or column) 0 of its 16-wide MFMA
// operand and the other lanes hold zeros.  Wave w takes 16-channel fragment
// w & 1 of the 32-channel side and tile rows (w >> 1) + 2 j.  Staging and
// shifts as in k_wgrad32; pixel tiles blockIdx.x, + gridDim.x, ...
template <bool OUT1>
__global__ void __launch_bounds__(kB) k_wgrad_one(const bf16 *dy, const bf16 *x, float *dw, float *db, int B, int H, int W)
{
    constexpr int NCO = OUT1 ? 1 : 32, NCI = OUT1 ? 32 : 1;
    __shared__ __attribute__((aligned(16))) bf16 sD[NCO * kDyPitch];
    __shared__ __attribute__((aligned(16))) bf16 sXt[NCI * kXPitch];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, kg = lane >> 4, fr = wave & 1;
    const int tilesX = (W + kWgTW - 1) / kWgTW, tilesY = (H + kWgTH - 1) / kWgTH, nTiles = B * tilesX * tilesY;
    f4 acc[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    const u4v zero = {0u, 0u, 0u, 0u};
    float bs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // bias gradient, as in k_wgrad32
    for (int tile = blockIdx.x; tile < nTiles; tile += gridDim.x) {
        const int tx = tile % tilesX, rest = tile / tilesX;
        const int x0 = tx * kWgTW, y0 = (rest % tilesY) * kWgTH, bimg = rest / tilesY;
        __syncthreads();
        // dY: units (row, 4-pixel group, 8-channel group); one channel: 4 scalars
        for (int u = tid; u < kWgTH * (kWgTW / 4) * ((NCO + 7) / 8); u += kB) {
            const int cg = u % ((NCO + 7) / 8), r2 = u / ((NCO + 7) / 8);
            const int x4 = r2 % (kWgTW / 4), r = r2 / (kWgTW / 4);
            const int yy = y0 + r;
            if (NCO == 1) {
                uint32_t h[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int xx = x0 + 4 * x4 + q;
                    h[q] = (yy < H && xx < W) ? (uint32_t)dy[((size_t)bimg * H + yy) * W + xx] : 0u;
                    bs[0] += bf2f((bf16)h[q]);
                }
                *reinterpret_cast<uint2 *>(&sD[r * kWgTW + 4 * x4]) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            } else {
                uint4 v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int xx = x0 + 4 * x4 + q;
                    v[q] = (yy < H && xx < W)
                               ? *reinterpret_cast<const uint4 *>(dy + (((size_t)bimg * H + yy) * W + xx) * NCO + 8 * cg)
                               : make_uint4(0u, 0u, 0u, 0u);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    auto h = [&](const uint4 &w) -> uint32_t {
                        const uint32_t d = e < 2 ? w.x : e < 4 ? w.y : e < 6 ? w.z : w.w;
                        return (e & 1) ? (d >> 16) : (d & 0xFFFFu);
                    };
                    *reinterpret_cast<uint2 *>(&sD[(8 * cg + e) * kDyPitch + r * kWgTW + 4 * x4]) =
                        make_uint2(h(v[0]) | (h(v[1]) << 16), h(v[2]) | (h(v[3]) << 16));
                    bs[e] += (bf2f(h(v[0])) + bf2f(h(v[1]))) + (bf2f(h(v[2])) + bf2f(h(v[3])));
                }
            }
        }
        // input with its halo: units (row, 4-column group, 8-channel group)
        for (int u = tid; u < (kWgTH + 2) * (kXCols / 4) * ((NCI + 7) / 8); u += kB) {
            const int ig = u % ((NCI + 7) / 8), r2 = u / ((NCI + 7) / 8);
            const int c4 = r2 % (kXCols / 4), r = r2 / (kXCols / 4);
            const int ys = y0 + r - 1;
            if (NCI == 1) {
                uint32_t h[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int xs = x0 - 1 + 4 * c4 + q;
                    h[q] = (ys >= 0 && ys < H && xs >= 0 && xs < W) ? (uint32_t)x[((size_t)bimg * H + ys) * W + xs] : 0u;
                }
                *reinterpret_cast<uint2 *>(&sXt[r * kXCols + 4 * c4]) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            } else {
                uint4 v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int xs = x0 - 1 + 4 * c4 + q;
                    v[q] = (ys >= 0 && ys < H && xs >= 0 && xs < W)
                               ? *reinterpret_cast<const uint4 *>(x + (((size_t)bimg * H + ys) * W + xs) * NCI + 8 * ig)
                               : make_uint4(0u, 0u, 0u, 0u);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    auto h = [&](const uint4 &w) -> uint32_t {
                        const uint32_t d = e < 2 ? w.x : e < 4 ? w.y : e < 6 ? w.z : w.w;
                        return (e & 1) ? (d >> 16) : (d & 0xFFFFu);
                    };
                    *reinterpret_cast<uint2 *>(&sXt[(8 * ig + e) * kXPitch + r * kXCols + 4 * c4]) =
                        make_uint2(h(v[0]) | (h(v[1]) << 16), h(v[2]) | (h(v[3]) << 16));
                }
            }
        }
        __syncthreads();
        // the one-channel side's operand: lane li = 0 only
        const bool one = li == 0;
#pragma unroll 1
        for (int j = 0; j < kWgTH / 2; ++j) {
            const int r = (wave >> 1) + 2 * j;
            bf8 av;
            if (OUT1) av = one ? *reinterpret_cast<const bf8 *>(&sD[r * kWgTW + 8 * kg]) : as_bf8(zero);
            else av = *reinterpret_cast<const bf8 *>(&sD[(16 * fr + li) * kDyPitch + r * kWgTW + 8 * kg]);
#pragma unroll
            for (int dyi = 0; dyi < 3; ++dyi) {
                u4v f0 = zero, f1 = zero;
                if (!OUT1 ? one : true) {
                    const bf16 *row = &sXt[(OUT1 ? (16 * fr + li) * kXPitch : 0) + (r + dyi) * kXCols + 8 * kg];
                    f0 = *reinterpret_cast<const u4v *>(row);
                    f1 = *reinterpret_cast<const u4v *>(row + 8);
                }
                u4v s1, s2;
                s1[0] = __builtin_amdgcn_alignbit(f0[1], f0[0], 16);
                s1[1] = __builtin_amdgcn_alignbit(f0[2], f0[1], 16);
                s1[2] = __builtin_amdgcn_alignbit(f0[3], f0[2], 16);
                s1[3] = __builtin_amdgcn_alignbit(f1[0], f0[3], 16);
                s2[0] = f0[1]; s2[1] = f0[2]; s2[2] = f0[3]; s2[3] = f1[0];
                acc[3 * dyi + 0] = mfma32(av, as_bf8(f0), acc[3 * dyi + 0]);
                acc[3 * dyi + 1] = mfma32(av, as_bf8(s1), acc[3 * dyi + 1]);
                acc[3 * dyi + 2] = mfma32(av, as_bf8(s2), acc[3 * dyi + 2]);
            }
        }
    }
    // The workgroup's sums meet in LDS, one atomic per weight and workgroup: all
    // workgroups add into the same 288 weights, and with an atomic per wave the
    // additions to one address took longer than the products.
    // D[4 kg + rr][li]: row = output channel (OUT1: only row 0), column = input channel (else: only column 0)
    __shared__ float sw[288], sb[kB * (OUT1 ? 1 : 8)];
    for (int q = tid; q < 288; q += kB) sw[q] = 0.f;
#pragma unroll
    for (int e = 0; e < (OUT1 ? 1 : 8); ++e) sb[tid * (OUT1 ? 1 : 8) + e] = bs[e];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        if (OUT1) {
            if (kg == 0) unsafeAtomicAdd(&sw[t * 32 + 16 * fr + li], acc[t][0]);
        } else if (li == 0) {
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) unsafeAtomicAdd(&sw[(16 * fr + 4 * kg + rr) * 9 + t], acc[t][rr]);
        }
    }
    __syncthreads();
    for (int q = tid; q < 288; q += kB) unsafeAtomicAdd(&dw[q], sw[q]);
    if (tid < NCO) {
        float t = 0.f;
        if (OUT1) {
            for (int q = 0; q < kB; ++q) t += sb[q];
        } else {
            for (int q = tid / 8; q < kB; q += NCO / 8) t += sb[q * 8 + tid % 8];
        }
        unsafeAtomicAdd(&db[tid], t);
    }
}

// Elementwise kernels take 8 channels (one 16-byte vector) per thread: every
// activation they touch has a channel count that is a multiple of 8.

// bias gradient for any C (layers whose weight gradient runs on k_conv_wgrad):
// one block per channel
__global__ void k_bias_grad(const bf16 *dy, float *db, int P, int C)
{
    __shared__ float sh[kB];
    const int c = blockIdx.y;
    float s = 0.f;
    for (int p = blockIdx.x * kB + threadIdx.x; p < P; p += gridDim.x * kB) s += bf2f(dy[(size_t)p * C + c]);
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = kB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) unsafeAtomicAdd(&db[c], sh[0]);
}

// 2x2 average pool (NHWC); H, W even; one thread per output pixel and 8 channels
__global__ void k_pool(const bf16 *x, bf16 *y, int B, int H, int W, int C)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
    if (k >= (size_t)B * Ho * Wo * C8) return;
    const int c = (int)(k % C8) * 8;
    size_t r = k / C8;
    const int xo = (int)(r % Wo); r /= Wo;
    const int yo = (int)(r % Ho);
    const int b = (int)(r / Ho);
    const bf16 *q = x + (((size_t)b * H + 2 * yo) * W + 2 * xo) * C + c;
    const V8 a = ld8(q), bb = ld8(q + C), cc = ld8(q + (size_t)W * C), d = ld8(q + (size_t)W * C + C);
    V8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = 0.25f * (a.v[i] + bb.v[i] + cc.v[i] + d.v[i]);
    st8(y + k * 8, o);
}

// Gradient at a skip activation y (a ReLU output that is pooled and also added to
// the decoder): dx = pool^T(dy) + ds where y is positive, 0 elsewhere.  0.25 dy
// is exact in bf16, so one rounding is left.
__global__ void k_skip_grad(const bf16 *dy, const bf16 *ds, const bf16 *y, bf16 *dx, int B, int H, int W, int C)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    const int C8 = C / 8;
    if (k >= (size_t)B * H * W * C8) return;
    const int c = (int)(k % C8) * 8;
    size_t r = k / C8;
    const int xx = (int)(r % W); r /= W;
    const int yy = (int)(r % H);
    const int b = (int)(r / H);
    V8 o = ld8(dy + (((size_t)b * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c);
    const V8 t = ld8(ds + k * 8), a = ld8(y + k * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = a.v[i] > 0.f ? 0.25f * o.v[i] + t.v[i] : 0.f;
    st8(dx + k * 8, o);
}

// nearest x2 upsample plus skip: y = up(x) + s
__global__ void k_up_add(const bf16 *x, const bf16 *s, bf16 *y, int B, int H, int W, int C)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    const int C8 = C / 8;
    if (k >= (size_t)B * H * W * C8) return;
    const int c = (int)(k % C8) * 8;
    size_t r = k / C8;
    const int xx = (int)(r % W); r /= W;
    const int yy = (int)(r % H);
    const int b = (int)(r / H);
    V8 o = ld8(x + (((size_t)b * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c);
    const V8 t = ld8(s + k * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] += t.v[i];
    st8(y + k * 8, o);
}

// gradient of up(x) at a ReLU output x: dx[y][x] = sum of the 2x2 block of dy
// where x is positive, 0 elsewhere
__global__ void k_up_grad(const bf16 *dy, const bf16 *x, bf16 *dx, int B, int Hs, int Ws, int C)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    const int C8 = C / 8;
    if (k >= (size_t)B * Hs * Ws * C8) return;
    const int c = (int)(k % C8) * 8;
    size_t r = k / C8;
    const int xx = (int)(r % Ws); r /= Ws;
    const int yy = (int)(r % Hs);
    const int b = (int)(r / Hs);
    const int W = 2 * Ws;
    const bf16 *q = dy + (((size_t)b * 2 * Hs + 2 * yy) * W + 2 * xx) * C + c;
    const V8 a = ld8(q), bb = ld8(q + C), cc = ld8(q + (size_t)W * C), d = ld8(q + (size_t)W * C + C);
    V8 o;
    const V8 xv = ld8(x + k * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = xv.v[i] > 0.f ? a.v[i] + bb.v[i] + cc.v[i] + d.v[i] : 0.f;
    st8(dx + k * 8, o);
}

__global__ void k_to_bf(const float *x, bf16 *y, size_t n, float scale)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    if (k < n) y[k] = f2bf(x[k] * scale);
}

// MSE loss of the fp32 output against the target; gradient 2 (o - t) / n in bf16
// (grid-stride over at most kMseBlocks blocks: one atomic per block)
constexpr int kMseBlocks = 1024;
__global__ void k_mse(const float *o, const float *t, bf16 *g, float *loss, size_t n)
{
    __shared__ float sh[kB];
    float acc = 0.f;
    for (size_t k = (size_t)blockIdx.x * kB + threadIdx.x; k < n; k += (size_t)gridDim.x * kB) {
        const float d = o[k] - t[k];
        g[k] = f2bf(2.f * d / (float)n);
        acc += d * d;
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) unsafeAtomicAdd(loss, sh[0] / (float)n);
}

// Adam on the fp32 master weights; refresh the bf16 copies (padded rows stay 0)
__global__ void k_adam(float *w, float *m, float *v, const float *g, size_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    if (k >= n) return;
    const float gg = g[k];
    const float mm = b1 * m[k] + (1.f - b1) * gg;
    const float vv = b2 * v[k] + (1.f - b2) * gg * gg;
    m[k] = mm;
    v[k] = vv;
    w[k] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
}

// bf16 copies of one layer: wf [Cout][9][Cin] -> wb [CoutP][9][Cin] and the
// transposed wt [CinP][9][Cout] (wt[ci][tap][co] = w[co][tap][ci]) used by the
// input gradient; padded rows are zero.
__global__ void k_wcopy(const float *wf, bf16 *wb, bf16 *wt, int Cin, int Cout, int CoutP, int CinP)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    const size_t nb = (size_t)CoutP * 9 * Cin, nt = (size_t)CinP * 9 * Cout;
    if (k < nb) {
        const int co = (int)(k / (9 * Cin));
        wb[k] = co < Cout ? f2bf(wf[k]) : (bf16)0;
    }
    if (k < nt) {
        const int ci = (int)(k / (9 * Cout)), rem = (int)(k % (9 * Cout)), tap = rem / Cout, co = rem % Cout;
        wt[k] = ci < Cin ? f2bf(wf[((size_t)co * 9 + tap) * Cin + ci]) : (bf16)0;
    }
}

int nb(size_t n) { return (int)((n + kB - 1) / kB); }
int pad16(int c) { return (c + 15) / 16 * 16; }

struct Layer {
    int cin, cout, relu;
    size_t woff, boff;       // offsets into the fp32 parameter vector
};

}  // namespace unet

using namespace unet;

struct csrst_warmstart {
    std::string err;
    hipStream_t s = nullptr;
    int H = 0, W = 0, base = 32, maxBatch = 0;
    hu::Stage stage;     // transfers on s of arrays in pageable memory
    std::vector<Layer> L;          // 15 convolutions
    size_t nparam = 0;
    DBuf<float> w, m, v, g;        // master weights, Adam moments, gradients
    DBuf<bf16> wb, wt;             // bf16 copies per layer (offsets below)
    std::vector<size_t> wbOff, wtOff;
    DBuf<bf16> act;                // activations and gradients arena
    DBuf<float> outf, tgt, scratchF, lossBuf;
    int steps = 0;
    // activation offsets
    struct Buf { size_t off; int h, w, c; };
    std::vector<Buf> A;            // forward activations
    std::vector<Buf> Gd;           // gradient buffers (same shapes)
    int batch = 0;
    // the multigrid of the grid H x W and the buffers of the network-in-the-loop
    // solve and of its training pairs
    struct Loop {
        pmg::Solver mg;
        bool ready = false;
        double hx = 0, hy = 0;
        std::vector<uint8_t> cls;      // host copy of the node classes of the hierarchy
        size_t unknowns = 0;
        DBuf<uint8_t> dcls;
        DBuf<double> b, phi, pstar, part;
        DBuf<double> pprev, rprev;     // the previous iterate and its residual (two-direction step)
        DBuf<float> dir;               // the network's direction as a level-0 array
        DBuf<bf16> pairIn;             // [maxBatch][H][W] r / rms(r)
        DBuf<float> pairTgt;           // [maxBatch][H][W] e / rms(e)
    } loop;

    bf16 *ptr(const Buf &b) { return act.p + b.off; }
};

namespace {

// conv indices in order: 0 c00 1->32, 1 c01, 2 c10 32->64, 3 c11, 4 c20 64->128,
// 5 c21, 6 c30 128->256, 7 c31, 8 c22 256->128, 9 c23, 10 c12 128->64, 11 c13,
// 12 c02 64->32, 13 c03, 14 out 32->1
void make_layers(csrst_warmstart *u)
{
    const int b = u->base;
    const int io[15][3] = {{1, b, 1},          {b, b, 1},          {b, 2 * b, 1},     {2 * b, 2 * b, 1},
                           {2 * b, 4 * b, 1},  {4 * b, 4 * b, 1},  {4 * b, 8 * b, 1}, {8 * b, 8 * b, 1},
                           {8 * b, 4 * b, 1},  {4 * b, 4 * b, 1},  {4 * b, 2 * b, 1}, {2 * b, 2 * b, 1},
                           {2 * b, b, 1},      {b, b, 1},          {b, 1, 0}};
    size_t off = 0;
    u->L.clear();
    for (auto &e : io) {
        Layer l;
        l.cin = e[0]; l.cout = e[1]; l.relu = e[2];
        l.woff = off; off += (size_t)l.cout * 9 * l.cin;
        l.boff = off; off += l.cout;
        u->L.push_back(l);
    }
    u->nparam = off;
}

void conv(csrst_warmstart *u, int li, const bf16 *x, bf16 *y, float *yf, int B, int H, int W)
{
    const Layer &l = u->L[li];
    ConvArgs a;
    a.x = x; a.w = u->wb.p + u->wbOff[li]; a.bias = u->w.p + l.boff; a.y = y; a.yf = yf;
    a.B = B; a.H = H; a.W = W; a.Cin = l.cin; a.Cout = l.cout; a.CoutP = pad16(l.cout); a.flip = 0; a.relu = l.relu; a.mask = nullptr;
    launch_conv(a, u->s);
}

// input gradient of conv li: dx[P][cin] from dpre[P][cout], zero where mask (the
// input, if a ReLU made it) is not positive
void conv_dgrad(csrst_warmstart *u, int li, const bf16 *dpre, bf16 *dx, const bf16 *mask, int B, int H, int W)
{
    const Layer &l = u->L[li];
    ConvArgs a;
    a.x = dpre; a.w = u->wt.p + u->wtOff[li]; a.bias = nullptr; a.y = dx; a.yf = nullptr;
    a.B = B; a.H = H; a.W = W; a.Cin = l.cout; a.Cout = l.cin; a.CoutP = pad16(l.cin); a.flip = 1; a.relu = 0; a.mask = mask;
    launch_conv(a, u->s);
}

void conv_wgrad(csrst_warmstart *u, int li, const bf16 *dpre, const bf16 *x, int B, int H, int W)
{
    const Layer &l = u->L[li];
    const int P = B * H * W;
    const int chunk = 1024;
    dim3 grid((9 * l.cin + 63) / 64, pad16(l.cout) / 16, (P + chunk - 1) / chunk);
    if (l.cin % 32 == 0 && l.cout % 32 == 0) {
        const int tiles = B * ((H + kWgTH - 1) / kWgTH) * ((W + kWgTW - 1) / kWgTW);
        auto go = [&](auto kern, int coBlk, int ciBlk) {
            const int nBlk = (l.cout / coBlk) * (l.cin / ciBlk);
            const int ksplit = std::max(1, std::min(tiles, kWgBlocks / nBlk));
            kern<<<nBlk * ksplit, kB, 0, u->s>>>(dpre, x, u->g.p + l.woff, u->g.p + l.boff, B, H, W, l.cin, l.cout, ksplit);
        };
        if (l.cin % 64 == 0) go(k_wgrad32<2, 1>, 32, 64);
        else if (l.cout % 64 == 0) go(k_wgrad32<2, 2>, 64, 32);
        else go(k_wgrad32<1, 2>, 32, 32);
    } else if ((l.cin == 1 && l.cout == 32) || (l.cin == 32 && l.cout == 1)) {
        const int tiles = B * ((H + kWgTH - 1) / kWgTH) * ((W + kWgTW - 1) / kWgTW);
        float *w = u->g.p + l.woff, *b = u->g.p + l.boff;
        if (l.cout == 1) k_wgrad_one<true><<<std::min(tiles, 1024), kB, 0, u->s>>>(dpre, x, w, b, B, H, W);
        else k_wgrad_one<false><<<std::min(tiles, 1024), kB, 0, u->s>>>(dpre, x, w, b, B, H, W);
    } else {
        k_conv_wgrad<<<grid, 64, 0, u->s>>>(dpre, x, u->g.p + l.woff, B, H, W, l.cin, l.cout, chunk);
        dim3 bg(std::min(64, (P + kB - 1) / kB), l.cout);
        k_bias_grad<<<bg, kB, 0, u->s>>>(dpre, u->g.p + l.boff, P, l.cout);
    }
}

void refresh_bf16(csrst_warmstart *u)
{
    for (size_t i = 0; i < u->L.size(); ++i) {
        const Layer &l = u->L[i];
        const size_t n = std::max((size_t)pad16(l.cout) * 9 * l.cin, (size_t)pad16(l.cin) * 9 * l.cout);
        k_wcopy<<<nb(n), kB, 0, u->s>>>(u->w.p + l.woff, u->wb.p + u->wbOff[i], u->wt.p + u->wtOff[i], l.cin, l.cout,
                                         pad16(l.cout), pad16(l.cin));
    }
    HU_LAUNCH_CHECK();
}

// activation plan for batch B: forward buffers A[0..] and gradient buffers
void plan(csrst_warmstart *u, int B)
{
    if (u->batch == B) return;
    const int H = u->H, W = u->W, b = u->base;
    u->A.clear();
    size_t off = 0;
    auto add = [&](std::vector<csrst_warmstart::Buf> &v, int h, int w, int c) {
        v.push_back({off, h, w, c});
        off += (size_t)B * h * w * c;
        off = (off + 63) / 64 * 64;
    };
    // forward: 0 in, 1 c00, 2 s0(c01), 3 p0, 4 c10, 5 s1(c11), 6 p1, 7 c20, 8 s2(c21), 9 p2, 10 c30, 11 c31,
    // 12 c22, 13 u2(up+s2), 14 c23, 15 c12, 16 u1, 17 c13, 18 c02, 19 u0, 20 c03, 21 out(bf16)
    const int sh[22][3] = {{H, W, 1},          {H, W, b},          {H, W, b},          {H / 2, W / 2, b},
                           {H / 2, W / 2, 2 * b}, {H / 2, W / 2, 2 * b}, {H / 4, W / 4, 2 * b}, {H / 4, W / 4, 4 * b},
                           {H / 4, W / 4, 4 * b}, {H / 8, W / 8, 4 * b}, {H / 8, W / 8, 8 * b}, {H / 8, W / 8, 8 * b},
                           {H / 8, W / 8, 4 * b}, {H / 4, W / 4, 4 * b}, {H / 4, W / 4, 4 * b}, {H / 4, W / 4, 2 * b},
                           {H / 2, W / 2, 2 * b}, {H / 2, W / 2, 2 * b}, {H / 2, W / 2, b},     {H, W, b},
                           {H, W, b},          {H, W, 1}};
    for (auto &e : sh) add(u->A, e[0], e[1], e[2]);
    u->Gd.clear();
    for (auto &e : sh) add(u->Gd, e[0], e[1], e[2]);
    // grow only: a smaller batch reuses the arena with its own offsets
    if (off > u->act.n) u->act.alloc(off);
    if ((size_t)B * H * W > u->outf.n) u->outf.alloc((size_t)B * H * W);
    if ((size_t)B * H * W > u->tgt.n) u->tgt.alloc((size_t)B * H * W);
    u->batch = B;
}

// the activations (of plan) that each convolution reads and writes
constexpr int kConvs = 15;
constexpr int kIn[kConvs] = {0, 1, 3, 4, 6, 7, 9, 10, 11, 13, 14, 16, 17, 19, 20};
constexpr int kOut[kConvs] = {1, 2, 4, 5, 7, 8, 10, 11, 12, 14, 15, 17, 18, 20, 21};

void forward(csrst_warmstart *u, int B)
{
    auto &A = u->A;
    auto P = [&](int i) { return u->ptr(A[i]); };
    auto pool = [&](int src, int dst) {
        const auto &d = A[dst];
        k_pool<<<nb((size_t)B * d.h * d.w * d.c / 8), kB, 0, u->s>>>(P(src), P(dst), B, A[src].h, A[src].w, d.c);
    };
    auto upadd = [&](int src, int skip, int dst) {
        const auto &d = A[dst];
        k_up_add<<<nb((size_t)B * d.h * d.w * d.c / 8), kB, 0, u->s>>>(P(src), P(skip), P(dst), B, d.h, d.w, d.c);
    };
    auto c = [&](int li) {
        const auto &d = A[kOut[li]];
        conv(u, li, P(kIn[li]), P(kOut[li]), li + 1 == kConvs ? u->outf.p : nullptr, B, d.h, d.w);
    };
    c(0);
    c(1);
    pool(2, 3);
    c(2);
    c(3);
    pool(5, 6);
    c(4);
    c(5);
    pool(8, 9);
    c(6);
    c(7);
    c(8);
    upadd(12, 8, 13);
    c(9);
    c(10);
    upadd(15, 5, 16);
    c(11);
    c(12);
    upadd(18, 2, 19);
    c(13);
    c(14);
    HU_LAUNCH_CHECK();
}

// backward from the bf16 output gradient in Gd[21]; fills u->g
void backward(csrst_warmstart *u, int B)
{
    auto &A = u->A;
    auto &G = u->Gd;
    auto P = [&](int i) { return u->ptr(A[i]); };
    auto D = [&](int i) { return u->ptr(G[i]); };
    HU_CHECK(hipMemsetAsync(u->g.p, 0, u->nparam * sizeof(float), u->s));
    // conv li, from D of its output to D of its input.  D of a ReLU's output is
    // the gradient before the ReLU: whatever produces a gradient there masks it.
    auto back = [&](int li) {
        const int x = kIn[li], y = kOut[li];
        const auto &d = A[y];
        conv_wgrad(u, li, D(y), P(x), B, d.h, d.w);
        if (li == 0) return;
        const bool relu = x == kOut[li - 1] && u->L[li - 1].relu;   // not a pooled or upsampled sum
        conv_dgrad(u, li, D(y), D(x), relu ? P(x) : nullptr, B, d.h, d.w);
    };
    auto upgrad = [&](int dstLow, int srcHigh) {      // D(dstLow) = up^T D(srcHigh)
        const auto &d = A[dstLow];
        k_up_grad<<<nb((size_t)B * d.h * d.w * d.c / 8), kB, 0, u->s>>>(D(srcHigh), P(dstLow), D(dstLow), B, d.h, d.w, d.c);
    };
    auto skipgrad = [&](int at, int low, int dec) {    // D(at) = pool^T D(low) + D(dec)
        const auto &d = A[at];
        k_skip_grad<<<nb((size_t)B * d.h * d.w * d.c / 8), kB, 0, u->s>>>(D(low), D(dec), P(at), D(at), B, d.h, d.w, d.c);
    };
    back(14);             // out -> D20
    back(13);             // -> D19 (= d(up(c02)) and d(s0))
    upgrad(18, 19);       // D18 = up^T D19
    back(12);
    back(11);
    upgrad(15, 16);
    back(10);
    back(9);
    upgrad(12, 13);
    back(8);
    back(7);
    back(6);
    skipgrad(8, 9, 13);
    back(5);
    back(4);
    skipgrad(5, 6, 16);
    back(3);
    back(2);
    skipgrad(2, 3, 19);
    back(1);
    back(0);
    HU_LAUNCH_CHECK();
}

void upload_input(csrst_warmstart *u, const float *rho, int B, float scale)
{
    const size_t n = (size_t)B * u->H * u->W;
    u->scratchF.alloc(std::max(u->scratchF.n, n));
    u->stage.in(u->scratchF.p, rho, n * sizeof(float), u->s);
    k_to_bf<<<nb(n), kB, 0, u->s>>>(u->scratchF.p, u->ptr(u->A[0]), n, scale);
    HU_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// The network between V-cycles.  At an iterate phi_k of the multigrid the
// residual r_k = b - A phi_k, scaled to unit RMS over the unknowns, goes
// through the network; its output c is taken as the direction of the error
// e_k = A^-1 r_k and the iterate moves by the step that minimises the energy
// norm of the error along it: phi += alpha c, alpha = (c . r) / (c . A c).  A
// V-cycle follows.  Training pairs are (r_k / rms(r_k), e_k / rms(e_k)) over
// the iterates of the solver itself, with e_k from a solve to round-off.

constexpr int kRed = 256;      // blocks of the fixed-order reductions

// The multigrid's arrays are in its own column order (pmg::Level::at), the
// network's images row-major: these kernels go between the two, a 32 x 32 tile per workgroup
// through LDS, so that both sides are read and written along their rows.
constexpr int kT = pmg::kTile;

// level value get(k) at the unknowns (0 elsewhere) to the image put(p, v)
template <class Get, class Put>
__device__ __forceinline__ void level_to_image(const pmg::Level &L, Get get, Put put)
{
    __shared__ float t[kT][kT + 1];
    const int a = threadIdx.x % kT, row = threadIdx.x / kT;
    int i0, j0;
    pmg::tile_origin(L.nx, i0, j0);
    for (int r = row; r < kT; r += kB / kT) {
        const int i = i0 + r, j = j0 + a;
        const size_t k = L.at(i, j);
        t[r][a] = i < L.nx && j < L.ny && L.act[k] ? get(k) : 0.f;
    }
    __syncthreads();
    for (int r = row; r < kT; r += kB / kT) {
        const int i = i0 + a, j = j0 + r;
        if (i < L.nx && j < L.ny) put((size_t)j * L.nx + i, t[a][r]);
    }
}

// r * inv as bf16 network input, zero off the unknowns
__global__ void __launch_bounds__(kB) k_res_in(pmg::Level L, bf16 *in, double inv)
{
    level_to_image(L, [&](size_t k) { return (float)(L.res[k] * inv); }, [&](size_t p, float v) { in[p] = f2bf(v); });
}

// (pstar - phi) * inv as float target, zero off the unknowns
__global__ void __launch_bounds__(kB) k_err_tgt(pmg::Level L, const double *pstar, float *t, double inv)
{
    level_to_image(L, [&](size_t k) { return (float)((pstar[k] - L.phi[k]) * inv); }, [&](size_t p, float v) { t[p] = v; });
}

// the network's output image as a level array
__global__ void __launch_bounds__(kB) k_dir_in(pmg::Level L, const float *img, float *c)
{
    __shared__ float t[kT][kT + 1];
    const int a = threadIdx.x % kT, row = threadIdx.x / kT;
    int i0, j0;
    pmg::tile_origin(L.nx, i0, j0);
    for (int r = row; r < kT; r += kB / kT) {
        const int i = i0 + a, j = j0 + r;
        t[r][a] = i < L.nx && j < L.ny ? img[(size_t)j * L.nx + i] : 0.f;
    }
    __syncthreads();
    for (int r = row; r < kT; r += kB / kT) {
        const int i = i0 + r, j = j0 + a;
        if (i < L.nx && j < L.pitch) c[L.at(i, j)] = t[a][r];
    }
}

unsigned tile_grid(const pmg::Level &L) { return pmg::num_tiles(L.nx, L.pitch); }

// c . A c's row k: the level's 5-point operator with the unknowns' couplings
// only, as the multigrid applies it
__device__ __forceinline__ double apply_dir(const pmg::Level &L, const float *c, size_t k)
{
    const int i = (int)(k / L.pitch), q = (int)(k % L.pitch), N = 64 * L.lane;
    const int j = q / N * N + (q % 128) / 2 * L.lane + 2 * (q % N / 128) + (q & 1);   // row_pos inverted
    double sx = 0.0, sy = 0.0;
    if (i > 0 && L.act[k - L.pitch]) sx += c[k - L.pitch];
    if (i + 1 < L.nx && L.act[k + L.pitch]) sx += c[k + L.pitch];
    const size_t d = L.at(i, j > 0 ? j - 1 : j), u = L.at(i, j + 1 < L.ny ? j + 1 : j);
    if (j > 0 && L.act[d]) sy += c[d];
    if (j + 1 < L.ny && L.act[u]) sy += c[u];
    return 2.0 * (L.cx + L.cy) * (double)c[k] - L.cx * sx - L.cy * sy;
}

__device__ __forceinline__ void block_sum2(double &a, double &b, double *part)
{
    __shared__ double sa[kB], sb[kB];
    sa[threadIdx.x] = a;
    sb[threadIdx.x] = b;
    __syncthreads();
    for (int o = kB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            sa[threadIdx.x] += sa[threadIdx.x + o];
            sb[threadIdx.x] += sb[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sa[0];
        part[2 * blockIdx.x + 1] = sb[0];
    }
}

// partial sums of (pstar - phi)^2 over the unknowns (second slot unused)
__global__ void __launch_bounds__(kB) k_err_sumsq(const double *pstar, const double *phi, const uint8_t *act, size_t n,
                                                 double *part)
{
    double s = 0.0, z = 0.0;
    for (size_t k = (size_t)blockIdx.x * kB + threadIdx.x; k < n; k += (size_t)gridDim.x * kB)
        if (act[k]) {
            const double d = pstar[k] - phi[k];
            s += d * d;
        }
    block_sum2(s, z, part);
}

// The step's sums: partial sums over the unknowns of c.Ac, c.Ad, d.Ad, c.r,
// d.r with d = phi - pprev (the previous iteration's change) and A d = rprev -
// r; c or pprev may be null (their sums are zero).  Five doubles per block.
__global__ void __launch_bounds__(kB) k_step_dots5(pmg::Level L, const float *c, const double *pprev,
                                                   const double *rprev, double *part)
{
    __shared__ double sh[5][kB];
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const size_t n = (size_t)L.nx * L.pitch;
    for (size_t k = (size_t)blockIdx.x * kB + threadIdx.x; k < n; k += (size_t)gridDim.x * kB) {
        if (!L.act[k]) continue;
        const double r = L.res[k];
        double ck = 0.0, ack = 0.0, d = 0.0, ad = 0.0;
        if (pprev) {
            d = L.phi[k] - pprev[k];
            ad = rprev[k] - r;
        }
        if (c) {
            ck = c[k];
            ack = apply_dir(L, c, k);
        }
        s[0] += ck * ack;
        s[1] += ck * ad;
        s[2] += d * ad;
        s[3] += ck * r;
        s[4] += d * r;
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) sh[q][threadIdx.x] = s[q];
    __syncthreads();
    for (int o = kB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
#pragma unroll
            for (int q = 0; q < 5; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x < 5) part[5 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}

// The step's coefficients from the kRed blocks' sums, on the device (the host
// would only hold the stream up for them): the energy-norm minimiser over
// span{c, d}, a 2 x 2 system, or over the one direction that is there and not
// degenerate.  coef = (alpha, beta).
__global__ void __launch_bounds__(kB) k_step_coef(const double *part, double *coef)
{
    static_assert(kRed == kB, "one partial per thread");
    __shared__ double sh[5][kB];
#pragma unroll
    for (int q = 0; q < 5; ++q) sh[q][threadIdx.x] = part[5 * threadIdx.x + q];
    __syncthreads();
    for (int o = kB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
#pragma unroll
            for (int q = 0; q < 5; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x) return;
    const double cac = sh[0][0], cad = sh[1][0], dad = sh[2][0], cr = sh[3][0], dr = sh[4][0];
    double alpha = 0.0, beta = 0.0;
    const bool hc = cac > 0, hd = dad > 0;
    const double det = cac * dad - cad * cad;
    if (hc && hd && det > 1e-12 * cac * dad) {
        alpha = (cr * dad - cad * dr) / det;
        beta = (cac * dr - cad * cr) / det;
    } else if (hc) {
        alpha = cr / cac;
    } else if (hd) {
        beta = dr / dad;
    }
    if (!isfinite(alpha) || !isfinite(beta)) alpha = beta = 0.0;
    coef[0] = alpha;
    coef[1] = beta;
}

// phi += alpha c + beta (phi - pprev) on the unknowns; pprev, rprev (if any)
// take the iterate and residual before the step
__global__ void k_step_update(pmg::Level L, const float *c, const double *coef, double *pprev, double *rprev)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    if (k >= (size_t)L.nx * L.pitch || !L.act[k]) return;
    const double ph = L.phi[k];
    double v = c ? ph + coef[0] * (double)c[k] : ph;
    if (pprev) {
        v += coef[1] * (ph - pprev[k]);
        pprev[k] = ph;
        rprev[k] = L.res[k];
    }
    L.phi[k] = v;
}

// the first of the kRed blocks' sums, on one workgroup
__global__ void __launch_bounds__(kB) k_sum2_final(double *part)
{
    __shared__ double sh[kB];
    sh[threadIdx.x] = part[2 * threadIdx.x];
    __syncthreads();
    for (int o = kB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[2 * kRed] = sh[0];
}

__global__ void k_copy_d(double *dst, const double *src, size_t n)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    if (k < n) dst[k] = src[k];
}

__global__ void k_zero_d(double *p, size_t n)
{
    const size_t k = (size_t)blockIdx.x * kB + threadIdx.x;
    if (k < n) p[k] = 0.0;
}

int ws_fail(csrst_warmstart *u, const std::exception &e)
{
    const Error *he = dynamic_cast<const Error *>(&e);
    if (u) u->err = e.what();
    hu::global_error() = e.what();
    return he ? he->code : CSRST_EINVAL;
}


// The hierarchy of the grid (hx, hy, cls), set up once and kept while the
// caller passes the same grid.
void loop_grid(csrst_warmstart *u, double hx, double hy, const uint8_t *cls)
{
    auto &Lp = u->loop;
    const size_t n = (size_t)u->H * u->W;
    if (!cls || !(hx > 0) || !(hy > 0)) throw Error(CSRST_EINVAL, "bad grid for the warm-start solve");
    if (Lp.ready && Lp.hx == hx && Lp.hy == hy && std::equal(Lp.cls.begin(), Lp.cls.end(), cls)) return;
    size_t unk = 0;
    for (size_t k = 0; k < n; ++k) {
        if (cls[k] > pmg::kKnown) throw Error(CSRST_EINVAL, hu::fmt("node class %d at %zu", cls[k], k));
        unk += cls[k] == pmg::kUnknown;
    }
    if (!unk) throw Error(CSRST_EINVAL, "the grid has no unknown nodes");
    Lp.ready = false;
    Lp.cls.assign(cls, cls + n);
    Lp.dcls.alloc(n);
    Lp.b.alloc(n); Lp.phi.alloc(n); Lp.part.alloc(5 * kRed + 2);
    HU_CHECK(hipMemcpyAsync(Lp.dcls.p, cls, n, hipMemcpyHostToDevice, u->s));
    Lp.mg.setup(u->W, u->H, hx, hy, Lp.dcls.p, u->s);
    const size_t nl = Lp.mg.level0_size();
    Lp.pstar.alloc(nl); Lp.pprev.alloc(nl); Lp.rprev.alloc(nl); Lp.dir.alloc(nl);
    Lp.hx = hx; Lp.hy = hy; Lp.unknowns = unk;
    Lp.ready = true;
}

// the sum of the last k_err_sumsq launch on the host
double loop_sum(csrst_warmstart *u)
{
    auto &Lp = u->loop;
    k_sum2_final<<<1, kB, 0, u->s>>>(Lp.part.p);
    HU_LAUNCH_CHECK();
    double h = 0.0;
    HU_CHECK(hipMemcpyAsync(&h, Lp.part.p + 2 * kRed, sizeof h, hipMemcpyDeviceToHost, u->s));
    HU_CHECK(hipStreamSynchronize(u->s));
    return h;
}

// The step at the current iterate, rn = ||r|| from resnorm(): over the
// network's direction (useNet), the previous iteration's change (usePrev), or
// both.  first: no previous iterate yet (d = 0).
void loop_step(csrst_warmstart *u, double rn, bool useNet, bool usePrev, bool first)
{
    auto &Lp = u->loop;
    const pmg::Level &L0 = Lp.mg.level0();
    const size_t nl = Lp.mg.level0_size();
    const double rms = rn / std::sqrt((double)Lp.unknowns);
    if (!(rms > 0)) return;
    if (usePrev && first) {
        k_copy_d<<<nb(nl), kB, 0, u->s>>>(Lp.pprev.p, L0.phi, nl);
        k_copy_d<<<nb(nl), kB, 0, u->s>>>(Lp.rprev.p, L0.res, nl);
    }
    const float *c = nullptr;
    if (useNet) {
        plan(u, 1);
        k_res_in<<<tile_grid(L0), kB, 0, u->s>>>(L0, u->ptr(u->A[0]), 1.0 / rms);
        forward(u, 1);
        k_dir_in<<<tile_grid(L0), kB, 0, u->s>>>(L0, u->outf.p, Lp.dir.p);
        c = Lp.dir.p;
    }
    double *pp = usePrev ? Lp.pprev.p : nullptr, *rp = usePrev ? Lp.rprev.p : nullptr;
    double *coef = Lp.part.p + 5 * kRed;
    k_step_dots5<<<kRed, kB, 0, u->s>>>(L0, c, pp, rp, Lp.part.p);
    k_step_coef<<<1, kB, 0, u->s>>>(Lp.part.p, coef);
    k_step_update<<<nb(nl), kB, 0, u->s>>>(L0, c, coef, pp, rp);
    HU_LAUNCH_CHECK();
}

// One Adam step on the first B staged pairs; returns the loss before it.
float loop_train(csrst_warmstart *u, int B, float lr)
{
    auto &Lp = u->loop;
    const size_t np = (size_t)B * u->H * u->W;
    plan(u, B);
    HU_CHECK(hipMemcpyAsync(u->ptr(u->A[0]), Lp.pairIn.p, np * sizeof(bf16), hipMemcpyDeviceToDevice, u->s));
    HU_CHECK(hipMemcpyAsync(u->tgt.p, Lp.pairTgt.p, np * sizeof(float), hipMemcpyDeviceToDevice, u->s));
    forward(u, B);
    HU_CHECK(hipMemsetAsync(u->lossBuf.p, 0, sizeof(float), u->s));
    k_mse<<<std::min(nb(np), kMseBlocks), kB, 0, u->s>>>(u->outf.p, u->tgt.p, u->ptr(u->Gd[21]), u->lossBuf.p, np);
    backward(u, B);
    ++u->steps;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)u->steps), c2 = 1.f - std::pow(b2, (float)u->steps);
    k_adam<<<nb(u->nparam), kB, 0, u->s>>>(u->w.p, u->m.p, u->v.p, u->g.p, u->nparam, lr, b1, b2, 1e-8f, c1, c2);
    refresh_bf16(u);
    float loss = 0.f;
    HU_CHECK(hipMemcpyAsync(&loss, u->lossBuf.p, sizeof(float), hipMemcpyDeviceToHost, u->s));
    HU_CHECK(hipStreamSynchronize(u->s));
    return loss;
}

}  // namespace

extern "C" {

int csrst_warmstart_create(int H, int W, int maxBatch, csrst_warmstart **out)
{
    std::unique_ptr<csrst_warmstart> u(new csrst_warmstart());
    try {
        if (!out || H < 16 || W < 16 || H % 8 || W % 8 || maxBatch < 1)
            throw Error(CSRST_EINVAL, "grid must be at least 16 x 16 and divisible by 8; batch >= 1");
        u->H = H; u->W = W; u->maxBatch = maxBatch;
        HU_CHECK(hipStreamCreateWithFlags(&u->s, hipStreamNonBlocking));
        make_layers(u.get());
        u->w.alloc(u->nparam); u->m.alloc(u->nparam); u->v.alloc(u->nparam); u->g.alloc(u->nparam);
        u->m.zero(u->s); u->v.zero(u->s); u->g.zero(u->s);
        size_t ob = 0, ot = 0;
        for (const Layer &l : u->L) {
            u->wbOff.push_back(ob); ob += (size_t)pad16(l.cout) * 9 * l.cin;
            u->wtOff.push_back(ot); ot += (size_t)pad16(l.cin) * 9 * l.cout;
        }
        u->wb.alloc(ob); u->wt.alloc(ot);
        u->lossBuf.alloc(1);
        // He initialisation from a fixed LCG (weights), zero biases
        std::vector<float> h(u->nparam, 0.f);
        uint64_t st = 0x9E3779B97F4A7C15ull;
        auto uni = [&]() {
            st = st * 6364136223846793005ull + 1442695040888963407ull;
            return ((st >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        };
        for (const Layer &l : u->L) {
            const double sd = std::sqrt(2.0 / (9.0 * l.cin));
            for (size_t k = 0; k < (size_t)l.cout * 9 * l.cin; ++k) {
                const double a = uni(), b = uni();
                h[l.woff + k] = (float)(sd * std::sqrt(-2 * std::log(a)) * std::cos(6.283185307179586 * b));
            }
        }
        HU_CHECK(hipMemcpyAsync(u->w.p, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice, u->s));
        refresh_bf16(u.get());
        HU_CHECK(hipStreamSynchronize(u->s));
        *out = u.release();
        return CSRST_OK;
    } catch (const std::exception &e) {
        if (u && u->s) { (void)hipStreamSynchronize(u->s); (void)hipStreamDestroy(u->s); u->s = nullptr; }
        return ws_fail(nullptr, e);
    }
}

int csrst_warmstart_destroy(csrst_warmstart *u)
{
    if (!u) return CSRST_OK;
    if (u->s) { (void)hipStreamSynchronize(u->s); (void)hipStreamDestroy(u->s); }
    delete u;
    return CSRST_OK;
}

int csrst_warmstart_num_params(csrst_warmstart *u, int *n)
{
    if (!u || !n) return CSRST_EINVAL;
    *n = (int)u->nparam;
    return CSRST_OK;
}

int csrst_warmstart_get_weights(csrst_warmstart *u, float *w, int n)
{
    try {
        if (!u || !w || n != (int)u->nparam) throw Error(CSRST_EINVAL, "weight count mismatch");
        HU_CHECK(hipMemcpyAsync(w, u->w.p, u->nparam * sizeof(float), hipMemcpyDeviceToHost, u->s));
        HU_CHECK(hipStreamSynchronize(u->s));
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}

int csrst_warmstart_set_weights(csrst_warmstart *u, const float *w, int n)
{
    try {
        if (!u || !w || n != (int)u->nparam) throw Error(CSRST_EINVAL, "weight count mismatch");
        HU_CHECK(hipMemcpyAsync(u->w.p, w, u->nparam * sizeof(float), hipMemcpyHostToDevice, u->s));
        u->m.zero(u->s); u->v.zero(u->s);
        u->steps = 0;
        refresh_bf16(u);
        HU_CHECK(hipStreamSynchronize(u->s));
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}

// Inference: rho [B][H][W] (host, float) scaled by `scale`, output [B][H][W].
int csrst_warmstart_infer(csrst_warmstart *u, const float *rho, float *out, int B, float scale)
{
    try {
        if (!u || !rho || !out || B < 1 || B > u->maxBatch) throw Error(CSRST_EINVAL, "bad inference arguments");
        plan(u, B);
        upload_input(u, rho, B, scale);
        forward(u, B);
        u->stage.out(out, u->outf.p, (size_t)B * u->H * u->W * sizeof(float), u->s);
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}

// Loss and parameter gradients of one batch (no update): grads [nparam].
int csrst_warmstart_gradients(csrst_warmstart *u, const float *rho, const float *phi, int B, float scale, float *loss,
                              float *grads, int n)
{
    try {
        if (!u || !rho || !phi || B < 1 || B > u->maxBatch) throw Error(CSRST_EINVAL, "bad gradient arguments");
        if (grads && n != (int)u->nparam) throw Error(CSRST_EINVAL, "gradient count mismatch");
        plan(u, B);
        upload_input(u, rho, B, scale);
        const size_t np = (size_t)B * u->H * u->W;
        u->stage.in(u->tgt.p, phi, np * sizeof(float), u->s);
        forward(u, B);
        HU_CHECK(hipMemsetAsync(u->lossBuf.p, 0, sizeof(float), u->s));
        k_mse<<<std::min(nb(np), kMseBlocks), kB, 0, u->s>>>(u->outf.p, u->tgt.p, u->ptr(u->Gd[21]), u->lossBuf.p, np);
        backward(u, B);
        if (loss) HU_CHECK(hipMemcpyAsync(loss, u->lossBuf.p, sizeof(float), hipMemcpyDeviceToHost, u->s));
        if (grads) u->stage.out(grads, u->g.p, u->nparam * sizeof(float), u->s);
        HU_CHECK(hipStreamSynchronize(u->s));
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}

// One Adam step on a batch; loss before the update.
int csrst_warmstart_train_step(csrst_warmstart *u, const float *rho, const float *phi, int B, float scale, float lr,
                               float *loss)
{
    try {
        const int rc = csrst_warmstart_gradients(u, rho, phi, B, scale, loss, nullptr, 0);
        if (rc) return rc;
        ++u->steps;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - std::pow(b1, (float)u->steps), c2 = 1.f - std::pow(b2, (float)u->steps);
        k_adam<<<nb(u->nparam), kB, 0, u->s>>>(u->w.p, u->m.p, u->v.p, u->g.p, u->nparam, lr, b1, b2, 1e-8f, c1, c2);
        refresh_bf16(u);
        HU_CHECK(hipStreamSynchronize(u->s));
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}


// Poisson solve on the network's H x W node grid (nx = W, ny = H) with the
// multigrid of csrst_poisson_solve.  mode 0: plain V-cycles from phi; 1: the
// network's step before every V-cycle; 2: before the first only (a one-shot
// start); 3: before every V-cycle the energy-norm minimiser over the
// network's direction and the previous iteration's change; 4: over the
// previous change alone (the same acceleration without the network).  phi: in the guess, out the solution; cycles and the final relative
// residual as csrst_poisson_solve reports them.
int csrst_warmstart_solve(csrst_warmstart *u, double hx, double hy, const uint8_t *cls, const double *b, double *phi,
                          double tol, int maxit, int mode, int *cycles, double *resid)
{
    try {
        if (!u || !b || !phi || maxit < 0 || !(tol >= 0) || mode < 0 || mode > 4)
            throw Error(CSRST_EINVAL, "bad warm-start solve arguments");
        loop_grid(u, hx, hy, cls);
        auto &Lp = u->loop;
        const size_t n = (size_t)u->H * u->W;
        u->stage.in(Lp.b.p, b, n * sizeof(double), u->s);
        u->stage.in(Lp.phi.p, phi, n * sizeof(double), u->s);
        const double bn = Lp.mg.begin(Lp.b.p, Lp.phi.p);
        double r = Lp.mg.resnorm();
        const double target = tol * (bn > 0 ? bn : 1.0);
        int cyc = 0, flat = 0;
        while (r > target && cyc < maxit && flat < 3) {
            if (mode >= 3 || mode == 1 || (mode == 2 && cyc == 0)) loop_step(u, r, mode != 4, mode >= 3, cyc == 0);
            Lp.mg.cycle();
            ++cyc;
            const double rn = Lp.mg.resnorm();
            if (!std::isfinite(rn)) throw Error(CSRST_EHIP, "multigrid diverged");
            flat = rn > 0.95 * r ? flat + 1 : 0;
            r = rn;
        }
        Lp.mg.store(Lp.b.p, Lp.phi.p);
        u->stage.out(phi, Lp.phi.p, n * sizeof(double), u->s);
        if (cycles) *cycles = cyc;
        if (resid) *resid = bn > 0 ? r / bn : r;
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}

// Training on the solver's own iterates.  For each of the nrhs right-hand
// sides b[nrhs][H][W]: a plain solve to a relative residual of 1e-13 gives
// phi*; then from phi = 0, at iterates k = 0 .. kmax-1 (until the residual
// reaches 1e-12), the pair (r_k / rms(r_k), (phi* - phi_k) / rms) is staged
// and the iterate advances by a V-cycle, preceded by the network's step when
// inloop is 1 (pairs from the learned loop itself).  Every maxBatch staged
// pairs make one Adam step of rate lr.  loss: mean loss of those steps;
// pairs: pairs used.
int csrst_warmstart_train_iterates(csrst_warmstart *u, double hx, double hy, const uint8_t *cls, const double *b,
                                   int nrhs, int kmax, int inloop, float lr, float *loss, int *pairs)
{
    try {
        if (!u || !b || nrhs < 1 || kmax < 1 || !(lr > 0)) throw Error(CSRST_EINVAL, "bad training arguments");
        loop_grid(u, hx, hy, cls);
        auto &Lp = u->loop;
        const size_t n = (size_t)u->H * u->W;
        const int MB = u->maxBatch;
        Lp.pairIn.alloc(std::max(Lp.pairIn.n, (size_t)MB * n));
        Lp.pairTgt.alloc(std::max(Lp.pairTgt.n, (size_t)MB * n));
        const pmg::Level &L0 = Lp.mg.level0();
        const size_t nl = Lp.mg.level0_size();
        int slot = 0, used = 0, nsteps = 0;
        double lsum = 0.0;
        for (int i = 0; i < nrhs; ++i) {
            u->stage.in(Lp.b.p, b + (size_t)i * n, n * sizeof(double), u->s);
            k_zero_d<<<nb(n), kB, 0, u->s>>>(Lp.phi.p, n);
            HU_LAUNCH_CHECK();
            const double bn = Lp.mg.begin(Lp.b.p, Lp.phi.p);
            if (!(bn > 0)) continue;
            double r = Lp.mg.resnorm();
            for (int c = 0, flat = 0; r > 1e-13 * bn && c < 200 && flat < 3; ++c) {
                Lp.mg.cycle();
                const double rn = Lp.mg.resnorm();
                flat = rn > 0.95 * r ? flat + 1 : 0;
                r = rn;
            }
            k_copy_d<<<nb(nl), kB, 0, u->s>>>(Lp.pstar.p, L0.phi, nl);
            Lp.mg.begin(Lp.b.p, Lp.phi.p);
            r = Lp.mg.resnorm();
            for (int k = 0; k < kmax && r > 1e-12 * bn; ++k) {
                k_err_sumsq<<<kRed, kB, 0, u->s>>>(Lp.pstar.p, L0.phi, L0.act, nl, Lp.part.p);
                const double e2 = loop_sum(u);
                const double rr = r / std::sqrt((double)Lp.unknowns), re = std::sqrt(e2 / (double)Lp.unknowns);
                if (rr > 0 && re > 0) {
                    k_res_in<<<tile_grid(L0), kB, 0, u->s>>>(L0, Lp.pairIn.p + (size_t)slot * n, 1.0 / rr);
                    k_err_tgt<<<tile_grid(L0), kB, 0, u->s>>>(L0, Lp.pstar.p, Lp.pairTgt.p + (size_t)slot * n, 1.0 / re);
                    HU_LAUNCH_CHECK();
                    if (++slot == MB) {
                        lsum += loop_train(u, slot, lr);
                        ++nsteps;
                        used += slot;
                        slot = 0;
                    }
                }
                if (inloop) loop_step(u, r, true, false, false);
                Lp.mg.cycle();
                r = Lp.mg.resnorm();
            }
        }
        if (slot) {
            lsum += loop_train(u, slot, lr);
            ++nsteps;
            used += slot;
        }
        HU_CHECK(hipStreamSynchronize(u->s));
        if (loss) *loss = nsteps ? (float)(lsum / nsteps) : 0.f;
        if (pairs) *pairs = used;
        return CSRST_OK;
    } catch (const std::exception &e) {
        return ws_fail(u, e);
    }
}

}  // extern "C"
