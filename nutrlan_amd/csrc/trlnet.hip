// trlnet.hip -- the learned start vector: a 4-layer 3x3 convolutional net
// (1 -> 32 -> 32 -> 32 -> 1 channels, ReLU between layers, periodic
// padding) that maps a lattice's on-site potential to a start vector for
// trlan().  Forward and backward run on BF16 MFMA (v_mfma_f32_16x16x32_bf16)
// with FP32 accumulation; master weights and Adam state are FP32.  No
// counterpart in the reference (it takes a start vector through
// info->guess = 1 and evec(:, nec)).
//
// Layout: activations NHWC, pixels flattened over (image, y, x), 32
// channels of BF16 (64 B) per pixel; the input potential and the output are
// one FP32 value per pixel.  A convolution is an implicit GEMM: M = 16
// pixels per MFMA tile, N = 16 output channels, K = 32 = one tap's 32 input
// channels (or, for the one-channel input layer, the 9 taps padded to 32).
//
// MFMA f32 16x16x32 bf16 operand layout (lane l): A row l%16 with K
// elements 8*(l/16) .. +7, B column l%16 with the same K elements, result
// D[4*(l/16) + i][l%16] in accumulator element i.
//
// A wave takes a strip of 16 pixels of one image row and walks down up to
// kRows rows: each input row is loaded once (three column shifts) and feeds the
// three output rows that use it, the layer's weights stay in registers, and
// the weights are the A operand, so a lane holds four consecutive channels
// of one pixel and stores them together.  What bounds the forward is the
// activations' HBM traffic; with nine loads a pixel, weights re-read per 16
// pixels and two-byte stores a 32 -> 32 layer took 0.89 ms for 7.3 M pixels
// (256 lattices, sides 64-256; 0.94 GB, 0.19 ms at copy rate), now 0.37; the
// first and last layers 0.54 and 0.44, now 0.18 each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "trlnet.h"

namespace {

#include "trl_strips.h"

constexpr int C = 32;          // hidden channels
constexpr int T = 9;           // 3x3 taps
constexpr int NB = 256;        // threads per block

// parameter offsets in the flat FP32 vector
constexpr int OW1 = 0, OB1 = OW1 + C * T;             // W1[co][t]
constexpr int OW2 = OB1 + C, OB2 = OW2 + C * T * C;   // W2[co][t][ci]
constexpr int OW3 = OB2 + C, OB3 = OW3 + C * T * C;   // W3[co][t][ci]
constexpr int OW4 = OB3 + C, OB4 = OW4 + T * C;       // W4[t][ci]
constexpr int NPARAM = OB4 + 1;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16_t;  // storage

__host__ __device__ inline bf16_t f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (bf16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(bf16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

__device__ inline __bf16 as_bf(bf16_t h) { return __builtin_bit_cast(__bf16, h); }

__device__ inline bf16x8 load8(const bf16_t *p)
{
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return __builtin_bit_cast(bf16x8, v);
}

__device__ inline bf16x8 zero8() { return __builtin_bit_cast(bf16x8, uint4{0, 0, 0, 0}); }

inline long conv_blocks(const Geo &g) { return (g.tasks + NB / 64 - 1) / (NB / 64); }

// Rows a wave walks for the images of all groups of a launch: shorter walks
// while there is at most a wave per SIMD.  Forward and backward of 8 images
// of 64 x 64 (1,024 waves of 2 rows, 256 of 8) 229 -> 207 us; with limits of
// 3,072 to 8,192 waves 32 and 64 such images are 0 to 9 % slower: every wave
// loads the layer's weights and two more rows.
constexpr long kConvWaves = 1024;
constexpr int kMinRows = 2;
inline int conv_rows(int ngroups, const int *nimg, const int *h, const int *w)
{
    int rows = kRows;
    while (rows > kMinRows) {
        long n = 0;
        for (int i = 0; i < ngroups; ++i) n += conv_tasks(nimg[i], h[i], w[i], rows / 2);
        if (n > kConvWaves) break;
        rows /= 2;
    }
    return rows;
}

__device__ __forceinline__ int wrap(int y, int h) { return y < 0 ? y + h : (y >= h ? y - h : y); }

__device__ __forceinline__ uint2 pack4(const float v[4])
{
    return uint2{(uint32_t)f2bf(v[0]) | (uint32_t)f2bf(v[1]) << 16,
                 (uint32_t)f2bf(v[2]) | (uint32_t)f2bf(v[3]) << 16};
}

// ---------------------------------------------------------------- forward

// Layer 1: one input channel (FP32 potential, rounded to BF16), K = the 9
// taps padded to 32.  out = relu(W1 * x + b1), BF16, 32 channels.  The
// wave's three input rows slide down in registers.
__device__ __forceinline__ void fwd1_body(const Geo &g, long bid, const float *__restrict__ x,
                                          const bf16_t *__restrict__ w1, const float *__restrict__ b1,
                                          bf16_t *__restrict__ out)
{
    const int lane = threadIdx.x & 63;
    Strip s;
    if (!strip_of(g, bid * (NB / 64) + (threadIdx.x >> 6), threadIdx.x & 15, s)) return;
    const int m = lane & 15, kq = lane >> 4;
    bf16x8 wt[2];
    float bs[2][4];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        wt[nt] = zero8();
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (8 * kq + j < T) wt[nt][j] = as_bf(w1[(16 * nt + m) * T + 8 * kq + j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) bs[nt][i] = b1[16 * nt + 4 * kq + i];
    }
    const float *xi = x + s.base;
    auto row = [&](int y, __bf16 r[3]) {
        const float *p = xi + (long)wrap(y, g.h) * g.w;
#pragma unroll
        for (int d = 0; d < 3; ++d) r[d] = as_bf(f2bf(p[s.xc[d]]));
    };
    __bf16 r0[3], r1[3], r2[3];
    row(s.y0 - 1, r0);
    row(s.y0, r1);
    const __bf16 z = as_bf(0);
    for (int y = s.y0; y < s.y1; ++y) {
        row(y + 1, r2);
        // taps 0..7 in the lanes of K 0..7, tap 8 in those of K 8..15
        bf16x8 a = zero8();
        const __bf16 t8[8] = {r0[0], r0[1], r0[2], r1[0], r1[1], r1[2], r2[0], r2[1]};
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = kq == 0 ? t8[j] : z;
        if (kq == 1) a[0] = r2[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            f4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[nt], a, acc, 0, 0, 0);
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = fmaxf(acc[i] + bs[nt][i], 0.f);
            if (s.ok)
                *reinterpret_cast<uint2 *>(out + (s.base + (long)y * g.w + s.x) * C + 16 * nt + 4 * kq) = pack4(v);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            r0[d] = r1[d];
            r1[d] = r2[d];
        }
    }
}

__global__ __launch_bounds__(NB) void k_fwd1(Geo g, const float *__restrict__ x,
                                             const bf16_t *__restrict__ w1, const float *__restrict__ b1,
                                             bf16_t *__restrict__ out)
{
    fwd1_body(g, blockIdx.x, x, w1, b1, out);
}

// A 32 -> 32 channel 3x3 convolution over a wave's strip, K = 9 taps x 32
// channels: forward (BWD = false: out = relu(W * in + bias)) or the data
// gradient (BWD: out = relu'(act) * W^T * in, taps mirrored, w transposed).
// Rows are walked so that each output row receives its taps in order 0..8:
// downwards, or upwards for the mirrored taps.  Input row r is the first
// tap row of the output row after it, the middle of its own and the last of
// the one before, so three rows of accumulators are open at a time.
template <bool BWD>
__device__ __forceinline__ void conv32_body(const Geo &g, long bid, const bf16_t *__restrict__ in,
                                            const bf16_t *__restrict__ w, const float *__restrict__ bias,
                                            const bf16_t *__restrict__ act, bf16_t *__restrict__ out)
{
    const int lane = threadIdx.x & 63;
    Strip s;
    if (!strip_of(g, bid * (NB / 64) + (threadIdx.x >> 6), threadIdx.x & 15, s)) return;
    const int m = lane & 15, kq = lane >> 4;
    bf16x8 wt[T][2];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) wt[t][nt] = load8(w + ((long)(16 * nt + m) * T + t) * C + 8 * kq);
    float bs[2][4];
    if constexpr (!BWD)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) bs[nt][i] = bias[16 * nt + 4 * kq + i];
    const bf16_t *pi = in + s.base * C + 8 * kq;
    const int nr = s.y1 - s.y0;
    // step k loads input row y0 - 1 + k, or y1 - k
    auto row = [&](int k) { return BWD ? s.y1 - k : s.y0 - 1 + k; };
    auto load = [&](int k, bf16x8 a[3]) {
        const bf16_t *p = pi + (long)wrap(row(k), g.h) * g.w * C;
#pragma unroll
        for (int d = 0; d < 3; ++d) a[d] = load8(p + s.xc[BWD ? 2 - d : d] * C);
    };
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 mid[2] = {zero, zero}, last[2] = {zero, zero};  // output rows k - 1 (middle taps next), k - 2
    bf16x8 a[3], nx[3];
    load(0, a);
    for (int k = 0; k < nr + 2; ++k) {
        if (k + 1 < nr + 2) load(k + 1, nx);
        f4 first[2] = {zero, zero};
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                first[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[d][nt], a[d], first[nt], 0, 0, 0);
                mid[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[3 + d][nt], a[d], mid[nt], 0, 0, 0);
                last[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[6 + d][nt], a[d], last[nt], 0, 0, 0);
            }
        if (k >= 2 && s.ok) {
            const long q = (s.base + (long)(BWD ? row(k) + 1 : row(k) - 1) * g.w + s.x) * C + 4 * kq;
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                float v[4];
                if constexpr (BWD) {
                    const uint2 av = *reinterpret_cast<const uint2 *>(act + q + 16 * nt);
                    const uint32_t h[4] = {av.x & 0xFFFFu, av.x >> 16, av.y & 0xFFFFu, av.y >> 16};
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = last[nt][i] * (bf2f((bf16_t)h[i]) > 0.f ? 1.f : 0.f);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = fmaxf(last[nt][i] + bs[nt][i], 0.f);
                }
                *reinterpret_cast<uint2 *>(out + q + 16 * nt) = pack4(v);
            }
        }
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            last[nt] = mid[nt];
            mid[nt] = first[nt];
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) a[d] = nx[d];
    }
}

__global__ __launch_bounds__(NB) void k_fwd32(Geo g, const bf16_t *__restrict__ in,
                                              const bf16_t *__restrict__ w, const float *__restrict__ bias,
                                              bf16_t *__restrict__ out)
{
    conv32_body<false>(g, blockIdx.x, in, w, bias, nullptr, out);
}

// Layer 4: 32 -> 1 channel (M padded to 16, row 0 real), FP32 output; rows
// walked as in conv32_body.
__device__ __forceinline__ void fwd4_body(const Geo &g, long bid, const bf16_t *__restrict__ in,
                                          const bf16_t *__restrict__ w4, const float *__restrict__ b4,
                                          float *__restrict__ out)
{
    const int lane = threadIdx.x & 63;
    Strip s;
    if (!strip_of(g, bid * (NB / 64) + (threadIdx.x >> 6), threadIdx.x & 15, s)) return;
    const int m = lane & 15, kq = lane >> 4;
    bf16x8 wt[T];
#pragma unroll
    for (int t = 0; t < T; ++t) wt[t] = m == 0 ? load8(w4 + (long)t * C + 8 * kq) : zero8();
    const float bias = b4[0];
    const bf16_t *pi = in + s.base * C + 8 * kq;
    const int nr = s.y1 - s.y0;
    auto load = [&](int k, bf16x8 a[3]) {
        const bf16_t *p = pi + (long)wrap(s.y0 - 1 + k, g.h) * g.w * C;
#pragma unroll
        for (int d = 0; d < 3; ++d) a[d] = load8(p + s.xc[d] * C);
    };
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 mid = zero, last = zero;
    bf16x8 a[3], nx[3];
    load(0, a);
    for (int k = 0; k < nr + 2; ++k) {
        if (k + 1 < nr + 2) load(k + 1, nx);
        f4 first = zero;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            first = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[d], a[d], first, 0, 0, 0);
            mid = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[3 + d], a[d], mid, 0, 0, 0);
            last = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[6 + d], a[d], last, 0, 0, 0);
        }
        if (k >= 2 && s.ok && kq == 0) out[s.base + (long)(s.y0 + k - 2) * g.w + s.x] = last[0] + bias;
        last = mid;
        mid = first;
#pragma unroll
        for (int d = 0; d < 3; ++d) a[d] = nx[d];
    }
}

__global__ __launch_bounds__(NB) void k_fwd4(Geo g, const bf16_t *__restrict__ in,
                                             const bf16_t *__restrict__ w4, const float *__restrict__ b4,
                                             float *__restrict__ out)
{
    fwd4_body(g, blockIdx.x, in, w4, b4, out);
}

// Groups of images of different sizes in one launch per layer: group i
// (geometry gg[i].g, first pixel gg[i].off) owns blocks [pre[i], pre[i+1]).
struct GroupGeo {
    Geo g;
    long off;
};

// The group owning block blk (pre increasing, pre[0] = 0): each wave
// narrows the range 64-fold per step with a ballot over 64 candidates.
__device__ __forceinline__ int group_of(const int *__restrict__ pre, int ng, int blk)
{
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = ng - 1;
    while (lo < hi) {
        const int step = (hi - lo + 64) / 64;
        const int k = lo + lane * step;
        const unsigned long long m = __ballot(k <= hi && pre[k] <= blk);
        lo += (63 - __clzll(m)) * step;
        hi = min(hi, lo + step - 1);
        if (step == 1) break;
    }
    return lo;
}

__global__ __launch_bounds__(NB) void k_fwd1_many(const GroupGeo *__restrict__ gg, const int *__restrict__ pre,
                                                  int ng, const float *__restrict__ x,
                                                  const bf16_t *__restrict__ w1, const float *__restrict__ b1,
                                                  bf16_t *__restrict__ out)
{
    const int i = group_of(pre, ng, blockIdx.x);
    const GroupGeo q = gg[i];
    fwd1_body(q.g, blockIdx.x - pre[i], x + q.off, w1, b1, out + q.off * C);
}

__global__ __launch_bounds__(NB) void k_fwd32_many(const GroupGeo *__restrict__ gg, const int *__restrict__ pre,
                                                   int ng, const bf16_t *__restrict__ in,
                                                   const bf16_t *__restrict__ w, const float *__restrict__ bias,
                                                   bf16_t *__restrict__ out)
{
    const int i = group_of(pre, ng, blockIdx.x);
    const GroupGeo q = gg[i];
    conv32_body<false>(q.g, blockIdx.x - pre[i], in + q.off * C, w, bias, nullptr, out + q.off * C);
}

__global__ __launch_bounds__(NB) void k_fwd4_many(const GroupGeo *__restrict__ gg, const int *__restrict__ pre,
                                                  int ng, const bf16_t *__restrict__ in,
                                                  const bf16_t *__restrict__ w4, const float *__restrict__ b4,
                                                  float *__restrict__ out)
{
    const int i = group_of(pre, ng, blockIdx.x);
    const GroupGeo q = gg[i];
    fwd4_body(q.g, blockIdx.x - pre[i], in + q.off * C, w4, b4, out + q.off);
}

// ------------------------------------------------------------ loss, grads

// Per image: c = (o.t)^2 / (|o|^2 |t|^2), loss += (1 - c) / nimg and
// dL/do = (2 / nimg) (c o / |o|^2 - (o.t) t / (|o|^2 |t|^2)).  One block
// per image; loss_part[img] = (1 - c) / nimg.
__global__ __launch_bounds__(NB) void k_loss(Geo g, const float *__restrict__ o,
                                             const float *__restrict__ tg, float *__restrict__ dout,
                                             double *__restrict__ loss_part)
{
    __shared__ double red[3][NB / 64];
    const long hw = (long)g.h * g.w;
    const long base = (long)blockIdx.x * hw;
    double ot = 0.0, oo = 0.0, tt = 0.0;
    for (long i = threadIdx.x; i < hw; i += NB) {
        const double ov = o[base + i], tv = tg[base + i];
        ot += ov * tv;
        oo += ov * ov;
        tt += tv * tv;
    }
    double v[3] = {ot, oo, tt};
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int k = 0; k < 3; ++k) {
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off);
        if (lane == 0) red[k][wv] = v[k];
    }
    __syncthreads();
    double s[3];
    for (int k = 0; k < 3; ++k) s[k] = (red[k][0] + red[k][1]) + (red[k][2] + red[k][3]);
    const double oo_ = s[1] > 1e-300 ? s[1] : 1e-300, tt_ = s[2] > 1e-300 ? s[2] : 1e-300;
    const double c = s[0] * s[0] / (oo_ * tt_);
    const double sc = 2.0 / g.nimg;
    for (long i = threadIdx.x; i < hw; i += NB)
        dout[base + i] = (float)(sc * (c * o[base + i] / oo_ - s[0] * tg[base + i] / (oo_ * tt_)));
    if (threadIdx.x == 0) loss_part[blockIdx.x] = (1.0 - c) / g.nimg;
}

// dX for layer 4's input: dA3[p][ci] = relu'(a3[p][ci]) * sum_t dO[nbr(p,-t)] W4[t][ci].
// K = the 9 taps padded to 32 (one output channel), M = 32 input channels;
// the three rows of dO slide down in registers (tap 0 reads the row below).
__global__ __launch_bounds__(NB) void k_bwd4(Geo g, const float *__restrict__ dout,
                                             const bf16_t *__restrict__ w4, const bf16_t *__restrict__ a3,
                                             bf16_t *__restrict__ da3)
{
    const int lane = threadIdx.x & 63;
    Strip s;
    if (!strip_of(g, (long)blockIdx.x * (NB / 64) + (threadIdx.x >> 6), threadIdx.x & 15, s)) return;
    const int m = lane & 15, kq = lane >> 4;
    bf16x8 wt[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        wt[nt] = zero8();
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (8 * kq + j < T) wt[nt][j] = as_bf(w4[(8 * kq + j) * C + 16 * nt + m]);
    }
    const float *di = dout + s.base;
    auto row = [&](int y, __bf16 r[3]) {
        const float *p = di + (long)wrap(y, g.h) * g.w;
#pragma unroll
        for (int d = 0; d < 3; ++d) r[d] = as_bf(f2bf(p[s.xc[2 - d]]));
    };
    __bf16 r0[3], r1[3], r2[3];  // rows y + 1, y, y - 1: taps 0..2, 3..5, 6..8
    row(s.y0 - 1, r2);
    row(s.y0, r1);
    const __bf16 z = as_bf(0);
    for (int y = s.y0; y < s.y1; ++y) {
        row(y + 1, r0);
        bf16x8 a = zero8();
        const __bf16 t8[8] = {r0[0], r0[1], r0[2], r1[0], r1[1], r1[2], r2[0], r2[1]};
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = kq == 0 ? t8[j] : z;
        if (kq == 1) a[0] = r2[2];
        const long q = (s.base + (long)y * g.w + s.x) * C + 4 * kq;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            f4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[nt], a, acc, 0, 0, 0);
            if (s.ok) {
                const uint2 av = *reinterpret_cast<const uint2 *>(a3 + q + 16 * nt);
                const uint32_t h[4] = {av.x & 0xFFFFu, av.x >> 16, av.y & 0xFFFFu, av.y >> 16};
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = acc[i] * (bf2f((bf16_t)h[i]) > 0.f ? 1.f : 0.f);
                *reinterpret_cast<uint2 *>(da3 + q + 16 * nt) = pack4(v);
            }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            r2[d] = r1[d];
            r1[d] = r0[d];
        }
    }
}

// dX for a 32 -> 32 layer: dA[p][ci] = relu'(a[p][ci]) * sum_t sum_co
// dY[nbr(p,-t)][co] W[co][t][ci], with wt = W transposed to [ci][t][co].
__global__ __launch_bounds__(NB) void k_bwd32(Geo g, const bf16_t *__restrict__ dy,
                                              const bf16_t *__restrict__ wt, const bf16_t *__restrict__ a,
                                              bf16_t *__restrict__ da)
{
    conv32_body<true>(g, blockIdx.x, dy, wt, nullptr, a, da);
}

// ------------------------------------------------------- weight gradients
//
// K = pixels, so both operands are needed pixel-contiguous per channel while
// the activations are channel-last.  Each wave transposes its own pixels
// through LDS: 32 pixels of a row x 32 channels are loaded with 16-byte
// loads, two pixels' channels interleaved by v_perm into dwords [channel]
// [pixel pair], and read back 8 pixels a lane.  Rows of kTr = 18 dwords put
// the writes of a wave on 64 different banks.  A wave walks down a strip of
// up to 32 columns and keeps its accumulators over all its strips (dw_rows).
// Gathering the operands two bytes at a time with a division per pixel and
// tap, the two layers took 330 us each at 64 images of 64 x 64 (now 19), and
// the first and last layers, one thread per weight over a serial pixel loop,
// 650 us each (now 17).
constexpr int kTr = 18;               // dwords per channel: 36 pixels
static_assert(kDwWaves == kDwBlocks * (NB / 64), "waves of the gradient kernels");
// Partials of the four layers, a row per block, and where each starts.  They
// are FP64: the sum over the waves' FP32 accumulators is rounded once, at its
// end.  Blocks without a strip are not launched.
constexpr int kRowMid = C * T * C + C, kRowEdge = C * T + C;
constexpr long kPart3 = 0, kPart2 = kPart3 + (long)kDwBlocks * kRowMid,
               kPart4 = kPart2 + (long)kDwBlocks * kRowMid,
               kPart1 = kPart4 + (long)kDwBlocks * kRowEdge, kPartCount = kPart1 + (long)kDwBlocks * kRowEdge;

// Column x0 + p of a row of w, periodic one pixel beyond either end; further
// out (a ragged strip's unused pixels) any column.
__device__ __forceinline__ int dw_col(int x, int w)
{
    x = x < 0 ? x + w : (x >= w ? x - w : x);
    return x < w ? x : 0;
}

// The lane's two pixels (2 pp, 2 pp + 1 after `x`) of row `row`, 8 channels.
struct Pair {
    uint4 a, b;
};

// Two pixels' 8 channels as 8 dwords [pixel 1 | pixel 0], to rows 8 cg + c.
__device__ __forceinline__ void put_pair(uint32_t *tr, int cg, int dw, const Pair &v)
{
    const uint32_t a[4] = {v.a.x, v.a.y, v.a.z, v.a.w}, b[4] = {v.b.x, v.b.y, v.b.z, v.b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        tr[(8 * cg + 2 * i) * kTr + dw] = __builtin_amdgcn_perm(b[i], a[i], 0x05040100u);
        tr[(8 * cg + 2 * i + 1) * kTr + dw] = __builtin_amdgcn_perm(b[i], a[i], 0x07060302u);
    }
}

__device__ __forceinline__ bf16x8 frag(const uint32_t d[4])
{
    return __builtin_bit_cast(bf16x8, uint4{d[0], d[1], d[2], d[3]});
}

// Weight gradient dW[co][t][ci] = sum_p dY[p][co] X[nbr(p,t)][ci] of a
// 32 -> 32 layer: M = co, N = ci.  Three rows of X stay in LDS (a row
// serves the dY rows above, at and below it); a lane reads 12 pixels of a
// channel and shifts them by one for the left and right taps.  The block's
// partial (co, t, ci) and bias sums (a product with ones), its four waves
// added in FP64, go to part[blockIdx] in FP64 (38 MB for 256 blocks, against
// 19 in FP32, 0.8 us of the kernel's 18.8 at 64 images of 64 x 64).
__global__ __launch_bounds__(NB) void k_dw32(Geo g, const bf16_t *__restrict__ dy,
                                             const bf16_t *__restrict__ x, double *__restrict__ part)
{
    constexpr int NW = C * T * C;
    constexpr int kSr = C + 4;
    __shared__ __align__(16) uint32_t lds[NB / 64][4][C * kTr];
    __shared__ float bs[NB / 64][C];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4;
    const int pp = lane >> 2, cg = lane & 3;
    uint32_t *ty = lds[wv][3];
    f4 acc[T][2][2], bacc[2];
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        bacc[mt] = zero;
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t][mt][0] = acc[t][mt][1] = zero;
    }
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = as_bf(0x3F80);
    const uint4 z4 = {0, 0, 0, 0};
    const long nt_ = dw_tasks(g);
    for (long task = (long)blockIdx.x * (NB / 64) + wv; task < nt_; task += (long)gridDim.x * (NB / 64)) {
        const DwStrip s = dw_strip(g, task);
        const int nr = s.y1 - s.y0;
        const int c0 = dw_col(s.x0 + 2 * pp, g.w), c1 = dw_col(s.x0 + 2 * pp + 1, g.w);
        // the pixels just left and right of the strip, lanes 0..7
        const int ch = dw_col(pp == 0 ? s.x0 - 1 : s.x0 + kDwW, g.w);
        const bool y0ok = s.x0 + 2 * pp < s.x1, y1ok = s.x0 + 2 * pp + 1 < s.x1;
        auto ldx = [&](int y, Pair &v, uint4 &h) {
            const bf16_t *p = x + (s.base + (long)wrap(y, g.h) * g.w) * C + 8 * cg;
            v.a = *reinterpret_cast<const uint4 *>(p + (long)c0 * C);
            v.b = *reinterpret_cast<const uint4 *>(p + (long)c1 * C);
            h = lane < 8 ? *reinterpret_cast<const uint4 *>(p + (long)ch * C) : z4;
        };
        auto ldy = [&](int y, Pair &v) {
            const bf16_t *p = dy + (s.base + (long)y * g.w) * C + 8 * cg;
            v.a = y0ok ? *reinterpret_cast<const uint4 *>(p + (long)c0 * C) : z4;
            v.b = y1ok ? *reinterpret_cast<const uint4 *>(p + (long)c1 * C) : z4;
        };
        // pixel p of the strip at half-word p + 2 of a channel's row
        auto putx = [&](int slot, const Pair &v, const uint4 &h) {
            uint32_t *tr = lds[wv][slot];
            put_pair(tr, cg, pp + 1, v);
            if (lane < 8) {
                Pair e;
                e.a = pp == 0 ? z4 : h;
                e.b = pp == 0 ? h : z4;
                put_pair(tr, cg, pp == 0 ? 0 : kDwW / 2 + 1, e);
            }
        };
        Pair vx, vy;
        uint4 hx;
        ldx(s.y0 - 1, vx, hx);
        putx(0, vx, hx);
        ldx(s.y0, vx, hx);
        putx(1, vx, hx);
        ldx(s.y0 + 1, vx, hx);
        ldy(s.y0, vy);
        for (int r = 0; r < nr; ++r) {
            putx((r + 2) % 3, vx, hx);
            put_pair(ty, cg, pp, vy);
            if (r + 1 < nr) {
                ldx(s.y0 + r + 2, vx, hx);
                ldy(s.y0 + r + 1, vy);
            }
            __builtin_amdgcn_wave_barrier();
            bf16x8 av[2];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                const uint32_t *p = ty + (16 * mt + m) * kTr + 4 * kq;
                const uint2 lo = *reinterpret_cast<const uint2 *>(p), hi = *reinterpret_cast<const uint2 *>(p + 2);
                const uint32_t d[4] = {lo.x, lo.y, hi.x, hi.y};
                av[mt] = frag(d);
                bacc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[mt], ones, bacc[mt], 0, 0, 0);
            }
#pragma unroll
            for (int dyi = 0; dyi < 3; ++dyi) {
                const uint32_t *tr = lds[wv][(r + dyi) % 3];
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) {
                    const uint32_t *p = tr + (16 * nt + m) * kTr + 4 * kq;
                    const uint2 q0 = *reinterpret_cast<const uint2 *>(p);
                    const uint2 q1 = *reinterpret_cast<const uint2 *>(p + 2);
                    const uint2 q2 = *reinterpret_cast<const uint2 *>(p + 4);
                    const uint32_t e[6] = {q0.x, q0.y, q1.x, q1.y, q2.x, q2.y};
                    uint32_t l[4], c[4], rr[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        l[i] = __builtin_amdgcn_alignbit(e[i + 1], e[i], 16);
                        c[i] = e[i + 1];
                        rr[i] = __builtin_amdgcn_alignbit(e[i + 2], e[i + 1], 16);
                    }
                    const bf16x8 b[3] = {frag(l), frag(c), frag(rr)};
#pragma unroll
                    for (int d = 0; d < 3; ++d)
#pragma unroll
                        for (int mt = 0; mt < 2; ++mt)
                            acc[3 * dyi + d][mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                av[mt], b[d], acc[3 * dyi + d][mt][nt], 0, 0, 0);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    // the four waves' sums, tap by tap through the two halves of the LDS
    // (rows of 36 put a wave's writes on different banks)
    static_assert(2 * (NB / 64) * C * kSr * sizeof(float) == sizeof(lds), "two taps' sums of four waves");
    float *sums = reinterpret_cast<float *>(&lds[0][0][0]);
    if (m == 0)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) bs[wv][16 * mt + 4 * kq + i] = bacc[mt][i];
    __syncthreads();
    double *out = part + (long)blockIdx.x * (NW + C);
    const int co = threadIdx.x / (C / 4), ci = 4 * (threadIdx.x % (C / 4));
#pragma unroll
    for (int t = 0; t < T; ++t) {
        float *b = sums + (t & 1) * (NB / 64) * C * kSr;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    b[(wv * C + 16 * mt + 4 * kq + i) * kSr + 16 * nt + m] = acc[t][mt][nt][i];
        __syncthreads();
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int w = 0; w < NB / 64; ++w) {
            const f4 v = *reinterpret_cast<const f4 *>(b + (w * C + co) * kSr + ci);
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += v[i];
        }
#pragma unroll
        for (int i = 0; i < 4; i += 2)
            *reinterpret_cast<double2 *>(out + (co * T + t) * C + ci + i) = make_double2(s[i], s[i + 1]);
    }
    if (threadIdx.x < C) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < NB / 64; ++w) s += bs[w][threadIdx.x];
        out[NW + threadIdx.x] = s;
    }
}

// Weight gradients of the layers with a one-channel side: M = the 32
// channels of v, N = the 9 taps of the FP32 one-channel u (rounded to BF16),
// K = pixels.
// Layer 1 (LAST = false): v = dA1, u = the potential x:
//   dW1[co][t] = sum_p dA1[p][co] x[nbr(p,t)], db1[co] = sum_p dA1[p][co]
//   (column 9: ones).
// Layer 4 (LAST): v = a3, u = dO:
//   dW4[t][ci] = sum_p a3[p][ci] dO[nbr(p,-t)], db4 = sum_p dO[p] in FP64
//   (dO's values nearly cancel).
// The block's partial, its four waves added in FP64, goes to part[blockIdx],
// C T + C values in the parameters' order.
template <bool LAST>
__global__ __launch_bounds__(NB) void k_dw_edge(Geo g, const bf16_t *__restrict__ v,
                                                const float *__restrict__ u, double *__restrict__ part)
{
    constexpr int NV = C * T + C;
    __shared__ __align__(16) uint32_t lds[NB / 64][C * kTr];
    __shared__ double bs[NB / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4;
    const int pp = lane >> 2, cg = lane & 3;
    const int sgn = LAST ? -1 : 1;
    const int ody = sgn * (m / 3 - 1), odx = sgn * (m % 3 - 1);  // the tap of column m < 9
    uint32_t *tv = lds[wv];
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 acc[2] = {zero, zero};
    double bsum = 0.0;
    const uint4 z4 = {0, 0, 0, 0};
    const long nt_ = dw_tasks(g);
    for (long task = (long)blockIdx.x * (NB / 64) + wv; task < nt_; task += (long)gridDim.x * (NB / 64)) {
        const DwStrip s = dw_strip(g, task);
        const int c0 = dw_col(s.x0 + 2 * pp, g.w), c1 = dw_col(s.x0 + 2 * pp + 1, g.w);
        const bool ok0 = s.x0 + 2 * pp < s.x1, ok1 = s.x0 + 2 * pp + 1 < s.x1;
        int uc[8];
        bool uok[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uok[j] = s.x0 + 8 * kq + j < s.x1;
            uc[j] = dw_col(s.x0 + 8 * kq + j + odx, g.w);
        }
        auto ldv = [&](int y, Pair &p) {
            const bf16_t *b = v + (s.base + (long)y * g.w) * C + 8 * cg;
            p.a = ok0 ? *reinterpret_cast<const uint4 *>(b + (long)c0 * C) : z4;
            p.b = ok1 ? *reinterpret_cast<const uint4 *>(b + (long)c1 * C) : z4;
        };
        auto ldu = [&](int y, float f[8]) {
            const float *b = u + s.base + (long)wrap(y + ody, g.h) * g.w;
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = m < T ? b[uc[j]] : 1.f;
        };
        Pair pv;
        float f[8];
        ldv(s.y0, pv);
        ldu(s.y0, f);
        for (int y = s.y0; y < s.y1; ++y) {
            put_pair(tv, cg, pp, pv);
            bf16x8 b;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                b[j] = as_bf(m <= T ? f2bf(f[j]) : (bf16_t)0);
                if (LAST && m == 4 && uok[j]) bsum += f[j];  // the centre tap's pixels
            }
            if (y + 1 < s.y1) {
                ldv(y + 1, pv);
                ldu(y + 1, f);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                const uint32_t *p = tv + (16 * mt + m) * kTr + 4 * kq;
                const uint2 lo = *reinterpret_cast<const uint2 *>(p), hi = *reinterpret_cast<const uint2 *>(p + 2);
                const uint32_t d[4] = {lo.x, lo.y, hi.x, hi.y};
                acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(d), b, acc[mt], 0, 0, 0);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    static_assert(sizeof(lds[0]) >= NV * sizeof(float), "a wave's sums in its part of the LDS");
    uint32_t *out = lds[wv];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = 16 * mt + 4 * kq + i;
            if (m < T) out[LAST ? m * C + ch : ch * T + m] = __float_as_uint(acc[mt][i]);
            if (!LAST && m == T) out[C * T + ch] = __float_as_uint(acc[mt][i]);
        }
    if (LAST) {
        bsum += __shfl_xor(bsum, 16);
        bsum += __shfl_xor(bsum, 32);
        if (lane == 4) bs[wv] = bsum;
    }
    __syncthreads();
    for (int j = threadIdx.x; j < (LAST ? C * T + 1 : NV); j += NB) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < NB / 64; ++w) t += LAST && j == C * T ? bs[w] : (double)__uint_as_float(lds[w][j]);
        part[(long)blockIdx.x * NV + j] = t;
    }
}

// grad = the sums over the partials' rows, in FP64, of all four layers in one
// launch: a block takes 32 columns of a layer, its 32 groups of threads every
// 32nd row, all their loads in flight, and the groups' sums are added in
// order.  (A launch per layer: 24 us and the gaps between them, of 340 for 64
// images of 64 x 64; 39 MB with 16 groups of 64 columns, and a row per wave of
// the first and last layers: 14.0 us, now 7.1.)
constexpr int kRedGroups = 32, kRedCols = 32;
struct RedSeg {
    long part;
    int len, stride, out, blk0;
};
struct RedArgs {
    RedSeg s[4];
    int blocks;
};
constexpr RedArgs red_args()
{
    RedArgs a{};
    a.s[0] = {kPart3, kRowMid, kRowMid, OW3, 0};
    a.s[1] = {kPart2, kRowMid, kRowMid, OW2, 0};
    a.s[2] = {kPart4, C * T + 1, kRowEdge, OW4, 0};  // layer 4 has one bias
    a.s[3] = {kPart1, kRowEdge, kRowEdge, OW1, 0};
    for (int i = 0; i < 4; ++i) {
        a.s[i].blk0 = a.blocks;
        a.blocks += (a.s[i].len + kRedCols - 1) / kRedCols;
    }
    return a;
}
__global__ __launch_bounds__(kRedCols * kRedGroups) void k_reduce(const double *__restrict__ part, int dwb,
                                                            float *__restrict__ grad)
{
    constexpr RedArgs a = red_args();
    __shared__ double sm[kRedGroups][kRedCols];
    const int c = threadIdx.x % kRedCols, gr = threadIdx.x / kRedCols;
    RedSeg q = a.s[0];
#pragma unroll
    for (int i = 1; i < 4; ++i)
        if ((int)blockIdx.x >= a.s[i].blk0) q = a.s[i];
    const int j = ((int)blockIdx.x - q.blk0) * kRedCols + c;
    double s = 0.0;
    if (j < q.len) {
        const double *p = part + q.part + j;
#pragma unroll 8
        for (int b = gr; b < dwb; b += kRedGroups) s += p[(long)b * q.stride];
    }
    sm[gr][c] = s;
    __syncthreads();
    if (gr == 0 && j < q.len) {
        double t = 0.0;
#pragma unroll
        for (int i = 0; i < kRedGroups; ++i) t += sm[i][c];
        grad[q.out + j] = (float)t;
    }
}

// Adam on the FP32 master parameters; refreshes the BF16 copies (W and
// the transposed W of layers 2/3 used by the backward data pass).
__global__ __launch_bounds__(NB) void k_adam(float *__restrict__ prm, const float *__restrict__ grad,
                                             float *__restrict__ m1, float *__restrict__ m2, int n,
                                             float lr, float b1t, float b2t)
{
    const int i = blockIdx.x * NB + threadIdx.x;
    if (i >= n) return;
    const float gr = grad[i];
    const float a = 0.9f * m1[i] + 0.1f * gr;
    const float b = 0.999f * m2[i] + 0.001f * gr * gr;
    m1[i] = a;
    m2[i] = b;
    prm[i] -= lr * (a / b1t) / (sqrtf(b / b2t) + 1e-8f);
}

__global__ __launch_bounds__(NB) void k_bf16_params(const float *__restrict__ prm, bf16_t *__restrict__ wb,
                                                    bf16_t *__restrict__ wt2, bf16_t *__restrict__ wt3)
{
    const int i = blockIdx.x * NB + threadIdx.x;
    if (i < NPARAM) wb[i] = f2bf(prm[i]);
    if (i < C * T * C) {
        // i = (co*T + t)*C + ci  ->  transposed (ci*T + t)*C + co
        const int co = i / (T * C), t = (i / C) % T, ci = i % C;
        const int j = (ci * T + t) * C + co;
        wt2[j] = f2bf(prm[OW2 + i]);
        wt3[j] = f2bf(prm[OW3 + i]);
    }
}

}  // namespace

struct trlnet {
    float *prm = nullptr, *grad = nullptr, *m1 = nullptr, *m2 = nullptr;
    bf16_t *wb = nullptr, *wt2 = nullptr, *wt3 = nullptr;
    int step = 0;
    // workspace
    long cap = 0;  // pixels
    float *x = nullptr, *tg = nullptr, *o = nullptr, *dO = nullptr;
    bf16_t *a1 = nullptr, *a2 = nullptr, *a3 = nullptr, *d1 = nullptr, *d2 = nullptr;
    double *part = nullptr;
    long partcap = 0;
    double *lpart = nullptr;
    int lcap = 0;
    float *hstage = nullptr;  // pinned staging of trlnet_forward_many (in, then out)
    long hcap = 0;            // floats
    char *hgeo = nullptr, *dgeo = nullptr;  // group table of the many-group launches (pinned / device)
    long geocap = 0;                        // bytes
    hipStream_t s = nullptr;
};

namespace {

#define NTRY(e)                                  \
    do {                                         \
        if ((e) != hipSuccess) return TRLNET_EHIP; \
    } while (0)

int ensure(trlnet *t, long np, int nimg)
{
    if (np > t->cap) {
        (void)hipStreamSynchronize(t->s);
        for (void *q : {(void *)t->x, (void *)t->tg, (void *)t->o, (void *)t->dO, (void *)t->a1,
                        (void *)t->a2, (void *)t->a3, (void *)t->d1, (void *)t->d2})
            if (q) (void)hipFree(q);
        t->cap = 0;
        NTRY(hipMalloc((void **)&t->x, sizeof(float) * np));
        NTRY(hipMalloc((void **)&t->tg, sizeof(float) * np));
        NTRY(hipMalloc((void **)&t->o, sizeof(float) * np));
        NTRY(hipMalloc((void **)&t->dO, sizeof(float) * np));
        NTRY(hipMalloc((void **)&t->a1, sizeof(bf16_t) * C * np));
        NTRY(hipMalloc((void **)&t->a2, sizeof(bf16_t) * C * np));
        NTRY(hipMalloc((void **)&t->a3, sizeof(bf16_t) * C * np));
        NTRY(hipMalloc((void **)&t->d1, sizeof(bf16_t) * C * np));
        NTRY(hipMalloc((void **)&t->d2, sizeof(bf16_t) * C * np));
        t->cap = np;
    }
    const long need = kPartCount;
    if (need > t->partcap) {
        if (t->part) (void)hipFree(t->part);
        t->partcap = 0;
        NTRY(hipMalloc((void **)&t->part, sizeof(double) * need));
        t->partcap = need;
    }
    if (nimg > t->lcap) {
        if (t->lpart) (void)hipFree(t->lpart);
        t->lcap = 0;
        NTRY(hipMalloc((void **)&t->lpart, sizeof(double) * nimg));
        t->lcap = nimg;
    }
    return 0;
}

int refresh_bf16(trlnet *t)
{
    hipLaunchKernelGGL(k_bf16_params, dim3((C * T * C + NB - 1) / NB > (NPARAM + NB - 1) / NB
                                               ? (C * T * C + NB - 1) / NB
                                               : (NPARAM + NB - 1) / NB),
                       dim3(NB), 0, t->s, t->prm, t->wb, t->wt2, t->wt3);
    return hipGetLastError() == hipSuccess ? 0 : TRLNET_EHIP;
}

// Forward pass of the images g at pixel offset off of the workspace
// (activations are channel-last, pixel p at p * C).
int forward(trlnet *t, const Geo &g, long off = 0)
{
    const int gb = (int)conv_blocks(g);
    const long oc = off * C;
    hipLaunchKernelGGL(k_fwd1, dim3(gb), dim3(NB), 0, t->s, g, t->x + off, t->wb + OW1, t->prm + OB1,
                       t->a1 + oc);
    hipLaunchKernelGGL(k_fwd32, dim3(gb), dim3(NB), 0, t->s, g, t->a1 + oc, t->wb + OW2, t->prm + OB2,
                       t->a2 + oc);
    hipLaunchKernelGGL(k_fwd32, dim3(gb), dim3(NB), 0, t->s, g, t->a2 + oc, t->wb + OW3, t->prm + OB3,
                       t->a3 + oc);
    hipLaunchKernelGGL(k_fwd4, dim3(gb), dim3(NB), 0, t->s, g, t->a3 + oc, t->wb + OW4, t->prm + OB4,
                       t->o + off);
    return hipGetLastError() == hipSuccess ? 0 : TRLNET_EHIP;
}

// The forward pass over groups back to back (inputs at t->x, outputs at
// t->o): one launch per layer for all groups, the same per-pixel
// arithmetic as forward() group by group.
int forward_groups(trlnet *t, int ngroups, const int *nimg, const int *h, const int *w)
{
    const size_t tab = sizeof(GroupGeo) * (size_t)ngroups;
    const size_t off_pre = (tab + 255) & ~(size_t)255;
    const size_t bytes = off_pre + sizeof(int) * (size_t)(ngroups + 1);
    if ((long)bytes > t->geocap) {
        if (t->hgeo) (void)hipHostFree(t->hgeo);
        if (t->dgeo) (void)hipFree(t->dgeo);
        t->hgeo = t->dgeo = nullptr;
        t->geocap = 0;
        NTRY(hipHostMalloc((void **)&t->hgeo, bytes, 0));
        NTRY(hipMalloc((void **)&t->dgeo, bytes));
        t->geocap = (long)bytes;
    }
    GroupGeo *gg = reinterpret_cast<GroupGeo *>(t->hgeo);
    int *pre = reinterpret_cast<int *>(t->hgeo + off_pre);
    const int rows = conv_rows(ngroups, nimg, h, w);
    long off = 0;
    pre[0] = 0;
    for (int i = 0; i < ngroups; ++i) {
        const Geo g = geo_of(nimg[i], h[i], w[i], rows);
        gg[i] = GroupGeo{g, off};
        const long nb = (long)pre[i] + conv_blocks(g);
        if (nb > 0x7fffffffL) return TRLNET_EINVAL;
        pre[i + 1] = (int)nb;
        off += g.np;
    }
    NTRY(hipMemcpyAsync(t->dgeo, t->hgeo, bytes, hipMemcpyHostToDevice, t->s));
    const GroupGeo *dg = reinterpret_cast<const GroupGeo *>(t->dgeo);
    const int *dp = reinterpret_cast<const int *>(t->dgeo + off_pre);
    const dim3 gb(pre[ngroups]);
    hipLaunchKernelGGL(k_fwd1_many, gb, dim3(NB), 0, t->s, dg, dp, ngroups, t->x, t->wb + OW1,
                       t->prm + OB1, t->a1);
    hipLaunchKernelGGL(k_fwd32_many, gb, dim3(NB), 0, t->s, dg, dp, ngroups, t->a1, t->wb + OW2,
                       t->prm + OB2, t->a2);
    hipLaunchKernelGGL(k_fwd32_many, gb, dim3(NB), 0, t->s, dg, dp, ngroups, t->a2, t->wb + OW3,
                       t->prm + OB3, t->a3);
    hipLaunchKernelGGL(k_fwd4_many, gb, dim3(NB), 0, t->s, dg, dp, ngroups, t->a3, t->wb + OW4,
                       t->prm + OB4, t->o);
    return hipGetLastError() == hipSuccess ? 0 : TRLNET_EHIP;
}

// loss and gradient into t->grad (device); *loss on the host
int backward(trlnet *t, const Geo &g, double *loss)
{
    const int gb = (int)conv_blocks(g);
    const int ndw = (int)std::min<long>(kDwBlocks, (dw_tasks(g) + NB / 64 - 1) / (NB / 64));
    const dim3 dwb(ndw), blk(NB);
    hipLaunchKernelGGL(k_loss, dim3(g.nimg), blk, 0, t->s, g, t->o, t->tg, t->dO, t->lpart);
    // layer 4
    hipLaunchKernelGGL((k_dw_edge<true>), dwb, blk, 0, t->s, g, t->a3, t->dO, t->part + kPart4);
    hipLaunchKernelGGL(k_bwd4, dim3(gb), blk, 0, t->s, g, t->dO, t->wb + OW4, t->a3, t->d2);
    // layer 3: dY = d2 (for a3), X = a2
    hipLaunchKernelGGL(k_dw32, dwb, blk, 0, t->s, g, t->d2, t->a2, t->part + kPart3);
    hipLaunchKernelGGL(k_bwd32, dim3(gb), blk, 0, t->s, g, t->d2, t->wt3, t->a2, t->d1);
    // layer 2: dY = d1 (for a2), X = a1
    hipLaunchKernelGGL(k_dw32, dwb, blk, 0, t->s, g, t->d1, t->a1, t->part + kPart2);
    hipLaunchKernelGGL(k_bwd32, dim3(gb), blk, 0, t->s, g, t->d1, t->wt2, t->a1, t->d2);
    // layer 1: dY = d2 (for a1), X = potential
    hipLaunchKernelGGL((k_dw_edge<false>), dwb, blk, 0, t->s, g, t->d2, t->x, t->part + kPart1);
    hipLaunchKernelGGL(k_reduce, dim3(red_args().blocks), dim3(kRedCols * kRedGroups), 0, t->s, t->part, ndw,
                       t->grad);
    if (hipGetLastError() != hipSuccess) return TRLNET_EHIP;
    std::vector<double> lp((size_t)g.nimg);
    NTRY(hipMemcpyAsync(lp.data(), t->lpart, sizeof(double) * g.nimg, hipMemcpyDeviceToHost, t->s));
    NTRY(hipStreamSynchronize(t->s));
    double l = 0.0;
    for (double v : lp) l += v;
    *loss = l;
    return 0;
}

int upload(trlnet *t, const Geo &g, const float *in, const float *target)
{
    if (int rc = ensure(t, g.np, g.nimg)) return rc;
    NTRY(hipMemcpyAsync(t->x, in, sizeof(float) * g.np, hipMemcpyHostToDevice, t->s));
    if (target) NTRY(hipMemcpyAsync(t->tg, target, sizeof(float) * g.np, hipMemcpyHostToDevice, t->s));
    return 0;
}

bool geo_ok(int nimg, int h, int w) { return nimg > 0 && h >= 3 && w >= 3 && (long)nimg * h * w < (1L << 40); }

}  // namespace

extern "C" {

int trlnet_param_count(void) { return NPARAM; }

int trlnet_create(trlnet **out, unsigned long long seed)
{
    if (!out) return TRLNET_EINVAL;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return TRLNET_ENODEV;
    trlnet *t = new (std::nothrow) trlnet();
    if (!t) return TRLNET_ENOMEM;
    int rc = 0;
    if (hipStreamCreate(&t->s) != hipSuccess) rc = TRLNET_EHIP;
    const size_t pb = sizeof(float) * NPARAM;
    if (!rc && (hipMalloc((void **)&t->prm, pb) != hipSuccess || hipMalloc((void **)&t->grad, pb) != hipSuccess ||
                hipMalloc((void **)&t->m1, pb) != hipSuccess || hipMalloc((void **)&t->m2, pb) != hipSuccess ||
                hipMalloc((void **)&t->wb, sizeof(bf16_t) * NPARAM) != hipSuccess ||
                hipMalloc((void **)&t->wt2, sizeof(bf16_t) * C * T * C) != hipSuccess ||
                hipMalloc((void **)&t->wt3, sizeof(bf16_t) * C * T * C) != hipSuccess))
        rc = TRLNET_ENOMEM;
    if (!rc) {
        // He-normal weights from a 64-bit xorshift stream (Box-Muller), zero biases
        std::vector<float> h(NPARAM, 0.f);
        uint64_t st = seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull;
        auto uni = [&]() {
            st ^= st >> 12;
            st ^= st << 25;
            st ^= st >> 27;
            return ((st * 0x2545F4914F6CDD1Dull) >> 11) * (1.0 / 9007199254740992.0);
        };
        auto gauss = [&]() {
            const double u1 = uni() + 1e-300, u2 = uni();
            return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
        };
        const struct { int off, n, fan_in; } L[4] = {
            {OW1, C * T, T}, {OW2, C * T * C, T * C}, {OW3, C * T * C, T * C}, {OW4, T * C, T * C}};
        for (const auto &l : L)
            for (int i = 0; i < l.n; ++i) h[(size_t)l.off + i] = (float)(gauss() * std::sqrt(2.0 / l.fan_in));
        if (hipMemcpy(t->prm, h.data(), pb, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemset(t->m1, 0, pb) != hipSuccess || hipMemset(t->m2, 0, pb) != hipSuccess ||
            hipMemset(t->grad, 0, pb) != hipSuccess)
            rc = TRLNET_EHIP;
    }
    if (!rc) rc = refresh_bf16(t);
    if (!rc && hipStreamSynchronize(t->s) != hipSuccess) rc = TRLNET_EHIP;
    if (rc) {
        trlnet_destroy(t);
        return rc;
    }
    *out = t;
    return 0;
}

int trlnet_destroy(trlnet *t)
{
    if (!t) return 0;
    if (t->s) (void)hipStreamSynchronize(t->s);
    for (void *p : {(void *)t->prm, (void *)t->grad, (void *)t->m1, (void *)t->m2, (void *)t->wb,
                    (void *)t->wt2, (void *)t->wt3, (void *)t->x, (void *)t->tg, (void *)t->o,
                    (void *)t->dO, (void *)t->a1, (void *)t->a2, (void *)t->a3, (void *)t->d1,
                    (void *)t->d2, (void *)t->part, (void *)t->lpart})
        if (p) (void)hipFree(p);
    if (t->hstage) (void)hipHostFree(t->hstage);
    if (t->hgeo) (void)hipHostFree(t->hgeo);
    if (t->dgeo) (void)hipFree(t->dgeo);
    if (t->s) (void)hipStreamDestroy(t->s);
    delete t;
    return 0;
}

int trlnet_get_params(trlnet *t, float *out, int n)
{
    if (!t || !out || n < NPARAM) return TRLNET_EINVAL;
    NTRY(hipMemcpyAsync(out, t->prm, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, t->s));
    NTRY(hipStreamSynchronize(t->s));
    return 0;
}

int trlnet_set_params(trlnet *t, const float *in, int n)
{
    if (!t || !in || n < NPARAM) return TRLNET_EINVAL;
    NTRY(hipMemcpyAsync(t->prm, in, sizeof(float) * NPARAM, hipMemcpyHostToDevice, t->s));
    if (int rc = refresh_bf16(t)) return rc;
    NTRY(hipStreamSynchronize(t->s));
    return 0;
}

int trlnet_forward(trlnet *t, int nimg, int h, int w, const float *in, float *out)
{
    if (!t || !in || !out || !geo_ok(nimg, h, w)) return TRLNET_EINVAL;
    const Geo g = geo_of(nimg, h, w, conv_rows(1, &nimg, &h, &w));
    if (int rc = upload(t, g, in, nullptr)) return rc;
    if (int rc = forward(t, g)) return rc;
    NTRY(hipMemcpyAsync(out, t->o, sizeof(float) * g.np, hipMemcpyDeviceToHost, t->s));
    NTRY(hipStreamSynchronize(t->s));
    return 0;
}

int trlnet_forward_many(trlnet *t, int ngroups, const int *nimg, const int *h, const int *w,
                        const float *in, float *out)
{
    if (!t || ngroups < 1 || !nimg || !h || !w || !in || !out) return TRLNET_EINVAL;
    long total = 0;
    for (int i = 0; i < ngroups; ++i) {
        if (!geo_ok(nimg[i], h[i], w[i])) return TRLNET_EINVAL;
        total += (long)nimg[i] * h[i] * w[i];
    }
    if (int rc = ensure(t, total, 1)) return rc;
    if (total > t->hcap) {  // pinned staging: the copies run as DMA, asynchronously
        if (t->hstage) (void)hipHostFree(t->hstage);
        t->hstage = nullptr;
        t->hcap = 0;
        NTRY(hipHostMalloc((void **)&t->hstage, sizeof(float) * total, 0));
        t->hcap = total;
    }
    memcpy(t->hstage, in, sizeof(float) * total);
    NTRY(hipMemcpyAsync(t->x, t->hstage, sizeof(float) * total, hipMemcpyHostToDevice, t->s));
    if (int rc = forward_groups(t, ngroups, nimg, h, w)) return rc;
    NTRY(hipMemcpyAsync(t->hstage, t->o, sizeof(float) * total, hipMemcpyDeviceToHost, t->s));
    NTRY(hipStreamSynchronize(t->s));
    memcpy(out, t->hstage, sizeof(float) * total);
    return 0;
}

}  // extern "C"

namespace {

// Validates the groups, sizes the device buffers and the pinned staging
// for `total` input floats.
int many_prepare(trlnet *t, int ngroups, const int *nimg, const int *h, const int *w, long *total)
{
    long tot = 0;
    for (int i = 0; i < ngroups; ++i) {
        if (!geo_ok(nimg[i], h[i], w[i])) return TRLNET_EINVAL;
        tot += (long)nimg[i] * h[i] * w[i];
    }
    if (int rc = ensure(t, tot, 1)) return rc;
    if (tot > t->hcap) {
        if (t->hstage) (void)hipHostFree(t->hstage);
        t->hstage = nullptr;
        t->hcap = 0;
        NTRY(hipHostMalloc((void **)&t->hstage, sizeof(float) * tot, 0));
        t->hcap = tot;
    }
    *total = tot;
    return 0;
}

// Uploads the staged inputs and runs every group; outputs stay on the device.
int many_run(trlnet *t, int ngroups, const int *nimg, const int *h, const int *w, long total,
             const float **out_device)
{
    NTRY(hipMemcpyAsync(t->x, t->hstage, sizeof(float) * total, hipMemcpyHostToDevice, t->s));
    if (int rc = forward_groups(t, ngroups, nimg, h, w)) return rc;
    NTRY(hipStreamSynchronize(t->s));
    *out_device = t->o;
    return 0;
}

}  // namespace

extern "C" {

int trlnet_forward_many_device(trlnet *t, int ngroups, const int *nimg, const int *h, const int *w,
                               const float *in, const float **out_device)
{
    if (!t || ngroups < 1 || !nimg || !h || !w || !in || !out_device) return TRLNET_EINVAL;
    long total = 0;
    if (int rc = many_prepare(t, ngroups, nimg, h, w, &total)) return rc;
    memcpy(t->hstage, in, sizeof(float) * total);
    return many_run(t, ngroups, nimg, h, w, total, out_device);
}

int trlnet_forward_many_device_f64(trlnet *t, int ngroups, const int *nimg, const int *h,
                                   const int *w, const double *const *img, double scale,
                                   const float **out_device)
{
    if (!t || ngroups < 1 || !nimg || !h || !w || !img || !out_device) return TRLNET_EINVAL;
    long total = 0;
    if (int rc = many_prepare(t, ngroups, nimg, h, w, &total)) return rc;
    // image i: its pointer, size and offset in the staging buffer
    std::vector<const double *> src;
    std::vector<long> len, off;
    long o = 0;
    for (int g = 0; g < ngroups; ++g)
        for (int k = 0; k < nimg[g]; ++k) {
            const long np = (long)h[g] * w[g];
            if (!img[src.size()]) return TRLNET_EINVAL;
            src.push_back(img[src.size()]);
            len.push_back(np);
            off.push_back(o);
            o += np;
        }
    // fl32(x * scale) into the staging, images dealt to up to 16 threads
    // by a shared counter
    const int nimgs = (int)src.size();
    unsigned hw = std::thread::hardware_concurrency();
    const int nthr = (int)std::min<long>(std::min<unsigned>(hw ? hw : 1, 16), std::max(1, nimgs));
    std::atomic<int> next{0};
    auto work = [&]() {
        for (int i; (i = next.fetch_add(1, std::memory_order_relaxed)) < nimgs;) {
            const double *p = src[i];
            float *q = t->hstage + off[i];
            for (long j = 0; j < len[i]; ++j) q[j] = (float)(p[j] * scale);
        }
    };
    std::vector<std::thread> th;
    for (int k = 1; k < nthr; ++k) th.emplace_back(work);
    work();
    for (auto &x : th) x.join();
    return many_run(t, ngroups, nimg, h, w, total, out_device);
}

int trlnet_loss_grad(trlnet *t, int nimg, int h, int w, const float *in, const float *target,
                     float *loss, float *grad)
{
    if (!t || !in || !target || !geo_ok(nimg, h, w)) return TRLNET_EINVAL;
    const Geo g = geo_of(nimg, h, w, conv_rows(1, &nimg, &h, &w));
    if (int rc = upload(t, g, in, target)) return rc;
    if (int rc = forward(t, g)) return rc;
    double l = 0.0;
    if (int rc = backward(t, g, &l)) return rc;
    if (loss) *loss = (float)l;
    if (grad) {
        NTRY(hipMemcpyAsync(grad, t->grad, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, t->s));
        NTRY(hipStreamSynchronize(t->s));
    }
    return 0;
}

int trlnet_train_step(trlnet *t, int nimg, int h, int w, const float *in, const float *target,
                      float lr, float *loss)
{
    float l = 0.f;
    if (int rc = trlnet_loss_grad(t, nimg, h, w, in, target, &l, nullptr)) return rc;
    ++t->step;
    const float b1t = 1.f - std::pow(0.9f, (float)t->step), b2t = 1.f - std::pow(0.999f, (float)t->step);
    hipLaunchKernelGGL(k_adam, dim3((NPARAM + NB - 1) / NB), dim3(NB), 0, t->s, t->prm, t->grad, t->m1,
                       t->m2, NPARAM, lr, b1t, b2t);
    if (int rc = refresh_bf16(t)) return rc;
    NTRY(hipStreamSynchronize(t->s));
    if (loss) *loss = l;
    return 0;
}

}  // extern "C"
