// A small fully connected cost model trained and evaluated on the GPU:
//   z1 = W1 x + b1, a1 = relu(z1)      (hidden H)
//   z2 = W2 a1 + b2, a2 = relu(z2)     (hidden H)
//   y  = W3 a2 + b3                    (scalar: predicted log2 time)
// trained with mean squared error and Adam. Parameters are one flat FP32
// array [W1 (H x D, row-major), b1 (H), W2 (H x H), b2 (H), W3 (H), b3 (1)].
// Every sum has one fixed order (no atomics): a layer's outputs over its
// inputs in increasing index, weight gradients over chunks of kChunk samples
// in increasing sample, then over the chunks. Two sets of kernels compute
// these same sums, bit for bit: networks up to kSmallD inputs and kSmallH
// hidden units take three launches per epoch (mlp_pass, grad_part, grad_sum);
// larger ones one plain kernel per layer and direction, one thread per output.
//
// No reference counterpart (an extension beside the reference's scans). Compiled with
// -ffp-contract=off so results are reproducible against the CPU oracle.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "handle.hpp"

using gps::fail;
using gps::hip_fail;

namespace {

constexpr int kThreads = 256;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

inline dim3 grid_of(uint64_t n) { return dim3((uint32_t)((n + kThreads - 1) / kThreads)); }

// Y[b, o] = act(b[o] + sum_i W[o, i] X[b, i]); Z keeps the pre-activation.
__global__ void linear_fwd(const float* X, const float* W, const float* bias, float* Z, float* Y, uint32_t B,
                           uint32_t Din, uint32_t Dout, int relu) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (uint64_t)B * Dout) return;
    const uint32_t b = (uint32_t)(t / Dout), o = (uint32_t)(t % Dout);
    float acc = bias[o];
    const float* x = X + (uint64_t)b * Din;
    const float* w = W + (uint64_t)o * Din;
    for (uint32_t i = 0; i < Din; ++i) acc += w[i] * x[i];
    if (Z) Z[t] = acc;
    Y[t] = relu ? fmaxf(acc, 0.f) : acc;
}

// dY = 2 (y - target) / B; per-block partial sums of (y - target)^2.
__global__ void mse_grad(const float* y, const float* target, float* dy, float* partial, uint32_t B) {
    __shared__ float s[kThreads];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    float e = 0.f;
    if (i < B) {
        const float d = y[i] - target[i];
        dy[i] = 2.f * d / (float)B;
        e = d * d;
    }
    s[threadIdx.x] = e;
    __syncthreads();
    for (uint32_t w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

__global__ void sum_partials(const float* partial, uint32_t n, float scale, float* out) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        float s = 0.f;
        for (uint32_t i = 0; i < n; ++i) s += partial[i];
        *out = s * scale;
    }
}

// Weight gradients in two deterministic passes. The batch is cut into chunks
// of kChunk samples; pass 1 writes, per chunk c and output t,
//   part[c, t] = sum_{b in chunk c} dZ[b, o] X[b, i]   (t = o Din + i), or
//   part[c, t] = sum_{b in chunk c} dZ[b, o]           (t = Dout Din + o, the bias),
// in increasing b; pass 2 sums the chunks of each output in increasing c.
// The summation order is fixed, so results do not depend on scheduling.
constexpr uint32_t kChunk = 128;

inline uint32_t chunks_of(uint32_t B) { return (B + kChunk - 1) / kChunk; }

__global__ void linear_bwd_w_part(const float* dZ, const float* X, float* part, uint32_t B, uint32_t Din,
                                  uint32_t Dout) {
    const uint64_t outs = (uint64_t)Dout * Din + Dout;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= outs) return;
    const uint32_t c = blockIdx.y;
    const uint32_t b0 = c * kChunk, b1 = min(B, b0 + kChunk);
    float acc = 0.f;
    if (t < (uint64_t)Dout * Din) {
        const uint32_t o = (uint32_t)(t / Din), i = (uint32_t)(t % Din);
        for (uint32_t b = b0; b < b1; ++b) acc += dZ[(uint64_t)b * Dout + o] * X[(uint64_t)b * Din + i];
    } else {
        const uint32_t o = (uint32_t)(t - (uint64_t)Dout * Din);
        for (uint32_t b = b0; b < b1; ++b) acc += dZ[(uint64_t)b * Dout + o];
    }
    part[(uint64_t)c * outs + t] = acc;
}

// dW (Dout x Din) and db (Dout) follow each other in the flat gradient array.
__global__ void linear_bwd_w_sum(const float* part, float* dWb, uint64_t outs, uint32_t chunks) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= outs) return;
    float acc = 0.f;
    for (uint32_t c = 0; c < chunks; ++c) acc += part[(uint64_t)c * outs + t];
    dWb[t] = acc;
}

// dZprev[b, i] = (sum_o dZ[b, o] W[o, i]) * (Zprev[b, i] > 0)   (through relu).
__global__ void linear_bwd_x(const float* dZ, const float* W, const float* Zprev, float* dZprev, uint32_t B,
                             uint32_t Din, uint32_t Dout) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (uint64_t)B * Din) return;
    const uint32_t b = (uint32_t)(t / Din), i = (uint32_t)(t % Din);
    float acc = 0.f;
    for (uint32_t o = 0; o < Dout; ++o) acc += dZ[(uint64_t)b * Dout + o] * W[(uint64_t)o * Din + i];
    dZprev[t] = Zprev[t] > 0.f ? acc : 0.f;
}

// Adam with decoupled weight decay (AdamW) on one parameter; bc1 and bc2 are
// the 1-based step's bias corrections.
struct AdamArgs {
    float lr, beta1, beta2, eps, wd, bc1, bc2;
};
__device__ __forceinline__ void adam_update(float& p, float& m, float& v, float g, const AdamArgs& a) {
    m = a.beta1 * m + (1.f - a.beta1) * g;
    v = a.beta2 * v + (1.f - a.beta2) * g * g;
    const float mh = m / a.bc1, vh = v / a.bc2;
    p -= a.lr * (mh / (sqrtf(vh) + a.eps) + a.wd * p);
}

__global__ void adam_step(float* p, const float* g, float* m, float* v, uint64_t count, AdamArgs a) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) adam_update(p[i], m[i], v[i], g[i], a);
}

// ---------------------------------------------------------------------------
// Small networks: three launches per epoch.
//
// mlp_pass takes a group of 32 samples through forward and backward. Each
// layer is a product on 4 x 2 register tiles (samples x units): per step of
// the sum a thread reads four samples' activations from LDS and two units'
// weights from a transposed copy that stays in L1, and layers meet in LDS. It
// leaves the activations and deltas unit-major, [unit][32 samples] per group.
// grad_part sums a chunk's weight gradients, a 2 x 4 tile of one gradient
// matrix per thread, from LDS rows read four samples at a time; grad_sum adds
// the chunks and takes the Adam step.
//
// The sums keep the plain kernels' order and rounding (one multiply, one add),
// which rules out the matrix cores: their products are fused and their order
// is their own, and 20 Adam epochs turn a last-bit difference near a zero
// gradient into a step of the learning rate. The bound is then the vector ALU:
// 14.8 k multiply-adds per sample at 18 inputs and 64 hidden units, 14 us an
// epoch at 18,808 samples. Measured there: 43 us an epoch (mlp_pass
// 20.8, grad_part 15.7, grad_sum 6.1), against 519 us for one
// plain kernel per layer and direction, which read their weights uncoalesced
// from memory for every product. (Weights as scalar loads, one sample to a
// lane and 64 samples to a workgroup: mlp_pass 32 us, waiting on the loads.)
// ---------------------------------------------------------------------------
constexpr uint32_t kSmallD = 64;
constexpr uint32_t kSmallH = 128;
constexpr uint32_t kGroup = 32;             // samples of a group
constexpr uint32_t kRow = kGroup + 4;       // LDS row of grad_part: eight rows' 16-byte reads fall in different banks
constexpr uint32_t kPartThreads = 256;

inline bool is_small(uint32_t D, uint32_t H) { return D <= kSmallD && H <= kSmallH; }
__host__ __device__ inline uint32_t groups_of(uint32_t B) { return (B + kGroup - 1) / kGroup; }

// Padded sizes and the places of the weights' packed copies: W1 and W2
// transposed, so that neighbouring units are neighbours, W2 as it is, and the
// vectors; rows of HP floats, zero in the padding.
struct Shape {
    uint32_t D, H, DP, HP;
    __host__ __device__ Shape(uint32_t d, uint32_t h) : D(d), H(h), DP((d + 3) / 4 * 4), HP((h + 15) / 16 * 16) {}
    __host__ __device__ uint32_t w1t() const { return 0; }
    __host__ __device__ uint32_t w2t() const { return DP * HP; }
    __host__ __device__ uint32_t w2() const { return w2t() + HP * HP; }
    __host__ __device__ uint32_t b1() const { return w2() + HP * HP; }
    __host__ __device__ uint32_t b2() const { return b1() + HP; }
    __host__ __device__ uint32_t w3() const { return b2() + HP; }
    __host__ __device__ uint32_t b3() const { return w3() + HP; }
    __host__ __device__ uint32_t packed() const { return b3() + 1; }
};

// Writes parameter i (flat order) to its packed places.
__device__ __forceinline__ void pack_param(const Shape& s, float* packed, uint32_t i, float value) {
    if (i < s.H * s.D) {
        packed[s.w1t() + i % s.D * s.HP + i / s.D] = value;
        return;
    }
    i -= s.H * s.D;
    if (i < s.H) {
        packed[s.b1() + i] = value;
        return;
    }
    i -= s.H;
    if (i < s.H * s.H) {
        packed[s.w2t() + i % s.H * s.HP + i / s.H] = value;
        packed[s.w2() + i / s.H * s.HP + i % s.H] = value;
        return;
    }
    i -= s.H * s.H;
    packed[(i < s.H ? s.b2() + i : i < 2 * s.H ? s.w3() + i - s.H : s.b3())] = value;
}

__global__ void pack_params(const float* p, float* packed, Shape s, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) pack_param(s, packed, i, p[i]);
}

// x (B x D) to [group][DP inputs][32 samples], zero beyond B and D.
__global__ void pack_inputs(const float* x, float* xt, uint32_t B, uint32_t D, uint32_t DP, uint64_t total) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const uint64_t b = t / (DP * kGroup) * kGroup + t % kGroup;
    const uint32_t k = (uint32_t)(t / kGroup % DP);
    xt[t] = b < B && k < D ? x[b * D + k] : 0.f;
}

struct PassArgs {
    const float* packed;
    const float* xt;
    const float* target;
    float* y;                     // forward
    float *a1, *a2, *dz1;         // training: [group][HP][32]
    float *dy, *sq;               // training: [groups * 32]
    uint32_t B;
    Shape s;
};

// Memory no kernel writes while it is read: loads at uniform indexes go through
// the scalar cache.
typedef __attribute__((address_space(4))) const float scalar_float;

// dZ of the second layer: dY through the output unit's weight and the relu.
__device__ __forceinline__ float delta2(float a2, float dy, float w3) { return a2 > 0.f ? 0.f + dy * w3 : 0.f; }

// z[u] += w[k][u] act[k] for k in [0, n): two units of four samples.
__device__ __forceinline__ void layer(f32x4 (&z)[2], const float* w, uint32_t stride, const float* act, uint32_t n) {
#pragma unroll 8
    for (uint32_t k = 0; k < n; ++k) {
        const f32x2 wk = *reinterpret_cast<const f32x2*>(w + k * stride);
        const f32x4 a = *reinterpret_cast<const f32x4*>(act + k * kGroup);
        z[0] += wk.x * a;
        z[1] += wk.y * a;
    }
}

// HP x 4 threads: 8 quads of samples, HP / 2 pairs of units.
template <uint32_t MAXH, bool TRAIN>
__global__ __launch_bounds__(MAXH * 4) void mlp_pass(PassArgs q) {
    __shared__ __align__(16) float s_a[MAXH * kGroup], s_b[MAXH * kGroup];
    __shared__ __align__(16) float s_dy[kGroup];
    const uint32_t HP = q.s.HP, DP = q.s.DP, group = blockIdx.x;
    const uint32_t m = threadIdx.x % 8 * 4, u = threadIdx.x / 8 * 2;  // first sample and unit of this thread's tile
    const uint32_t b = group * kGroup + m;
    const uint64_t at = (uint64_t)group * HP * kGroup + u * kGroup + m;
    bool valid[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) valid[j] = b + j < q.B;
    for (uint32_t t = threadIdx.x; t < DP * kGroup / 4; t += blockDim.x)
        reinterpret_cast<f32x4*>(s_b)[t] = reinterpret_cast<const f32x4*>(q.xt + (uint64_t)group * DP * kGroup)[t];
    __syncthreads();

    f32x4 a1[2], a2[2], z[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) z[j] = (f32x4){} + q.packed[q.s.b1() + u + j];
    layer(z, q.packed + q.s.w1t() + u, HP, s_b + m, DP);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) a1[j][e] = fmaxf(z[j][e], 0.f);
        *reinterpret_cast<f32x4*>(s_a + (u + j) * kGroup + m) = a1[j];
        if (TRAIN) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = valid[e] ? a1[j][e] : 0.f;
            __builtin_nontemporal_store(o, reinterpret_cast<f32x4*>(q.a1 + at + j * kGroup));
        }
        z[j] = (f32x4){} + q.packed[q.s.b2() + u + j];
    }
    __syncthreads();
    layer(z, q.packed + q.s.w2t() + u, HP, s_a + m, HP);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) a2[j][e] = fmaxf(z[j][e], 0.f);
        *reinterpret_cast<f32x4*>(s_b + (u + j) * kGroup + m) = a2[j];
        if (TRAIN) __builtin_nontemporal_store(a2[j], reinterpret_cast<f32x4*>(q.a2 + at + j * kGroup));
    }
    __syncthreads();
    // The output unit, and dY = 2 (y - target) / B: one thread per sample.
    if (threadIdx.x < kGroup) {
        const uint32_t sample = group * kGroup + threadIdx.x;
        float y = q.packed[q.s.b3()];
        scalar_float* w3 = (scalar_float*)(uintptr_t)(q.packed + q.s.w3());
#pragma unroll 16
        for (uint32_t k = 0; k < HP; ++k) y += w3[k] * s_b[k * kGroup + threadIdx.x];
        if (TRAIN) {
            const float d = sample < q.B ? y - q.target[sample] : 0.f;
            const float dy = 2.f * d / (float)q.B;
            s_dy[threadIdx.x] = dy;
            q.dy[sample] = dy;
            q.sq[sample] = d * d;
        } else if (sample < q.B) {
            q.y[sample] = y;
        }
    }
    if (!TRAIN) return;

    // Back through W3 and the second relu, then W2 and the first.
    __syncthreads();
    const f32x4 dy = *reinterpret_cast<const f32x4*>(s_dy + m);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const float w3 = q.packed[q.s.w3() + u + j];
        f32x4 dz;
#pragma unroll
        for (int e = 0; e < 4; ++e) dz[e] = delta2(a2[j][e], dy[e], w3);
        *reinterpret_cast<f32x4*>(s_a + (u + j) * kGroup + m) = dz;
        z[j] = (f32x4){};
    }
    __syncthreads();
    layer(z, q.packed + q.s.w2() + u, HP, s_a + m, HP);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        f32x4 dz;
#pragma unroll
        for (int e = 0; e < 4; ++e) dz[e] = valid[e] && a1[j][e] > 0.f ? z[j][e] : 0.f;
        __builtin_nontemporal_store(dz, reinterpret_cast<f32x4*>(q.dz1 + at + j * kGroup));
    }
}

struct PartArgs {
    const float *packed, *a1, *a2, *dz1, *xt, *dy;
    float* part;  // [chunk][count], parameters' order
    uint32_t B, chunks, jobs;
    uint64_t count;
    Shape s;
};

// Jobs of one chunk, 256 threads each: first over the 2 x 4 tiles of W2's
// gradient (dZ2 x a1), then of W1's (dZ1 x x), then one for W3 and b3. Tile
// (o, i) of a matrix holds rows o and o + R and columns i + C c (half the
// rows, a quarter of the columns apart), so that neighbouring threads read
// neighbouring LDS rows. A matrix's first job also sums its delta rows: the
// bias gradient. (4 x 4 tiles read a third less LDS per product but leave
// half as many waves, two to some SIMDs and none to others; workgroups of 128
// threads stage each group's rows twice as often: 16.2 us each, against 15.7.)
__host__ __device__ inline uint32_t w2_jobs(const Shape& s) {
    return (s.HP / 2 * (s.HP / 4) + kPartThreads - 1) / kPartThreads;
}
__host__ __device__ inline uint32_t w1_jobs(const Shape& s) {
    return (s.HP / 2 * (s.DP / 4) + kPartThreads - 1) / kPartThreads;
}
enum PartKind { kPartW2, kPartW1, kPartW3 };

// A group's rows (contiguous in memory) to registers, and from there to LDS:
// the next group's loads overlap this one's arithmetic.
template <int N>
__device__ __forceinline__ void load_rows(f32x4 (&r)[N], const float* src, uint32_t rows, uint32_t group) {
    const f32x4* p = reinterpret_cast<const f32x4*>(src + (uint64_t)group * rows * kGroup);
#pragma unroll
    for (int n = 0; n < N; ++n)
        if (n * kPartThreads < rows * (kGroup / 4)) {
            const uint32_t t = threadIdx.x + n * kPartThreads;
            r[n] = p[t < rows * (kGroup / 4) ? t : 0];
        }
}
template <int N>
__device__ __forceinline__ void store_rows(float* dst, const f32x4 (&r)[N], uint32_t rows) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const uint32_t t = threadIdx.x + n * kPartThreads;
        if (t < rows * (kGroup / 4)) *reinterpret_cast<f32x4*>(dst + t / (kGroup / 4) * kRow + t % (kGroup / 4) * 4) = r[n];
    }
}

// MAXH: most padded units, which fixes the LDS and the prefetch registers.
template <uint32_t MAXH>
__global__ __launch_bounds__(kPartThreads) void grad_part(PartArgs q) {
    constexpr int N = (MAXH * (kGroup / 4) + kPartThreads - 1) / kPartThreads;
    __shared__ __align__(16) float s_u[MAXH * kRow], s_v[MAXH * kRow];
    // A chunk's jobs run on one XCD (workgroups go to the eight in turn), so
    // its rows are fetched into one L2.
    const uint32_t slot = blockIdx.x / 8;
    const uint32_t chunk = slot / q.jobs * 8 + blockIdx.x % 8;
    if (chunk >= q.chunks) return;
    const uint32_t D = q.s.D, H = q.s.H, HP = q.s.HP, R = HP / 2;
    const uint32_t job = slot % q.jobs, first1 = w2_jobs(q.s), first3 = first1 + w1_jobs(q.s);
    const PartKind kind = job < first1 ? kPartW2 : job < first3 ? kPartW1 : kPartW3;
    const float* u = kind == kPartW1 ? q.dz1 : q.a2;                        // rows: dZ1, or a2 on its way to dZ2 or dY a2
    const float* v = kind == kPartW2 ? q.a1 : kind == kPartW1 ? q.xt : q.dy;  // columns
    const uint32_t vrows = kind == kPartW2 ? HP : kind == kPartW1 ? q.s.DP : 1;
    const uint32_t cols = kind == kPartW2 ? H : kind == kPartW1 ? D : 0;
    const uint32_t tile0 = kind == kPartW2 ? job : kind == kPartW1 ? job - first1 : 0;
    // The parameters' order: W1, b1, W2, b2, W3, b3.
    float* const out = q.part + (uint64_t)chunk * q.count + (kind == kPartW2 ? H * D + H : 0);
    float* const bias = kind == kPartW3 ? out + H * D + H + H * H + H : out + H * cols;
    const uint32_t C = vrows / 4, t = tile0 * kPartThreads + threadIdx.x;
    const uint32_t o = C ? t / C : R, i = C ? t % C : 0;
    const bool has_tile = o < R, has_row = tile0 == 0 && threadIdx.x < HP, has_dy = kind == kPartW3 && threadIdx.x == 0;
    const uint32_t g0 = chunk * (kChunk / kGroup), g1 = min(groups_of(q.B), g0 + kChunk / kGroup);

    float w3[N];  // of the rows this thread stages
    if (kind == kPartW2) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const uint32_t h = (threadIdx.x + n * kPartThreads) / (kGroup / 4);
            w3[n] = h < HP ? q.packed[q.s.w3() + h] : 0.f;
        }
    }
    float acc[2][4] = {}, row = 0.f, sum_dy = 0.f;
    f32x4 ru[N], rv[N], rdy = {};
    load_rows<N>(ru, u, HP, g0);
    load_rows<N>(rv, v, vrows, g0);
    if (kind != kPartW1) rdy = *reinterpret_cast<const f32x4*>(q.dy + g0 * kGroup + threadIdx.x % (kGroup / 4) * 4);
    for (uint32_t g = g0; g < g1; ++g) {
        if (kind != kPartW1) {
#pragma unroll
            for (int n = 0; n < N; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    ru[n][e] = kind == kPartW2 ? delta2(ru[n][e], rdy[e], w3[n]) : rdy[e] * ru[n][e];
        }
        store_rows<N>(s_u, ru, HP);
        store_rows<N>(s_v, rv, vrows);
        __syncthreads();
        if (g + 1 < g1) {
            load_rows<N>(ru, u, HP, g + 1);
            load_rows<N>(rv, v, vrows, g + 1);
            if (kind != kPartW1)
                rdy = *reinterpret_cast<const f32x4*>(q.dy + (g + 1) * kGroup + threadIdx.x % (kGroup / 4) * 4);
        }
        if (has_tile) {
#pragma unroll 2
            for (uint32_t k = 0; k < kGroup; k += 4) {
                f32x4 x[2], y[4];
#pragma unroll
                for (int a = 0; a < 2; ++a) x[a] = *reinterpret_cast<const f32x4*>(s_u + (o + R * a) * kRow + k);
#pragma unroll
                for (int c = 0; c < 4; ++c) y[c] = *reinterpret_cast<const f32x4*>(s_v + (i + C * c) * kRow + k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int c = 0; c < 4; ++c) acc[a][c] += x[a][e] * y[c][e];
            }
        }
        if (has_row) {
#pragma unroll
            for (uint32_t k = 0; k < kGroup; k += 4) {
                const f32x4 x = *reinterpret_cast<const f32x4*>(s_u + threadIdx.x * kRow + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) row += x[e];
            }
        }
        if (has_dy)
            for (uint32_t k = 0; k < kGroup; ++k) sum_dy += s_v[k];
        __syncthreads();
    }
    if (has_tile) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (o + R * a < H && i + C * c < cols) out[(o + R * a) * cols + i + C * c] = acc[a][c];
    }
    if (has_row && threadIdx.x < H) bias[threadIdx.x] = row;
    if (has_dy) bias[H] = sum_dy;
}

// Adds the chunks' rows in increasing chunk and stores the gradients (grads)
// or takes the Adam step. 64 parameters per workgroup: 16 waves bring 256 rows
// to LDS at a time, so the loads are all in flight together, and the first
// wave adds them in order. The last workgroup adds the squared errors: per 256
// samples by halves, then those sums in order.
constexpr uint32_t kSumThreads = 1024;
constexpr uint32_t kSumRows = 256;
__global__ __launch_bounds__(kSumThreads) void grad_sum(const float* part, uint32_t chunks, uint32_t count,
                                                        const float* sq, uint32_t B, float loss_scale, float* loss,
                                                        float* grads, float* p, float* m, float* v, float* packed, Shape s,
                                                        AdamArgs a) {
    constexpr uint32_t kWaves = kSumThreads / 64;
    __shared__ float s_rows[kSumRows][64];
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    float total = 0.f;
    if (blockIdx.x == gridDim.x - 1) {
        float* s_sums = &s_rows[0][0];
        const uint32_t blocks = (B + 255) / 256;
        for (uint32_t r0 = 0; r0 < blocks; r0 += kSumRows * 64) {
            const uint32_t rows = min(kSumRows * 64, blocks - r0);
            for (uint32_t r = wave; r < rows; r += kWaves) {
                float e[4];
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const uint32_t b = (r0 + r) * 256 + 64 * k + lane;
                    e[k] = b < B ? sq[b] : 0.f;
                }
                float t = (e[0] + e[2]) + (e[1] + e[3]);
                for (uint32_t w = 32; w > 0; w >>= 1) t += __shfl_down(t, w);
                if (lane == 0) s_sums[r] = t;
            }
            __syncthreads();
            if (threadIdx.x == 0)
#pragma unroll 8
                for (uint32_t r = 0; r < rows; ++r) total += s_sums[r];
            __syncthreads();
        }
        if (threadIdx.x == 0) *loss = total * loss_scale;
        return;
    }
    const uint32_t i = blockIdx.x * 64 + lane;
    const bool update = wave == 0 && i < count && !grads;
    float pi = 0.f, mi = 0.f, vi = 0.f;  // loaded beside the rows
    if (update) {
        pi = p[i];
        mi = m[i];
        vi = v[i];
    }
    for (uint32_t r0 = 0; r0 < chunks; r0 += kSumRows) {
        const uint32_t rows = min(kSumRows, chunks - r0);
#pragma unroll
        for (uint32_t k = 0; k < kSumRows / kWaves; ++k) {
            const uint32_t r = wave + k * kWaves;
            if (r < rows && i < count) s_rows[r][lane] = part[(uint64_t)(r0 + r) * count + i];
        }
        __syncthreads();
        if (wave == 0)
#pragma unroll 16
            for (uint32_t r = 0; r < rows; ++r) total += s_rows[r][lane];
        __syncthreads();
    }
    if (wave != 0 || i >= count) return;
    if (!update) {
        grads[i] = total;
        return;
    }
    adam_update(pi, mi, vi, total, a);
    p[i] = pi;
    m[i] = mi;
    v[i] = vi;
    pack_param(s, packed, i, pi);
}

}  // namespace

struct gps_mlp {
    uint32_t D = 0, H = 0, max_batch = 0;
    uint64_t count = 0;
    uint64_t step = 0;
    float *params = nullptr, *grads = nullptr, *m = nullptr, *v = nullptr;
    float *x = nullptr, *t = nullptr, *z1 = nullptr, *a1 = nullptr, *z2 = nullptr, *a2 = nullptr, *y = nullptr;
    float *dy = nullptr, *dz2 = nullptr, *dz1 = nullptr, *partial = nullptr, *loss = nullptr;
    float* wpart = nullptr;  // per-chunk weight-gradient partial sums
    bool small = false;      // the three-launch kernels, with a1, a2 and dz1 as [group][HP][32]
    float *packed = nullptr, *xt = nullptr, *sq = nullptr;
    float* curve = nullptr;  // epoch losses of a training call, grown on demand
    uint32_t curve_len = 0;

    float* W1() const { return params; }
    float* b1() const { return params + (uint64_t)H * D; }
    float* W2() const { return b1() + H; }
    float* b2() const { return W2() + (uint64_t)H * H; }
    float* W3() const { return b2() + H; }
    float* b3() const { return W3() + H; }
    float* gW1() const { return grads; }
    float* gb1() const { return grads + (uint64_t)H * D; }
    float* gW2() const { return gb1() + H; }
    float* gb2() const { return gW2() + (uint64_t)H * H; }
    float* gW3() const { return gb2() + H; }
    float* gb3() const { return gW3() + H; }
};

namespace {

uint64_t param_count(uint32_t D, uint32_t H) { return (uint64_t)H * D + H + (uint64_t)H * H + H + H + 1; }

void free_mlp(gps_mlp* m) {
    if (!m) return;
    float* ptrs[] = {m->params, m->grads, m->m, m->v,  m->x,       m->t,    m->z1,   m->a1, m->z2,
                     m->a2,     m->y,     m->dy, m->dz2, m->dz1, m->partial, m->loss, m->wpart,
                     m->packed, m->xt,    m->sq, m->curve};
    for (float* p : ptrs) (void)hipFree(p);
    delete m;
}

template <bool TRAIN>
hipError_t launch_pass(gps_mlp* m, uint32_t B) {
    const Shape s(m->D, m->H);
    const PassArgs q{m->packed, m->xt, m->t, m->y, m->a1, m->a2, m->dz1, m->dy, m->sq, B, s};
    const dim3 grid(groups_of(B)), block(s.HP * 4);
    if (s.HP <= 64)
        hipLaunchKernelGGL((mlp_pass<64, TRAIN>), grid, block, 0, nullptr, q);
    else
        hipLaunchKernelGGL((mlp_pass<kSmallH, TRAIN>), grid, block, 0, nullptr, q);
    return hipGetLastError();
}

// One pass over the staged batch: the loss into `loss`, and the gradients
// into m->grads or, with `adam`, the Adam step.
hipError_t small_step(gps_mlp* m, uint32_t B, float* loss, const AdamArgs* adam) {
    const hipError_t e = launch_pass<true>(m, B);
    if (e != hipSuccess) return e;
    const Shape s(m->D, m->H);
    const uint32_t chunks = chunks_of(B), jobs = w2_jobs(s) + w1_jobs(s) + 1;
    const PartArgs q{m->packed, m->a1, m->a2, m->dz1, m->xt, m->dy, m->wpart, B, chunks, jobs, m->count, s};
    const dim3 grid((chunks + 7) / 8 * 8 * jobs);
    if (s.HP <= 64)
        hipLaunchKernelGGL(grad_part<64>, grid, dim3(kPartThreads), 0, nullptr, q);
    else
        hipLaunchKernelGGL(grad_part<kSmallH>, grid, dim3(kPartThreads), 0, nullptr, q);
    hipLaunchKernelGGL(grad_sum, dim3((uint32_t)((m->count + 63) / 64) + 1), dim3(kSumThreads), 0, nullptr, m->wpart,
                       chunks, (uint32_t)m->count, m->sq, B, 1.f / (float)B, loss, adam ? nullptr : m->grads, m->params, m->m, m->v, m->packed, s, adam ? *adam : AdamArgs{});
    return hipGetLastError();
}

hipError_t forward(gps_mlp* m, uint32_t B) {
    if (m->small) return launch_pass<false>(m, B);
    const uint32_t D = m->D, H = m->H;
    hipLaunchKernelGGL(linear_fwd, grid_of((uint64_t)B * H), dim3(kThreads), 0, nullptr, m->x, m->W1(), m->b1(),
                       m->z1, m->a1, B, D, H, 1);
    hipLaunchKernelGGL(linear_fwd, grid_of((uint64_t)B * H), dim3(kThreads), 0, nullptr, m->a1, m->W2(), m->b2(),
                       m->z2, m->a2, B, H, H, 1);
    hipLaunchKernelGGL(linear_fwd, grid_of(B), dim3(kThreads), 0, nullptr, m->a2, m->W3(), m->b3(), nullptr, m->y,
                       B, H, 1u, 0);
    return hipGetLastError();
}

// dW and db of one layer (Din inputs, Dout outputs) into the flat gradient
// array at dWb, through the per-chunk partials.
void linear_bwd_w(gps_mlp* m, const float* dZ, const float* X, float* dWb, uint32_t B, uint32_t Din, uint32_t Dout) {
    const uint64_t outs = (uint64_t)Dout * Din + Dout;
    const uint32_t chunks = chunks_of(B);
    const dim3 g1((uint32_t)((outs + kThreads - 1) / kThreads), chunks);
    hipLaunchKernelGGL(linear_bwd_w_part, g1, dim3(kThreads), 0, nullptr, dZ, X, m->wpart, B, Din, Dout);
    hipLaunchKernelGGL(linear_bwd_w_sum, grid_of(outs), dim3(kThreads), 0, nullptr, m->wpart, dWb, outs, chunks);
}

// Loss (device scalar at `loss`) and all parameter gradients for the batch in m->x / m->t.
hipError_t loss_and_grads(gps_mlp* m, uint32_t B, float* loss) {
    if (m->small) return small_step(m, B, loss, nullptr);
    const uint32_t D = m->D, H = m->H;
    hipError_t e = forward(m, B);
    if (e != hipSuccess) return e;
    const dim3 gb = grid_of(B);
    hipLaunchKernelGGL(mse_grad, gb, dim3(kThreads), 0, nullptr, m->y, m->t, m->dy, m->partial, B);
    hipLaunchKernelGGL(sum_partials, dim3(1), dim3(64), 0, nullptr, m->partial, gb.x, 1.f / (float)B, loss);
    // layer 3: dz3 = dy
    linear_bwd_w(m, m->dy, m->a2, m->gW3(), B, H, 1u);
    hipLaunchKernelGGL(linear_bwd_x, grid_of((uint64_t)B * H), dim3(kThreads), 0, nullptr, m->dy, m->W3(), m->z2,
                       m->dz2, B, H, 1u);
    // layer 2
    linear_bwd_w(m, m->dz2, m->a1, m->gW2(), B, H, H);
    hipLaunchKernelGGL(linear_bwd_x, grid_of((uint64_t)B * H), dim3(kThreads), 0, nullptr, m->dz2, m->W2(), m->z1,
                       m->dz1, B, H, H);
    // layer 1 (no gradient into x)
    linear_bwd_w(m, m->dz1, m->x, m->gW1(), B, D, H);
    return hipGetLastError();
}

int stage_batch(gps_mlp* m, const float* h_x, const float* h_t, uint32_t batch) {
    if (!m || !h_x || batch == 0) return fail(GPS_ERR_INVALID, "bad MLP arguments");
    if (batch > m->max_batch) return fail(GPS_ERR_TOO_LARGE, "batch %u exceeds max_batch %u", batch, m->max_batch);
    HIP_TRY(hipMemcpy(m->x, h_x, (size_t)batch * m->D * sizeof(float), hipMemcpyHostToDevice));
    if (h_t) HIP_TRY(hipMemcpy(m->t, h_t, (size_t)batch * sizeof(float), hipMemcpyHostToDevice));
    if (m->small) {
        const Shape s(m->D, m->H);
        const uint64_t total = (uint64_t)groups_of(batch) * s.DP * kGroup;
        hipLaunchKernelGGL(pack_inputs, grid_of(total), dim3(kThreads), 0, nullptr, m->x, m->xt, batch, s.D, s.DP, total);
        HIP_TRY(hipGetLastError());
    }
    return GPS_OK;
}

}  // namespace

extern "C" {

uint64_t gps_mlp_param_count(uint32_t in_dim, uint32_t hidden) { return param_count(in_dim, hidden); }

int gps_mlp_create(uint32_t in_dim, uint32_t hidden, uint32_t max_batch, gps_mlp** out) {
    if (!out) return fail(GPS_ERR_INVALID, "null output pointer");
    *out = nullptr;
    if (!in_dim || !hidden || !max_batch || in_dim > 4096 || hidden > 4096)
        return fail(GPS_ERR_INVALID, "bad MLP dimensions");
    if (chunks_of(max_batch) > 65535u)  // the chunk index is the weight-gradient grid's y dimension
        return fail(GPS_ERR_TOO_LARGE, "max_batch %u exceeds %u samples", max_batch, 65535u * kChunk);
    gps_mlp* m = new (std::nothrow) gps_mlp();
    if (!m) return fail(GPS_ERR_INVALID, "out of host memory");
    m->D = in_dim;
    m->H = hidden;
    m->max_batch = max_batch;
    m->count = param_count(in_dim, hidden);
    m->small = is_small(in_dim, hidden);
    const Shape s(in_dim, hidden);
    const uint64_t B = max_batch;
    const uint32_t nblocks = (max_batch + kThreads - 1) / kThreads;
    // Samples and units per activation array: whole groups and padded units
    // for the small networks.
    const uint64_t PB = m->small ? (uint64_t)groups_of(max_batch) * kGroup : B;
    const uint64_t act = PB * (m->small ? s.HP : hidden);
    const uint64_t zs = m->small ? 0 : act;  // what the small kernels do not keep
    struct A {
        float** p;
        uint64_t n;
    } allocs[] = {{&m->params, m->count}, {&m->grads, m->count}, {&m->m, m->count}, {&m->v, m->count},
                  {&m->x, B * in_dim},    {&m->t, B},            {&m->z1, zs},      {&m->a1, act},
                  {&m->z2, zs},           {&m->a2, act},         {&m->y, B},        {&m->dy, PB},
                  {&m->dz2, zs},          {&m->dz1, act},        {&m->partial, nblocks}, {&m->loss, 1},
                  {&m->wpart, (m->small ? m->count : (uint64_t)hidden * std::max(in_dim, hidden) + hidden) *
                                  chunks_of(max_batch)},
                  {&m->packed, m->small ? s.packed() : 0},
                  {&m->xt, m->small ? PB * s.DP : 0},
                  {&m->sq, m->small ? PB : 0}};
    for (auto& a : allocs) {
        if (a.n == 0) continue;
        const hipError_t e = hipMalloc(a.p, a.n * sizeof(float));
        if (e != hipSuccess) {
            free_mlp(m);
            return hip_fail(e, "gps_mlp_create");
        }
    }
    hipError_t e = hipMemset(m->params, 0, m->count * sizeof(float));
    if (e == hipSuccess) e = hipMemset(m->m, 0, m->count * sizeof(float));
    if (e == hipSuccess) e = hipMemset(m->v, 0, m->count * sizeof(float));
    if (e == hipSuccess && m->small) e = hipMemset(m->packed, 0, s.packed() * sizeof(float));
    if (e != hipSuccess) {
        free_mlp(m);
        return hip_fail(e, "gps_mlp_create");
    }
    *out = m;
    return GPS_OK;
}

int gps_mlp_destroy(gps_mlp* m) {
    if (!m) return fail(GPS_ERR_INVALID, "null MLP");
    free_mlp(m);
    return GPS_OK;
}

int gps_mlp_set_params(gps_mlp* m, const float* h_params) {
    if (!m || !h_params) return fail(GPS_ERR_INVALID, "null argument");
    HIP_TRY(hipMemcpy(m->params, h_params, m->count * sizeof(float), hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(m->m, 0, m->count * sizeof(float)));
    HIP_TRY(hipMemset(m->v, 0, m->count * sizeof(float)));
    if (m->small) {
        hipLaunchKernelGGL(pack_params, grid_of(m->count), dim3(kThreads), 0, nullptr, m->params, m->packed,
                           Shape(m->D, m->H), (uint32_t)m->count);
        HIP_TRY(hipGetLastError());
    }
    m->step = 0;
    return GPS_OK;
}

int gps_mlp_get_params(gps_mlp* m, float* h_params) {
    if (!m || !h_params) return fail(GPS_ERR_INVALID, "null argument");
    HIP_TRY(hipMemcpy(h_params, m->params, m->count * sizeof(float), hipMemcpyDeviceToHost));
    return GPS_OK;
}

int gps_mlp_forward(gps_mlp* m, const float* h_x, uint32_t batch, float* h_y) {
    if (!h_y) return fail(GPS_ERR_INVALID, "null output");
    int rc = stage_batch(m, h_x, nullptr, batch);
    if (rc) return rc;
    HIP_TRY(forward(m, batch));
    HIP_TRY(hipMemcpy(h_y, m->y, (size_t)batch * sizeof(float), hipMemcpyDeviceToHost));
    return GPS_OK;
}

int gps_mlp_loss_grad(gps_mlp* m, const float* h_x, const float* h_t, uint32_t batch, float* h_loss,
                      float* h_grad) {
    if (!h_t) return fail(GPS_ERR_INVALID, "null targets");
    int rc = stage_batch(m, h_x, h_t, batch);
    if (rc) return rc;
    HIP_TRY(loss_and_grads(m, batch, m->loss));
    if (h_loss) HIP_TRY(hipMemcpy(h_loss, m->loss, sizeof(float), hipMemcpyDeviceToHost));
    if (h_grad) HIP_TRY(hipMemcpy(h_grad, m->grads, m->count * sizeof(float), hipMemcpyDeviceToHost));
    HIP_TRY(hipDeviceSynchronize());
    return GPS_OK;
}

int gps_mlp_train(gps_mlp* m, const float* h_x, const float* h_t, uint32_t batch, uint32_t epochs, float lr,
                  float weight_decay, float* h_loss_curve) {
    int rc = stage_batch(m, h_x, h_t, batch);
    if (rc) return rc;
    if (!h_t) return fail(GPS_ERR_INVALID, "null targets");
    const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
    // The epoch losses stay on the device until the end (one copy, no
    // per-epoch synchronisation), in a buffer the model keeps between calls.
    if (h_loss_curve && epochs > m->curve_len) {
        (void)hipFree(m->curve);
        m->curve = nullptr;
        m->curve_len = 0;
        HIP_TRY(hipMalloc(&m->curve, (size_t)epochs * sizeof(float)));
        m->curve_len = epochs;
    }
    hipError_t e = hipSuccess;
    for (uint32_t ep = 0; ep < epochs && e == hipSuccess; ++ep) {
        float* const loss = h_loss_curve ? m->curve + ep : m->loss;
        if (!m->small) e = loss_and_grads(m, batch, loss);
        if (e != hipSuccess) break;
        ++m->step;
        const float bc1 = 1.f - std::pow(beta1, (float)m->step);
        const float bc2 = 1.f - std::pow(beta2, (float)m->step);
        const AdamArgs adam{lr, beta1, beta2, eps, weight_decay, bc1, bc2};
        if (m->small) {
            e = small_step(m, batch, loss, &adam);
        } else {
            hipLaunchKernelGGL(adam_step, grid_of(m->count), dim3(kThreads), 0, nullptr, m->params, m->grads, m->m,
                               m->v, m->count, adam);
            e = hipGetLastError();
        }
    }
    if (e == hipSuccess && h_loss_curve && epochs)
        e = hipMemcpy(h_loss_curve, m->curve, (size_t)epochs * sizeof(float), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) return hip_fail(e, "gps_mlp_train");
    return GPS_OK;
}

}  // extern "C"
