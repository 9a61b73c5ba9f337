// bn_common.hpp -- what the batch-norm layer passes share (batchnorm.hip,
// batchnorm_ragged.hip): per-channel values and their finalisation, workgroup
// sums, and the element expressions' channel parts.
#pragma once

#include "dkz_channel.hpp"

namespace dkz {

struct Shape {
    uint32_t B, F, S, n;
};

struct FwdArgs {
    Shape sh;
    bool train;
    const float *input;
    float *output, *x, *x_norm, *mean, *variance, *rolling_mean, *rolling_variance;
    const float *scales, *biases;
};

struct BwdArgs {
    Shape sh;
    const float *y;
    float *delta;
    const float *x, *x_norm, *mean, *variance, *scales;
    float *bias_updates, *scale_updates, *mean_delta, *variance_delta;
};

namespace {

constexpr float kMomentum = 0.99f;          // rolling_momentum, batchnorm.zig:16 (f32)
constexpr float kAlpha = 1.0f - kMomentum;  // batchnorm.zig:141: an f32 subtraction, exact

template <int NS>
struct Sums {
    double s[NS];
};

// NS sums over a BS-thread workgroup; the result is valid in wave 0. Each
// wave's sums go through LDS (lds holds NS * BS/64 doubles) and wave 0 adds
// them with one more DPP reduction, so the order is fixed by the shape.
template <int NS, int BS>
__device__ __forceinline__ Sums<NS> block_sums(const double (&a)[NS], double *lds) {
    constexpr int W = BS / kWave;
    const int w = threadIdx.x / kWave, l = threadIdx.x & (kWave - 1);
    Sums<NS> r;
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        const double v = wave_sum(a[q]);
        if (l == 0) lds[q * W + w] = v;
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
        for (int q = 0; q < NS; ++q) r.s[q] = wave_sum(l < W ? lds[q * W + l] : 0.0);
    }
    return r;
}

// Partial sums of workgroup (f, k) go to partials[(q*F + f)*K + k].
template <int NS, int BS>
__device__ __forceinline__ void store_partials(const Sums<NS> &r, const RedGeom &g, uint32_t f, uint32_t k,
                                               double *partials) {
    if (threadIdx.x == 0) {
        const uint32_t F = g.div_filters.d;
#pragma unroll
        for (int q = 0; q < NS; ++q) partials[((uint32_t)q * F + f) * g.K + k] = r.s[q];
    }
}

// Second launch: one wave per channel adds its K partials of each sum in
// index order, then finalises.
template <int NS, class Fin>
__global__ __launch_bounds__(kBlock) void bn_finalize_kernel(Fin fin, const double *partials, uint32_t F,
                                                             uint32_t K) {
    const uint32_t f = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (f >= F) return;  // whole waves leave together
    const uint32_t l = threadIdx.x & (kWave - 1);
    Sums<NS> r;
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        const double *p = partials + ((uint64_t)q * F + f) * K;
        double s = 0.0;
        for (uint32_t i = l; i < K; i += kWave) s += p[i];
        r.s[q] = wave_sum(s);
    }
    if (l == 0) fin(f, r);
}

// mean, variance and the rolling averages of channel f from s1 = sum(x - c),
// s2 = sum((x - c)^2) over its n elements, c = the channel's first element.
// The split statistics pass stores c beside the partials (shift[f]): the
// apply pass may overwrite the input in place before every workgroup has
// finalised.
struct FwdFin {
    const double *shift;
    float *mean, *variance, *rolling_mean, *rolling_variance;
    double n;
    float mean_scale;  // 1/(B*S) in f32 (blas.zig:107)
    float var_scale;   // 1/(B*S - 1) in f32 (blas.zig:122)
    __device__ void stats(const Sums<2> &r, double c, float &m, float &v) const {
        const double s1 = r.s[0], s2 = r.s[1];
        m = (float)(n * c + s1) * mean_scale;  // blas.zig:114: sum * (1/(B*S))
        const double dm = (c + s1 / n) - (double)m;
        double m2 = s2 - s1 * (s1 / n);
        m2 = m2 > 0.0 ? m2 : 0.0;
        v = (float)(m2 + n * dm * dm) * var_scale;  // blas.zig:133
    }
    // met == false (a one-launch pass whose channel barrier gave up): the
    // batch statistics are written (NaN) but the rolling averages, which
    // carry over to the next call, are left as they were.
    __device__ void write(uint32_t f, float m, float v, bool met = true) const {
        mean[f] = m;
        variance[f] = v;
        if (!met) return;
        // batchnorm.zig:140-143: scal(0.99) then axpy(1 - 0.99) -- axpy is an fma (blas.zig:22)
        rolling_mean[f] = __builtin_fmaf(kAlpha, m, rolling_mean[f] * kMomentum);
        rolling_variance[f] = __builtin_fmaf(kAlpha, v, rolling_variance[f] * kMomentum);
    }
    __device__ void operator()(uint32_t f, const Sums<2> &r) const {  // after a split pass
        float m, v;
        stats(r, shift[f], m, v);
        write(f, m, v);
    }
};

struct FwdParams {
    const float *mean, *variance, *scales, *biases;
};

// What the forward apply pass needs of channel f.
struct FwdChan {
    float m, inv, gam, bet;
};

__device__ __forceinline__ FwdChan fwd_chan(float m, float v, float gam, float bet) {
    return {m, 1.0f / (sqrtf(v) + 1e-6f), gam, bet};  // blas.zig:141-143
}

// Per channel: s0 = sum(d1), s1 = sum(d1 * x_norm), s2 = sum(d2),
// s3 = sum(d2 * (x - m)), where d1 = delta * gradient(y) (activations.zig:
// 127-143) and d2 = d1 * scale (the scale_bias on delta, batchnorm.zig:165).
struct BwdFin {
    const float *variance;
    float *bias_updates, *scale_updates, *mean_delta, *variance_delta;
    __device__ void values(uint32_t f, const Sums<4> &r, float &md, float &vd) const {
        const float v = variance[f];
        md = (float)r.s[2] * (-1.0f / sqrtf(v + 1e-5f));            // blas.zig:155
        vd = ((float)r.s[3] * -0.5f) * pow_m1p5(v + 1e-5f);          // blas.zig:176
    }
    // met == false (a one-launch pass whose channel barrier gave up):
    // mean_delta and variance_delta are written (NaN), but nothing is added
    // to the updates, which accumulate across calls.
    __device__ void write(uint32_t f, const Sums<4> &r, float md, float vd, bool met = true) const {
        if (met) {
            bias_updates[f] = bias_updates[f] + (float)r.s[0];   // blas.zig:79
            scale_updates[f] = scale_updates[f] + (float)r.s[1]; // blas.zig:98
        }
        mean_delta[f] = md;
        variance_delta[f] = vd;
    }
    __device__ void operator()(uint32_t f, const Sums<4> &r) const {
        float md, vd;
        values(f, r, md, vd);
        write(f, r, md, vd);
    }
};

template <int A>
__device__ __forceinline__ float grad_delta(float d, float y) {
    if constexpr (A == kLinear) return d;  // activations.zig:129: linear leaves delta alone
    else return d * gradient<A>(y);
}

struct BwdParams {
    const float *mean, *variance, *mean_delta, *variance_delta, *scales;
    float denom;  // f32(spatial * batch), blas.zig:191
};

// What the backward apply pass needs of channel f.
struct BwdChan {
    float m, inv, vd2, mdn, gam;
};

__device__ __forceinline__ BwdChan bwd_chan(const BwdParams &p, uint32_t f, float md, float vd) {
    return {p.mean[f], 1.0f / sqrtf(p.variance[f] + 1e-5f), vd * 2.0f, md / p.denom, p.scales[f]};
}

// delta = d2 * inv + ((vd * 2) * (x - m)) / N + md / N (blas.zig:180-204) on
// d2 = delta * gradient(y) * scale.
}  // namespace

// batchnorm_ragged.hip: the passes over tensors whose channel rows are no whole
// float4s (spatial % 4 != 0, or a tensor not 16-byte aligned). Return true with
// the status in *rc, or false, launching nothing, for a call left to the per-op
// sequence.
bool bn_forward_ragged(int activation, const FwdArgs &a, int *rc);
bool bn_backward_ragged(int activation, const BwdArgs &a, int *rc);

}  // namespace dkz
