// batchnorm_ragged.hip -- the fused batch-norm layer passes (batchnorm.hip) over
// channels whose rows are no whole float4s: spatial % 4 != 0 (13x13, 19x19 and
// 7x7 maps), or a tensor not 16-byte aligned. The per-op sequence moves 56
// bytes an element in 11 to 13 launches; these are memory bound at
//   * 16 (forward) and 20 (backward) bytes an element in one launch where a
//     workgroup holds its whole channel in registers, one float at a time;
//   * 20 and 32 in a reduction pass, its finalisation and an apply pass
//     otherwise (the apply pass streams float4s over the flat tensor and looks
//     each element's channel up in LDS).
// A channel is one workgroup's alone in the first form, so nothing meets and no
// grid has to be resident at once. Loads are one float a lane (a row starts at
// any alignment; 64 lanes read 256 consecutive bytes), enough of them in flight:
// [64,512,13,13] forward 82 -> 19 us, [64,1024,13,13] backward 124 -> 53.
//
// Element results are the per-op sequence's, bit for bit, given the same
// per-channel values, and the backward's sums add the same f32 terms in f64.
// The forward's statistics are batchnorm.hip's shifted sums, with a shift of 0
// where the channel's first element is not finite.
#include "bn_common.hpp"
#include "dkz_hints.hpp"

namespace dkz {
namespace {

template <bool NT>
__device__ __forceinline__ float ld1(const float *p, uint32_t i) {
    return NT ? __builtin_nontemporal_load(p + i) : p[i];
}
template <bool NT>
__device__ __forceinline__ void st1(float *p, uint32_t i, float v) {
    if constexpr (NT) __builtin_nontemporal_store(v, p + i);
    else p[i] = v;
}

__device__ __forceinline__ double shift_of(float first) {
    return fabsf(first) < __builtin_inff() ? (double)first : 0.0;
}

template <int A>
__device__ __forceinline__ void fwd_elem1(float v, const FwdChan &c, float &xn, float &o) {
    xn = (v - c.m) * c.inv;                    // blas.zig:137-146
    o = activate<A>(xn * c.gam + c.bet);       // blas.zig:53-71, activations.zig:107-125
}

__device__ __forceinline__ float bwd_elem1(float d2, float xm, const BwdChan &c, float denom) {
    return (d2 * c.inv + (c.vd2 * xm) / denom) + c.mdn;  // blas.zig:180-204
}

// ---- one launch: workgroup f holds channel f ---------------------------------

// H: bit 0 = input load, bit 1 = x store, bit 2 = x_norm store, bit 3 = output store.
template <int A, int H, int BS, int U>
__global__ __launch_bounds__(BS) void bn_fwd_chan_kernel(const float *input, float *output, float *x, float *x_norm,
                                                         FwdParams p, RedGeom g, FwdFin fin) {
    __shared__ double lds[2 * (BS / kWave)];
    __shared__ FwdChan chan_sh;
    const uint32_t f = blockIdx.x, fbase = f * g.spatial, L = g.chan_len;
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t j = threadIdx.x + u * BS;
        if (j < L) v[u] = ld1<(H & 1) != 0>(input, chan_addr(fbase, j, g));
    }
    const double c = shift_of(input[fbase]);
    double a[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (threadIdx.x + u * BS >= L) continue;
        const double d = (double)v[u] - c;
        a[0] += d;
        a[1] += d * d;
    }
    const Sums<2> sums = block_sums<2, BS>(a, lds);
    if (threadIdx.x == 0) {
        float m, var;
        fin.stats(sums, c, m, var);
        chan_sh = fwd_chan(m, var, p.scales[f], p.biases[f]);
        fin.write(f, m, var);
    }
    __syncthreads();
    const FwdChan ch = chan_sh;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t j = threadIdx.x + u * BS;
        if (j >= L) continue;
        const uint32_t at = chan_addr(fbase, j, g);
        float xn, o;
        fwd_elem1<A>(v[u], ch, xn, o);
        st1<(H & 2) != 0>(x, at, v[u]);
        st1<(H & 4) != 0>(x_norm, at, xn);
        st1<(H & 8) != 0>(output, at, o);
    }
}

// Holds d2 = delta * gradient(y) * scale and x - mean of U elements a lane.
// H: bit 0 = y, bit 1 = delta, bit 2 = x_norm, bit 3 = x loads, bit 4 = delta store.
constexpr int kBwdGroup = 4;  // elements whose four loads are in flight together
template <int A, int H, int BS, int U>
__global__ __launch_bounds__(BS) void bn_bwd_chan_kernel(const float *y, float *delta, const float *x_norm,
                                                         const float *x, BwdParams p, RedGeom g, BwdFin fin) {
    static_assert(U % kBwdGroup == 0, "whole groups");
    constexpr bool kLin = A == kLinear;
    __shared__ double lds[4 * (BS / kWave)];
    __shared__ BwdChan chan_sh;
    const uint32_t f = blockIdx.x, fbase = f * g.spatial, L = g.chan_len;
    const float m = p.mean[f], gam = p.scales[f];
    float d2[U], xm[U];
    double a[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += kBwdGroup) {
        float vy[kBwdGroup], vd[kBwdGroup], vn[kBwdGroup], vx[kBwdGroup];
#pragma unroll
        for (int q = 0; q < kBwdGroup; ++q) {
            const uint32_t j = threadIdx.x + (u0 + q) * BS;
            if (j >= L) continue;
            const uint32_t at = chan_addr(fbase, j, g);
            vd[q] = ld1<(H & 2) != 0>(delta, at);
            vy[q] = kLin ? 0.0f : ld1<(H & 1) != 0>(y, at);
            vn[q] = ld1<(H & 4) != 0>(x_norm, at);
            vx[q] = ld1<(H & 8) != 0>(x, at);
        }
#pragma unroll
        for (int q = 0; q < kBwdGroup; ++q) {
            if (threadIdx.x + (u0 + q) * BS >= L) continue;
            const float d1 = grad_delta<A>(vd[q], vy[q]);
            d2[u0 + q] = d1 * gam;
            xm[u0 + q] = vx[q] - m;
            a[0] += (double)d1;
            a[1] += (double)(d1 * vn[q]);                // blas.zig:96
            a[2] += (double)d2[u0 + q];
            a[3] += (double)(d2[u0 + q] * xm[u0 + q]);   // blas.zig:174
        }
    }
    const Sums<4> sums = block_sums<4, BS>(a, lds);
    if (threadIdx.x == 0) {
        float md, vd;
        fin.values(f, sums, md, vd);
        chan_sh = bwd_chan(p, f, md, vd);
        fin.write(f, sums, md, vd);
    }
    __syncthreads();
    const BwdChan ch = chan_sh;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t j = threadIdx.x + u * BS;
        if (j < L) st1<(H & 16) != 0>(delta, chan_addr(fbase, j, g), bwd_elem1(d2[u], xm[u], ch, p.denom));
    }
}

// ---- two passes -----------------------------------------------------------------

// Chunk k of channel f; K == 1 (FIN): the workgroup finalises its channel.
constexpr int kRaggedUnroll = 8;

template <int BS, bool FIN>
__global__ __launch_bounds__(BS) void bn_stats_ragged_kernel(const float *input, RedGeom g, FwdFin fin, double *partials) {
    __shared__ double lds[2 * (BS / kWave)];
    const uint32_t f = fdiv(blockIdx.x, g.div_k), k = blockIdx.x - f * g.K;
    const uint32_t j0 = k * g.chunk, j1 = min(j0 + g.chunk, g.chan_len), fbase = f * g.spatial;
    const double c = shift_of(input[fbase]);
    double a[2] = {0.0, 0.0};
    for (uint32_t j = j0 + threadIdx.x; j < j1; j += BS * kRaggedUnroll) {
        float v[kRaggedUnroll];
#pragma unroll
        for (int u = 0; u < kRaggedUnroll; ++u)  // past the chunk: its last element again, not added
            v[u] = ld1<(DKZ_HINT_BN_STATS & 1) != 0>(input, chan_addr(fbase, min(j + u * BS, j1 - 1), g));
#pragma unroll
        for (int u = 0; u < kRaggedUnroll; ++u) {
            if (j + u * BS >= j1) continue;
            const double d = (double)v[u] - c;
            a[0] += d;
            a[1] += d * d;
        }
    }
    const Sums<2> r = block_sums<2, BS>(a, lds);
    if constexpr (FIN) {
        if (threadIdx.x == 0) {
            float m, v;
            fin.stats(r, c, m, v);
            fin.write(f, m, v);
        }
    } else {
        store_partials<2, BS>(r, g, f, k, partials);
        if (k == 0 && threadIdx.x == 0) partials[2u * g.div_filters.d * g.K + f] = c;  // = fin.shift[f]
    }
}

template <int A, int BS, bool FIN>
__global__ __launch_bounds__(BS) void bn_bwd_sums_ragged_kernel(const float *y, const float *delta, const float *x_norm,
                                                                const float *x, const float *mean, const float *scales,
                                                                RedGeom g, BwdFin fin, double *partials) {
    constexpr int H = DKZ_HINT_BN_BWD_SUMS, kU = 4;
    constexpr bool kLin = A == kLinear;
    __shared__ double lds[4 * (BS / kWave)];
    const uint32_t f = fdiv(blockIdx.x, g.div_k), k = blockIdx.x - f * g.K;
    const uint32_t j0 = k * g.chunk, j1 = min(j0 + g.chunk, g.chan_len), fbase = f * g.spatial;
    const float m = mean[f], gam = scales[f];
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    for (uint32_t j = j0 + threadIdx.x; j < j1; j += BS * kU) {
        float vy[kU], vd[kU], vn[kU], vx[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const uint32_t at = chan_addr(fbase, min(j + u * BS, j1 - 1), g);
            vd[u] = ld1<(H & 2) != 0>(delta, at);
            vy[u] = kLin ? 0.0f : ld1<(H & 1) != 0>(y, at);
            vn[u] = ld1<(H & 4) != 0>(x_norm, at);
            vx[u] = ld1<(H & 8) != 0>(x, at);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            if (j + u * BS >= j1) continue;
            const float d1 = grad_delta<A>(vd[u], vy[u]), d2 = d1 * gam;
            a[0] += (double)d1;
            a[1] += (double)(d1 * vn[u]);
            a[2] += (double)d2;
            a[3] += (double)(d2 * (vx[u] - m));
        }
    }
    const Sums<4> r = block_sums<4, BS>(a, lds);
    if constexpr (FIN) {
        if (threadIdx.x == 0) fin(f, r);
    } else {
        store_partials<4, BS>(r, g, f, k, partials);
    }
}

// The apply passes: a workgroup's tile of kTile elements spans at most kRows
// rows (spatial >= kMinSpatial), whose channel values it works out once.
constexpr int kApplyUnroll = 4;
constexpr uint32_t kTile = kBlock * kApplyUnroll * 4, kMinSpatial = 4, kRows = kTile / kMinSpatial + 2;

// Row of element e and how far along it e is.
struct RowOf {
    uint32_t row, rem;
    __device__ __forceinline__ RowOf(uint32_t e, const ChanGeom &g) : row(fdiv(e, g.spatial)), rem(e - row * g.spatial.d) {}
};

template <int A, bool TRAIN>
__global__ __launch_bounds__(kBlock) void bn_fwd_apply_ragged_kernel(const float *input, float *output, float *x,
                                                                     float *x_norm, FwdParams p, ChanGeom g, uint32_t n) {
    constexpr int H = DKZ_HINT_BN_FWD_APPLY;
    __shared__ FwdChan slot[kRows];
    const uint32_t nv = n >> 2, e0 = blockIdx.x * kTile, base = (e0 >> 2) + threadIdx.x;
    float4 v[kApplyUnroll];
#pragma unroll
    for (int u = 0; u < kApplyUnroll; ++u)
        if (base + u * kBlock < nv) v[u] = ld4<(H & 1) != 0>(input, base + u * kBlock);
    const uint32_t r0 = fdiv(e0, g.spatial), rows = fdiv(min(e0 + kTile, n) - 1, g.spatial) - r0 + 1;
    for (uint32_t s = threadIdx.x; s < rows; s += kBlock) {
        const uint32_t f = r0 + s - fdiv(r0 + s, g.filters) * g.filters.d;
        slot[s] = fwd_chan(p.mean[f], p.variance[f], p.scales[f], p.biases[f]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kApplyUnroll; ++u) {
        const uint32_t i = base + u * kBlock;
        if (i >= nv) continue;
        const RowOf r(i << 2, g);
        float4 xn, o;
#pragma unroll
        for (int l = 0; l < 4; ++l)
            fwd_elem1<A>(lane(v[u], l), slot[r.row - r0 + (r.rem + l >= g.spatial.d)], lane(xn, l), lane(o, l));
        st4<(H & 2) != 0>(x, i, v[u]);
        if constexpr (TRAIN) st4<(H & 4) != 0>(x_norm, i, xn);
        st4<(H & 8) != 0>(output, i, o);
    }
    // the last n % 4 elements
    const uint32_t e = (nv << 2) + threadIdx.x;
    if (e >= e0 && e < n && e - e0 < kTile) {
        const float t = input[e];
        float xn, o;
        fwd_elem1<A>(t, slot[fdiv(e, g.spatial) - r0], xn, o);
        x[e] = t;
        if constexpr (TRAIN) x_norm[e] = xn;
        output[e] = o;
    }
}

template <int A>
__global__ __launch_bounds__(kBlock) void bn_bwd_apply_ragged_kernel(const float *y, float *delta, const float *x,
                                                                     BwdParams p, ChanGeom g, uint32_t n) {
    constexpr int H = DKZ_HINT_BN_BWD_APPLY;
    constexpr bool kLin = A == kLinear;
    __shared__ BwdChan slot[kRows];
    const uint32_t nv = n >> 2, e0 = blockIdx.x * kTile, base = (e0 >> 2) + threadIdx.x;
    float4 vy[kApplyUnroll], vd[kApplyUnroll], vx[kApplyUnroll];
#pragma unroll
    for (int u = 0; u < kApplyUnroll; ++u) {
        const uint32_t i = base + u * kBlock;
        if (i >= nv) continue;
        vd[u] = ld4<(H & 2) != 0>(delta, i);
        if constexpr (kLin) vy[u] = vd[u];
        else vy[u] = ld4<(H & 1) != 0>(y, i);
        vx[u] = ld4<(H & 4) != 0>(x, i);
    }
    const uint32_t r0 = fdiv(e0, g.spatial), rows = fdiv(min(e0 + kTile, n) - 1, g.spatial) - r0 + 1;
    for (uint32_t s = threadIdx.x; s < rows; s += kBlock) {
        const uint32_t f = r0 + s - fdiv(r0 + s, g.filters) * g.filters.d;
        slot[s] = bwd_chan(p, f, p.mean_delta[f], p.variance_delta[f]);
    }
    __syncthreads();
    const auto elem = [&](float fy, float fd, float fx, const BwdChan &c) {
        return bwd_elem1(grad_delta<A>(fd, fy) * c.gam, fx - c.m, c, p.denom);
    };
#pragma unroll
    for (int u = 0; u < kApplyUnroll; ++u) {
        const uint32_t i = base + u * kBlock;
        if (i >= nv) continue;
        const RowOf r(i << 2, g);
        float4 o;
#pragma unroll
        for (int l = 0; l < 4; ++l)
            lane(o, l) = elem(lane(vy[u], l), lane(vd[u], l), lane(vx[u], l), slot[r.row - r0 + (r.rem + l >= g.spatial.d)]);
        st4<(H & 8) != 0>(delta, i, o);
    }
    const uint32_t e = (nv << 2) + threadIdx.x;
    if (e >= e0 && e < n && e - e0 < kTile)
        delta[e] = elem(kLin ? 0.0f : y[e], delta[e], x[e], slot[fdiv(e, g.spatial) - r0]);
}

// Rows of one to three floats: neighbouring channels share every line, and a
// workgroup per channel fetches and writes a line for each float. The tensor
// has to be small enough that the lines stay in L2: forward / backward us
// against the per-op sequence, [256,1000,1] 24 / 26 against 43 / 65, [128,4096,1]
// (2 MB) 47 / 53 against 53 / 95, [2048,2048,1] 358 / 407 against 127 / 193.
constexpr uint32_t kMaxThin = 1u << 19;
inline bool chan_fits(const Shape &sh, uint32_t most) {
    return sh.B * sh.S <= most && (sh.S >= kMinSpatial || sh.n <= kMaxThin);
}

// ---- host -------------------------------------------------------------------------

// A reduction pass over K chunks a channel (partials and a finalize launch),
// or one workgroup a channel.
template <int NS, class Fin, class KFin, class KPart, class... Args>
int run_sums(const char *name, const RedGeom &g, uint32_t F, const Fin &fin, KFin kfin, KPart kpart, Args... args) {
    if (g.K == 1) return launch(name, kfin, dim3(F), dim3(kWideBlock), args..., g, fin, (double *)nullptr);
    Scratch sc{};
    DKZ_TRY(device_scratch(&sc));
    DKZ_TRY(launch(name, kpart, dim3(F * g.K), dim3(kBlock), args..., g, fin, sc.partials));
    return launch(name, bn_finalize_kernel<NS, Fin>, dim3(div_up(F, kBlock / kWave)), dim3(kBlock), fin,
                  (const double *)sc.partials, F, g.K);
}

// Whether the apply passes take a tensor: rows of at least kMinSpatial,
// float4s over the flat tensor.
inline bool apply_fits(const Shape &sh, bool aligned) { return aligned && sh.S >= kMinSpatial; }

// Everything cached but the backward's delta store: rows share lines with their
// neighbours' rows, which nontemporal accesses fetch and write twice.
// [64,512,13,13] / [64,1024,7,7] forward 26.3 / 23.0 us with nontemporal loads and
// x, x_norm stores, 19.0 / 14.4 cached; backward 29.2 / 24.2 all nontemporal,
// 27.4 / 20.0 all cached, 25.7 / 19.5 so.
constexpr int kFwdHint = 0, kBwdHint = 16;

// Tensors past this run the forward in two passes, whose float4 stores make up
// for reading the input twice: [64,512,13,13] (22 MB) 19.2 us in one launch, 23.5
// in two passes, [64,1024,13,13] (44 MB) 54.2 and 41.7, [128,1024,13,13] 108 and
// 84. The backward stores one tensor, not three, and stays ahead in one
// launch: 23.1 / 52.7 / 104 us against 37.7 / 65.8 / 126.
constexpr uint32_t kMaxOneLaunch = 1u << 23;

template <int A, int BS, int U>
int fwd_chan_launch(const FwdArgs &a, const RedGeom &g, const FwdFin &fin) {
    const FwdParams p{a.mean, a.variance, a.scales, a.biases};
    return launch("batchnorm_forward", bn_fwd_chan_kernel<A, kFwdHint, BS, U>, dim3(a.sh.F), dim3(BS), a.input,
                  a.output, a.x, a.x_norm, p, g, fin);
}

template <int A>
bool forward(const FwdArgs &a, int *rc) {
    const Shape &sh = a.sh;
    const uint32_t L = sh.B * sh.S;
    const ChanGeom cg{make_fastdiv(sh.S), make_fastdiv(sh.F)};
    const dim3 grid(div_up(sh.n, kTile)), block(kBlock);
    const bool apply = apply_fits(sh, aligned16(a.input) && aligned16(a.output) && aligned16(a.x) &&
                                          (!a.train || aligned16(a.x_norm)));
    if (!a.train) {
        if (!apply) return false;
        const FwdParams p{a.rolling_mean, a.rolling_variance, a.scales, a.biases};
        *rc = launch("batchnorm_forward_apply", bn_fwd_apply_ragged_kernel<A, false>, grid, block, a.input, a.output, a.x,
                     a.x_norm, p, cg, sh.n);
        return true;
    }
    FwdFin fin{nullptr, a.mean, a.variance, a.rolling_mean, a.rolling_variance, (double)L, 1.0f / (float)L,
               1.0f / (float)(L - 1u)};
    // The channel in one workgroup's registers where it fits (the smallest
    // workgroup that holds it), except for the largest tensors. With few
    // channels that leaves CUs idle, but is well ahead of the per-op sequence at
    // every count: [32,F,75,75] forward 35.5 / 50.5 / 76.9 / 127 / 246 us in the
    // sequence and 9.8 / 15.5 / 26.9 / 41.8 / 84.1 so, backward 31.5 / 49.2 / 69.8
    // / 121 / 201 and 12.8 / 22.1 / 40.1 / 67.2 / 123, for F = 1, 16, 32, 64, 128;
    // [1,F,207,207] forward 39 and 16 to 19 us for F up to 64.
    const RedGeom whole = make_red_geom(sh.F, sh.S, L, 1, false);
    if (chan_fits(sh, 64 * 1024) && (sh.n <= kMaxOneLaunch || !apply)) {
        if (L <= 4 * 256) *rc = fwd_chan_launch<A, 256, 4>(a, whole, fin);
        else if (L <= 4 * 1024) *rc = fwd_chan_launch<A, 1024, 4>(a, whole, fin);
        else if (L <= 12 * 1024) *rc = fwd_chan_launch<A, 1024, 12>(a, whole, fin);
        else if (L <= 32 * 1024) *rc = fwd_chan_launch<A, 1024, 32>(a, whole, fin);
        else *rc = fwd_chan_launch<A, 1024, 64>(a, whole, fin);
        return true;
    }
    if (!apply) return false;
    const RedGeom g = make_red_geom(sh.F, sh.S, L, pick_split(sh.F, L, 1, 3), false);
    if (g.K > 1) {
        Scratch sc{};
        *rc = device_scratch(&sc);
        if (*rc != 0) return true;
        fin.shift = sc.partials + 2u * sh.F * g.K;  // after the partials (pick_split was asked for three sums)
    }
    *rc = run_sums<2>("batchnorm_forward_stats", g, sh.F, fin, bn_stats_ragged_kernel<kWideBlock, true>,
                      bn_stats_ragged_kernel<kBlock, false>, a.input);
    if (*rc != 0) return true;
    const FwdParams p{a.mean, a.variance, a.scales, a.biases};
    *rc = launch("batchnorm_forward_apply", bn_fwd_apply_ragged_kernel<A, true>, grid, block, a.input, a.output, a.x,
                 a.x_norm, p, cg, sh.n);
    return true;
}

template <int A, int BS, int U>
int bwd_chan_launch(const BwdArgs &a, const BwdParams &p, const RedGeom &g, const BwdFin &fin) {
    return launch("batchnorm_backward", bn_bwd_chan_kernel<A, kBwdHint, BS, U>, dim3(a.sh.F), dim3(BS), a.y,
                  a.delta, a.x_norm, a.x, p, g, fin);
}

template <int A>
bool backward(const BwdArgs &a, int *rc) {
    const Shape &sh = a.sh;
    const uint32_t L = sh.B * sh.S;
    const BwdFin fin{a.variance, a.bias_updates, a.scale_updates, a.mean_delta, a.variance_delta};
    const BwdParams p{a.mean, a.variance, a.mean_delta, a.variance_delta, a.scales, (float)((uint64_t)sh.S * (uint64_t)sh.B)};
    const RedGeom whole = make_red_geom(sh.F, sh.S, L, 1, false);
    if (chan_fits(sh, 32 * 1024)) {
        if (L <= 4 * 256) *rc = bwd_chan_launch<A, 256, 4>(a, p, whole, fin);
        else if (L <= 4 * 1024) *rc = bwd_chan_launch<A, 1024, 4>(a, p, whole, fin);
        else if (L <= 12 * 1024) *rc = bwd_chan_launch<A, 512, 24>(a, p, whole, fin);
        else *rc = bwd_chan_launch<A, 1024, 32>(a, p, whole, fin);
        return true;
    }
    const bool aligned = aligned16(a.delta) && aligned16(a.x) && (A == kLinear || aligned16(a.y));
    if (!apply_fits(sh, aligned)) return false;
    const RedGeom g = make_red_geom(sh.F, sh.S, L, pick_split(sh.F, L, A == kLinear ? 3 : 4, 4), false);
    *rc = run_sums<4>("batchnorm_backward_sums", g, sh.F, fin, bn_bwd_sums_ragged_kernel<A, kWideBlock, true>,
                      bn_bwd_sums_ragged_kernel<A, kBlock, false>, a.y, (const float *)a.delta, a.x_norm, a.x, a.mean,
                      a.scales);
    if (*rc != 0) return true;
    const ChanGeom cg{make_fastdiv(sh.S), make_fastdiv(sh.F)};
    *rc = launch("batchnorm_backward_apply", bn_bwd_apply_ragged_kernel<A>, dim3(div_up(sh.n, kTile)), dim3(kBlock), a.y,
                 a.delta, a.x, p, cg, sh.n);
    return true;
}

typedef bool (*FwdFn)(const FwdArgs &, int *);
typedef bool (*BwdFn)(const BwdArgs &, int *);
template <int... As>
struct RaggedTables {
    static constexpr FwdFn fwd[] = {forward<As>...};
    static constexpr BwdFn bwd[] = {backward<As>...};
};
using Tables = RaggedTables<0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13>;

}  // namespace

bool bn_forward_ragged(int activation, const FwdArgs &a, int *rc) { return Tables::fwd[activation](a, rc); }
bool bn_backward_ragged(int activation, const BwdArgs &a, int *rc) { return Tables::bwd[activation](a, rc); }

}  // namespace dkz
