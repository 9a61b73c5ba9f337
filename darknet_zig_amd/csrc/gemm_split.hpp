// gemm_split.hpp -- the matrix-product kernel behind dkz_gemm and the
// convolution entry points (gemm.hip): fp32 products on the bf16 matrix cores.
//
// An fp32 value is the sum of three bf16 values, x = h + m + l (8 significant
// bits each, rounded to nearest, so 24 bits in all): exact for |x| >= 2^-109.
// A product of two such sums keeps six of its nine terms,
//     hh | hm + mh + mm + hl + lh,
// the rest being below 2^-25 of it. v_mfma_f32_32x32x16_bf16 forms the
// products exactly and adds them in fp32 with round to nearest. hh has an
// accumulator of its own and the five small terms another, so the large one is
// rounded once per 16 k (the fp32 matrix instruction rounds it at every k):
// over K = 32 .. 9216 the relative error against f64 is 0.36e-7 .. 6.4e-7 where
// v_mfma_f32_32x32x2_f32 leaves 1e-7 .. 1.7e-6 (normal, leaky and positive
// data). Six bf16 products cost 6/16 of the fp32 instruction's time.
//
// Where the split is not exact the tile is computed again with
// v_mfma_f32_32x32x2_f32 from the same loads (redo): when an accumulator is
// not finite (an infinity, a NaN, a value that rounds to a bf16 infinity: its
// l is a NaN) or when all of a thread's share of some row is tiny (its largest
// magnitude within (0, 2^-85)). Infinities, NaNs and tiny operands so give
// what fp32 products give.
//
// A workgroup of four waves owns a BM x BN tile of C, each wave a quarter of
// it. K advances in slabs of 16: each thread holds its share of the next slab
// in registers while the waves run the current one's MFMAs out of LDS, then
// splits it and stores the three planes to the other LDS buffer: one barrier a
// slab. A plane is kept as [k half][row][8 k], so a lane's operand (eight
// consecutive k of its row) is one 128-bit read, and the 32 rows a half wave
// reads are contiguous; halves sit 64 bytes off a multiple of 128 so the stores
// of both halves fall in distinct banks.
#pragma once

#include <type_traits>

#include "dkz_device.hpp"
#include "dkz_internal.hpp"

namespace dkz {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kBK = 16;
constexpr int kGroupM = 8;
constexpr int kXcds = 8;
constexpr int kPlanes = 3;
constexpr int kF32Pitch = kBK + 4;  // LDS row pitch of the fp32 pass, in words
constexpr float kTiny = 0x1p-85f;

// LDS words of one half (8 k) of a plane of R rows, and of an operand's slab.
template <int R>
constexpr int half_words() { return R * 4 + 16; }
template <int R>
constexpr int slab_words() { return kPlanes * 2 * half_words<R>(); }

// Operand kinds. kRowMajor: rows along the tile dimension, k contiguous (A
// row-major, B transposed). kColMajor: k along the rows, the tile dimension
// contiguous (A transposed, B row-major), also the (image, position) columns of
// a 1x1 convolution.
enum Operand { kRowMajor, kColMajor };

struct SplitArgs {
    const float *a;
    const float *b;
    float *c;
    float *partial;  // splits > 1: [splits][m][n] partial tiles
    uint32_t m, n, k, lda, ldb, ldc;
    float alpha, beta;
    uint32_t tiles_m, tiles_n, splits, k_chunk;
    // Batched launches (z = blockIdx.y): A at a + (z % zgroups) * a_z, B at
    // b + z * b_z, C at c + z * c_z.
    uint32_t zgroups;
    uint64_t a_z, b_z, c_z;
    // Columns over (image, position): npos positions per image (0: one matrix),
    // element strides from one image to the next of B and C.
    uint32_t npos, b_img, c_img;
    FastDiv div_npos;
};

__device__ __forceinline__ void tile_of(uint32_t w, const SplitArgs &g, uint32_t &tm, uint32_t &tn, uint32_t &split) {
    const uint32_t tiles = g.tiles_m * g.tiles_n;
    const uint32_t total = tiles * g.splits;
    uint32_t t = w;
    if (total % kXcds == 0) t = (w % kXcds) * (total / kXcds) + w / kXcds;
    split = t / tiles;
    t -= split * tiles;
    const uint32_t per_group = kGroupM * g.tiles_n;
    const uint32_t first_m = (t / per_group) * kGroupM;
    const uint32_t gsize = g.tiles_m - first_m < (uint32_t)kGroupM ? g.tiles_m - first_m : (uint32_t)kGroupM;
    const uint32_t in_group = t % per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// x and y as three packed bf16 pairs (x in the low half).
struct Split2 {
    uint32_t w[kPlanes];
};
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
    const f32x2 v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// x minus a half of the packed pair h: one v_dot2_f32_bf16 with (-1, 0) or
// (0, -1), exact (the difference is a float), where unpacking the half and
// subtracting takes two instructions.
__device__ __forceinline__ float minus_half(uint32_t h, uint32_t sel, float x) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, h), __builtin_bit_cast(bf16x2, sel), x, false);
}
__device__ __forceinline__ Split2 split2(float x, float y) {
    // In scalar registers: as a literal, (-1, 0) becomes the inline constant
    // -1 of both halves.
    uint32_t lo, hi;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(lo));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(hi));
    Split2 s;
    s.w[0] = pack_bf16(x, y);
    x = minus_half(s.w[0], lo, x);
    y = minus_half(s.w[0], hi, y);
    s.w[1] = pack_bf16(x, y);
    x = minus_half(s.w[1], lo, x);
    y = minus_half(s.w[1], hi, y);
    s.w[2] = pack_bf16(x, y);
    return s;
}

// Largest magnitude seen in one row's share; tiny() says the split loses bits.
struct RowMax {
    float mx = 0.0f;
    __device__ __forceinline__ void see(float x, float y) { mx = fmaxf(fmaxf(mx, fabsf(x)), fabsf(y)); }
    __device__ __forceinline__ bool tiny() const { return mx > 0.0f && mx < kTiny; }
};

// ---- operand loaders: `load` takes a whole slab, `load_tail` one that ends at
// kend (missing k read as 0); rows past the operand repeat its last row, whose
// results are not stored. `store` writes the planes, `store_f32` the fp32 slab.

template <int R>
struct RowLoad {
    static constexpr int kL = R * kBK / 4 / kBlock;  // float4s per thread
    const float *p[kL];
    float4 v[kL];
    RowMax mx[kL];

    __device__ __forceinline__ void init(const float *base, uint32_t ld, uint32_t r0, uint32_t rows, int tid) {
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const uint32_t f = tid + l * kBlock, r = f / 4 < rows ? f / 4 : rows - 1;
            p[l] = base + (size_t)(r0 + r) * ld + 4 * (f % 4);
        }
    }
    // One 16-byte load whatever the alignment (global loads need 4).
    __device__ __forceinline__ void load(uint32_t k0) {
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const f32x4u t = *reinterpret_cast<const f32x4u *>(p[l] + k0);
            v[l] = make_float4(t.x, t.y, t.z, t.w);
        }
    }
    __device__ __forceinline__ void load_tail(uint32_t k0, uint32_t kend, int tid) {
        const uint32_t kk = k0 + 4 * (tid % 4);
#pragma unroll
        for (int l = 0; l < kL; ++l)
#pragma unroll
            for (int j = 0; j < 4; ++j) ::dkz::lane(v[l], j) = kk + j < kend ? p[l][k0 + j] : 0.0f;
    }
    __device__ __forceinline__ void store(uint32_t *s, int tid) {
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const int f = tid + l * kBlock, r = f / 4, q = f % 4;
            const Split2 x = split2(v[l].x, v[l].y), y = split2(v[l].z, v[l].w);
            mx[l].see(v[l].x, v[l].y);
            mx[l].see(v[l].z, v[l].w);
            uint32_t *d = s + (q >> 1) * half_words<R>() + r * 4 + (q & 1) * 2;
#pragma unroll
            for (int u = 0; u < kPlanes; ++u)
                *reinterpret_cast<uint2 *>(d + u * 2 * half_words<R>()) = make_uint2(x.w[u], y.w[u]);
        }
    }
    __device__ __forceinline__ void store_f32(float *s, int tid) const {
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const int f = tid + l * kBlock;
            *reinterpret_cast<float4 *>(s + (f / 4) * kF32Pitch + 4 * (f % 4)) = v[l];
        }
    }
    __device__ __forceinline__ bool tiny() const {
        bool t = false;
#pragma unroll
        for (int l = 0; l < kL; ++l) t |= mx[l].tiny();
        return t;
    }
};

// One row of the tile and kT consecutive k of each slab per thread: a wave's
// loads of one k are 64 consecutive elements, its k the same in every lane
// (scalar address arithmetic), whatever the alignment.
template <int R>
struct ColBase {
    static constexpr int kT = R * kBK / kBlock;
    float v[kT];
    RowMax mx;
    uint32_t kq;  // wave-uniform: this wave's k start at kq * kT of the slab

    __device__ __forceinline__ void store(uint32_t *s, int tid) {
        Split2 w[kT / 2];
#pragma unroll
        for (int j = 0; j < kT / 2; ++j) {
            w[j] = split2(v[2 * j], v[2 * j + 1]);
            mx.see(v[2 * j], v[2 * j + 1]);
        }
        const int r = tid % R;
#pragma unroll
        for (int u = 0; u < kPlanes; ++u) {
            uint32_t *d = s + u * 2 * half_words<R>() + r * 4;
            if constexpr (kT == 8)
                *reinterpret_cast<uint4 *>(d + kq * half_words<R>()) = make_uint4(w[0].w[u], w[1].w[u], w[2].w[u], w[3].w[u]);
            else
                *reinterpret_cast<uint2 *>(d + (kq >> 1) * half_words<R>() + (kq & 1) * 2) = make_uint2(w[0].w[u], w[1].w[u]);
        }
    }
    __device__ __forceinline__ void store_f32(float *s, int tid) const {
        float *d = s + (tid % R) * kF32Pitch + kq * kT;
#pragma unroll
        for (int j = 0; j < kT; j += 4) *reinterpret_cast<float4 *>(d + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
    }
    __device__ __forceinline__ bool tiny() const { return mx.tiny(); }
};

template <int R>
struct ColLoad : ColBase<R> {
    using ColBase<R>::kT;
    using ColBase<R>::v;
    using ColBase<R>::kq;
    const float *base;  // wave-uniform
    uint32_t off, ld;   // this lane's byte offset

    // g.npos != 0: the columns run over (image, position).
    __device__ __forceinline__ void init(const float *b, uint32_t ld_, uint32_t r0, uint32_t rows, int tid,
                                         const SplitArgs &g, bool span) {
        kq = __builtin_amdgcn_readfirstlane(tid / R);
        ld = ld_;
        const uint32_t r = (uint32_t)(tid % R) < rows ? tid % R : rows - 1;
        if (span) {
            const uint32_t i0 = fdiv(r0, g.div_npos), i = fdiv(r0 + r, g.div_npos);
            base = b + (size_t)i0 * g.b_img;
            off = 4 * ((i - i0) * g.b_img + (r0 + r - i * g.npos));
        } else {
            base = b + r0;
            off = 4 * r;
        }
    }
    __device__ __forceinline__ const float *at(uint32_t k) const { return base + (size_t)k * ld; }
    __device__ __forceinline__ float get(const float *row) const {
        return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(row) + off);
    }
    __device__ __forceinline__ void load(uint32_t k0) {
        const float *row = at(k0 + kq * kT);
#pragma unroll
        for (int j = 0; j < kT; ++j, row += ld) v[j] = get(row);
    }
    __device__ __forceinline__ void load_tail(uint32_t k0, uint32_t kend) {
        const uint32_t kk = k0 + kq * kT;
#pragma unroll
        for (int j = 0; j < kT; ++j) v[j] = kk + j < kend ? get(at(kk + j)) : 0.0f;
    }
};

// C(i, j) = beta-applied C + alpha * s (gemm.zig:121-131: beta == 0 clears C,
// NaN included).
__device__ __forceinline__ float gemm_out(const float *cp, float s, float alpha, float beta) {
    float cv = 0.0f;
    if (beta != 0.0f) cv = (beta == 1.0f) ? *cp : *cp * beta;
    return cv + alpha * s;
}

// Interleaves a step's VALU work with its MFMAs (each occupies the matrix core
// for the time of eight VALU instructions).
#ifndef DKZ_SPLIT_VALU
#define DKZ_SPLIT_VALU 4
#endif
#ifndef DKZ_SPLIT_SCHED
#define DKZ_SPLIT_SCHED()                                     \
    do {                                                      \
        _Pragma("unroll") for (int i_ = 0; i_ < 6 * TM * TN; ++i_) { \
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   \
            __builtin_amdgcn_sched_group_barrier(0x002, DKZ_SPLIT_VALU, 0);   \
        }                                                     \
    } while (0)
#endif

// Waves a SIMD should hold: the accumulators of a 64x64 wave tile (128
// registers) leave room for two, smaller tiles for more.
template <int BM, int BN>
constexpr int min_waves() { return BM * BN >= 128 * 128 ? 2 : BM * BN >= 128 * 64 ? 3 : 4; }

template <int BM, int BN, Operand AK, Operand BK>
__global__ __launch_bounds__(kBlock, (min_waves<BM, BN>())) void gemm_split_kernel(SplitArgs g) {
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int kA = slab_words<BM>(), kB = slab_words<BN>();
    __shared__ __align__(16) uint32_t lds[2 * (kA + kB)];
    static_assert((BM + BN) * kF32Pitch <= 2 * (kA + kB), "the fp32 pass uses the same LDS");

    const uint32_t z = blockIdx.y;
    uint32_t tm, tn, split;
    tile_of(blockIdx.x, g, tm, tn, split);
    const float *ga = g.a + (size_t)(z % g.zgroups) * g.a_z;
    const float *gb = g.b + (size_t)z * g.b_z;
    float *gc = g.c + (size_t)z * g.c_z;
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t kbeg = split * g.k_chunk;
    const uint32_t kend = kbeg + g.k_chunk < g.k ? kbeg + g.k_chunk : g.k;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave >> 1) * WM, wn0 = (wave & 1) * WN;
    const int half = lane >> 5, l32 = lane & 31;

    std::conditional_t<AK == kRowMajor, RowLoad<BM>, ColLoad<BM>> sa[2];
    std::conditional_t<BK == kRowMajor, RowLoad<BN>, ColLoad<BN>> sb[2];
    // Two register sets: slab s is loaded into set s & 1.
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        if constexpr (AK == kRowMajor) sa[d].init(ga, g.lda, m0, g.m - m0, tid);
        else sa[d].init(ga, g.lda, m0, g.m - m0, tid, g, false);
        if constexpr (BK == kRowMajor) sb[d].init(gb, g.ldb, n0, g.n - n0, tid);
        else sb[d].init(gb, g.ldb, n0, g.n - n0, tid, g, g.npos != 0);
    }
    auto load = [&](int d, uint32_t k0) {
        sa[d].load(k0);
        sb[d].load(k0);
    };
    auto load_tail = [&](uint32_t k0) {
        if constexpr (AK == kRowMajor) sa[0].load_tail(k0, kend, tid);
        else sa[0].load_tail(k0, kend);
        if constexpr (BK == kRowMajor) sb[0].load_tail(k0, kend, tid);
        else sb[0].load_tail(k0, kend);
    };
    auto store = [&](int d) {  // set d to LDS buffer d
        uint32_t *to = lds + d * (kA + kB);
        sa[d].store(to, tid);
        sb[d].store(to + kA, tid);
    };

    f32x16 big[TM][TN], small[TM][TN];
#pragma unroll
    for (int ti = 0; ti < TM; ++ti)
#pragma unroll
        for (int tj = 0; tj < TN; ++tj)
#pragma unroll
            for (int r = 0; r < 16; ++r) big[ti][tj][r] = small[ti][tj][r] = 0.0f;

    auto compute = [&](int cur) {
        bf16x8 af[TM][kPlanes], bf[TN][kPlanes];
        const uint32_t *pa = lds + cur * (kA + kB) + half * half_words<BM>() + (wm0 + l32) * 4;
        const uint32_t *pb = lds + cur * (kA + kB) + kA + half * half_words<BN>() + (wn0 + l32) * 4;
#pragma unroll
        for (int u = 0; u < kPlanes; ++u) {
#pragma unroll
            for (int ti = 0; ti < TM; ++ti)
                af[ti][u] = *reinterpret_cast<const bf16x8 *>(pa + u * 2 * half_words<BM>() + ti * 128);
#pragma unroll
            for (int tj = 0; tj < TN; ++tj)
                bf[tj][u] = *reinterpret_cast<const bf16x8 *>(pb + u * 2 * half_words<BN>() + tj * 128);
        }
        // hh, then the small terms; tiles innermost, so that successive MFMAs
        // write different accumulators.
        constexpr int kTa[6] = {0, 0, 1, 1, 0, 2}, kTb[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int ti = 0; ti < TM; ++ti)
#pragma unroll
                for (int tj = 0; tj < TN; ++tj) {
                    f32x16 &acc = t == 0 ? big[ti][tj] : small[ti][tj];
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ti][kTa[t]], bf[tj][kTb[t]], acc, 0, 0, 0);
                }
    };
    // Whole slabs: a step multiplies slab s out of LDS, splits and stores slab
    // s + 1 and loads slab s + 3 into the registers that held it (past the last
    // slab the last one again, unused): one basic block whose VALU work the
    // scheduler is told to place between the MFMAs.
    const uint32_t whole = kend > kbeg ? (kend - kbeg) / kBK : 0;
    const bool tail = kend > kbeg && (kend - kbeg) % kBK != 0;
    if (whole > 0) {
        const auto slab_k = [&](uint32_t x) { return kbeg + (x < whole ? x : whole - 1) * kBK; };
        const auto step = [&](auto d, uint32_t s) {
            constexpr int kD = decltype(d)::value;
            compute(kD);
            store(kD ^ 1);
            load(kD ^ 1, slab_k(s + 3));
            DKZ_SPLIT_SCHED();
            __syncthreads();
        };
        load(0, slab_k(0));
        load(1, slab_k(1));
        store(0);
        load(0, slab_k(2));
        __syncthreads();
        uint32_t s = 0;
#pragma unroll 1
        for (; s + 1 < whole; s += 2) {
            step(std::integral_constant<int, 0>{}, s);
            step(std::integral_constant<int, 1>{}, s + 1);
        }
        if (s < whole) {
            compute(0);
            __syncthreads();
        }
    }
    if (tail) {
        load_tail(kbeg + whole * kBK);
        store(0);
        __syncthreads();
        compute(0);
        __syncthreads();
    }

    // Sum the accumulators; a value that is not finite, or a row whose share
    // is tiny, sends the whole tile through the fp32 instruction.
    bool redo = sa[0].tiny() || sa[1].tiny() || sb[0].tiny() || sb[1].tiny();
#pragma unroll
    for (int ti = 0; ti < TM; ++ti)
#pragma unroll
        for (int tj = 0; tj < TN; ++tj) {
            big[ti][tj] += small[ti][tj];
#pragma unroll
            for (int r = 0; r < 16; ++r) redo |= !(fabsf(big[ti][tj][r]) < __builtin_inff());
        }
    if (__syncthreads_or(redo)) {
        float *as = reinterpret_cast<float *>(lds), *bs = as + BM * kF32Pitch;
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int tj = 0; tj < TN; ++tj)
#pragma unroll
                for (int r = 0; r < 16; ++r) big[ti][tj][r] = 0.0f;
#pragma unroll 1
        for (uint32_t k0 = kbeg; k0 < kend; k0 += kBK) {
            if (k0 + kBK <= kend) load(0, k0);
            else load_tail(k0);
            sa[0].store_f32(as, tid);
            sb[0].store_f32(bs, tid);
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int ti = 0; ti < TM; ++ti)
#pragma unroll
                    for (int tj = 0; tj < TN; ++tj)
                        big[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                            as[(wm0 + ti * 32 + l32) * kF32Pitch + 8 * half + q],
                            bs[(wn0 + tj * 32 + l32) * kF32Pitch + 8 * half + q], big[ti][tj], 0, 0, 0);
            __syncthreads();
        }
    }

    // big[ti][tj][r] is C(row, col) of the wave's block (ti, tj) with
    // row = 8*(r/4) + 4*(lane/32) + r%4 and col = lane%32.
#pragma unroll
    for (int tj = 0; tj < TN; ++tj) {
        const uint32_t j = n0 + wn0 + tj * 32 + l32;
        if (j >= g.n) continue;
        float *ccol = gc + j;
        if (g.npos != 0) {
            const uint32_t img = fdiv(j, g.div_npos);
            ccol = gc + (size_t)img * g.c_img + (j - img * g.npos);
        }
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t i = m0 + wm0 + ti * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
                if (i >= g.m) continue;
                if (g.splits > 1) {
                    g.partial[((size_t)split * g.m + i) * g.n + j] = big[ti][tj][r];
                } else {
                    float *cp = ccol + (size_t)i * g.ldc;
                    *cp = gemm_out(cp, big[ti][tj][r], g.alpha, g.beta);
                }
            }
    }
}

}  // namespace
}  // namespace dkz
