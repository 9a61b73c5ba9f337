// gemm_split.hpp -- the matrix-product kernel behind dkz_gemm and the
// convolution entry points (gemm.hip): fp32 products on the bf16 matrix cores.
//
// An fp32 value is the sum of three bf16 values, x = h + m + l (8 significant
// bits each, rounded to nearest, so 24 bits in all): exact for |x| >= 2^-109.
// A product of two such sums keeps six of its nine terms,
//     hh | hm + mh + mm + hl + lh,
// the rest (ml, lm, ll) being up to 2^-24 of it, 2^-27.5 rms.
// v_mfma_f32_32x32x16_bf16 forms the
// products exactly and adds them in fp32, rounding twice per 16 k. hh has an
// accumulator of its own and the five small terms another, so the large one is
// rounded once per 8 k (the fp32 matrix instruction rounds it at every k): over
// K = 2 .. 9216 the relative error against f64 is 0.26e-7 .. 6.4e-7 on data of
// both signs where v_mfma_f32_32x32x2_f32 leaves 0.37e-7 .. 1.7e-6. (Spread over
// four accumulators, as 64x64 tiles of that instruction were, sums of one sign
// came closer: 1.35e-7 over K = 1152, 1.88e-7 here.) Six bf16 products cost 6/16
// of the fp32 instruction's time.
//
// Where the split is not exact the tile is computed again with
// v_mfma_f32_32x32x2_f32 from the same loads (redo): when an accumulator is
// not finite (an infinity, a NaN, a value that rounds to a bf16 infinity: its
// l is a NaN) or when any of the tile's operands lies within (0, 2^-109).
// Infinities, NaNs and tiny operands so give what fp32 products give. Products
// with one k, where the fp32 instruction rounds but once, take it straight away:
// 2.53e-8 rms and 6.0e-8 at most of the result, the split 2.60e-8 and 9.4e-8.
// From two k on the split's rms error is the smaller one (3.67e-8 and 2.63e-8).
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

// LDS words of one half (8 k) of a plane of R rows, and of an operand's slab.
template <int R>
constexpr int half_words() { return R * 4 + 16; }
template <int R>
constexpr int slab_words() { return kPlanes * 2 * half_words<R>(); }

// Operand kinds. kRowMajor: rows along the tile dimension, k contiguous (A
// row-major, B transposed). kColMajor: k along the rows, the tile dimension
// contiguous (A transposed, B row-major), also the (image, position) columns of
// a 1x1 convolution. kGather: the same columns of a convolution's im2col, each
// element read from the image (kGatherWide: images or windows too large for
// kGather's 32-bit byte offsets and masks). kSeg, kTap: the operands of a weight
// gradient, whose k runs over (image, position) -- row f of delta (or of a 1x1
// convolution's input), and a tap's elements (kSegOdd: the positions per image
// are no multiple of four; kTapWide and kSegWide: 64-bit addresses).
enum Operand { kRowMajor, kColMajor, kGather, kGatherWide, kSeg, kSegOdd, kTap, kSegWide, kTapWide };

// The image behind a gathered operand: B[k][p] = im2col(image)[k][p] for
// k = (c, kh, kw) over a group's channels and p = (h, w) over the output
// positions (im2col.zig:13-49).
struct ConvGeom {
    uint32_t H, W, stride, rows, cols;  // rows x cols: the window
    int32_t pad, pad_x;                 // rows and columns (negative: the window starts inside the image)
    FastDiv div_kk, div_k, div_wo;      // rows*cols, cols, output width
};

// One phase of a strided data gradient: its flipped taps (A, `k` = filters x
// taps per group), their window over delta, and the pixels it writes:
// (s*yq + py, s*xq + px) for its column (yq, xq).
struct PhaseDesc {
    const float *a;
    uint32_t k, rows, cols, py, px;
    int32_t pad, pad_x;
    FastDiv div_kk, div_k;
};
constexpr int kMaxPhases = 4;

struct SplitArgs {
    const float *a;
    const float *b;
    float *c;
    float *partial;  // splits > 1: [splits][m][n] partial tiles
    uint32_t m, n, k, lda, ldb, ldc;
    float alpha, beta;
    uint32_t tiles_m, tiles_n, splits, k_chunk;
    // stream_len != 0 (splits 1, one grid row): tiles from full_tiles on are
    // streamed, stream_len slabs of the line (tile, slab) a workgroup.
    uint32_t full_tiles, stream_len, stream_slabs, runs;  // stream_slabs: the whole line's; runs: its workgroups
    FastDiv div_tile_slabs;
    uint32_t tile_bm, tile_bn_log2;
    // Groups (z = blockIdx.y): A at a + z * a_z, B at b + z * b_z, C at c + z * c_z.
    uint64_t a_z, b_z, c_z;
    // Columns over (image, position): npos positions per image (0: one matrix),
    // element strides from one image to the next of B and C.
    uint32_t npos;
    uint64_t b_img, c_img;
    FastDiv div_npos;
    ConvGeom cv;  // gathered operands and taps only
    // Weight gradient: positions per image, and those rounded up to a multiple
    // of four (k = image * kpos4 + position, so that four consecutive k lie in
    // one image; the positions past kpos read as 0). krow: a row's elements (of
    // delta, or of a 1x1 convolution's input), kpos but for a band of an image.
    // a_img: delta's element stride from one image to the next; the input's is
    // b_img.
    uint32_t kpos, krow;
    uint64_t a_img;
    FastDiv div_kpos4;
    // phases != 0: grid row y runs phase y / zrows over group y % zrows, its
    // columns (yq, xq) of an image ph_w wide.
    uint32_t phases, zrows, ph_s, ph_w;
    FastDiv div_wp;
    PhaseDesc ph[kMaxPhases];
};

// Column j's place in C.
__device__ __forceinline__ float *c_column(float *c, uint32_t j, const SplitArgs &g, uint32_t py, uint32_t px) {
    if (g.npos == 0) return c + j;
    const uint32_t img = fdiv(j, g.div_npos), p = j - img * g.npos;
    c += (size_t)img * g.c_img;
    if (g.phases == 0) return c + p;
    const uint32_t yq = fdiv(p, g.div_wp), xq = p - yq * g.div_wp.d;
    return c + (size_t)(g.ph_s * yq + py) * g.ph_w + g.ph_s * xq + px;
}

// Consecutive workgroups go round the XCDs: gives each XCD a run of neighbours.
__device__ __forceinline__ uint32_t xcd_order(uint32_t w, uint32_t total) {
    return total % kXcds == 0 ? (w % kXcds) * (total / kXcds) + w / kXcds : w;
}

// Tile t's row and column of tiles: groups of kGroupM rows, column by column.
__device__ __forceinline__ void tile_at(uint32_t t, const SplitArgs &g, uint32_t &tm, uint32_t &tn) {
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
// The differences are exact (a value minus its rounding is a float). They are
// taken by unpacking and subtracting: one v_dot2_f32_bf16 with (-1, 0) does the
// same, but runs on the matrix core, where it holds up the MFMAs (four of them
// an MFMA: 26 ns instead of the 16 that four shifts or subtractions leave it).
__device__ __forceinline__ Split2 split2(float x, float y) {
    Split2 s;
#pragma unroll
    for (int u = 0; u < kPlanes; ++u) {
        s.w[u] = pack_bf16(x, y);
        x -= __uint_as_float(s.w[u] << 16);
        y -= __uint_as_float(s.w[u] & 0xffff0000u);
    }
    return s;
}

// Looks for values the split is not exact for: the smallest of 2|x| - 1, x taken
// as its bits, in which zeros are the largest. (Three instructions a pair; the
// largest magnitude of a row's share took one, but let a tiny value pass beside
// a normal one, which is all of a sum where zeros lie opposite the normal ones.)
struct Smallest {
    uint32_t lo = ~0u;
    static __device__ __forceinline__ uint32_t rank(float x) { return (__float_as_uint(x) << 1) - 1; }
    __device__ __forceinline__ void see(float x, float y) { lo = min(min(lo, rank(x)), rank(y)); }
    __device__ __forceinline__ bool tiny() const { return lo < rank(0x1p-109f); }
};

// ---- operand loaders: `load` takes a whole slab, `load_tail` one that ends at
// kend (missing k read as 0); rows past the operand repeat its last row, whose
// results are not stored. `store` writes the planes and shows `seen` the values,
// `store_f32` writes the fp32 slab.

template <int R>
struct RowLoad {
    static constexpr int kL = R * kBK / 4 / kBlock;  // float4s per thread
    const float *p[kL];
    float4 v[kL];

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
    __device__ __forceinline__ void store(uint32_t *s, int tid, Smallest &seen) const {
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const int f = tid + l * kBlock, r = f / 4, q = f % 4;
            const Split2 x = split2(v[l].x, v[l].y), y = split2(v[l].z, v[l].w);
            seen.see(v[l].x, v[l].y);
            seen.see(v[l].z, v[l].w);
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
};

// One row of the tile and kT consecutive k of each slab per thread: a wave's
// loads of one k are 64 consecutive elements, its k the same in every lane
// (scalar address arithmetic), whatever the alignment.
template <int R>
struct ColBase {
    static constexpr int kT = R * kBK / kBlock;
    float v[kT];
    uint32_t kq;  // wave-uniform: this wave's k start at kq * kT of the slab

    __device__ __forceinline__ void store(uint32_t *s, int tid, Smallest &seen) const {
        Split2 w[kT / 2];
#pragma unroll
        for (int j = 0; j < kT / 2; ++j) {
            w[j] = split2(v[2 * j], v[2 * j + 1]);
            seen.see(v[2 * j], v[2 * j + 1]);
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
            off = 4 * ((i - i0) * (uint32_t)g.b_img + (r0 + r - i * g.npos));
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

// fdiv without its branch on a divisor of 1.
__device__ __forceinline__ uint32_t fdiv_select(uint32_t n, const FastDiv &f) {
    const uint32_t one = 0u - (uint32_t)(f.mul == 0), q = umulhi32(n, f.mul) >> f.shr;
    return (q & ~one) | (n & one);
}

// The im2col columns of a convolution, one output position a lane. The
// position is taken apart once; the k of a load is the same in every lane of
// the wave, so its channel and tap are scalar arithmetic. A tap outside the
// image reads as 0: its bit in the lane's row or column mask sends the load's
// offset past the buffer's end, where buffer loads return 0.
template <int R>
struct GatherLoad : ColBase<R> {
    using ColBase<R>::kT;
    using ColBase<R>::v;
    using ColBase<R>::kq;
    __amdgpu_buffer_rsrc_t buf;
    uint32_t off;        // byte offset of the window's first tap
    uint32_t rout, cout; // bit kh (kw) set: that row (column) of the window is outside
    uint32_t hw;         // H * W

    static __device__ __forceinline__ uint32_t outside(int first, uint32_t window, uint32_t size) {
        const int lo = first < 0 ? -first : 0, hi = min((int)window, (int)size - first);
        if (hi <= lo) return ~0u;
        return ~((hi >= 32 ? ~0u : (1u << hi) - 1) & ~((1u << lo) - 1));
    }
    __device__ __forceinline__ void init(const float *b, const ConvGeom &cv, uint32_t r0, int tid, const SplitArgs &g) {
        kq = __builtin_amdgcn_readfirstlane(tid / R);
        hw = cv.H * cv.W;
        const uint32_t r = r0 + tid % R, rr = r < g.n ? r : g.n - 1;
        const uint32_t i0 = fdiv(r0, g.div_npos), i = fdiv(rr, g.div_npos), p = rr - i * g.npos;
        const uint32_t h = fdiv(p, cv.div_wo), w = p - h * cv.div_wo.d;
        rout = r < g.n ? outside((int)(h * cv.stride) - cv.pad, cv.rows, cv.H) : ~0u;
        cout = outside((int)(w * cv.stride) - cv.pad_x, cv.cols, cv.W);
        off = 4 * ((i - i0) * (uint32_t)g.b_img + h * cv.stride * cv.W + w * cv.stride);
        const float *first = b + (size_t)i0 * g.b_img - ((int64_t)cv.pad * cv.W + cv.pad_x);
        buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(first), 0, 0x80000000u, 0x00020000);
    }
    template <bool TAIL>
    __device__ __forceinline__ void load_taps(const ConvGeom &cv, uint32_t k0, uint32_t kend) {
        const uint32_t k = k0 + kq * kT;
        const uint32_t c = fdiv_select(k, cv.div_kk), t = k - c * cv.div_kk.d;
        uint32_t kh = fdiv_select(t, cv.div_k), kw = t - kh * cv.cols;
        uint32_t at = 4 * (c * hw + kh * cv.W + kw);
        const uint32_t next_row = 4 * (cv.W - cv.cols), next_chan = 4 * (hw - cv.rows * cv.W);
#pragma unroll
        for (int j = 0; j < kT; ++j) {
            if (!TAIL || k + j < kend) {
                const uint32_t out = (uint32_t)(__builtin_amdgcn_sbfe((int)rout, kh, 1) | __builtin_amdgcn_sbfe((int)cout, kw, 1));
                v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buf, off | out, at, 0));
            } else {
                v[j] = 0.0f;
            }
            // The next tap, without branches (the loads stay in one basic block).
            const uint32_t row = 0u - (uint32_t)(kw + 1 == cv.cols);
            const uint32_t chan = row & (0u - (uint32_t)(kh + 1 == cv.rows));
            kw = (kw + 1) & ~row;
            kh = (kh - row) & ~chan;
            at += 4 + (row & next_row) + (chan & next_chan);
        }
    }
    __device__ __forceinline__ void load(uint32_t k0, const ConvGeom &cv) { load_taps<false>(cv, k0, 0); }
    __device__ __forceinline__ void load_tail(uint32_t k0, uint32_t kend, const ConvGeom &cv) { load_taps<true>(cv, k0, kend); }
};

// The same with 64-bit addresses and compared bounds.
template <int R>
struct GatherWideLoad : ColBase<R> {
    using ColBase<R>::kT;
    using ColBase<R>::v;
    using ColBase<R>::kq;
    const float *img;
    int y, x;
    bool in;

    __device__ __forceinline__ void init(const float *b, const ConvGeom &cv, uint32_t r0, int tid, const SplitArgs &g) {
        kq = __builtin_amdgcn_readfirstlane(tid / R);
        const uint32_t r = r0 + tid % R, rr = r < g.n ? r : g.n - 1;
        const uint32_t i = fdiv(rr, g.div_npos), p = rr - i * g.npos;
        const uint32_t h = fdiv(p, cv.div_wo), w = p - h * cv.div_wo.d;
        in = r < g.n;
        y = (int)(h * cv.stride) - cv.pad;
        x = (int)(w * cv.stride) - cv.pad_x;
        img = b + (size_t)i * g.b_img;
    }
    __device__ __forceinline__ void load_tail(uint32_t k0, uint32_t kend, const ConvGeom &cv) {
#pragma unroll
        for (int j = 0; j < kT; ++j) {
            const uint32_t k = k0 + kq * kT + j;
            const uint32_t c = fdiv(k, cv.div_kk), t = k - c * cv.div_kk.d;
            const uint32_t kh = fdiv(t, cv.div_k), kw = t - kh * cv.cols;
            const int yy = y + (int)kh, xx = x + (int)kw;
            const bool ok = in && k < kend && yy >= 0 && yy < (int)cv.H && xx >= 0 && xx < (int)cv.W;
            v[j] = ok ? img[((size_t)c * cv.H + yy) * cv.W + xx] : 0.0f;
        }
    }
    __device__ __forceinline__ void load(uint32_t k0, const ConvGeom &cv) { load_tail(k0, ~0u, cv); }
};

// The quad of k at k0 + 4 * (tid % 4) of a weight gradient: its image (from the
// split's first one on) and first position; `in` says whether it is there. The
// host gives the narrow loaders images, positions and image sides below 2^24, so
// that all their products but those with the image stride are 24-bit ones; WIDE
// takes any.
template <bool WIDE>
struct Quad {
    uint32_t img, p;
    bool in;
    __device__ __forceinline__ Quad(uint32_t k0, uint32_t kend, uint32_t img0, int tid, const SplitArgs &g) {
        const uint32_t k = k0 + 4 * (tid % 4);
        const uint32_t i = fdiv_select(k, g.div_kpos4);
        in = k < kend;
        img = i - img0;
        p = k - (WIDE ? i * g.div_kpos4.d : __umul24(i, g.div_kpos4.d));
    }
};

// Where the four floats of thread tid's float4 l of a slab go: as RowLoad's.
template <int R>
struct QuadBase {
    static constexpr int kL = RowLoad<R>::kL;
    RowLoad<R> row;  // v only
    __device__ __forceinline__ void store(uint32_t *s, int tid, Smallest &seen) const { row.store(s, tid, seen); }
    __device__ __forceinline__ void store_f32(float *s, int tid) const { row.store_f32(s, tid); }
};

// Rows of delta (row stride krow): four positions in one 16-byte load. ODD: an
// image's last quad has fewer; it is loaded from kpos - 4 and shifted.
template <int R, bool ODD>
struct SegLoad : QuadBase<R> {
    using QuadBase<R>::kL;
    using QuadBase<R>::row;
    __amdgpu_buffer_rsrc_t buf;
    uint32_t at[kL], img0;

    __device__ __forceinline__ void init(const float *base, uint32_t r0, uint32_t rows, uint32_t kbeg, int tid,
                                         uint64_t img_stride, const SplitArgs &g) {
        img0 = fdiv_select(kbeg, g.div_kpos4);
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const uint32_t f = tid + l * kBlock, r = f / 4 < rows ? f / 4 : rows - 1;
            at[l] = 4 * r * g.krow;
        }
        buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base + (size_t)img0 * img_stride + (size_t)r0 * g.krow), 0,
                                                0x80000000u, 0x00020000);
    }
    __device__ __forceinline__ void load(uint32_t k0, uint32_t kend, int tid, uint64_t img_stride, const SplitArgs &g) {
        const Quad<false> q(k0, kend, img0, tid, g);
        const uint32_t p = ODD ? min(q.p, g.kpos - 4) : q.p, d = q.p - p;
        const uint32_t off = 4 * (q.img * (uint32_t)img_stride + p);
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const auto t = __builtin_amdgcn_raw_buffer_load_b128(buf, (off + at[l]) | (q.in ? 0u : 0x80000000u), 0, 0);
            float4 v = make_float4(__uint_as_float(t[0]), __uint_as_float(t[1]), __uint_as_float(t[2]), __uint_as_float(t[3]));
            if constexpr (ODD) {
                if (d & 1) v = make_float4(v.y, v.z, v.w, 0.0f);
                if (d & 2) v = make_float4(v.z, v.w, 0.0f, 0.0f);
            }
            row.v[l] = v;
        }
    }
};

// Rows of the input's im2col: one tap of one channel a row (fixed for the
// thread), its element at each position of the quad.
template <int R>
struct TapLoad : QuadBase<R> {
    using QuadBase<R>::kL;
    using QuadBase<R>::row;
    __amdgpu_buffer_rsrc_t buf;
    uint32_t img0;
    int at[kL], dy[kL], dx[kL];

    __device__ __forceinline__ void init(const float *base, const ConvGeom &cv, uint32_t r0, uint32_t rows, uint32_t kbeg,
                                         int tid, const SplitArgs &g) {
        img0 = fdiv_select(kbeg, g.div_kpos4);
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const uint32_t f = tid + l * kBlock, r = r0 + (f / 4 < rows ? f / 4 : rows - 1);
            const uint32_t c = fdiv_select(r, cv.div_kk), t = r - c * cv.div_kk.d;
            const uint32_t kh = fdiv_select(t, cv.div_k);
            dy[l] = (int)kh - cv.pad;
            dx[l] = (int)(t - kh * cv.cols) - cv.pad_x;
            at[l] = (int)(c * cv.H * cv.W) + dy[l] * (int)cv.W + dx[l];
        }
        buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base + (size_t)img0 * g.b_img), 0, 0x80000000u, 0x00020000);
    }
    __device__ __forceinline__ void load(uint32_t k0, uint32_t kend, int tid, const ConvGeom &cv, const SplitArgs &g) {
        const Quad<false> q(k0, kend, img0, tid, g);
        const uint32_t h = fdiv_select(q.p, cv.div_wo), last = __umul24(cv.div_wo.d - 1, cv.stride);
        uint32_t y = __umul24(h, cv.stride), x = __umul24(q.p - __umul24(h, cv.div_wo.d), cv.stride);
        uint32_t pos = q.img * (uint32_t)g.b_img + __umul24(y, cv.W) + x;
        const uint32_t wrap_pos = cv.stride * cv.W - last;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool in = q.in & (q.p + j < g.kpos);
#pragma unroll
            for (int l = 0; l < kL; ++l) {
                // Unsigned: below 0 is out too. No branches (see the step's one basic block).
                const bool ok = in & (y + dy[l] < cv.H) & (x + dx[l] < cv.W);
                ::dkz::lane(row.v[l], j) =
                    __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buf, 4 * (pos + at[l]) | (ok ? 0u : 0x80000000u), 0, 0));
            }
            const bool wrap = x == last;
            x = wrap ? 0 : x + cv.stride;
            y += wrap ? cv.stride : 0;
            pos += wrap ? wrap_pos : cv.stride;
        }
    }
};

// Both with 64-bit addresses: img + r * krow + p, and the tap's element.
template <int R, bool TAP>
struct QuadWideLoad : QuadBase<R> {
    using QuadBase<R>::kL;
    using QuadBase<R>::row;
    __device__ __forceinline__ void load(const float *base, uint32_t r0, uint32_t rows, uint32_t k0, uint32_t kend, int tid,
                                         uint64_t img_stride, const ConvGeom &cv, const SplitArgs &g) {
        const Quad<true> q(k0, kend, 0, tid, g);
#pragma unroll
        for (int l = 0; l < kL; ++l) {
            const uint32_t f = tid + l * kBlock, r = r0 + (f / 4 < rows ? f / 4 : rows - 1);
            const uint32_t c = fdiv(r, cv.div_kk), t = r - c * cv.div_kk.d, kh = fdiv(t, cv.div_k), kw = t - kh * cv.cols;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t p = q.p + j;
                bool ok = q.in && p < g.kpos;
                size_t e = (size_t)q.img * img_stride;
                if constexpr (TAP) {
                    const uint32_t h = fdiv(p, cv.div_wo), w = p - h * cv.div_wo.d;
                    const int y = (int)(h * cv.stride + kh) - cv.pad, x = (int)(w * cv.stride + kw) - cv.pad_x;
                    ok = ok && y >= 0 && y < (int)cv.H && x >= 0 && x < (int)cv.W;
                    e += ((size_t)c * cv.H + y) * cv.W + x;
                } else {
                    e += (size_t)r * g.krow + p;
                }
                ::dkz::lane(row.v[l], j) = ok ? base[e] : 0.0f;
            }
        }
    }
};

// C(i, j) = beta-applied C + alpha * s (gemm.zig:121-131: beta == 0 clears C,
// NaN included).
__device__ __forceinline__ float gemm_out(const float *cp, float s, float alpha, float beta) {
    float cv = 0.0f;
    if (beta != 0.0f) cv = (beta == 1.0f) ? *cp : *cp * beta;
    return cv + alpha * s;
}

template <Operand K, int R>
struct Loader;
template <int R> struct Loader<kRowMajor, R> { using type = RowLoad<R>; };
template <int R> struct Loader<kColMajor, R> { using type = ColLoad<R>; };
template <int R> struct Loader<kGather, R> { using type = GatherLoad<R>; };
template <int R> struct Loader<kGatherWide, R> { using type = GatherWideLoad<R>; };
template <int R> struct Loader<kSeg, R> { using type = SegLoad<R, false>; };
template <int R> struct Loader<kSegOdd, R> { using type = SegLoad<R, true>; };
template <int R> struct Loader<kTap, R> { using type = TapLoad<R>; };
template <int R> struct Loader<kSegWide, R> { using type = QuadWideLoad<R, false>; };
template <int R> struct Loader<kTapWide, R> { using type = QuadWideLoad<R, true>; };

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

// ORDERED: a workgroup takes all of a tile's K ranges or pieces, one behind the
// other, and keeps their sum in f64 as the reductions do, so that no scratch is
// needed and the results are the same. Tiles are 64x64 (their sums take 32
// registers; a 128x128 tile's would take 128), each a part of the g.tile_bm x
// g.tile_bn tile whose pieces it adds up, or the 32x128 ones.
template <int BM, int BN, Operand AK, Operand BK, bool ORDERED = false>
__global__ __launch_bounds__(kBlock, (min_waves<BM, BN>() - (ORDERED ? 2 : 0))) void gemm_split_kernel(SplitArgs g) {
    constexpr int kRowsOfWaves = BM == 32 ? 1 : 2;  // 32-row tiles: four waves side by side
    constexpr int WM = BM / kRowsOfWaves, WN = BN * kRowsOfWaves / 4, TM = WM / 32, TN = WN / 32;
    constexpr int RA = BM == 32 ? 64 : BM;  // rows of A staged (of a 32-row tile, the last row again)
    constexpr int kA = slab_words<RA>(), kB = slab_words<BN>();
    __shared__ __align__(16) uint32_t lds[2 * (kA + kB)];
    __shared__ uint32_t votes[kBlock / kWave];
    static_assert((RA + BN) * kF32Pitch <= 2 * (kA + kB), "the fp32 pass uses the same LDS");

    constexpr bool kGa = BK == kGather || BK == kGatherWide;
    constexpr bool kQuads = AK >= kSeg;  // a weight gradient: quads past kend load as zeros
    uint32_t z = blockIdx.y;
    // A phase's row of a strided data gradient takes its taps, window and
    // pixel offsets (fields picked with constant indexes, so the arguments
    // stay where they are).
    const float *a_base = g.a;
    uint32_t k_all = g.k, k_chunk = g.k_chunk, lda = g.lda, py = 0, px = 0;
    uint64_t a_z = g.a_z;
    ConvGeom cv = g.cv;
    if (kGa && g.phases != 0) {
        const uint32_t p = z / g.zrows;
        z -= p * g.zrows;
#define DKZ_PHASE_FIELD(f) (p == 0 ? g.ph[0].f : p == 1 ? g.ph[1].f : p == 2 ? g.ph[2].f : g.ph[3].f)
        a_base = DKZ_PHASE_FIELD(a);
        k_all = DKZ_PHASE_FIELD(k);
        cv.rows = DKZ_PHASE_FIELD(rows);
        cv.cols = DKZ_PHASE_FIELD(cols);
        cv.pad = DKZ_PHASE_FIELD(pad);
        cv.pad_x = DKZ_PHASE_FIELD(pad_x);
        cv.div_kk = DKZ_PHASE_FIELD(div_kk);
        cv.div_k = DKZ_PHASE_FIELD(div_k);
        py = DKZ_PHASE_FIELD(py);
        px = DKZ_PHASE_FIELD(px);
#undef DKZ_PHASE_FIELD
        k_chunk = lda = k_all;
        a_z = (uint64_t)g.m * k_all;
    }
    const float *ga = a_base + (size_t)z * a_z;
    const float *gb = g.b + (size_t)z * g.b_z;
    float *gc = g.c + (size_t)z * g.c_z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = BM == 32 ? 0 : (wave >> 1) * WM, wn0 = (BM == 32 ? wave : wave & 1) * WN;
    const int half = lane >> 5, l32 = lane & 31;

    // One K range of one tile; or a run of the streamed line: the last slabs of
    // a tile, the first ones of the next. Piece (workgroup b, tile t) has
    // partial tile b + t (along the line at least one of the two advances).
    const bool streams = !ORDERED && g.stream_len != 0 && blockIdx.x >= g.full_tiles;
    uint32_t block = blockIdx.x, line = 0, line_end = 0, run = 0;
    [[maybe_unused]] double total[ORDERED ? TM : 1][ORDERED ? TN : 1][ORDERED ? 16 : 1] = {};
    [[maybe_unused]] uint32_t own_m0 = 0, own_n0 = 0;
    if constexpr (ORDERED) {  // the tile's slabs along the line, or from 0; cut at multiples of run
        const uint32_t subs_n = g.tile_bn_log2 == 7 && BN == 64 ? 2 : 1, subs = subs_n * (g.tile_bm == 128 ? 2 : 1);
        block = xcd_order(block, (g.tiles_m * g.tiles_n - g.full_tiles) * subs);
        const uint32_t sub = block % subs;
        block /= subs;
        uint32_t tm, tn;
        tile_at(g.full_tiles + block, g, tm, tn);
        own_m0 = tm * g.tile_bm + sub / subs_n * BM;
        own_n0 = (tn << g.tile_bn_log2) + sub % subs_n * BN;
        if (own_m0 >= g.m || own_n0 >= g.n) return;
        const uint32_t slabs = (k_all + kBK - 1) / kBK;
        run = g.stream_len != 0 ? g.stream_len : k_chunk / kBK;
        line = g.stream_len != 0 ? block * slabs : 0;
        line_end = line + slabs;
    } else if (streams) {
        block = xcd_order(block - g.full_tiles, g.runs);
        line = block * g.stream_len;
        line_end = min(line + g.stream_len, g.stream_slabs);
    }
#pragma unroll 1
    do {
    uint32_t tm, tn, kbeg, kend, slot = 0;
    if constexpr (ORDERED) {
        const uint32_t len = min(run - line % run, line_end - line);
        tm = tn = 0;
        kbeg = (line + (k_all + kBK - 1) / kBK - line_end) * kBK;
        kend = min(kbeg + len * kBK, k_all);
        line += len;
    } else if (streams) {
        const uint32_t t = fdiv(line, g.div_tile_slabs), first = line - t * g.div_tile_slabs.d;
        const uint32_t len = min(g.div_tile_slabs.d - first, line_end - line);
        tile_at(g.full_tiles + t, g, tm, tn);
        kbeg = first * kBK;
        kend = min(kbeg + len * kBK, k_all);
        slot = block + t;
        line += len;
    } else {
        const uint32_t tiles = g.stream_len != 0 ? g.full_tiles : g.tiles_m * g.tiles_n;
        uint32_t t = xcd_order(block, tiles * g.splits);
        slot = t / tiles;
        tile_at(t - slot * tiles, g, tm, tn);
        kbeg = slot * k_chunk;
        kend = kbeg + k_chunk < k_all ? kbeg + k_chunk : k_all;
    }
    const uint32_t m0 = ORDERED ? own_m0 : tm * BM, n0 = ORDERED ? own_n0 : tn * BN;

    // Two register sets: slab s is loaded into set s & 1.
    typename Loader<AK, RA>::type sa[2];
    typename Loader<BK, BN>::type sb[2];
    const uint32_t rows_a = BM == 32 ? min(g.m - m0, 32u) : g.m - m0, rows_b = g.n - n0;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        if constexpr (AK == kRowMajor) sa[d].init(ga, lda, m0, rows_a, tid);
        else if constexpr (AK == kColMajor) sa[d].init(ga, lda, m0, rows_a, tid, g, false);
        else if constexpr (AK == kSeg || AK == kSegOdd) sa[d].init(ga, m0, rows_a, kbeg, tid, g.a_img, g);
        if constexpr (BK == kRowMajor) sb[d].init(gb, g.ldb, n0, rows_b, tid);
        else if constexpr (BK == kColMajor) sb[d].init(gb, g.ldb, n0, rows_b, tid, g, g.npos != 0);
        else if constexpr (kGa) sb[d].init(gb, cv, n0, tid, g);
        else if constexpr (BK == kSeg || BK == kSegOdd) sb[d].init(gb, n0, rows_b, kbeg, tid, g.b_img, g);
        else if constexpr (BK == kTap) sb[d].init(gb, cv, n0, rows_b, kbeg, tid, g);
    }
    auto load = [&](int d, uint32_t k0) {
        if constexpr (AK == kSeg || AK == kSegOdd) sa[d].load(k0, kend, tid, g.a_img, g);
        else if constexpr (AK == kSegWide) sa[d].load(ga, m0, rows_a, k0, kend, tid, g.a_img, cv, g);
        else sa[d].load(k0);
        if constexpr (kGa) sb[d].load(k0, cv);
        else if constexpr (BK == kSeg || BK == kSegOdd) sb[d].load(k0, kend, tid, g.b_img, g);
        else if constexpr (BK == kTap) sb[d].load(k0, kend, tid, cv, g);
        else if constexpr (BK == kTapWide) sb[d].load(gb, n0, rows_b, k0, kend, tid, g.b_img, cv, g);
        else sb[d].load(k0);
    };
    auto load_tail = [&](int d, uint32_t k0) {
        if constexpr (kQuads) {
            load(d, k0);
        } else {
            if constexpr (AK == kRowMajor) sa[d].load_tail(k0, kend, tid);
            else sa[d].load_tail(k0, kend);
            if constexpr (BK == kRowMajor) sb[d].load_tail(k0, kend, tid);
            else if constexpr (kGa) sb[d].load_tail(k0, kend, cv);
            else sb[d].load_tail(k0, kend);
        }
    };
    Smallest seen;
    auto store = [&](int d) {  // set d to LDS buffer d
        uint32_t *to = lds + d * (kA + kB);
        sa[d].store(to, tid, seen);
        sb[d].store(to + kA, tid, seen);
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
        const uint32_t *pa = lds + cur * (kA + kB) + half * half_words<RA>() + (wm0 + l32) * 4;
        const uint32_t *pb = lds + cur * (kA + kB) + kA + half * half_words<BN>() + (wn0 + l32) * 4;
#pragma unroll
        for (int u = 0; u < kPlanes; ++u) {
#pragma unroll
            for (int ti = 0; ti < TM; ++ti)
                af[ti][u] = *reinterpret_cast<const bf16x8 *>(pa + u * 2 * half_words<RA>() + ti * 128);
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
    const bool one_k = kQuads ? g.kpos == 1 && k_all == 4 : k_all == 1;
    const uint32_t whole = kend > kbeg && !one_k ? (kend - kbeg + (kQuads ? kBK - 1 : 0)) / kBK : 0;
    const bool tail = !kQuads && !one_k && kend > kbeg && (kend - kbeg) % kBK != 0;
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
        // One slab alone loads no others (where registers are left for the branches).
        constexpr bool kLean = kQuads && TM * TN == 1;
        load(0, slab_k(0));
        if (tail && whole == 1) load_tail(1, kbeg + kBK);  // a first layer's 27 k: both slabs at once
        else if (!kLean || whole > 1) load(1, slab_k(1));
        store(0);
        if (!kLean || whole > 1) load(0, slab_k(2));
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
        if (whole == 1) {
            store(1);
        } else {
            load_tail(0, kbeg + whole * kBK);
            store(0);
        }
        __syncthreads();
        compute(whole == 1);
        __syncthreads();
    }

    // Sum the accumulators; a value that is not finite, or a tiny operand,
    // sends the whole tile through the fp32 instruction.
    bool redo = one_k || seen.tiny();
#pragma unroll
    for (int ti = 0; ti < TM; ++ti)
#pragma unroll
        for (int tj = 0; tj < TN; ++tj) {
            big[ti][tj] += small[ti][tj];
#pragma unroll
            for (int r = 0; r < 16; ++r) redo |= !(fabsf(big[ti][tj][r]) < __builtin_inff());
        }
    // One barrier (__syncthreads_or takes three, and a load of the workgroup's size).
    const bool any = __builtin_amdgcn_ballot_w64(redo) != 0;
    if (lane == 0) votes[wave] = any;
    __syncthreads();
    if ((votes[0] | votes[1] | votes[2] | votes[3]) != 0) {
        float *as = reinterpret_cast<float *>(lds), *bs = as + RA * kF32Pitch;
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int tj = 0; tj < TN; ++tj)
#pragma unroll
                for (int r = 0; r < 16; ++r) big[ti][tj][r] = 0.0f;
#pragma unroll 1
        for (uint32_t k0 = kbeg; k0 < kend; k0 += kBK) {
            if (k0 + kBK <= kend) load(0, k0);
            else load_tail(0, k0);
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

    if constexpr (ORDERED) {
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int tj = 0; tj < TN; ++tj)
#pragma unroll
                for (int r = 0; r < 16; ++r) total[ti][tj][r] += (double)big[ti][tj][r];
        if (line < line_end) continue;
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int tj = 0; tj < TN; ++tj)
#pragma unroll
                for (int r = 0; r < 16; ++r) big[ti][tj][r] = (float)total[ti][tj][r];
    }

    // big[ti][tj][r] is C(row, col) of the wave's block (ti, tj) with
    // row = 8*(r/4) + 4*(lane/32) + r%4 and col = lane%32. A block's sixteen
    // values of C are loaded together (rows past m read row m - 1), then stored.
#pragma unroll
    for (int tj = 0; tj < TN; ++tj) {
        const uint32_t j = n0 + wn0 + tj * 32 + l32;
        if (j >= g.n) continue;
        float *ccol = c_column(gc, j, g, py, px);
#pragma unroll
        for (int ti = 0; ti < TM; ++ti) {
            const uint32_t i0 = m0 + wm0 + ti * 32 + half * 4;
            const auto row = [&](int r) { return i0 + (r >> 2) * 8 + (r & 3); };
            // A K range's partial is a whole m x n one, a streamed piece's its tile.
            const bool part = !ORDERED && (streams || g.splits > 1);
            float *to = !part     ? ccol
                        : streams ? g.partial + (size_t)slot * (BM * BN) + (j - n0) - (size_t)m0 * BN
                                  : g.partial + (size_t)slot * g.m * g.n + j;
            const uint32_t ld = !part ? g.ldc : streams ? BN : g.n;
            float out[16];
            if (part) {
#pragma unroll
                for (int r = 0; r < 16; ++r) out[r] = big[ti][tj][r];
            } else if (g.beta == 0.0f) {
#pragma unroll
                for (int r = 0; r < 16; ++r) out[r] = 0.0f + g.alpha * big[ti][tj][r];
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) out[r] = to[(size_t)min(row(r), g.m - 1) * ld];
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    out[r] = (g.beta == 1.0f ? out[r] : out[r] * g.beta) + g.alpha * big[ti][tj][r];
            }
            if (m0 + BM <= g.m) {
#pragma unroll
                for (int r = 0; r < 16; ++r) to[(size_t)row(r) * ld] = out[r];
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (row(r) < g.m) to[(size_t)row(r) * ld] = out[r];
            }
        }
    }
    } while (line < line_end);
}

// The split-K epilogue: adds a tile's partials in split order, then as the
// kernel's own epilogue. The sum is kept in f64 and rounded once: with hundreds
// of partials their fp32 sum was most of the error ([42,75,31,31]->18 1x1 weight
// gradient: 4.5e-7 of the result with 255 partials in fp32, 0.7e-7 with 507 in
// f64). V4: a lane takes four consecutive columns of one row (one image's,
// 16-byte aligned).
//
// GROUPS lanes share an output, lane g taking partials g, g + GROUPS, ..., and
// the first adds the others' sums in order: one lane an output up to 32
// partials, 16 beyond, where one lane's loads would take a round trip to memory
// for every few partials ([1,50176]x[50176,9], 448 of them: 50 us with one lane,
// 3.2 with 16).
template <bool V4, int GROUPS>
__global__ __launch_bounds__(kBlock) void split_reduce_kernel(SplitArgs g) {
    using T = std::conditional_t<V4, float4, float>;
    constexpr uint32_t kW = V4 ? 4 : 1, kOuts = kBlock / GROUPS;
    constexpr int kInFlight = 8;
    const uint32_t mn = g.m * g.n, v = blockIdx.x * kOuts + threadIdx.x % kOuts, first = threadIdx.x / kOuts;
    const bool in = v < mn / kW;
    double s[kW] = {};
    if (in) {
        for (uint32_t t = first; t < g.splits; t += GROUPS * kInFlight) {
            T p[kInFlight];  // past the last partial: that one again, not added
#pragma unroll
            for (int u = 0; u < kInFlight; ++u)
                p[u] = reinterpret_cast<const T *>(g.partial + (size_t)min(t + u * GROUPS, g.splits - 1) * mn)[v];
#pragma unroll
            for (int u = 0; u < kInFlight; ++u)
#pragma unroll
                for (uint32_t x = 0; x < kW; ++x)
                    s[x] += t + u * GROUPS < g.splits ? (double)reinterpret_cast<const float *>(&p[u])[x] : 0.0;
        }
    }
    if constexpr (GROUPS > 1) {
        __shared__ double sums[kW][kBlock];
#pragma unroll
        for (uint32_t x = 0; x < kW; ++x) sums[x][threadIdx.x] = s[x];
        __syncthreads();
        if (first != 0) return;
#pragma unroll
        for (int u = 1; u < GROUPS; ++u)
#pragma unroll
            for (uint32_t x = 0; x < kW; ++x) s[x] += sums[x][threadIdx.x + u * kOuts];
    }
    if (!in) return;
    const uint32_t e = v * kW, i = e / g.n, j = e - i * g.n;
    float *cp = c_column(g.c, j, g, 0, 0) + (size_t)i * g.ldc;
    T o;
#pragma unroll
    for (uint32_t x = 0; x < kW; ++x) reinterpret_cast<float *>(&o)[x] = gemm_out(cp + x, (float)s[x], g.alpha, g.beta);
    *reinterpret_cast<T *>(cp) = o;
}

// The streamed tiles' epilogue: adds a tile's pieces in k order (in f64), then as above.
// A lane takes four consecutive columns of one row, eight pieces in flight; V4:
// they are 16 aligned bytes of C.
template <bool V4>
__global__ __launch_bounds__(kBlock) void stream_reduce_kernel(SplitArgs g) {
    constexpr int kPieces = 8;
    const uint32_t tile_floats = g.tile_bm << g.tile_bn_log2;
    const uint32_t e = 4 * (blockIdx.x * kBlock + threadIdx.x), t = e / tile_floats, at = e - t * tile_floats;
    uint32_t tm, tn;
    tile_at(g.full_tiles + t, g, tm, tn);
    const uint32_t i = tm * g.tile_bm + (at >> g.tile_bn_log2);
    const uint32_t j = (tn << g.tile_bn_log2) + (at & ((1u << g.tile_bn_log2) - 1));
    if (i >= g.m || j >= g.n) return;
    const uint32_t slabs = g.div_tile_slabs.d;
    const uint32_t first = t * slabs / g.stream_len, last = ((t + 1) * slabs - 1) / g.stream_len;
    const float *from = g.partial + at + (size_t)t * tile_floats;
    double s[4] = {};
    for (uint32_t b = first; b <= last; b += kPieces) {
        float4 p[kPieces];  // past the last piece: that one again, not added
#pragma unroll
        for (int u = 0; u < kPieces; ++u)
            p[u] = *reinterpret_cast<const float4 *>(from + (size_t)min(b + u, last) * tile_floats);
#pragma unroll
        for (int u = 0; u < kPieces; ++u)
#pragma unroll
            for (int x = 0; x < 4; ++x) s[x] += b + u <= last ? (double)::dkz::lane(p[u], x) : 0.0;
    }
    if constexpr (V4) {
        float *cp = c_column(g.c, j, g, 0, 0) + (size_t)i * g.ldc;
        float4 o;
#pragma unroll
        for (int x = 0; x < 4; ++x) ::dkz::lane(o, x) = gemm_out(cp + x, (float)s[x], g.alpha, g.beta);
        *reinterpret_cast<float4 *>(cp) = o;
    } else {
#pragma unroll
        for (uint32_t x = 0; x < 4; ++x) {
            if (j + x >= g.n) break;
            float *cp = c_column(g.c, j + x, g, 0, 0) + (size_t)i * g.ldc;
            *cp = gemm_out(cp, (float)s[x], g.alpha, g.beta);
        }
    }
}

}  // namespace
}  // namespace dkz
