// gemm.hip -- C = alpha*op(A)*op(B) + beta*C, row-major (src/gpu.zig:671-719,
// CPU twin src/gemm.zig:47-278), and a convolutional layer's three per-image
// loops as one call each (dkz_convolution_forward, _data_gradient,
// _weight_gradient), whose im2col operands are gathered inside the product.
// The kernel is gemm_split.hpp's; here each entry point checks its arguments,
// describes its operands and picks tiles and K ranges.
//
// Products too small to fill the chip split K: the grid holds `splits` copies of
// the tile grid, each summing one range of K into a partial tile in the
// library's scratch, and a second kernel adds a tile's partials in split order
// and applies alpha and beta -- deterministic, no atomics. The epilogue follows
// gemm.zig:121-131 then :180-184 (so do the streamed tiles' pieces, see
// pick_tiling): beta == 0 clears C (NaN included), beta == 1
// keeps it, anything else scales it; then C += alpha*acc.
//
// Workgroups take tiles in groups of 8 tile-rows, so that the tiles running
// at once share A and B panels, and neighbouring tile numbers are placed on
// one XCD (workgroups are dealt to the 8 XCDs round robin) so that they share
// its L2.
#include <algorithm>
#include <mutex>
#include <vector>

#include "dkz_device.hpp"
#include "dkz_internal.hpp"
#include "gemm_split.hpp"
#include "gemm_tiling.hpp"

namespace dkz {
namespace {

static_assert(kSlab == kBK, "the tilings count the kernel's slabs");

// Held from a null-stream product's launch to its reduction's (see launch_split).
std::mutex g_own_mutex;

template <Operand AK, Operand BK>
int launch_tiles(hipStream_t stream, const char *name, uint32_t bm, uint32_t bn, dim3 grid, const SplitArgs &g) {
    const dim3 block(kBlock);
    if constexpr (BK != kGatherWide && BK != kTapWide) {
        if (bm == 128 && bn == 128) return launch_on(stream, name, gemm_split_kernel<128, 128, AK, BK>, grid, block, g);
        if (bm == 128) return launch_on(stream, name, gemm_split_kernel<128, 64, AK, BK>, grid, block, g);
        if (bm == 64 && bn == 128) return launch_on(stream, name, gemm_split_kernel<64, 128, AK, BK>, grid, block, g);
        if (bm == 32) return launch_on(stream, name, gemm_split_kernel<32, 128, AK, BK>, grid, block, g);
    }
    return launch_on(stream, name, gemm_split_kernel<64, 64, AK, BK>, grid, block, g);
}

// The tiles from full_tiles on, a workgroup taking all of a tile's pieces.
template <Operand AK, Operand BK>
int launch_ordered(hipStream_t stream, const char *name, const SplitArgs &g) {
    const uint32_t tiles = g.tiles_m * g.tiles_n - g.full_tiles;
    const dim3 block(kBlock);
    if constexpr (BK != kGatherWide)
        if (g.tile_bm == 32) return launch_on(stream, name, gemm_split_kernel<32, 128, AK, BK, true>, dim3(tiles), block, g);
    const dim3 grid(tiles * (g.tile_bm / 64) * ((1u << g.tile_bn_log2) / 64));
    return launch_on(stream, name, gemm_split_kernel<64, 64, AK, BK, true>, grid, block, g);
}

// Runs a product of g's operands over `z` grid rows (one when K may be split).
//
// The partials of K ranges and pieces go to g.partial, in the device's scratch
// (null: K is not split), which calls on several streams must not share at the
// same time. OWN: a product of which calls may overlap on any streams, threads
// and captured graphs (a convolution's forward, its 1x1 data gradient). On the
// null stream, where calls run one behind the other, its partials have a block
// of the scratch to themselves, and a mutex keeps another thread's product from
// between a product and its reduction; on other streams a workgroup takes all of
// a tile's pieces itself (launch_ordered), with the same results. Null stream /
// another, us, and the unsplit fp32 kernel this replaced: [1,64,52,52]->128 3x3
// 16.8 / 25.5 / 38; [64,128,56,56]->128 367 / 402 / 688; [32,512,13,13]->1024 337 /
// 482 / 622; [1,512,13,13]->1024 28 / 146 / 249, where 48 tiles leave most CUs idle.
template <Operand AK, Operand BK, bool OWN = false>
int launch_split(const char *name, SplitArgs g, uint32_t z) {
    uint64_t left = 0;
    if (z == 1 && g.phases == 0 && g.k >= 8 * kBK && (OWN || g.partial != nullptr)) {
        if constexpr (OWN) {
            left = kScratchOwnFloats;
        } else {
            Scratch sc{};
            DKZ_TRY(device_scratch(&sc));
            left = (uint64_t)(sc.gemm + sc.gemm_floats - g.partial);
        }
    }
    const Tiling t = pick_tiling(g.m, g.n, g.k, z, left, BK == kGatherWide || BK == kTapWide);
    g.tiles_m = div_up(g.m, t.bm);
    g.tiles_n = div_up(g.n, t.bn);
    g.tile_bm = t.bm;
    g.tile_bn_log2 = t.bn == 128 ? 7 : 6;
    g.splits = t.splits;
    g.k_chunk = t.k_chunk;
    uint64_t total = (uint64_t)g.tiles_m * g.tiles_n * g.splits;
    const uint32_t streamed = t.stream ? (uint32_t)(total - t.full_tiles) : 0;
    if (t.stream) {
        const uint32_t slabs = div_up(g.k, kBK);
        g.full_tiles = t.full_tiles;
        g.stream_len = t.stream;
        g.stream_slabs = streamed * slabs;
        g.div_tile_slabs = make_fastdiv(slabs);
        g.runs = div_up(g.stream_slabs, t.stream);
        total = t.full_tiles + g.runs;
    }
    DKZ_REQUIRE(total <= 0x7fffffffull);
    const hipStream_t stream = current_stream();
    std::unique_lock<std::mutex> lock(g_own_mutex, std::defer_lock);
    if constexpr (OWN) {
        if (t.stream || g.splits > 1) {
            g.partial = stream == nullptr ? null_stream_scratch() : nullptr;
            if (g.partial == nullptr) {
                if (g.full_tiles != 0) DKZ_TRY((launch_tiles<AK, BK>(stream, name, t.bm, t.bn, dim3(g.full_tiles), g)));
                return launch_ordered<AK, BK>(stream, name, g);
            }
            lock.lock();
        }
    }
    DKZ_TRY((launch_tiles<AK, BK>(stream, name, t.bm, t.bn, dim3((uint32_t)total, z), g)));
    const bool v4 = g.n % 4 == 0 && g.ldc % 4 == 0 && aligned16(g.c) && g.npos % 4 == 0 && g.c_img % 4 == 0;
    const dim3 block(kBlock);
    if (t.stream) {
        const dim3 blocks(streamed * (t.bm * t.bn / 4 / kBlock));
        return v4 ? launch_on(stream, name, stream_reduce_kernel<true>, blocks, block, g)
                  : launch_on(stream, name, stream_reduce_kernel<false>, blocks, block, g);
    }
    if (g.splits == 1) return 0;
    const uint64_t vecs = (uint64_t)g.m * g.n / (v4 ? 4 : 1);
    const bool many = g.splits > 32;
    const dim3 blocks(div_up(vecs, many ? kBlock / 16 : kBlock));
    if (v4)
        return many ? launch_on(stream, name, split_reduce_kernel<true, 16>, blocks, block, g)
                    : launch_on(stream, name, split_reduce_kernel<true, 1>, blocks, block, g);
    return many ? launch_on(stream, name, split_reduce_kernel<false, 16>, blocks, block, g)
                : launch_on(stream, name, split_reduce_kernel<false, 1>, blocks, block, g);
}

// The data gradient's A: at[j][c][(f*ks + kh)*ks + kw] = w[j][f][c][ks-1-kh][ks-1-kw]
// for group j, channel c < cg and filter f < m -- the group's weights with
// channels as rows and the window flipped, so that the product with the
// implicit gather of delta is col2im(w^T x delta) (im2col.zig:51-79).
__global__ __launch_bounds__(kBlock) void flip_weights_kernel(const float *w, float *at, uint32_t kk, FastDiv div_kk,
                                                             FastDiv div_mkk, FastDiv div_cgmkk, uint32_t cg,
                                                             uint32_t total) {
    const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= total) return;
    const uint32_t j = fdiv(e, div_cgmkk), r = e - j * div_cgmkk.d;
    const uint32_t c = fdiv(r, div_mkk), q = r - c * div_mkk.d;
    const uint32_t f = fdiv(q, div_kk), t = q - f * kk;
    at[e] = w[(size_t)j * div_cgmkk.d + (size_t)f * cg * kk + c * kk + (kk - 1 - t)];
}

// One phase's A of a strided data gradient: at[j][c][(f*na + a)*nb + b] =
// w[j][f][c][kh0 + s*(na-1-a)][kw0 + s*(nb-1-b)], the taps of the phase
// (kh = kh0 mod s, kw = kw0 mod s) with channels as rows, flipped.
struct PhaseTaps {
    uint32_t ks, s, kh0, kw0, na, nb, m, cg;
    FastDiv div_nb, div_nab, div_mnab, div_cgmnab;
};
__global__ __launch_bounds__(kBlock) void flip_phase_kernel(const float *w, float *at, PhaseTaps t, uint32_t total) {
    const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= total) return;
    const uint32_t j = fdiv(e, t.div_cgmnab), r = e - j * t.div_cgmnab.d;
    const uint32_t c = fdiv(r, t.div_mnab), q = r - c * t.div_mnab.d;
    const uint32_t f = fdiv(q, t.div_nab), u = q - f * t.div_nab.d;
    const uint32_t a = fdiv(u, t.div_nb), b = u - a * t.nb;
    const uint32_t kh = t.kh0 + t.s * (t.na - 1 - a), kw = t.kw0 + t.s * (t.nb - 1 - b);
    const size_t kk = (size_t)t.ks * t.ks;
    at[e] = w[((size_t)j * t.m + f) * t.cg * kk + c * kk + kh * t.ks + kw];
}

// The largest byte offset that the 32-bit loaders may form from an operand's
// tile or split base: below the buffers' 2^31 bytes.
constexpr uint64_t kMaxOffset = 1ull << 31;

// Whether the columns of one tile (at most 128 consecutive (image, position)
// pairs) of a product over images b_img elements apart, `extent` elements read
// from each, stay within 32-bit byte offsets.
inline bool span_fits(uint64_t npos, uint64_t b_img, uint64_t extent) {
    return ((127 / npos + 1) * b_img + extent) * 4 < kMaxOffset;
}

// Columns over (image, position) of every image, one grid row a group: the
// tiles are full whatever an image's size, and a column's place is worked out
// once. B and C advance b_img and c_img elements from one image to the next.
void set_span(SplitArgs &g, uint64_t npos, uint64_t batch, uint64_t b_img, uint64_t c_img) {
    g.n = (uint32_t)(npos * batch);
    g.npos = (uint32_t)npos;
    g.div_npos = make_fastdiv((uint32_t)npos);
    g.b_img = b_img;
    g.c_img = c_img;
}

// The gather geometry of a rows x cols window over an H x W image.
ConvGeom conv_geom(uint64_t H, uint64_t W, uint64_t wo, uint32_t rows, uint32_t cols, uint32_t stride, int pad, int pad_x) {
    return {(uint32_t)H,   (uint32_t)W, stride, rows, cols, pad, pad_x, make_fastdiv(rows * cols), make_fastdiv(cols),
            make_fastdiv((uint32_t)wo)};
}

// A product whose B is gathered from images of `in_group` elements each.
template <bool OWN>
int launch_gather(const char *name, const SplitArgs &g, uint32_t z, uint64_t in_group) {
    // kGather's offsets count from a window's first tap at position (0, 0), so
    // the image's last element lies pad rows and pad_x elements further on.
    const auto fits = [&](uint32_t rows, uint32_t cols, int pad, int pad_x) {
        return rows <= 32 && cols <= 32 &&
               span_fits(g.npos, g.b_img, in_group + (uint64_t)std::max(pad, 0) * g.cv.W + (uint64_t)std::max(pad_x, 0));
    };
    bool narrow = fits(g.cv.rows, g.cv.cols, g.cv.pad, g.cv.pad_x);
    for (uint32_t p = 0; p < g.phases; ++p) narrow = narrow && fits(g.ph[p].rows, g.ph[p].cols, g.ph[p].pad, g.ph[p].pad_x);
    return narrow ? launch_split<kRowMajor, kGather, OWN>(name, g, z) : launch_split<kRowMajor, kGatherWide, OWN>(name, g, z);
}

// Extent in elements of a rows x cols row-major view with leading dimension ld.
inline uint64_t extent(uint64_t rows, uint64_t cols, uint64_t ld) {
    return rows == 0 || cols == 0 ? 0 : (rows - 1) * ld + cols;
}

}  // namespace
}  // namespace dkz

using namespace dkz;

extern "C" {

int dkz_gemm(int ta, int tb, int m, int n, int k, float alpha, const float *a, int lda, const float *b, int ldb,
             float beta, float *c, int ldc) {
    DKZ_REQUIRE(m >= 0 && n >= 0 && k >= 0 && lda >= 0 && ldb >= 0 && ldc >= 0);
    if (m == 0 || n == 0) return 0;  // gpu.zig:686
    DKZ_REQUIRE(c != nullptr && ldc >= n);
    DKZ_REQUIRE(extent(m, n, ldc) <= kMaxElems);
    if (k > 0) {
        DKZ_REQUIRE(a != nullptr && b != nullptr);
        DKZ_REQUIRE(lda >= (ta ? m : k) && ldb >= (tb ? k : n));
        DKZ_REQUIRE(extent(ta ? k : m, ta ? m : k, lda) + 3 <= kMaxElems);
        DKZ_REQUIRE(extent(tb ? n : k, tb ? k : n, ldb) + 3 <= kMaxElems);
    }
    SplitArgs g{};
    g.a = a;
    g.b = b;
    g.c = c;
    g.m = (uint32_t)m;
    g.n = (uint32_t)n;
    g.k = (uint32_t)k;
    g.lda = (uint32_t)lda;
    g.ldb = (uint32_t)ldb;
    g.ldc = (uint32_t)ldc;
    g.alpha = alpha;
    g.beta = beta;

    Scratch sc{};
    if (k >= 8 * kBK) DKZ_TRY(device_scratch(&sc));
    g.partial = sc.gemm;
    if (!ta && !tb) return launch_split<kRowMajor, kColMajor>("gemm_nn", g, 1);
    if (ta && !tb) return launch_split<kColMajor, kColMajor>("gemm_tn", g, 1);
    if (!ta && tb) return launch_split<kRowMajor, kRowMajor>("gemm_nt", g, 1);
    return launch_split<kColMajor, kRowMajor>("gemm_tt", g, 1);
}

// convolutional.zig:240-260 in one launch: for image i and group j,
// output(i, j) (m x n, m = filters/groups, n = out_h*out_w) += weights(j)
// (m x k, k = ksize^2 * channels/groups) x im2col(input(i, j)) (k x n), with
// out_h = (height + 2*pad - ksize)/stride + 1 as outHeight computes it. The
// layer zero-fills the output first; this adds to it (beta = 1), as its gemm
// calls do. ksize 1 multiplies by the input itself (ldb = n), as the layer
// does. No workspace: the im2col operand is gathered inside the product.
int dkz_convolution_forward(int batch, int groups, int channels, int height, int width, int filters, int ksize,
                            int stride, int pad, const float *weights, const float *input, float *output) {
    DKZ_REQUIRE(batch >= 0 && groups >= 1 && groups <= 65535 && channels >= 0 && height >= 0 && width >= 0 &&
                filters >= 0);
    DKZ_REQUIRE(ksize >= 1 && stride >= 1 && pad >= 0);
    DKZ_REQUIRE(channels % groups == 0 && filters % groups == 0);
    DKZ_REQUIRE((int64_t)height + 2 * (int64_t)pad >= ksize && (int64_t)width + 2 * (int64_t)pad >= ksize);
    const uint64_t m = (uint64_t)filters / groups, cg = (uint64_t)channels / groups;
    const uint64_t ho = ((uint64_t)height + 2 * (uint64_t)pad - ksize) / stride + 1;
    const uint64_t wo = ((uint64_t)width + 2 * (uint64_t)pad - ksize) / stride + 1;
    const uint64_t n = ho * wo, k = (uint64_t)ksize * ksize * cg;
    const uint64_t zcount = (uint64_t)batch * groups, in_group = cg * height * width;
    if (zcount == 0 || m == 0 || n == 0 || k == 0) return 0;
    DKZ_REQUIRE(weights && input && output);
    DKZ_REQUIRE(zcount * m * n <= kMaxElems && zcount * in_group <= kMaxElems && (uint64_t)groups * m * k <= kMaxElems);
    DKZ_REQUIRE(ksize != 1 || n <= (uint64_t)height * width);  // the input is read as a k x n matrix
    SplitArgs g{};
    g.a = weights;
    g.b = input;
    g.c = output;
    g.m = (uint32_t)m;
    g.k = (uint32_t)k;
    g.lda = (uint32_t)k;
    g.ldb = (uint32_t)n;
    g.ldc = (uint32_t)n;
    g.alpha = 1.0f;
    g.beta = 1.0f;
    g.a_z = m * k;
    g.b_z = in_group;
    g.c_z = m * n;
    set_span(g, n, (uint64_t)batch, (uint64_t)groups * in_group, (uint64_t)groups * m * n);
    constexpr const char *kName = "convolution_forward";
    if (ksize == 1 && span_fits(n, g.b_img, 0)) 
        return launch_split<kRowMajor, kColMajor, true>(kName, g, (uint32_t)groups);
    // ksize 1 reads the input as a k x n matrix: rows of n positions.
    g.cv = ksize == 1 ? conv_geom(1, n, n, 1, 1, 1, 0, 0)
                      : conv_geom((uint64_t)height, (uint64_t)width, wo, (uint32_t)ksize, (uint32_t)ksize, (uint32_t)stride, pad, pad);
    return launch_gather<true>(kName, g, (uint32_t)groups, in_group);
}

// convolutional.zig:299-305 (the data-gradient half of the per-image
// backward loop) in one call. For image i and group j, with m, n, k, the
// offsets and out_h, out_w as in dkz_convolution_forward and
// input_delta(i, j) = input_delta + (i*groups + j)*in_group:
//   ksize 1: input_delta(i, j), read as a k x n matrix as the layer reads it,
//            = weights(j)^T (k x m) x delta(i, j) (m x n) -- overwritten
//            (the layer's gemm with beta 0);
//   else:    input_delta(i, j) += col2im(weights(j)^T x delta(i, j)) -- the
//            layer's gemm into the workspace, then col2im, which adds.
// With stride 1 and pad < ksize the second is one product per image and
// group: input channels by input positions, k = (filter, tap) over the
// group's flipped weights (transposed once into the library's scratch) and
// delta gathered at each tap's output position, so col2im's adds join the
// product's sum. Otherwise the same per phase of the input pixels (y mod
// stride, x mod stride), each over its own taps. No workspace.
int dkz_convolution_data_gradient(int batch, int groups, int channels, int height, int width, int filters, int ksize,
                                  int stride, int pad, const float *weights, const float *delta,
                                  float *input_delta) {
    DKZ_REQUIRE(batch >= 0 && groups >= 1 && groups <= 65535 && channels >= 0 && height >= 0 && width >= 0 &&
                filters >= 0);
    DKZ_REQUIRE(ksize >= 1 && stride >= 1 && pad >= 0);
    DKZ_REQUIRE(channels % groups == 0 && filters % groups == 0);
    DKZ_REQUIRE((int64_t)height + 2 * (int64_t)pad >= ksize && (int64_t)width + 2 * (int64_t)pad >= ksize);
    const uint64_t m = (uint64_t)filters / groups, cg = (uint64_t)channels / groups;
    const uint64_t ho = ((uint64_t)height + 2 * (uint64_t)pad - ksize) / stride + 1;
    const uint64_t wo = ((uint64_t)width + 2 * (uint64_t)pad - ksize) / stride + 1;
    const uint64_t npos = ho * wo, kk = (uint64_t)ksize * ksize, kw = kk * cg;
    const uint64_t zcount = (uint64_t)batch * groups, in_group = cg * height * width;
    if (zcount == 0 || cg == 0 || npos == 0 || in_group == 0) return 0;
    DKZ_REQUIRE(weights && delta && input_delta);
    DKZ_REQUIRE(zcount * m * npos <= kMaxElems && zcount * in_group <= kMaxElems &&
                (uint64_t)groups * m * kw <= kMaxElems);
    DKZ_REQUIRE(ksize != 1 || npos <= (uint64_t)height * width);  // the k x n view stays inside the image
    SplitArgs g{};
    g.c = input_delta;
    g.b = delta;
    g.m = (uint32_t)cg;
    g.alpha = 1.0f;
    g.b_z = m * npos;
    g.c_z = in_group;
    const uint64_t b_img = (uint64_t)groups * m * npos, c_img = (uint64_t)groups * in_group;
    constexpr const char *kName = "convolution_data_gradient";
    if (ksize == 1) {
        // C(i, j) = A^T x B with A = weights(j) (m x cg, k-major), B = delta(i, j);
        // with m == 0 the sum is empty and beta 0 leaves zeros (gemm.zig:121-131).
        g.a = weights;
        g.k = (uint32_t)m;
        g.lda = (uint32_t)cg;
        g.ldb = (uint32_t)npos;
        g.ldc = (uint32_t)npos;
        g.beta = 0.0f;
        g.a_z = m * cg;
        set_span(g, npos, (uint64_t)batch, b_img, c_img);
        if (span_fits(npos, b_img, 0)) return launch_split<kColMajor, kColMajor, true>(kName, g, (uint32_t)groups);
        g.cv = conv_geom(1, npos, npos, 1, 1, 1, 0, 0);
        return launch_split<kColMajor, kGatherWide, true>(kName, g, (uint32_t)groups);
    }
    if (m == 0) return 0;  // col2im adds an empty sum
    Scratch sc;
    DKZ_TRY(device_scratch(&sc));
    g.beta = 1.0f;
    if (stride == 1 && pad <= ksize - 1) {
        // input_delta(i, j) += A x im2col(delta(i, j)) with A the group's
        // weights flipped and transposed (flip_weights_kernel, into the
        // scratch) and the im2col of delta (out_h x out_w, pad ksize-1-pad)
        // gathered inside the product: out_h + 2*(ksize-1-pad) - ksize + 1 =
        // height, and tap (kh, kw) of input position (y, x) reads delta at
        // (y + kh - (ksize-1-pad), ...), i.e. the layer's col2im term of tap
        // (ksize-1-kh, ksize-1-kw).
        const uint64_t at_floats = (uint64_t)groups * cg * m * kk;
        DKZ_REQUIRE(at_floats <= sc.gemm_floats);
        DKZ_TRY(launch("convolution_data_gradient", flip_weights_kernel, dim3(div_up(at_floats, kBlock)),
                       dim3(kBlock), weights, sc.gemm, (uint32_t)kk, make_fastdiv((uint32_t)kk),
                       make_fastdiv((uint32_t)(m * kk)), make_fastdiv((uint32_t)(cg * m * kk)), (uint32_t)cg,
                       (uint32_t)at_floats));
        const uint64_t n = (uint64_t)height * width, k = m * kk;
        g.a = sc.gemm;
        g.partial = sc.gemm + (at_floats + 63) / 64 * 64;  // behind the flipped weights
        g.k = (uint32_t)k;
        g.lda = (uint32_t)k;
        g.ldc = (uint32_t)n;
        g.a_z = cg * k;
        set_span(g, n, (uint64_t)batch, b_img, c_img);
        const int back = ksize - 1 - pad;
        g.cv = conv_geom(ho, wo, (uint64_t)width, (uint32_t)ksize, (uint32_t)ksize, 1, back, back);
        return launch_gather<false>(kName, g, (uint32_t)groups, m * npos);
    }
    // Strided (or pad >= ksize): the im2col of delta would have holes between
    // the strided outputs. Input pixel (y, x) takes tap (kh, kw) only when
    // y + pad - kh is a multiple of stride, so the pixels split into stride^2
    // phases (y mod stride, x mod stride), each taking the taps kh = kh0 + s*a,
    // kw = kw0 + s*b with kh0 = (py + pad) mod s: per phase one product over
    // the phase's pixels whose A is those taps flipped (flip_phase_kernel) and
    // whose B is a stride-1 im2col of delta with window na x nb and pads
    // na-1-qy, nb-1-qx (qy = (py + pad - kh0) / s), written to the phase's
    // pixels. The same multiply-adds as the layer's gemm, no column buffer.
    const int s = stride;
    const uint64_t at_all = (uint64_t)groups * cg * m * kk;
    DKZ_REQUIRE(at_all <= sc.gemm_floats);
    // The phases that some tap reaches, most taps first (their workgroups
    // are the longest, so they start first).
    struct Phase {
        int py, px, kh0, kw0, na, nb, hp, wp, qy, qx;
    };
    std::vector<Phase> phases;
    for (int py = 0; py < s; ++py) {
        for (int px = 0; px < s; ++px) {
            Phase q{};
            q.py = py;
            q.px = px;
            q.kh0 = (py + pad) % s;
            q.kw0 = (px + pad) % s;
            q.na = q.kh0 < ksize ? (ksize - q.kh0 + s - 1) / s : 0;
            q.nb = q.kw0 < ksize ? (ksize - q.kw0 + s - 1) / s : 0;
            q.hp = py < height ? (height - py + s - 1) / s : 0;
            q.wp = px < width ? (width - px + s - 1) / s : 0;
            if (q.na == 0 || q.nb == 0 || q.hp == 0 || q.wp == 0) continue;  // no tap reaches these pixels
            q.qy = (py + pad - q.kh0) / s;
            q.qx = (px + pad - q.kw0) / s;
            phases.push_back(q);
        }
    }
    std::stable_sort(phases.begin(), phases.end(),
                     [](const Phase &x, const Phase &y) { return x.na * x.nb > y.na * y.nb; });
    // Phases share a launch (grid row = phase x (image, group)) when they
    // cover equal pixel grids, i.e. the stride divides the input, and a
    // launch's rows can hold every group of an image for each phase.
    const bool merge = height % s == 0 && width % s == 0 && (uint64_t)groups * kMaxPhases <= 65535;
    uint64_t at_off = 0;
    for (size_t i0 = 0; i0 < phases.size();) {
        const size_t cnt = merge ? std::min<size_t>(kMaxPhases, phases.size() - i0) : 1;
        const int hp = phases[i0].hp, wp = phases[i0].wp;
        const uint64_t n = (uint64_t)hp * wp;
        SplitArgs gp = g;
        for (size_t u = 0; u < cnt; ++u) {
            const Phase &q = phases[i0 + u];
            const uint64_t nab = (uint64_t)q.na * q.nb, k = m * nab;
            const uint64_t at_n = (uint64_t)groups * cg * k;
            PhaseTaps t{(uint32_t)ksize, (uint32_t)s, (uint32_t)q.kh0, (uint32_t)q.kw0, (uint32_t)q.na,
                        (uint32_t)q.nb, (uint32_t)m, (uint32_t)cg, make_fastdiv((uint32_t)q.nb),
                        make_fastdiv((uint32_t)nab), make_fastdiv((uint32_t)(m * nab)),
                        make_fastdiv((uint32_t)(cg * k))};
            float *at = sc.gemm + at_off;
            DKZ_TRY(launch("convolution_data_gradient", flip_phase_kernel, dim3(div_up(at_n, kBlock)), dim3(kBlock),
                           weights, at, t, (uint32_t)at_n));
            gp.ph[u] = PhaseDesc{at,
                                 (uint32_t)k,
                                 (uint32_t)q.na,
                                 (uint32_t)q.nb,
                                 (uint32_t)q.py,
                                 (uint32_t)q.px,
                                 q.na - 1 - q.qy,
                                 q.nb - 1 - q.qx,
                                 make_fastdiv((uint32_t)nab),
                                 make_fastdiv((uint32_t)q.nb)};
            at_off += at_n;
        }
        gp.a = gp.ph[0].a;
        gp.k = gp.ph[0].k;
        gp.lda = gp.k;
        gp.ldc = (uint32_t)((uint64_t)height * width);
        gp.a_z = cg * gp.k;
        gp.phases = (uint32_t)cnt;
        gp.zrows = (uint32_t)groups;
        gp.ph_s = (uint32_t)s;
        gp.ph_w = (uint32_t)width;
        gp.div_wp = make_fastdiv((uint32_t)wp);
        set_span(gp, n, (uint64_t)batch, b_img, c_img);
        gp.cv = conv_geom(ho, wo, (uint64_t)wp, gp.ph[0].rows, gp.ph[0].cols, 1, gp.ph[0].pad, gp.ph[0].pad_x);
        DKZ_TRY(launch_gather<false>(kName, gp, (uint32_t)(cnt * groups), m * npos));
        i0 += cnt;
    }
    return 0;
}

// convolutional.zig:288-297 (the weight-gradient half of the per-image
// backward loop) in one product: for group j,
//     weight_updates(j) (m x k) += sum over images i of delta(i, j) (m x n) x im2col(input(i, j))^T (n x k)
// with the same m, n, k, offsets and ksize-1 reading of the input as
// dkz_convolution_forward, delta(i, j) = delta + (i*groups + j)*m*n and
// weight_updates(j) = weight_updates + j*m*k. One NT product per group whose
// k runs over (image, position), split into ranges of k that are added in
// order.
int dkz_convolution_weight_gradient(int batch, int groups, int channels, int height, int width, int filters,
                                    int ksize, int stride, int pad, const float *delta, const float *input,
                                    float *weight_updates) {
    DKZ_REQUIRE(batch >= 0 && groups >= 1 && channels >= 0 && height >= 0 && width >= 0 && filters >= 0);
    DKZ_REQUIRE(ksize >= 1 && stride >= 1 && pad >= 0);
    DKZ_REQUIRE(channels % groups == 0 && filters % groups == 0);
    DKZ_REQUIRE((int64_t)height + 2 * (int64_t)pad >= ksize && (int64_t)width + 2 * (int64_t)pad >= ksize);
    const uint64_t m = (uint64_t)filters / groups, cg = (uint64_t)channels / groups;
    const uint64_t ho = ((uint64_t)height + 2 * (uint64_t)pad - ksize) / stride + 1;
    const uint64_t wo = ((uint64_t)width + 2 * (uint64_t)pad - ksize) / stride + 1;
    const uint64_t npos = ho * wo, kw = (uint64_t)ksize * ksize * cg, in_group = cg * height * width;
    if (batch == 0 || m == 0 || kw == 0 || npos == 0) return 0;
    DKZ_REQUIRE(delta && input && weight_updates);
    const uint64_t images = (uint64_t)batch * groups;
    DKZ_REQUIRE(images * m * npos <= kMaxElems && images * in_group <= kMaxElems && (uint64_t)groups * m * kw <= kMaxElems);
    DKZ_REQUIRE((uint64_t)batch * npos <= kMaxElems);
    DKZ_REQUIRE(ksize != 1 || npos <= (uint64_t)height * width);  // the input is read as a k x n matrix
    Scratch sc;
    DKZ_TRY(device_scratch(&sc));
    SplitArgs g{};
    g.m = (uint32_t)m;
    g.n = (uint32_t)kw;
    g.ldc = (uint32_t)kw;
    g.alpha = 1.0f;
    g.beta = 1.0f;
    g.partial = sc.gemm;
    g.krow = (uint32_t)npos;
    g.a_img = (uint64_t)groups * m * npos;
    g.b_img = (uint64_t)groups * in_group;
    constexpr const char *kName = "convolution_weight_gradient";
    // One position an image (a classifier's 1x1 layer behind a global average
    // pool): images are rows of delta and input, a plain TN product whose k are
    // the images. [256,2048,1,1]->1000 43.5 us on the fp32 instruction, 54.8
    // through the 64-bit quad loaders, which pad its k to four, 14.0 so.
    if (npos == 1 && ksize == 1) {
        g.k = (uint32_t)batch;
        g.lda = (uint32_t)g.a_img;
        g.ldb = (uint32_t)g.b_img;
        for (int j = 0; j < groups; ++j) {
            SplitArgs gj = g;
            gj.a = delta + (uint64_t)j * m;
            gj.b = input + (uint64_t)j * in_group;
            gj.c = weight_updates + (uint64_t)j * m * kw;
            DKZ_TRY((launch_split<kColMajor, kColMajor>(kName, gj, 1)));
        }
        return 0;
    }
    // The narrow loaders: an image within 2^31 bytes, at least one whole quad
    // an image, and 24-bit products: a map of 2^24 positions or more goes
    // through them in bands of output rows (of positions, where ksize 1 reads
    // the input as a k x n matrix). The others take 64-bit addresses element by
    // element: half the speed or less.
    constexpr uint64_t k24 = 1u << 24, kBand = k24 - 4;
    const uint64_t img_bytes = 4 * std::max(g.a_img, g.b_img), row = ksize == 1 ? 4 : wo;
    const bool narrow = npos >= 4 && row <= kBand && img_bytes < kMaxOffset &&
                        (ksize == 1 || ((uint64_t)height < k24 && (uint64_t)width < k24 && (uint64_t)stride < k24));
    const uint64_t rows = div_up(npos, row), bands = narrow && npos > kBand ? div_up(rows, kBand / row) : 1;
    const uint64_t band = std::min(npos, div_up(rows, bands) * row);
    // k = image * band4 + position, each band's positions rounded up to a
    // multiple of four. As many images a product as keep k below 2^31 and, for
    // the narrow loaders, the images below 2^24 and within 2^31 bytes; later
    // ones add to the same updates. [64,3,416,416]->64 3x3 (2.8 GB of delta) in
    // two products 1.2 ms, where one through the 64-bit loaders took 820 ms.
    // (band4 may be 2^31, of a single image.)
    const auto up4 = [](uint64_t x) { return (x + 3) / 4 * 4; };
    uint64_t most = std::min<uint64_t>((uint64_t)batch, std::max<uint64_t>(kMaxElems / up4(band), 1));
    if (narrow) most = std::min({most, k24 - 1, (kMaxOffset - 1) / img_bytes});
    if (bands > 1) most = 1;
    for (int j = 0; j < groups; ++j) {
        for (uint64_t i0 = 0; i0 < (uint64_t)batch; i0 += most) {
            for (uint64_t p0 = 0; p0 < npos; p0 += band) {
                SplitArgs gj = g;
                const uint64_t kpos = std::min(band, npos - p0), kpos4 = up4(kpos);
                gj.kpos = (uint32_t)kpos;
                gj.div_kpos4 = make_fastdiv((uint32_t)kpos4);
                gj.k = (uint32_t)(std::min<uint64_t>(most, (uint64_t)batch - i0) * kpos4);
                gj.a = delta + i0 * g.a_img + (uint64_t)j * m * npos + p0;
                gj.b = input + i0 * g.b_img + (uint64_t)j * in_group + (ksize == 1 ? p0 : 0);
                gj.c = weight_updates + (uint64_t)j * m * kw;
                // A band starts p0 / wo output rows down (modulo 2^32, as the
                // loaders' bounds tests are).
                gj.cv = ksize == 1 ? conv_geom(1, npos, npos, 1, 1, 1, 0, 0)
                                   : conv_geom((uint64_t)height, (uint64_t)width, wo, (uint32_t)ksize, (uint32_t)ksize, (uint32_t)stride,
                                               (int)(uint32_t)((uint64_t)pad - p0 / wo * (uint64_t)stride), pad);
                if (!narrow) DKZ_TRY((launch_split<kSegWide, kTapWide>(kName, gj, 1)));
                else if (ksize == 1 && kpos % 4 == 0) DKZ_TRY((launch_split<kSeg, kSeg>(kName, gj, 1)));
                else if (ksize == 1) DKZ_TRY((launch_split<kSegOdd, kSegOdd>(kName, gj, 1)));
                else if (kpos % 4 == 0) DKZ_TRY((launch_split<kSeg, kTap>(kName, gj, 1)));
                else DKZ_TRY((launch_split<kSegOdd, kTap>(kName, gj, 1)));
            }
        }
    }
    return 0;
}

}  // extern "C"
