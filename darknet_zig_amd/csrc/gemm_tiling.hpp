// gemm_tiling.hpp -- which tiles and K ranges a matrix product runs in
// (gemm.hip). Host code without HIP, so that tests can ask which tiles a shape
// takes.
#pragma once

#include <algorithm>
#include <cstdint>

namespace dkz {
namespace {

constexpr uint32_t kCus = 256;
constexpr uint32_t kSlab = 16;  // k of a slab

// Tiles and K ranges of one m x n x k product (`z` of them in the launch), by
// the time a CU takes, in cycles: workgroups a CU x slabs x the cycles a slab
// of that tile costs in a full CU, but at least the cycles a slab takes a
// workgroup that has its CU to itself; K ranges add the partials' traffic and a
// launch. The cycles, measured at 2048^3 and 4096^3 (128x128 alone 120 us, two
// a CU 92 us + 17 for the partials, 64x64 126, 128x64 116): a 128x128 slab
// 1450 of them (4 x 362), 128x64 and 64x128 900 (2 x 450), 64x64 520; alone 1900,
// 1300 and 900. Smaller tiles fill the chip at the price of more LDS traffic
// and splitting per product.
//
// stream != 0: tiles that fill no whole round of the chip (`occupancy`
// workgroups a CU) have their slabs laid end to end and cut into equal runs of
// `stream` slabs, one a workgroup, so that the round ends everywhere at once.
// Where whole tiles or uniform ranges leave some CUs with a workgroup more than
// others, or the last round nearly empty, that costs more than the pieces'
// traffic and the second launch: [64,128,56,56]->128 3x3 (1568 tiles, 3.06
// rounds) 435 us in whole tiles, 402 streamed; [32,512,13,13]->1024 (172 and 288
// tiles) both gradients 851 us in uniform ranges, 729 streamed. Below one round,
// where a uniform range a workgroup fits (2048^3 in two, [256,4096]x[4096,1000]
// in eight), the two cost the same and the uniform one is taken.
struct Tiling {
    uint32_t bm, bn, splits, k_chunk, full_tiles, stream;
};
// K ranges go to 1024 of them: weight gradients over large maps have K in the
// millions and a tile or two ([2,3,2048,2048]->16 3x3: 525 thousand slabs, one tile).
//
// partial_floats: room for partials; 0, z > 1 or under eight slabs: K stays whole.
// wide: the kernels with 64-bit addresses, built for 64x64 tiles alone.
constexpr uint64_t kMaxSplits = 1024;
inline Tiling pick_tiling(uint64_t m, uint64_t n, uint64_t k, uint64_t z, uint64_t partial_floats, bool wide) {
    const bool cut = z == 1 && k >= 8 * kSlab && partial_floats > 0;
    const uint64_t max_splits = cut ? std::min(kMaxSplits, partial_floats / (m * n)) : 1;
    struct Cost {
        uint32_t bm, bn, occupancy;
        double full, alone;
        // Of `slabs` slabs in each of per_cu workgroups.
        double cycles(uint64_t slabs, uint64_t per_cu) const {
            const uint64_t rest = per_cu % occupancy;
            return (double)slabs * ((double)(per_cu - rest) * full + (rest ? std::max(alone, (double)rest * full) : 0.0));
        }
    };
    static constexpr Cost kTiles[] = {
        {128, 128, 2, 1450, 1900}, {128, 64, 3, 900, 1300}, {64, 128, 3, 900, 1300}, {64, 64, 4, 520, 900}, {32, 128, 4, 520, 900}};
    static constexpr uint16_t kSplits[] = {1,  2,  3,  4,  5,  6,   7,   8,   10,  12,  14,  16,  20,  24,  28,  32,        40,
                                           48, 56, 64, 80, 96, 112, 128, 160, 192, 224, 256, 320, 384, 512, 640, 768, kMaxSplits};
    constexpr double kFloats = 2.0 * 4 / 2000;  // cycles a float of partials: ~4.2 TB/s at 2.1 GHz
    const uint64_t slabs = (k + kSlab - 1) / kSlab;
    Tiling best{64, 64, 1, (uint32_t)slabs * kSlab, 0, 0};
    double least = 1e300;
    for (const Cost &t : kTiles) {
        if (wide && (t.bm != 64 || t.bn != 64)) continue;
        const uint64_t tiles = (m + t.bm - 1) / t.bm * ((n + t.bn - 1) / t.bn) * z;
        for (const uint32_t want : kSplits) {
            const uint64_t chunk = (slabs + want - 1) / want, splits = chunk ? (slabs + chunk - 1) / chunk : 1;
            if (want > 1 && (want > max_splits || chunk < 4 || tiles * splits > 4 * kCus + tiles)) break;
            double cycles = 3000 + t.cycles(chunk, (tiles * splits + kCus - 1) / kCus);
            if (splits > 1) cycles += 6000 + kFloats * m * n * splits;
            if (cycles < least) {
                least = cycles;
                best = {t.bm, t.bn, (uint32_t)splits, (uint32_t)chunk * kSlab, 0, 0};
            }
        }
        // Runs of at least four slabs, at most 34 pieces a tile.
        const uint64_t slots = kCus * t.occupancy, rest = tiles % slots, line = rest * slabs;
        const uint64_t run = std::max<uint64_t>({(line + slots - 1) / slots, (slabs + 31) / 32, 4});
        if (!cut || rest == 0 || run >= slabs || line + run >= 1ull << 31) continue;
        const uint64_t runs = (line + run - 1) / run, floats = (runs + rest) * t.bm * t.bn;
        if (floats > partial_floats) continue;
        const double cycles = 3000 + t.cycles(slabs, (tiles - rest) / kCus) + t.cycles(run, (runs + kCus - 1) / kCus) + 6000 +
                              2000.0 * (double)((slabs / run + 9) / 8) + kFloats * floats;
        if (cycles < least) {
            least = cycles;
            best = {t.bm, t.bn, 1, (uint32_t)slabs * kSlab, (uint32_t)(tiles - rest), (uint32_t)run};
        }
    }
    return best;
}

}  // namespace
}  // namespace dkz
