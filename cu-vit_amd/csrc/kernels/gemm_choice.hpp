// Which GEMM kernel and tile a problem takes: the rules alone, from sizes and
// the number of compute units, on the host. gemm.hip asks them after checking
// what each kernel needs of the operands (alignment, strides, spans).
#pragma once

#include "launch.hpp"

#include <cstddef>
#include <cstdint>

namespace cuvit::detail {

/// Dispatch order puts workgroup x on XCD x % 8.
constexpr int kXcds = 8;

/// Batch entries of one launch: within a grid's y extent (65535), and a multiple
/// of the XCDs, over which entries are spread.
constexpr int kMaxGridY = 65528;

/// Runs launch(first, entries) over a batch of @p count entries, as many at a
/// time as a grid takes, up to the first that fails. (`first` steps past
/// INT_MAX behind the last entries of the largest batches.)
template <typename Launch> hipError_t for_entries(int count, Launch&& launch) {
    for (std::int64_t first = 0; first < count; first += kMaxGridY) {
        const std::int64_t left = count - first;
        const hipError_t launched =
            launch(static_cast<int>(first), static_cast<int>(left < kMaxGridY ? left : kMaxGridY));
        if (launched != hipSuccess) {
            return launched;
        }
    }
    return hipSuccess;
}

inline std::int64_t tile_count(const GemmArgs& args, int bm, int bn) {
    return static_cast<std::int64_t>((args.m + bm - 1) / bm) * ((args.n + bn - 1) / bn) * args.count;
}

/// The px x py split of an entry's tile grid among the 8 XCDs (px * py = 8)
/// that moves the fewest bytes into their L2 caches, A being read once per
/// column block and B once per row block, counting B double when its block
/// would not fit comfortably in one XCD's 4 MB L2. Measured on the ViT-Base
/// bf16 GEMMs: FC1 183 -> 173 us, FC2 129 -> 120 us. The fp32 ViT-Tiny GEMMs
/// (a few MB in all) gained nothing from it, so they keep row-major order.
inline gemm::TileMap tile_map(const GemmArgs& args, int bm, int bn, std::size_t element) {
    gemm::TileMap map{0, 0};
    const int tiles_m = (args.m + bm - 1) / bm;
    const int tiles_n = (args.n + bn - 1) / bn;
    if (element != 2 || static_cast<std::int64_t>(tiles_m) * tiles_n < 64) {
        return map;
    }
    const double a_bytes = static_cast<double>(tiles_m) * bm * args.k * element;
    const double b_bytes = static_cast<double>(tiles_n) * bn * args.k * element;
    constexpr double kL2Budget = 3.0 * (1 << 20);
    double best = 0.0;
    for (const int px : {8, 4, 2, 1}) {
        const int py = 8 / px;
        if (px > tiles_m || py > tiles_n) {
            continue;
        }
        double cost = py * a_bytes + px * b_bytes;
        if (b_bytes / py > kL2Budget) {
            cost *= 2.0;
        }
        if (map.px == 0 || cost < best) {
            best = cost;
            map = gemm::TileMap{px, py};
        }
    }
    return map;
}

/// Whether a batch of @p tiles tiles an entry has its entries dealt to the XCDs
/// whole (TileMap, px < 0), so that each operand is read into one L2 only and
/// lines of C that two tiles share are merged there: where no XCD gets more
/// than a tenth above its share. Entries spread over all XCDs against this, us:
/// bf16 577 x 168 x 384 in 192 entries 63 -> 41, 295 x 296 x 768 in 256 134 ->
/// 77, fp32 196 x 200 x 384 in 192 118 -> 75; against it, 9 entries for 8 XCDs:
/// fp32 562 x 128 x 768 12 -> 15.
inline bool entries_by_xcd(int count, std::int64_t tiles) {
    const std::int64_t dealt = (static_cast<std::int64_t>(count) + kXcds - 1) / kXcds * kXcds;
    // (Tiles within a grid's y extent.)
    return count > 1 && tiles < 16384 && 10 * (dealt - count) <= count;
}

/// Tiles of the XCD that @p map gives the most, over all batch entries.
inline std::int64_t largest_share(const GemmArgs& args, const gemm::TileMap& map, int bm, int bn) {
    const std::int64_t tiles_m = (args.m + bm - 1) / bm;
    const std::int64_t tiles_n = (args.n + bn - 1) / bn;
    if (map.px < 0) {
        return tiles_m * tiles_n * ((static_cast<std::int64_t>(args.count) + kXcds - 1) / kXcds);
    }
    if (map.px == 0) {
        return (tiles_m * tiles_n * args.count + kXcds - 1) / kXcds;
    }
    return (tiles_m + map.px - 1) / map.px * ((tiles_n + map.py - 1) / map.py) * args.count;
}

/// The XCD split for a persistent kernel whose @p turns workgroups per XCD
/// take an XCD's tiles in turn: fewest rounds (the largest block's tiles over
/// @p turns), then the fewest bytes moved into the L2 caches (tile_map's
/// measure). Measured at ViT-Base FC2 on 192 x 256 tiles: a byte-only choice
/// left one XCD 34 tiles for its 32 workgroups, 139 against 88 us.
inline gemm::TileMap balanced_map(const GemmArgs& args, int bm, int bn, int turns, int* rounds_out) {
    const int tiles_m = (args.m + bm - 1) / bm;
    const int tiles_n = (args.n + bn - 1) / bn;
    const double a_bytes = static_cast<double>(tiles_m) * bm * args.k * 2;
    const double b_bytes = static_cast<double>(tiles_n) * bn * args.k * 2;
    constexpr double kL2Budget = 3.0 * (1 << 20);
    gemm::TileMap best{0, 0};
    double best_cost = 0.0;
    int best_rounds = 0;
    for (const int px : {8, 4, 2, 1}) {
        const int py = 8 / px;
        if (px > tiles_m || py > tiles_n) {
            continue;
        }
        const int block = ((tiles_m + px - 1) / px) * ((tiles_n + py - 1) / py);
        const int rounds = (block + turns - 1) / turns;
        double cost = py * a_bytes + px * b_bytes;
        if (b_bytes / py > kL2Budget) {
            cost *= 2.0;
        }
        if (best.px == 0 || rounds < best_rounds || (rounds == best_rounds && cost < best_cost)) {
            best = gemm::TileMap{px, py};
            best_cost = cost;
            best_rounds = rounds;
        }
    }
    *rounds_out = best_rounds;
    return best;
}

/// Relative times of the bf16 kernels with B as [N, K], one 64 x 64 ring tile
/// per CU without GELU being 1, all proportional to K: a ring kernel's busiest
/// CU takes its rounds (the tiles of the XCD with the most, over its CUs) times
/// the tile's cost, the persistent kernel rounds x BM times its cost per row of
/// a 256-wide tile. Fitted to MI355X times at K = 384 and 768, M from 197 to
/// 12608 (us at K = 768: a 64 x 64 tile 2.65, 128 x 64 4.4, 128 x 128 7.7, a
/// persistent 192-row tile 16.7; at K = 384: 1.6, 2.6, 4.2). The GELU weighs
/// more where fewer wavefronts share a SIMD.
constexpr double kRingCost[3] = {1.0, 1.65, 2.9};
constexpr double kRingCostGelu[3] = {1.1, 1.85, 3.3};
/// A tile alone on its CU, with nothing beside it to cover its waits (128 x 64:
/// 4616 x 384 x 384 5.7 us against 5.3 with two 64 x 64 tiles per CU).
constexpr double kRingCostAlone[3] = {1.3, 2.1, 3.0};
/// With GELU and a long K two 64 x 64 tiles with three stages are the faster
/// ones (6504 x 240 x 3072: 30.8 us on 128 x 64, 21.9 on 64 x 64, 41 and 31 with
/// operands from HBM; but 6338 x 264 x 384 7.8 and 8.7).
constexpr double kRingCostAloneGeluLongK[3] = {1.3, 2.3, 3.0};
constexpr double kDmaRow = 0.035;
constexpr double kDmaRowGelu = 0.043;
/// What a round that fills an XCD's slots but for one or none costs more: a
/// workgroup that finds its slot late makes its CU take another tile. 394 x
/// 4096 x 1024 on 128 x 64 tiles, 32 for the 32 CUs: 12.7 us with its operands
/// in the caches, 16.2 without; the 64 x 64 tiles taken so 11.6 and 11.6.
constexpr double kFullRound = 1.15;
/// The ring kernel takes what the persistent kernel could only where its cost
/// is this much smaller. The persistent kernel's time is the same on every card
/// and from wherever its operands come, the ring's is not: 3152 x 2304 x 768,
/// 63 tiles of 128 x 128 for an XCD's 64 slots, took 15.8 to 22.8 us by card
/// against 17.8 to 18.1, and 18.2 to 19.5 against 18.7 to 20.1 with operands
/// from HBM. Below K = 384 the ring has too few stages to hide such operands
/// (9232 x 768 x 256: 10.8 us against 11.2 from the caches, 11.7 against 10.9
/// from HBM).
constexpr double kRingMargin = 0.9;
constexpr double kRingMarginShortK = 0.85;

/// The ring kernel's XCD split: tile_map's where an entry has tiles enough for
/// one, else whole entries where they divide evenly.
inline gemm::TileMap ring_map(const GemmArgs& args, int bm, int bn, std::size_t element) {
    const gemm::TileMap map = tile_map(args, bm, bn, element);
    const std::int64_t tiles = static_cast<std::int64_t>((args.m + bm - 1) / bm) * ((args.n + bn - 1) / bn);
    return map.px == 0 && entries_by_xcd(args.count, tiles) ? gemm::TileMap{-1, -1} : map;
}

struct RingChoice {
    RingTile tile;
    int bm;
    int bn;
    gemm::TileMap map;
    double cost;
};

/// The bf16 ring kernel's cheapest tile for a problem. Where a CU has few tiles and
/// K is long, the tile's own loads are all there is to hide behind, and it
/// takes three stages: 64 x 64 tiles up to two per CU (768 x 3072 on 1576 rows
/// 24.0 -> 19.3 us; FC2 of 4616 rows, 384 x 1536, two microseconds inside its
/// forward), 128 x 128 alone on a CU (768 x 3072 on 4616 rows 31 -> 27 us; two
/// with two stages each beat one at a time with three, 40 against 51 us on 6304
/// rows). Tiles that are alone on their CUs have loading wavefronts beside the
/// computing ones (64 x 32 tiles: 197 x 768 x 768 5.3 -> 4.4 us, 197 x 768 x 3072
/// 11.6 -> 8.5; 64 x 64 from K = 768 on: 197 x 2304 x 768 5.5 -> 4.7; at K = 384
/// 788 x 1152 lost, 4.7 -> 5.3).
inline RingChoice choose_ring(const GemmArgs& args, int units) {
    constexpr RingTile kTiles[3] = {RingTile::k64x64, RingTile::k128x64, RingTile::k128x128};
    constexpr int kHeights[3] = {64, 128, 128};
    constexpr int kWidths[3] = {64, 64, 128};
    const std::int64_t slots = units >= kXcds ? units / kXcds : 1;  // CUs of an XCD
    RingChoice best{RingTile::k64x64, 64, 64, {0, 0}, 0.0};
    for (int i = 0; i < 3; ++i) {
        const std::int64_t tiles = tile_count(args, kHeights[i], kWidths[i]);
        const gemm::TileMap map = ring_map(args, kHeights[i], kWidths[i], 2);
        const std::int64_t share = largest_share(args, map, kHeights[i], kWidths[i]);
        const std::int64_t rounds = (share + slots - 1) / slots;
        double cost = rounds <= 1 ? (args.gelu && args.k >= 1024 ? kRingCostAloneGeluLongK[i] : kRingCostAlone[i])
                                  : static_cast<double>(rounds) * (args.gelu ? kRingCostGelu[i] : kRingCost[i]);
        if (32 * share > 31 * rounds * slots) {
            cost *= kFullRound;
        }
        if (i == 0 || cost < best.cost) {
            best = RingChoice{kTiles[i], kHeights[i], kWidths[i], map, cost};
            if (i == 0 && tile_count(args, 64, 32) <= units) {
                best = RingChoice{RingTile::k64x32Alone, 64, 32, ring_map(args, 64, 32, 2), cost};
            } else if (i == 0 && tiles <= units && args.k >= 768) {
                best.tile = RingTile::k64x64Alone;
            } else if (i == 0 && tiles <= 2 * units && args.k >= 1024) {
                best.tile = RingTile::k64x64Deep;
            } else if (i == 2 && tiles <= units && args.k >= 1024) {
                best.tile = RingTile::k128x128Deep;
            }
        }
    }
    return best;
}

/// The persistent kernel's tile height (0: too few tiles for it), XCD split and
/// cost.
struct DmaChoice {
    int rows;
    gemm::TileMap map;
    double cost;
};

/// BM x 256 tiles for at least half the CUs, BM the height with the fewest
/// rounds x BM, the rounds as balanced_map's split gives them (ViT-Base b64:
/// 320 for FC1, 256 for QKV, 192 for FC2 and the projection).
inline DmaChoice choose_dma(const GemmArgs& args, int units) {
    DmaChoice best{0, {0, 0}, 0.0};
    int best_rounds = 0;
    for (const int height : {192, 256, 320}) {
        if (args.addend != nullptr && height == 320) {
            continue;  // the addend's registers would spill at 320 rows
        }
        if (2 * tile_count(args, height, 256) < units) {
            continue;  // fewer tiles than half the CUs: the ring kernel
        }
        int rounds = 0;
        const gemm::TileMap map = balanced_map(args, height, 256, units / kXcds, &rounds);
        if (best.rows == 0 || rounds * height < best_rounds * best.rows) {
            best = DmaChoice{height, map, 0.0};
            best_rounds = rounds;
        }
    }
    best.cost = best_rounds * best.rows * (args.gelu ? kDmaRowGelu : kDmaRow);
    return best;
}

/// Whether the ring kernel takes a problem that the persistent one could.
inline bool ring_beats_dma(const GemmArgs& args, const RingChoice& ring, const DmaChoice& dma) {
    return dma.rows == 0 || ring.cost < dma.cost * (args.k < 384 ? kRingMarginShortK : kRingMargin);
}

struct RingChoiceF32 {
    RingTileF32 tile;
    gemm::TileMap map;
};

/// The fp32 ring kernel's tile for a problem, by relative times of a CU's row
/// of tiles fitted to MI355X at K = 768 (us: 32 x 32 3.8, 64 x 32 6.9, 64 x 64
/// 13.7 each, more for a tile alone on its CU; these are MFMA-bound, so larger
/// tiles gain little and lose it to a last row of tiles that is not full).
/// While 32 x 16 tiles are alone on their CUs, those, with loading wavefronts
/// beside the computing ones (197 x 192 x 768 7.6 -> 6.6, 197 x 576 x 192 4.0 ->
/// 3.6).
///
/// Two stages hide the L2 but not HBM, which with K above 128 costs more than a
/// larger tile gains: 9182 x 96 x 3072, operands from HBM, 90 us on 64 x 32 tiles,
/// 78 on 32 x 32 with two stages, 66 with three (from the caches 65, 61, 62);
/// 12608 x 320 x 384 41 us on 64 x 64, 36 on 32 x 32 with three. So three stages
/// there, but for many tiles a CU, where more workgroups hide as much (1576 x
/// 2304 x 768 54 us with two, 57 with three), and a larger tile only with a long
/// K and many tiles (10602 x 744 x 3072: 386 us on 64 x 64, 429 on 32 x 32) or
/// with more of them than the tiled kernel leaves to the ring.
/// Entries dealt to the XCDs whole come from the L2 (196 x 200 x 384 in 192
/// entries: 75 us with two stages), and take three for few tiles a CU only.
inline RingChoiceF32 choose_ring_f32(const GemmArgs& args, int units) {
    constexpr RingTileF32 kTiles[3] = {RingTileF32::k32x32, RingTileF32::k64x32, RingTileF32::k64x64};
    constexpr int kHeights[3] = {32, 64, 64};
    constexpr int kWidths[3] = {32, 32, 64};
    constexpr double kCost[3] = {1.0, 1.8, 3.56};
    constexpr double kAlone[3] = {1.5, 2.45, 4.0};
    if (tile_count(args, 32, 16) <= units) {
        return {RingTileF32::k32x16Alone, ring_map(args, 32, 16, 4)};
    }
    const std::int64_t slots = units >= kXcds ? units / kXcds : 1;  // CUs of an XCD
    const gemm::TileMap map = ring_map(args, 32, 32, 4);
    const bool by_entry = map.px < 0;
    const std::int64_t small_rounds = (largest_share(args, map, 32, 32) + slots - 1) / slots;
    const bool larger = by_entry || args.k <= 128 || small_rounds > (args.k >= 1024 ? 6 : 32);
    const int candidates = larger ? 3 : 1;
    RingChoiceF32 best{RingTileF32::k32x32, map};
    double best_cost = 0.0;
    for (int i = 0; i < candidates; ++i) {
        const std::int64_t rounds = (largest_share(args, map, kHeights[i], kWidths[i]) + slots - 1) / slots;
        const double cost = rounds <= 1 ? kAlone[i] : static_cast<double>(rounds) * kCost[i];
        if (i == 0 || cost < best_cost) {
            best.tile = kTiles[i];
            best_cost = cost;
        }
    }
    if (best.tile == RingTileF32::k32x32 && (args.k >= 1024 || (args.k > 128 && small_rounds <= (by_entry ? 4 : 12)))) {
        best.tile = RingTileF32::k32x32Deep;
    }
    return best;
}

/// Whether an fp32 problem that the ring kernel could take runs on the tiled
/// kernel: with many tiles a CU and operands that come from several XCDs' worth
/// of L2 (12507 x 1928 x 512: 224 to 232 us against 235 to 262 by tile; 8221 x
/// 1376 x 768 159 against 160 to 174). At K = 64 the ring is ahead, and at K of
/// 1024 its 64 x 64 tiles are (10602 x 744 x 3072: 386 against 440). Entries run
/// as one problem are the ring's unless they are whole 64-row tiles, since the
/// tiled kernel's stop at each (768 x 588 on 64 entries of 196 rows 151 us there,
/// 126 on the ring; of 256 rows 136 and 149).
inline bool tiled_beats_ring_f32(const GemmArgs& args, int units) {
    return args.rows_per_entry % 64 == 0 && args.k > 64 && (args.count > 1 || args.k < 1024) &&
           tile_count(args, 32, 32) > 32 * static_cast<std::int64_t>(units) && ring_map(args, 32, 32, 4).px >= 0;
}

} // namespace cuvit::detail
