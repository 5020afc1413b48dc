// How the long tiles of the FP32 pair kernel are cut into parts (pp32.hip).
#pragma once

#include <cstdint>

namespace cuco {

constexpr uint32_t kPartShare = 32768;  // parts of a box's work
constexpr uint32_t kPartMin = 4096;     // candidates of a part, at least
constexpr uint32_t kPartMost = 1024;    // parts of a tile, at most

// Estimated candidates of one part in a box whose tiles have total of them
// together, and uniform each were they spread evenly.  At most 32 bits: a
// share of more holds any tile whole (a tile's candidates are particles).
constexpr uint32_t tile_part_size(uint64_t total, uint32_t uniform)
{
    uint64_t size = total / kPartShare;
    if (size < kPartMin) size = kPartMin;
    if (size < uniform) size = uniform;
    return size < 0xffffffffull ? (uint32_t)size : 0xffffffffu;
}

// Parts of a tile of e estimated candidates.
constexpr uint32_t tile_parts(uint32_t e, uint32_t size)
{
    return e / size + 1u < kPartMost ? e / size + 1u : kPartMost;
}

// Most parts the tiles of a box of n particles can be listed in.  A tile is
// listed once, and e / size (rounded down) more times.  Over a box these add
// up to at most work / size <= kPartShare (1 + 1 / kPartMin) (size >= work /
// kPartShare - 1 and >= kPartMin; where size is cut to 32 bits, no tile is
// longer), and, as a tile's estimate counts a particle once at most, to at
// most tiles x n / kPartMin.
constexpr uint64_t tile_parts_bound(uint64_t n, uint64_t nblocks)
{
    const uint64_t tiles = (n + 63) / 64 + nblocks;
    const uint64_t all = tiles * (n / kPartMin);
    const uint64_t shares = kPartShare + kPartShare / kPartMin + 1;
    return tiles + (shares < all ? shares : all) + 1;
}

}  // namespace cuco
