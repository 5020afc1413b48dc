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

// Workgroups of a launch of at most most_tiles tiles, limit at most (the
// tuning's per compute unit, over the chip).
//
// Of k_pp32, a tile per wave: no more waves than tiles, but a workgroup for
// every compute unit: 512 tiles of 32^3 particles took 167 us on 2048
// workgroups and 86 us on 256.
constexpr uint32_t wave_tile_workgroups(uint32_t most_tiles, uint32_t waves, uint32_t limit)
{
    const uint32_t tiles = (most_tiles + waves - 1u) / waves;
    const uint32_t want = tiles < 256u ? 256u : tiles;
    return want < limit ? want : limit;
}

// Of k_pp32_team, a tile per workgroup: two fill a compute unit.
constexpr uint32_t team_tile_workgroups(uint32_t most_tiles, uint32_t limit)
{
    const uint32_t most = limit < 512u ? limit : 512u;
    return most_tiles < 1u ? 1u : most_tiles < most ? most_tiles : most;
}

}  // namespace cuco
