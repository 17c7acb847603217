// The tiles of the segmented reduce (convert.hip): which sorted entries a
// workgroup's tile holds.  m is at most 2^31 - 1, so an entry of the last tile
// and of the tail staged past it needs one bit more than int32_t has: unsigned
// throughout.
#pragma once
#include <cstdint>

namespace mi
{
constexpr int kSegTile = 256;  // sorted entries per tile
constexpr int kSegTail = 96;   // entries past the tile staged with it

// the tiles of m entries
constexpr uint32_t seg_tiles(uint32_t m)
{
    return (m + (uint32_t)kSegTile - 1u) / (uint32_t)kSegTile;
}
// entry k of tile t (k < kSegTile + kSegTail; t = seg_tiles(m) too, past the last tile)
constexpr uint32_t seg_entry(uint32_t t, int k)
{
    return t * (uint32_t)kSegTile + (uint32_t)k;
}
}  // namespace mi
