// Entry of a tile's candidate queue: a triangle (any index below 2^31, more
// than 32 bits hold beside the list) and the list it is in, 0 for the cell
// boxes or 1 + a for the rays along axis a.
#pragma once

#include <cstdint>

namespace octlb {

using VoxEntry = uint64_t;

constexpr VoxEntry MakeVoxEntry(int64_t triangle, int list) {
  return static_cast<VoxEntry>(triangle) << 2 | static_cast<VoxEntry>(list);
}
constexpr int64_t VoxTriangle(VoxEntry e) { return static_cast<int64_t>(e >> 2); }
constexpr int VoxList(VoxEntry e) { return static_cast<int>(e & 3); }

}  // namespace octlb
