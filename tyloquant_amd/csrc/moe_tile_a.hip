// Plain results of the routed experts' tile kernel (moe_tile.hpp).
#include "moe_tile.hpp"

namespace mfq {
int moe_tile_plain(const MoeTileArgs &t, unsigned grid, hipStream_t st) { return moe_tile_start<false>(t, grid, st); }
}  // namespace mfq
