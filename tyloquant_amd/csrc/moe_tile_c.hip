// Plain results of the routed experts' tile kernel for few pairs an expert (moe_tile.hpp).
#include "moe_tile.hpp"

namespace mfq {
int moe_tile_few_plain(const MoeTileArgs &t, unsigned grid, hipStream_t st) { return moe_tile_few_start<false>(t, grid, st); }
}  // namespace mfq
