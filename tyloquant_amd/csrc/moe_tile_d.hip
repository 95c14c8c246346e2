// act(gate) * up of the routed experts' tile kernel for few pairs an expert (moe_tile.hpp).
#include "moe_tile.hpp"

namespace mfq {
int moe_tile_few_glu(const MoeTileArgs &t, unsigned grid, hipStream_t st) { return moe_tile_few_start<true>(t, grid, st); }
}  // namespace mfq
