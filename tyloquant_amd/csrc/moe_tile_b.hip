// act(gate) * up of the routed experts' tile kernel (moe_tile.hpp).
#include "moe_tile.hpp"

namespace mfq {
int moe_tile_glu(const MoeTileArgs &t, unsigned grid, hipStream_t st) { return moe_tile_start<true>(t, grid, st); }
}  // namespace mfq
