// Tile kernels of some NINT profiles (nint_tile.hpp); the profiles are dealt out over several files to compile side by side.
#include "nint_tile.hpp"

namespace mfq {
int nint_tile_5_28(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    return nint_tile_launch<GenericUnit<5, 28>>(a, shape, glu, splits, st);
}
int nint_tile_6_24(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    return nint_tile_launch<GenericUnit<6, 24>>(a, shape, glu, splits, st);
}
int nint_tile_8_48(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    return nint_tile_launch<GenericUnit<8, 48>>(a, shape, glu, splits, st);
}
}  // namespace mfq
