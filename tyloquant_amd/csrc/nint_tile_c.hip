// Tile kernels of some NINT profiles (nint_tile.hpp); the profiles are dealt out over several files to compile side by side.
#include "nint_tile.hpp"

namespace mfq {
int nint_tile_3_24(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    return nint_tile_launch<PairedUnit<3, 24>>(a, shape, glu, splits, st);
}
int nint_tile_2_16(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    return nint_tile_launch<PairedUnit<2, 16>>(a, shape, glu, splits, st);
}
int nint_tile_2_32(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    return nint_tile_launch<PairedUnit<2, 32>>(a, shape, glu, splits, st);
}
}  // namespace mfq
