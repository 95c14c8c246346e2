// Tile kernels of one family of row-major payloads (row_tile.hpp), in files of their own to compile side by side.
#include "row_tile.hpp"

namespace mfq {
int row_tile_mx8(const RowTileArgs &a, bool f16, int shape, int splits, hipStream_t st) {
    return f16 ? row_tile_launch<kRowMx8F16>(a, shape, splits, st) : row_tile_launch<kRowMx8>(a, shape, splits, st);
}
}  // namespace mfq
