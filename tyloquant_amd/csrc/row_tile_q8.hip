// Tile kernels of one family of row-major payloads (row_tile.hpp), in files of their own to compile side by side.
#include "row_tile.hpp"

namespace mfq {
int row_tile_q8(const RowTileArgs &a, int shape, int splits, hipStream_t st) { return row_tile_launch<kRowQ8>(a, shape, splits, st); }
}  // namespace mfq
