// pairs_tile_wxyz.hip -- matrix-core pair kernels, kModeWXYZ variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeWXYZ>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
