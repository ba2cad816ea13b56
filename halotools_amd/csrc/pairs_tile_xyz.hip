// pairs_tile_xyz.hip -- matrix-core pair kernels, kModeXYZ variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeXYZ>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
