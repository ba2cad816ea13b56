// pairs_tile_proj.hip -- matrix-core pair kernels, kModeProj variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeProj>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
