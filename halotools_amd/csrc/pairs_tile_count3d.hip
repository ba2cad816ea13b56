// pairs_tile_count3d.hip -- matrix-core pair kernels, kModeCount3D variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeCount3D>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
