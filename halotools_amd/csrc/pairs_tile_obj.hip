// pairs_tile_obj.hip -- matrix-core pair kernels, kModeObj variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeObj>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
