// pairs_tile_wsum.hip -- matrix-core pair kernels, kModeWSum variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeWSum>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
