// pairs_tile_jack.hip -- matrix-core pair kernels, kModeJack variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeJack>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
