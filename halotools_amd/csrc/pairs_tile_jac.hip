// pairs_tile_jac.hip -- matrix-core pair kernels, kModeJac variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeJac>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
