// pairs_tile_tan.hip -- matrix-core pair kernels, kModeTan variants (pairs_tile.h).
#include "pairs_tile.h"

namespace hp {
template int launch_tiles_mode<kModeTan>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
}  // namespace hp
