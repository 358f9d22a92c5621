// The 192x256 and 224x256 tiles.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_WHOLE_K_LAUNCHER(, Tile192x256)
HGEMM_WHOLE_K_LAUNCHER(, Tile224x256)

}  // namespace hgemm
