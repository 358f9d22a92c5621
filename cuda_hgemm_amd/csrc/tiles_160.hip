// The 160-row tiles.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_WHOLE_K_LAUNCHER(, Tile160x128)
HGEMM_WHOLE_K_LAUNCHER(, Tile160x160)
HGEMM_WHOLE_K_LAUNCHER(, Tile160x256)

}  // namespace hgemm
