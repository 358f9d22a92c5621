// The 192-row tiles.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_PIPE_LAUNCHERS(, Tile192)
HGEMM_PIPE_LAUNCHERS(, Row192x128)

}  // namespace hgemm
