// The 64-row tiles.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_PIPE_LAUNCHERS(, Small64)
HGEMM_PIPE_LAUNCHERS(, Row64x128)

}  // namespace hgemm
