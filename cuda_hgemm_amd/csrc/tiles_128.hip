// The 128x128 tile in its two ring depths.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_PIPE_LAUNCHERS(, Mid128)
HGEMM_WHOLE_K_LAUNCHER(, Mid128S2)

}  // namespace hgemm
