// The 256x256 tile, and launches whose last round goes to smaller tiles.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_PIPE_LAUNCHERS(, Big256)
HGEMM_SUBTILE_LAUNCHER(, Rect256x128)
HGEMM_SUBTILE_LAUNCHER(, Mid128)
HGEMM_SUBTILE_LAUNCHER(, Small64)

}  // namespace hgemm
