// The 128x128 tile in its two ring depths.
#include "pipe_tiles.h"

namespace hgemm {

HGEMM_PIPE_LAUNCHERS(, Mid128)
template void launch_pipelined<Mid128S2>(const void *, const void *, void *, size_t, size_t, size_t, const char *, PipeKernel);

}  // namespace hgemm
