// The kernel that reads unaligned rows where they lie, every tile.
#include "mfma_unaligned.h"

namespace hgemm {

HGEMM_UNALIGNED_LAUNCHERS()

}  // namespace hgemm
