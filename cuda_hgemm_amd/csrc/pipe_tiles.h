// The pipelined kernels' tiles, and where their launchers are instantiated: one source file per group of tiles, so that
// they compile side by side.
#pragma once

#include "mfma_pipelined.h"

namespace hgemm {

// 256x256x64 tile on v_mfma_f32_16x16x32_f16, two B buffers and three A buffers (all 160 KB of LDS)
using Big256 = PipeConfig<256, 256, 64, 2, 2, 2, 16, 1>;
using Mid128 = PipeConfig<128, 128, 64, 2, 2, 5, 16>;
// two LDS buffers (64 KB): two workgroups fit a CU, and one's C tile goes out while the other multiplies.  Pays where
// a workgroup's K loop is shorter than its epilogue and C outgrows the Infinity Cache: 16384^2 x 256 201 -> 170 us.
using Mid128S2 = PipeConfig<128, 128, 64, 2, 2, 2, 16>;
using Small64 = PipeConfig<64, 64, 64, 1, 1, 3, 16>;
// one row of tiles for M <= 64: four waves side by side, 64x32 each
using Row64x128 = PipeConfig<64, 128, 64, 1, 4, 5, 16>;
// one row of tiles for M = 129 ... 192: four stages of 24 + 16 KB are the whole LDS
using Row192x128 = PipeConfig<192, 128, 64, 2, 2, 4, 16>;
using Tile192 = PipeConfig<192, 192, 64, 2, 2, 3, 16>;
using Rect256x128 = PipeConfig<256, 128, 64, 2, 2, 3, 16>;
// Sizes between those, for products whose tiles of the sizes above leave part of the chip idle in their last round or run
// past M: 600 x 14336 x 4096 is 168 tiles of 256x256 (84 us on operands that stay cached, 83 on operands that change from call
// to call), 224 of 160x256 (60, 67).  Wave tiles are any multiple
// of the 16x16 MFMA tile.  The rings are as deep as 160 KB allow (192 and 224 rows: two B buffers, three A buffers).
using Tile160x128 = PipeConfig<160, 128, 64, 2, 2, 4, 16>;
using Tile160x160 = PipeConfig<160, 160, 64, 2, 2, 4, 16>;
using Tile160x256 = PipeConfig<160, 256, 64, 2, 2, 3, 16>;
using Tile192x256 = PipeConfig<192, 256, 64, 2, 2, 2, 16, 1>;
using Tile224x256 = PipeConfig<224, 256, 64, 2, 2, 2, 16, 1>;

#define HGEMM_PIPE_LAUNCHERS(LINKAGE, Cfg)                                                                              \
    LINKAGE template void launch_pipelined<Cfg>(const void *, const void *, void *, size_t, size_t, size_t, const char *, \
                                                PipeKernel);                                                            \
    LINKAGE template void launch_pipelined_split<Cfg>(const void *, const void *, float *, size_t, size_t, size_t, int,   \
                                                      const char *);                                                    \
    LINKAGE template void launch_pipelined_with_tail<Cfg>(const void *, const void *, void *, float *, size_t, size_t,    \
                                                          size_t, int, int, const char *);
#define HGEMM_WHOLE_K_LAUNCHER(LINKAGE, Cfg)                                                                              \
    LINKAGE template void launch_pipelined<Cfg>(const void *, const void *, void *, size_t, size_t, size_t, const char *, \
                                                PipeKernel);
#define HGEMM_SUBTILE_LAUNCHER(LINKAGE, Child)                                                                          \
    LINKAGE template void launch_pipelined_with_subtiles<Big256, Child>(const void *, const void *, void *, size_t, size_t, \
                                                                        size_t, int, const char *);

HGEMM_PIPE_LAUNCHERS(extern, Big256)        // tiles_256.hip
HGEMM_PIPE_LAUNCHERS(extern, Tile192)       // tiles_192.hip
HGEMM_PIPE_LAUNCHERS(extern, Row192x128)
HGEMM_PIPE_LAUNCHERS(extern, Mid128)        // tiles_128.hip
HGEMM_WHOLE_K_LAUNCHER(extern, Mid128S2)
HGEMM_PIPE_LAUNCHERS(extern, Small64)       // tiles_64.hip
HGEMM_PIPE_LAUNCHERS(extern, Row64x128)
HGEMM_WHOLE_K_LAUNCHER(extern, Tile160x128)  // tiles_160.hip
HGEMM_WHOLE_K_LAUNCHER(extern, Tile160x160)
HGEMM_WHOLE_K_LAUNCHER(extern, Tile160x256)
HGEMM_WHOLE_K_LAUNCHER(extern, Tile192x256)  // tiles_224.hip
HGEMM_WHOLE_K_LAUNCHER(extern, Tile224x256)
HGEMM_SUBTILE_LAUNCHER(extern, Rect256x128)  // tiles_256.hip
HGEMM_SUBTILE_LAUNCHER(extern, Mid128)
HGEMM_SUBTILE_LAUNCHER(extern, Small64)

}  // namespace hgemm
