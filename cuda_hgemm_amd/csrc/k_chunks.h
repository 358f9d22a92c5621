// K in chunks of `bk`, and the chunks in slices.  Plain integer functions, usable on the host too.  K goes up to 2^31 - 1,
// so what rounds up does so in unsigned arithmetic.
#pragma once

#include "tile_order.h"

namespace hgemm {

// chunks that hold K elements, the last one perhaps not full
HGEMM_HOST_DEVICE int chunks_of(int K, int bk) { return (int)(((unsigned)K + (unsigned)bk - 1u) / (unsigned)bk); }

// K in slices of whole chunks, as even as that allows: the first `chunks % slices` slices walk one chunk more.
// Slice `slice` starts at chunk `first` and walks `count`.
HGEMM_HOST_DEVICE void slice_of_k(int chunks, int slices, int slice, int &first, int &count) {
    const int base = chunks / slices, longer = chunks % slices;
    first = slice * base + (slice < longer ? slice : longer);
    count = base + (slice < longer ? 1 : 0);
}

// ---- K that ends inside a chunk (K % 8 == 0, so rows still start on 16-byte boundaries).  The last chunk is read from
// K - 64 on instead of from its own beginning: every copy stays inside the matrix and as aligned as the others, and
// only a wave-uniform base address changes.  The chunk then starts with `tail_dup` 16-byte pieces that the chunk
// before it has already multiplied; both operands' registers of those pieces are cleared before the last chunk's MFMAs
// (both, because a product of a cleared and an infinite element would be NaN).  Padding the operands instead cost two
// launches and 4 (M + N) K bytes: 1000^3 16.4 -> 7.8 us.
HGEMM_HOST_DEVICE int tail_pieces(int K, int bk) {
    return (int)(((unsigned)K + (unsigned)bk - 1u) / (unsigned)bk * (unsigned)bk - (unsigned)K) >> 3;
}

}  // namespace hgemm
