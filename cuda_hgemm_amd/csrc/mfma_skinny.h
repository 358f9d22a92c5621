// Small-M ("decode shaped") product: M <= 128 rows of A against a large B.
//
// The work is streaming B (N x K halves) from HBM exactly once; MFMA throughput is
// irrelevant.  A workgroup owns BN rows of B and one slice of K, keeps a deep ring of
// direct-to-LDS copies in flight, and multiplies against the (L2-resident) A rows with the
// same LDS layout and fragment scheme as the big-tile kernels.  Rows of the tile beyond M
// are loaded from row M-1 (valid memory) and never stored.
//
// When N alone does not give enough workgroups to fill 256 CUs, K is split: each slice
// writes fp32 partial sums to a workspace and a second kernel adds the slices in index
// order and rounds to fp16, so the result does not depend on scheduling (no float
// atomics) and is bit-identical from run to run.
//
// The reference has no kernel for these shapes: its tiled kernels need M % 256 == 0
// (src/mma/mma_async_stage4.cu:64-66,93-94).
#pragma once

#include "mfma_tiled.h"

namespace hgemm {

// LOOKAHEAD: see the loop
template <int BM_, int BN_, int WAVES_M_, int WAVES_N_, int STAGES_, bool LOOKAHEAD_ = true>
struct SkinnyConfig : TileConfig<BM_, BN_, 64, WAVES_M_, WAVES_N_, STAGES_, LOAD_DMA, LDS_SWIZZLE, true, LOOKAHEAD_> {};

// STREAM_B: B is copied with the non-temporal hint.  Every byte of B is read once; when B is larger than the
// Infinity Cache keeps (N = 28672, K = 4096: 235 MB) the hint is worth 11-12 % (M = 16 ... 64: 64.5 -> 72.6 %, 63.6 ->
// 70.5 %, 57.6 -> 64.7 % of 8 TB/s), when B fits (N = K = 4096) it costs up to 7 %, so the launcher decides by size.
// EDGE: N ends anywhere inside a tile and K % 8 == 0 anywhere inside a chunk: rows of B beyond the last are copied from
// it, columns beyond N are not stored, the last chunk is treated as `tail_pieces` says.
template <class Cfg, bool STREAM_B = false, bool EDGE = false>
__global__ void __launch_bounds__(Cfg::THREADS)
    hgemm_skinny_kernel(const half_t *__restrict__ A, const half_t *__restrict__ B, half_t *__restrict__ C,
                        float *__restrict__ partial, int M, int N, int K, int splits, int tiles_n) {
    constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK;
    constexpr int TM = Cfg::TM, TN = Cfg::TN, KSTEPS = Cfg::KSTEPS, CPR = Cfg::CPR;
    constexpr int ROW_BYTES = Cfg::ROW_BYTES, STAGES = Cfg::STAGES;
    constexpr int L = Cfg::A_DMA + Cfg::B_DMA;
    static_assert(Cfg::WM % 32 == 0 && Cfg::WN % 32 == 0, "wave tile must be a multiple of the 32x32 MFMA tile");

    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / Cfg::WAVES_N, wn = wave % Cfg::WAVES_N;

    // One-dimensional grid, slice-major.  Up to two workgroups of a look-ahead tile to each of the 256 CUs are dealt so that those an XCD runs
    // together are neighbours in a slice (32x64, M = 9 ... 16: 1.01 ... 1.05x).  More of them go round the XCDs, and so do the wider
    // tiles (0.94 ... 1.0x the other way).
    // K of one chunk against a large C lives by what a workgroup does beside its loads and stores: no division for what is not sliced or
    // has at most two rows of tiles (each is 100 clocks and more of one chain), and operands of a k-step at a time in the loop below:
    // 7505 x 8832 x 64 69.2 -> 58.5 us, 8768 x 11971 x 64 136 -> 110, 1664 x 12032 x 64 23.8 -> 20.5 (divisions alone 67.2, 116, 22.9).
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * tiles_n;
    int split = 0, slot = (int)blockIdx.x, tile_m, tile_n;
    if (Cfg::LOOKAHEAD && gridDim.x <= 512)
        slice_and_slot_of_workgroup((int)blockIdx.x, tiles, splits, split, slot);
    else if (splits > 1)
        split = (int)blockIdx.x / tiles, slot = (int)blockIdx.x - split * tiles;
    few_rows_tile(slot, tiles_m, tiles_n, tile_m, tile_n);
    split = __builtin_amdgcn_readfirstlane(split);
    tile_m = __builtin_amdgcn_readfirstlane(tile_m), tile_n = __builtin_amdgcn_readfirstlane(tile_n);
    const int m0 = tile_m * BM;
    const int chunks = EDGE ? chunks_of(K, BK) : K / BK;
    int first_chunk = 0, num_k = chunks;  // K's chunks are dealt to the slices as evenly as whole chunks allow
    if (splits > 1) slice_of_k(chunks, splits, split, first_chunk, num_k);
    const int k_begin = first_chunk * BK;
    const int tail_dup = EDGE && first_chunk + num_k == chunks ? tail_pieces(K, BK) : 0;
    const int last_koff = (num_k - 1) * BK - tail_dup * 8;  // where the last chunk is read from, relative to k_begin

    // ---- copy set-up (rows of A clamped to the last valid row)
    constexpr int DMA_ROW_STEP = Cfg::WAVES * Cfg::ROWS_PER_DMA;
    const int cp_row = wave * Cfg::ROWS_PER_DMA + lane / CPR;
    const int cp_ch = (lane % CPR) ^ swizzle_of_row<Cfg>(cp_row);
    const half_t *a_src[Cfg::A_DMA];
    const half_t *b_src[Cfg::B_DMA];
#pragma unroll
    for (int it = 0; it < Cfg::A_DMA; ++it) {
        int r = m0 + cp_row + it * DMA_ROW_STEP;
        r = r < M ? r : M - 1;
        a_src[it] = A + (size_t)r * K + k_begin + cp_ch * 8;
    }
#pragma unroll
    for (int it = 0; it < Cfg::B_DMA; ++it) {
        int r = tile_n * BN + cp_row + it * DMA_ROW_STEP;
        if constexpr (EDGE) r = r < N ? r : N - 1;
        b_src[it] = B + (size_t)r * K + k_begin + cp_ch * 8;
    }
    const uint32_t cp_lds = (uint32_t)(uintptr_t)lds + wave * 1024;

    auto dma_fetch = [&](int kt, int stage) {
        const int koff = EDGE && kt == num_k - 1 ? last_koff : kt * BK;
        const uint32_t base = cp_lds + stage * Cfg::STAGE_BYTES;
#pragma unroll
        for (int it = 0; it < Cfg::A_DMA; ++it) dma_load16(a_src[it] + koff, base + it * Cfg::WAVES * 1024);
#pragma unroll
        for (int it = 0; it < Cfg::B_DMA; ++it)
            if constexpr (STREAM_B)
                dma_load16_streaming(b_src[it] + koff, base + Cfg::A_BYTES + it * Cfg::WAVES * 1024);
            else
                dma_load16(b_src[it] + koff, base + Cfg::A_BYTES + it * Cfg::WAVES * 1024);
    };

    // ---- fragments
    const int frag_row = lane & 31;
    const int frag_x = (lane >> 5) ^ swizzle_of_row<Cfg>(frag_row);
    const uint32_t a_frag_off = (wm * Cfg::WM + frag_row) * ROW_BYTES;
    const uint32_t b_frag_off = Cfg::A_BYTES + (wn * Cfg::WN + frag_row) * ROW_BYTES;

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // Operands of k-step kk of a chunk.  drop: 16-byte pieces at the chunk's start that must not count (EDGE, last chunk)
    auto load_step = [&](int stage, int drop, int kk, half8 (&a)[TM], half8 (&b)[TN]) __attribute__((always_inline)) {
        const unsigned char *s = lds + stage * Cfg::STAGE_BYTES;
        const uint32_t chunk = (uint32_t)((kk * 2) ^ frag_x) << 4;
#pragma unroll
        for (int i = 0; i < TM; ++i)
            a[i] = *reinterpret_cast<const half8 *>(s + a_frag_off + i * 32 * ROW_BYTES + chunk);
#pragma unroll
        for (int j = 0; j < TN; ++j)
            b[j] = *reinterpret_cast<const half8 *>(s + b_frag_off + j * 32 * ROW_BYTES + chunk);
        if constexpr (EDGE) {
            if (drop > 0) {
                const bool keep = kk * 2 + (lane >> 5) >= drop;
#pragma unroll
                for (int i = 0; i < TM; ++i) a[i] = keep_or_zero(a[i], keep);
#pragma unroll
                for (int j = 0; j < TN; ++j) b[j] = keep_or_zero(b[j], keep);
            }
        }
    };
    auto multiply_step = [&](half8 (&a)[TM], half8 (&b)[TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[j], a[i], acc[i][j], 0, 0, 0);
    };

    // ---- ring of STAGES buffers, STAGES-1 chunks in flight, barrier one chunk ahead (as the look-ahead loop of mfma_tiled.h,
    // for any number of chunks): at the top of iteration kt every operand of chunk kt is on its way into registers; the wait
    // and the barrier confirm chunk kt+1 and retire every wave's reads of chunk kt-1, whose buffer the new copy refills; then
    // the wave issues all operand reads of chunk kt+1, the copy, and only then the MFMAs of chunk kt.  Against a loop that reads a
    // chunk's operands behind its own barrier, at the best slice counts of both: 32x64 1.02 ... 1.05x, 64x64 1.05x (14 ... 18 shapes a
    // class of M; 64 x 4096 x 4096 11.2 -> 10.3 us, unsliced 19.9 -> 14.6).  That loop (!LOOKAHEAD) stays for a few
    // chunks, where it is 0.2 ... 0.3 us ahead (38 x 40 x 136 3.0 us, 3.4), and on the wider tiles, whose waves have more
    // than one MFMA to a k-step (128x64 0.87 ... 1.0x, 64x128 0.89 ... 1.0x, 128x128 1.01x by ring depth).
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < num_k) dma_fetch(s, s);
    int cur = 0, fill = STAGES - 1, kt = 0;
    if constexpr (!Cfg::LOOKAHEAD) {
        for (; kt < num_k; ++kt) {
            if (num_k - 1 - kt >= STAGES - 2)
                wait_vmcnt<(STAGES - 2) * L>();
            else
                wait_vmcnt<0>();
            __syncthreads();
            if (kt + STAGES - 1 < num_k) dma_fetch(kt + STAGES - 1, fill);
            const int drop = kt == num_k - 1 ? tail_dup : 0;
#pragma unroll
            for (int kk = 0; kk < KSTEPS; ++kk) {
                half8 a[TM], b[TN];
                load_step(cur, drop, kk, a, b);
                multiply_step(a, b);
            }
            cur = (cur + 1 == STAGES) ? 0 : cur + 1;
            fill = (fill + 1 == STAGES) ? 0 : fill + 1;
        }
    } else {
        if (num_k >= STAGES - 1)
            wait_vmcnt<(STAGES - 2) * L>();
        else
            wait_vmcnt<0>();
        __syncthreads();
        half8 af[2][KSTEPS][TM], bf[2][KSTEPS][TN];
        auto load_chunk = [&](int stage, int drop, half8 (&a)[KSTEPS][TM], half8 (&b)[KSTEPS][TN]) __attribute__((always_inline)) {
#pragma unroll
            for (int kk = 0; kk < KSTEPS; ++kk) load_step(stage, drop, kk, a[kk], b[kk]);
        };
        load_chunk(0, num_k == 1 ? tail_dup : 0, af[0], bf[0]);
        // STEADY: the copy of chunk kt+STAGES-1 exists (so does chunk kt+1, and the wait count is the full one)
        auto iteration = [&](auto steady, int kt, half8 (&ca)[KSTEPS][TM], half8 (&cb)[KSTEPS][TN], half8 (&na)[KSTEPS][TM],
                             half8 (&nb)[KSTEPS][TN]) __attribute__((always_inline)) {
            constexpr bool STEADY = decltype(steady)::value;
            const int nxt = (cur + 1 == STAGES) ? 0 : cur + 1;
            if (STEADY || kt + 1 < num_k) {
                // copies issued so far: chunks up to min(kt+STAGES-2, num_k-1); all but those beyond kt+1 must land
                if (STEADY || num_k - 1 - (kt + 1) >= STAGES - 3)
                    wait_vmcnt<(STAGES - 3) * L>();
                else
                    wait_vmcnt<0>();
                // a bare barrier: the fence of __syncthreads() would wait for this wave's own operand reads of chunk kt, which
                // nothing behind the barrier overwrites
                __builtin_amdgcn_sched_barrier(0);  // the MFMAs of chunk kt-1 (and their waits) stay in front
                asm volatile("s_barrier" ::: "memory");
                load_chunk(nxt, !STEADY && kt + 1 == num_k - 1 ? tail_dup : 0, na, nb);
            }
            if (STEADY || kt + STAGES - 1 < num_k) dma_fetch(kt + STAGES - 1, fill);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kk = 0; kk < KSTEPS; ++kk) multiply_step(ca[kk], cb[kk]);
            cur = nxt;
            fill = (fill + 1 == STAGES) ? 0 : fill + 1;
        };
        const int steady_end = num_k - (STAGES - 1);
        for (; kt + 2 <= steady_end; kt += 2) {
            iteration(std::true_type{}, kt, af[0], bf[0], af[1], bf[1]);
            iteration(std::true_type{}, kt + 1, af[1], bf[1], af[0], bf[0]);
        }
        for (; kt < num_k; kt += 2) {
            iteration(std::false_type{}, kt, af[0], bf[0], af[1], bf[1]);
            if (kt + 1 < num_k) iteration(std::false_type{}, kt + 1, af[1], bf[1], af[0], bf[0]);
        }
    }

    // ---- epilogue.  Lane l holds row l%32 of each 32x32 tile and four consecutive n per
    // register group: 8 bytes of fp16, or 16 bytes of an fp32 partial sum.
    const int row_in_wave = lane & 31;
    const int col_in_tile = (lane >> 5) << 2;
    const size_t ld = EDGE ? partial_ld(N) : (size_t)N;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + wm * Cfg::WM + i * 32 + row_in_wave;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = tile_n * BN + wn * Cfg::WN + j * 32 + col_in_tile;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (partial) {
                    floatx4 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = acc[i][j][g * 4 + r];
                    if (!EDGE || (size_t)(n + g * 8) < ld)
                        *reinterpret_cast<floatx4 *>(partial + ((size_t)split * M + m) * ld + n + g * 8) = v;
                } else {
                    half4 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = (half_t)acc[i][j][g * 4 + r];
                    if constexpr (EDGE)
                        store_quad_edge(C + (size_t)m * N + n + g * 8, v, n + g * 8, N);
                    else
                        *reinterpret_cast<half4 *>(C + (size_t)m * N + n + g * 8) = v;
                }
            }
        }
    }
}

// C[i] = fp16( partial[0][i] + partial[1][i] + ... ), always added in slice order, VEC
// outputs per thread.  The loads of four slices are issued together before their adds, so
// the kernel is not one memory round trip per slice; small outputs use a small VEC so the
// reduction still spreads over the chip.
// EDGE: N is no multiple of 8: rows of the partial sums are partial_ld(N) apart (`elems` counts them so), rows of C
// start anywhere.
template <int VEC, bool EDGE = false>
__global__ void __launch_bounds__(256)
    splitk_reduce_kernel(const float *__restrict__ partial, half_t *__restrict__ C, size_t elems, int splits, int N) {
    typedef float vec_t __attribute__((ext_vector_type(VEC)));
    typedef half_t hvec_t __attribute__((ext_vector_type(VEC)));
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    if (i >= elems) return;
    const float *src = partial + i;
    vec_t acc = *reinterpret_cast<const vec_t *>(src);
    int s = 1;
    for (; s + 4 <= splits; s += 4) {
        const vec_t v0 = *reinterpret_cast<const vec_t *>(src + (size_t)s * elems);
        const vec_t v1 = *reinterpret_cast<const vec_t *>(src + (size_t)(s + 1) * elems);
        const vec_t v2 = *reinterpret_cast<const vec_t *>(src + (size_t)(s + 2) * elems);
        const vec_t v3 = *reinterpret_cast<const vec_t *>(src + (size_t)(s + 3) * elems);
        acc += v0;
        acc += v1;
        acc += v2;
        acc += v3;
    }
    for (; s < splits; ++s) acc += *reinterpret_cast<const vec_t *>(src + (size_t)s * elems);
    hvec_t out;
#pragma unroll
    for (int r = 0; r < VEC; ++r) out[r] = (half_t)acc[r];
    if constexpr (EDGE) {
        // 32 bits hold the index: the launcher checks
        const uint32_t ld = (uint32_t)partial_ld(N), row = (uint32_t)i / ld;
        const int col = (int)((uint32_t)i - row * ld);
        half_t *dst = C + (size_t)row * N + col;
        typedef hvec_t hvec_any __attribute__((aligned(2)));
        if (col + VEC <= N) {
            *reinterpret_cast<hvec_any *>(dst) = out;
        } else {
#pragma unroll
            for (int r = 0; r < VEC; ++r)
                if (col + r < N) dst[r] = out[r];
        }
    } else {
        (void)N;
        store_streaming(reinterpret_cast<hvec_t *>(C + i), out);
    }
}

template <int VEC>
void launch_splitk_reduce_vec(const float *partial, half_t *C, size_t M, size_t N, int splits) {
    const size_t elems = M * partial_ld(N);
    const dim3 grid((unsigned)div_ceil(elems / VEC, 256)), block(256);
    if (N % 8 == 0)
        splitk_reduce_kernel<VEC, false><<<grid, block, 0, nullptr>>>(partial, C, elems, splits, (int)N);
    else
        splitk_reduce_kernel<VEC, true><<<grid, block, 0, nullptr>>>(partial, C, elems, splits, (int)N);
    HGEMM_CHECK_HIP_ERROR(hipGetLastError());
}
// partial: [splits][M][partial_ld(N)]
inline void launch_splitk_reduce(const float *partial, half_t *C, size_t M, size_t N, int splits) {
    const size_t elems = M * partial_ld(N);
    HGEMM_CHECK(elems < ((size_t)1 << 32));
    if (elems >= (size_t)2 << 20)
        launch_splitk_reduce_vec<8>(partial, C, M, N, splits);
    else if (elems >= (size_t)512 << 10)
        launch_splitk_reduce_vec<4>(partial, C, M, N, splits);
    else
        launch_splitk_reduce_vec<2>(partial, C, M, N, splits);
}

}  // namespace hgemm
