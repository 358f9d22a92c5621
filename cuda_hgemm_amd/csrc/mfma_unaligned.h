// Products whose rows of A and B start on 2-byte boundaries (K % 8 != 0), read where they lie instead of being copied to
// aligned rows first, which is a launch and (M + N) K elements there and back before the first product.
//
// Direct-to-LDS copies want an aligned source, so these rows travel through registers: 16-byte loads at the rows' own
// alignment, one chunk ahead, then 16-byte LDS writes, a share of each in front of every MFMA step so that neither blocks
// the other.  What a row on a 2-byte boundary costs is the load path: a CU takes 30 bytes a clock of such rows, in pieces of 256 bytes as
// in pieces of 128, where it takes 53 of rows on 16-byte boundaries and 63 of rows of whole lines (operands in the L2s,
// profiles/l2_load_rates_by_row_alignment.txt).  64x64: 0.55 us a chunk, of which 0.46 are its 32 KB at that rate.  A chunk is 128 of K, twice
// the other kernels', for half as many barriers and twice the loads in flight; with one wave on a SIMD the loads' latency counts too, which
// is why the wider tiles have eight waves.
// Two chunks ahead in registers measured 0 ... 10 % slower.
#pragma once

#include "mfma_pipelined.h"
#include "mfma_skinny.h"

namespace hgemm {

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_>
struct UnalignedConfig {
    static constexpr int BM = BM_, BN = BN_, BK = 128;
    static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, WAVES = WAVES_M * WAVES_N, THREADS = WAVES * 64;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    static constexpr int MI = 16, PTM = WM / MI, PTN = WN / MI;
    static constexpr int ROW_BYTES = BK * 2, PIECES = BK / 8;  // 16-byte pieces of a row
    static constexpr int ROW_STEP = THREADS / PIECES;          // rows between two loads of a thread
    static constexpr int A_LOADS = BM / ROW_STEP, B_LOADS = BN / ROW_STEP, LOADS = A_LOADS + B_LOADS;
    static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
    static constexpr int C_STRIP_BYTES = 32 * (WN * 2 + 16);
    static constexpr int LDS_BYTES = 2 * STAGE_BYTES > WAVES * C_STRIP_BYTES ? 2 * STAGE_BYTES : WAVES * C_STRIP_BYTES;
    static_assert(BM % ROW_STEP == 0 && BN % ROW_STEP == 0 && ROW_STEP % 8 == 0, "rows are dealt evenly, eight apart at least");
    static_assert(WM % MI == 0 && WN % MI == 0 && LDS_BYTES <= 160 * 1024, "tile");
};

// K of at least one chunk, and short enough that a byte offset inside 128 rows fits 32 bits
inline bool unaligned_runs(size_t K) { return K >= 128 && K <= ((size_t)1 << 23); }

template <class Cfg, bool SPLIT>
__global__ void __launch_bounds__(Cfg::THREADS)
    hgemm_unaligned_kernel(const half_t *__restrict__ A, const half_t *__restrict__ B, half_t *__restrict__ C,
                           float *__restrict__ partial, int M, int N, int K, int slices, int tiles_m, int tiles_n) {
    constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, TM = Cfg::PTM, TN = Cfg::PTN;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / Cfg::WAVES_N, wn = wave % Cfg::WAVES_N;

    int tile_m, tile_n, slice = 0;
    if constexpr (SPLIT) {
        int slot;
        slice_and_slot_of_workgroup((int)blockIdx.x, tiles_m * tiles_n, slices, slice, slot);
        tile_of_position(blocked_order(N, K), slot, tiles_m, tiles_n, tile_m, tile_n);
        slice = __builtin_amdgcn_readfirstlane(slice);
    } else {
        tile_of_workgroup(blocked_order(N, K), 0, (int)blockIdx.x, (int)gridDim.x, tiles_m, tiles_n, tile_m, tile_n);
    }
    tile_m = __builtin_amdgcn_readfirstlane(tile_m);
    tile_n = __builtin_amdgcn_readfirstlane(tile_n);

    // The last chunk is read from K - BK on; the elements that the chunk before it has already multiplied are cleared
    // in both operands (a product of a cleared and an infinite element would be NaN) on their way into LDS.
    int first_chunk, num_k;
    const int chunks = chunks_of(K, BK);
    slice_of_k(chunks, slices, slice, first_chunk, num_k);
    const int drop = first_chunk + num_k == chunks ? (int)((unsigned)chunks * (unsigned)BK - (unsigned)K) : 0;
    const int last_off = (num_k - 1) * BK - drop;
    const half_t *a_base = A + (size_t)tile_m * BM * K + (size_t)first_chunk * BK;
    const half_t *b_base = B + (size_t)tile_n * BN * K + (size_t)first_chunk * BK;

    const int row0 = tid / Cfg::PIECES, piece = tid % Cfg::PIECES;
    const int last_a = M - 1 - tile_m * BM, last_b = N - 1 - tile_n * BN;  // rows beyond the matrix are read from its last row
    uint32_t voff[Cfg::LOADS];
#pragma unroll
    for (int i = 0; i < Cfg::LOADS; ++i) {
        const int r = row0 + (i < Cfg::A_LOADS ? i : i - Cfg::A_LOADS) * Cfg::ROW_STEP, last = i < Cfg::A_LOADS ? last_a : last_b;
        voff[i] = ((uint32_t)(r < last ? r : last) * (uint32_t)K + (uint32_t)piece * 8u) * 2u;
    }
    // XOR of a row's piece index: the 16 lanes that one cycle of a ds_read_b128 serves are eight rows at pieces p and p ^ 2,
    // and 256-byte rows put every row's piece p on the same banks
    auto swizzle = [](int row) { return (row & 5) | ((row & 2) << 2); };
    unsigned char *const wr = lds + row0 * Cfg::ROW_BYTES + ((piece ^ swizzle(row0)) << 4);

    // register i of chunk c: its load, and its way into LDS buffer `stage`
    u32x4 v[Cfg::LOADS];
    auto fetch = [&](int c, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        const int off = c * BK < last_off ? c * BK : last_off;
        const unsigned char *src = reinterpret_cast<const unsigned char *>((i < Cfg::A_LOADS ? a_base : b_base) + off);
        v[i] = *reinterpret_cast<const u32x4_any *>(src + voff[i]);
    };
    u32x4 keep;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        keep[r] = (piece * 8 + 2 * r >= drop ? 0xffffu : 0u) | (piece * 8 + 2 * r + 1 >= drop ? 0xffff0000u : 0u);
    auto commit = [&](bool last, int stage, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if (last) v[i] &= keep;
        *reinterpret_cast<u32x4 *>(wr + stage * Cfg::STAGE_BYTES + i * Cfg::ROW_STEP * Cfg::ROW_BYTES) = v[i];
    };
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const int frag_row = lane % 16, frag_x = (lane / 16) ^ swizzle(frag_row);
    const unsigned char *const ard = lds + (wm * Cfg::WM + frag_row) * Cfg::ROW_BYTES;
    const unsigned char *const brd = lds + (BM + wn * Cfg::WN + frag_row) * Cfg::ROW_BYTES;
    half8 af[2][TM], bf[2][TN];
    auto read = [&](int stage, auto kk_c) __attribute__((always_inline)) {
        constexpr int kk = decltype(kk_c)::value;
        const int off = stage * Cfg::STAGE_BYTES + ((kk * 4) ^ frag_x) * 16;
#pragma unroll
        for (int i = 0; i < TM; ++i) af[kk & 1][i] = *reinterpret_cast<const half8 *>(ard + off + i * 16 * Cfg::ROW_BYTES);
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[kk & 1][j] = *reinterpret_cast<const half8 *>(brd + off + j * 16 * Cfg::ROW_BYTES);
    };
    // step kk of the loop moves registers [first(kk), first(kk + 1)) of the chunks to come
    constexpr int STEPS = BK / 32;
    auto share = [](int kk) constexpr -> int { return kk * Cfg::LOADS / STEPS; };

    static_for<Cfg::LOADS>([&](auto i) { fetch(0, i); });
    static_for<Cfg::LOADS>([&](auto i) { commit(num_k == 1, 0, i); });
    if (num_k > 1) static_for<Cfg::LOADS>([&](auto i) { fetch(1, i); });
    meet();
    // chunk c in LDS buffer u.  STEADY: chunk c + 2 exists, so nothing is asked at run time (a branch around a load
    // would have the compiler wait for the loads of both its sides).
    auto iteration = [&](auto steady, auto u_c, int c) __attribute__((always_inline)) {
        constexpr bool STEADY = decltype(steady)::value;
        constexpr int u = decltype(u_c)::value;
        const bool next = STEADY || c + 1 < num_k, more = STEADY || c + 2 < num_k;
        read(u, std::integral_constant<int, 0>{});
        static_for<STEPS>([&](auto kk_c) __attribute__((always_inline)) {
            constexpr int kk = decltype(kk_c)::value;
            if constexpr (kk + 1 < STEPS) read(u, std::integral_constant<int, kk + 1>{});
            static_for<share(kk + 1) - share(kk)>([&](auto q) __attribute__((always_inline)) {
                using I = std::integral_constant<int, share(kk) + decltype(q)::value>;
                if (next) commit(!STEADY && c + 2 == num_k, u ^ 1, I{});
                if (more) fetch(c + 2, I{});
            });
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[kk & 1][j], af[kk & 1][i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
        meet();
    };
    int c = 0;
    for (; c + 3 < num_k; c += 2) {
        iteration(std::true_type{}, std::integral_constant<int, 0>{}, c);
        iteration(std::true_type{}, std::integral_constant<int, 1>{}, c + 1);
    }
    static_for<3>([&](auto t) {
        if (c + decltype(t)::value < num_k) iteration(std::false_type{}, std::integral_constant<int, decltype(t)::value & 1>{}, c + decltype(t)::value);
    });

    const int m0 = tile_m * BM + wm * Cfg::WM, n0 = tile_n * BN + wn * Cfg::WN;
    if constexpr (SPLIT) {
        const int ld = (int)partial_ld(N);
        store_wave_tile_f32<Cfg, true>([&](auto i_c, auto j_c) -> floatx4 { return acc[decltype(i_c)::value][decltype(j_c)::value]; }, lds,
                                       partial + ((size_t)slice * M + m0) * ld + n0, ld, M - m0, ld - n0, wave, lane);
    } else {
        (void)partial;
        store_wave_tile<Cfg, floatx4, EDGE_ANY>(acc, lds, C, M, N, m0, n0, wave, lane);
    }
}

// partial: splits > 1 only, fp32 [splits][M][partial_ld(N)]
template <class Cfg>
void launch_unaligned(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, int splits, float *partial) {
    static bool configured = [] {
        HGEMM_CHECK_HIP_ERROR(hipFuncSetAttribute(reinterpret_cast<const void *>(&hgemm_unaligned_kernel<Cfg, false>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES));
        HGEMM_CHECK_HIP_ERROR(hipFuncSetAttribute(reinterpret_cast<const void *>(&hgemm_unaligned_kernel<Cfg, true>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES));
        return true;
    }();
    (void)configured;
    const size_t tiles_m = div_ceil(M, (size_t)Cfg::BM), tiles_n = div_ceil(N, (size_t)Cfg::BN), grid = tiles_m * tiles_n * (size_t)splits;
    HGEMM_CHECK(unaligned_runs(K) && splits >= 1 && div_ceil(K, (size_t)Cfg::BK) >= (size_t)splits && grid < ((size_t)1 << 31));
    HGEMM_CHECK(splits == 1 || partial != nullptr);
    auto kernel = splits > 1 ? &hgemm_unaligned_kernel<Cfg, true> : &hgemm_unaligned_kernel<Cfg, false>;
    kernel<<<dim3((unsigned)grid), dim3(Cfg::THREADS), Cfg::LDS_BYTES, nullptr>>>(
        reinterpret_cast<const half_t *>(A), reinterpret_cast<const half_t *>(B), reinterpret_cast<half_t *>(C), partial,
        (int)M, (int)N, (int)K, splits, (int)tiles_m, (int)tiles_n);
    HGEMM_CHECK_HIP_ERROR(hipGetLastError());
    if (splits > 1) launch_splitk_reduce(partial, reinterpret_cast<half_t *>(C), M, N, splits);
}

using Unaligned64 = UnalignedConfig<64, 64, 2, 2>;
using Unaligned96 = UnalignedConfig<96, 96, 2, 2>;
using Unaligned128x64 = UnalignedConfig<128, 64, 4, 2>;
using Unaligned128 = UnalignedConfig<128, 128, 2, 4>;
#define HGEMM_UNALIGNED_LAUNCHERS(LINKAGE)                                                                                     \
    LINKAGE template void launch_unaligned<Unaligned64>(const void *, const void *, void *, size_t, size_t, size_t, int, float *); \
    LINKAGE template void launch_unaligned<Unaligned96>(const void *, const void *, void *, size_t, size_t, size_t, int, float *); \
    LINKAGE template void launch_unaligned<Unaligned128x64>(const void *, const void *, void *, size_t, size_t, size_t, int, float *); \
    LINKAGE template void launch_unaligned<Unaligned128>(const void *, const void *, void *, size_t, size_t, size_t, int, float *);
HGEMM_UNALIGNED_LAUNCHERS(extern)  // tiles_unaligned.hip

}  // namespace hgemm
