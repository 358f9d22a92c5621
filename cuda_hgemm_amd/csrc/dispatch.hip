// hgemm_skinny and hgemm_auto: shape-driven choice among the tuned kernels.
#include "../../include/hgemm.h"
#include "mfma_decode.h"
#include "mfma_decode_ring.h"
#include "mfma_decode_resident.h"
#include "pipe_tiles.h"
#include "mfma_ragged.h"
#include "mfma_skinny.h"
#include "mfma_unaligned.h"
#include "plan.h"

#include <atomic>
#include <map>
#include <mutex>

namespace hgemm {

namespace {

constexpr size_t MAX_PARTIAL_BYTES = PlanLimits().partial_bytes;
constexpr size_t MAX_PADDED_BYTES = PlanLimits().operand_bytes;
constexpr size_t SMALL_PADDED_BYTES = (size_t)64 << 20;
constexpr int MAX_DEVICES = 64;

int current_device() {
    int dev = 0;
    HGEMM_CHECK_HIP_ERROR(hipGetDevice(&dev));
    HGEMM_CHECK_MSG(dev >= 0 && dev < MAX_DEVICES, "device %d beyond the %d this library keeps state for", dev, MAX_DEVICES);
    return dev;
}

// Heap workspaces of hgemm_auto / hgemm_skinny, one pair per device, kept for the life of
// the process (the reference keeps its vendor handle the same way,
// src/cublas_tensor_op.cu:18).  Each is allocated once, at its cap, the first time a plan
// needs it (or by hgemm_reserve_workspace).  Operand copies have two buffers: most calls that need one copy a few MB
// (192 x 192 x 1001: 0.8 MB) and are no reason to hold 1 GiB, so copies of up to 64 MiB get a buffer of that size, unless the
// large one is there.  If the cap cannot be had, the size asked for is
// tried, and sizes hipMalloc has refused are remembered so that no later call asks again.
// An entry point never frees or replaces a buffer: a plan that needs more than the buffer
// holds (possible only after such a refusal) is not run, the caller plans again without a
// workspace.  Only hgemm_reserve_workspace and hgemm_release_workspace replace or free, after
// waiting for the device.
//
// g_heap_mutex guards the table AND is held while the launches of a plan that uses a
// workspace are enqueued: every launch goes to the null stream, which runs them in the order
// they were enqueued, so with the lock held two host threads cannot interleave one plan's
// partial-sum kernel with the other's reduction, and no thread holds a workspace pointer
// while another frees it.
struct HeapState {
    Workspace ws;  // partial sums, large operand copies
    unsigned char *small_operands = nullptr;
    size_t small_bytes = 0, small_refused = SIZE_MAX;
    size_t partial_refused = SIZE_MAX, operand_refused = SIZE_MAX;  // smallest size hipMalloc has refused
};
std::mutex g_heap_mutex;
HeapState g_heap[MAX_DEVICES];

// Caller holds g_heap_mutex.  `may_replace`: an existing, smaller buffer may be freed (after a device synchronisation).
bool grow(void **ptr, size_t *have, size_t need, size_t cap, size_t *refused, bool may_replace) {
    if (need <= *have) return true;
    if (need >= *refused) return false;
    if (*ptr) {
        if (!may_replace) return false;
        HGEMM_CHECK_HIP_ERROR(hipDeviceSynchronize());
        HGEMM_CHECK_HIP_ERROR(hipFree(*ptr));
        *ptr = nullptr;
        *have = 0;
    }
    for (size_t want : {need > cap ? need : cap, need}) {
        if (want >= *refused) continue;
        if (hipMalloc(ptr, want) == hipSuccess) {
            *have = want;
            return true;
        }
        (void)hipGetLastError();  // clear the allocation failure
        *ptr = nullptr;
        *refused = want;
    }
    return false;
}

// The device's heap workspace with at least the given sizes; false if it does not hold them and
// cannot be made to.  Caller holds g_heap_mutex.
bool heap_workspace(size_t partial_bytes, size_t operand_bytes, Workspace *out, bool may_replace) {
    HeapState &h = g_heap[current_device()];
    Workspace &w = h.ws;
    bool ok = true;
    if (partial_bytes > w.partial_bytes)
        ok = grow(reinterpret_cast<void **>(&w.partial), &w.partial_bytes, partial_bytes, MAX_PARTIAL_BYTES,
                  &h.partial_refused, may_replace) && ok;
    const bool small = !may_replace && operand_bytes > w.operand_bytes && operand_bytes <= SMALL_PADDED_BYTES;
    if (small)
        ok = grow(reinterpret_cast<void **>(&h.small_operands), &h.small_bytes, operand_bytes, SMALL_PADDED_BYTES,
                  &h.small_refused, false) && ok;
    else if (operand_bytes > w.operand_bytes)
        ok = grow(reinterpret_cast<void **>(&w.operands), &w.operand_bytes, operand_bytes, MAX_PADDED_BYTES,
                  &h.operand_refused, may_replace) && ok;
    *out = w;
    if (small) out->operands = h.small_operands, out->operand_bytes = h.small_bytes;
    return ok;
}

// Scratch of the entry point that allocates nothing: a fixed array in the code object, one
// copy per device, partial sums first and padded operands behind them.  In host code the
// array's name is only a handle for hipGetSymbolAddress; kernels get the device address.
constexpr size_t STATIC_WORKSPACE_BYTES = HGEMM_STATIC_WORKSPACE_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_WORKSPACE_BYTES];
std::mutex g_scratch_mutex;
unsigned char *g_scratch_ptr[MAX_DEVICES];

unsigned char *static_scratch() {
    const int dev = current_device();
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        HGEMM_CHECK_HIP_ERROR(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        HGEMM_CHECK(ptr != nullptr);
        g_scratch_ptr[dev] = reinterpret_cast<unsigned char *>(ptr);
    }
    return g_scratch_ptr[dev];
}

int compute_units() {
    static int cus = [] {
        // A planning query must also work where no GPU is visible: assume one MI355X.
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 256;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 256;
        return n > 0 ? n : 256;
    }();
    return cus;
}

template <class Cfg, bool EDGE>
void launch_splitk_form(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, int splits,
                        const Workspace &ws) {
    static bool configured = [] {
        HGEMM_CHECK_HIP_ERROR(hipFuncSetAttribute(reinterpret_cast<const void *>(&hgemm_skinny_kernel<Cfg, false, EDGE>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES));
        HGEMM_CHECK_HIP_ERROR(hipFuncSetAttribute(reinterpret_cast<const void *>(&hgemm_skinny_kernel<Cfg, true, EDGE>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES));
        return true;
    }();
    (void)configured;
    HGEMM_CHECK(EDGE ? K % 8 == 0 && K >= 64 : N % Cfg::BN == 0 && K % (size_t)Cfg::BK == 0);
    HGEMM_CHECK(splits >= 1 && div_ceil(K, (size_t)Cfg::BK) >= (size_t)splits);
    const size_t tiles_n = div_ceil(N, (size_t)Cfg::BN), tiles = tiles_n * div_ceil(M, (size_t)Cfg::BM);  // < 2^31
    HGEMM_CHECK(tiles * (size_t)splits < ((size_t)1 << 31));
    const dim3 grid((unsigned)(tiles * (size_t)splits));
    float *partial = nullptr;
    if (splits > 1) {
        HGEMM_CHECK(ws.partial != nullptr && ws.partial_bytes >= (size_t)splits * M * partial_ld(N) * sizeof(float));
        partial = ws.partial;
    }
    // a B of 48 MB or more is streamed past the caches: +2-12 % from 64 MB up (N = 8192 ... 28672 at K = 4096),
    // 0-7 % slower at 32 MB (N = K = 4096), where the next call finds parts of B in the Infinity Cache otherwise
    const bool stream_b = div_ceil(M, Cfg::BM) == 1 && N * K >= ((size_t)24 << 20);
    auto kernel = stream_b ? &hgemm_skinny_kernel<Cfg, true, EDGE> : &hgemm_skinny_kernel<Cfg, false, EDGE>;
    kernel<<<grid, dim3(Cfg::THREADS), Cfg::LDS_BYTES, nullptr>>>(
        reinterpret_cast<const half_t *>(A), reinterpret_cast<const half_t *>(B), reinterpret_cast<half_t *>(C),
        partial, (int)M, (int)N, (int)K, splits, (int)tiles_n);
    HGEMM_CHECK_HIP_ERROR(hipGetLastError());
    if (splits > 1) launch_splitk_reduce(partial, reinterpret_cast<half_t *>(C), M, N, splits);
}
template <class Cfg>
void launch_splitk(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, int splits, const Workspace &ws) {
    if (N % Cfg::BN == 0 && K % (size_t)Cfg::BK == 0)
        launch_splitk_form<Cfg, false>(A, B, C, M, N, K, splits, ws);
    else
        launch_splitk_form<Cfg, true>(A, B, C, M, N, K, splits, ws);
}

//                             BM   BN  WM WN stages look-ahead
// Six and five stages leave a CU room for two workgroups (72 and 80 KB).
using Split32x64 = SkinnyConfig<32, 64, 1, 2, 6>;
using Split64x64 = SkinnyConfig<64, 64, 2, 2, 5>;
// ... and for slices of few chunks; 32x64 also for more than two workgroups to a CU, of which three share one at a time
// (18 x 59328 x 2624 52.5 us, 55.7 on six stages; 16 x 9689 x 14912 in five slices 47.0, 54.4)
using Split32x64Short = SkinnyConfig<32, 64, 1, 2, 4, false>;
using Split64x64Short = SkinnyConfig<64, 64, 2, 2, 4, false>;
using Split64x128 = SkinnyConfig<64, 128, 2, 2, 4, false>;
using Split128x64 = SkinnyConfig<128, 64, 2, 2, 4, false>;
using Split128x128 = SkinnyConfig<128, 128, 2, 2, 4, false>;

constexpr size_t SPLIT_SHORT_MAX_CHUNKS = 8;
template <class Cfg, class Short>
void launch_splitk_by_length(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, int splits, const Workspace &ws) {
    const size_t wgs = div_ceil(M, (size_t)Cfg::BM) * div_ceil(N, (size_t)Cfg::BN) * (size_t)splits;
    if (div_ceil(div_ceil(K, (size_t)64), (size_t)splits) <= SPLIT_SHORT_MAX_CHUNKS || (Cfg::BM == 32 && wgs > 2 * (size_t)compute_units()))
        launch_splitk<Short>(A, B, C, M, N, K, splits, ws);
    else
        launch_splitk<Cfg>(A, B, C, M, N, K, splits, ws);
}

// 64x64x64 on four waves (one 32x32 MFMA tile each) with the ladder's kernel: a small tile whose chunk takes a quarter
// of the one-wave tile's matrix-pipe time; for grids that give a CU at most one tile.  Three forms by the number of
// chunks a workgroup walks: the plain 3-stage ring up to 4 (the look-ahead prologue costs more than it returns),
// the look-ahead loop on 5 stages (also the entry point hgemm_mfma_tiled_64x64; 4 stages are 1-2 % ahead while the
// operands sit in L2 and 15-25 % behind once they do not: 512 x 512 x 4096), and on 6 stages from 40 chunks
// (K >= 2560 per slice), where one more chunk in flight pays.
using Small64W4Short = TileConfig<64, 64, 64, 2, 2, 3, LOAD_DMA, LDS_SWIZZLE, true>;
using Small64W4 = TileConfig<64, 64, 64, 2, 2, 5, LOAD_DMA, LDS_SWIZZLE, true, true>;
using Small64W4Deep = TileConfig<64, 64, 64, 2, 2, 6, LOAD_DMA, LDS_SWIZZLE, true, true>;
// two workgroups per CU (grids of one to two tiles per CU): the 4-stage form, 64 KB each, 0-6 % ahead of 5 stages there
using Small64W4Pair = TileConfig<64, 64, 64, 2, 2, 4, LOAD_DMA, LDS_SWIZZLE, true, true>;
constexpr size_t W4_SHORT_MAX_CHUNKS = 4, W4_DEEP_MIN_CHUNKS = 40;

// Pipelined kernel with K cut into `splits` slices: fp32 partial sums per slice, then the
// ordered reduction (the same one the small-M kernel uses), so the result is bit-identical
// from run to run.
template <class Cfg>
void launch_pipelined_plan(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, const Plan &plan,
                           const Workspace &ws) {
    const int splits = plan.splits;
    if constexpr (Cfg::BM == 256 && Cfg::BN == 256) {
        switch (plan.tail_kernel) {
            case KERNEL_R256x128:
                launch_pipelined_with_subtiles<Cfg, Rect256x128>(A, B, C, M, N, K, plan.tail_tiles, "hgemm_auto");
                return;
            case KERNEL_MID128:
                launch_pipelined_with_subtiles<Cfg, Mid128>(A, B, C, M, N, K, plan.tail_tiles, "hgemm_auto");
                return;
            case KERNEL_SMALL64:
                launch_pipelined_with_subtiles<Cfg, Small64>(A, B, C, M, N, K, plan.tail_tiles, "hgemm_auto");
                return;
            default: break;
        }
    }
    if (plan.tail_splits > 1) {
        HGEMM_CHECK(ws.partial != nullptr &&
                    ws.partial_bytes >= (size_t)plan.tail_splits * plan.tail_tiles * Cfg::BM * Cfg::BN * sizeof(float));
        launch_pipelined_with_tail<Cfg>(A, B, C, ws.partial, M, N, K, plan.tail_tiles, plan.tail_splits, "hgemm_auto");
        return;
    }
    if (splits <= 1) {
        launch_pipelined<Cfg>(A, B, C, M, N, K, "hgemm_auto");
        return;
    }
    HGEMM_CHECK(ws.partial != nullptr && ws.partial_bytes >= (size_t)splits * M * partial_ld(N) * sizeof(float));
    launch_pipelined_split<Cfg>(A, B, ws.partial, M, N, K, splits, "hgemm_auto");
    launch_splitk_reduce(ws.partial, reinterpret_cast<half_t *>(C), M, N, splits);
}

// The four-wave 64x64 tile in the form that suits the number of chunks a workgroup walks; EDGE: sizes that end inside a
// tile or chunk.
template <bool EDGE>
void launch_small64_w4(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, int splits, const Workspace &ws) {
    const size_t chunks = div_ceil(K, (size_t)64) / (size_t)(splits > 1 ? splits : 1);
    if (splits <= 1) {
        if (chunks <= W4_SHORT_MAX_CHUNKS)
            launch_tiled<Small64W4Short, EDGE>(A, B, C, M, N, K, "hgemm_auto");
        else if (div_ceil(M, (size_t)64) * div_ceil(N, (size_t)64) > (size_t)compute_units())
            launch_tiled<Small64W4Pair, EDGE>(A, B, C, M, N, K, "hgemm_auto");
        else if (chunks < W4_DEEP_MIN_CHUNKS)
            launch_tiled<Small64W4, EDGE>(A, B, C, M, N, K, "hgemm_auto");
        else
            launch_tiled<Small64W4Deep, EDGE>(A, B, C, M, N, K, "hgemm_auto");
        return;
    }
    check_operands(A, B, C, M, N, K);
    HGEMM_CHECK(ws.partial != nullptr && ws.partial_bytes >= (size_t)splits * M * partial_ld(N) * sizeof(float));
    if (chunks <= W4_SHORT_MAX_CHUNKS)
        launch_tiled_split<Small64W4Short, EDGE>(A, B, ws.partial, M, N, K, splits, "hgemm_auto");
    else if (chunks < W4_DEEP_MIN_CHUNKS)
        launch_tiled_split<Small64W4, EDGE>(A, B, ws.partial, M, N, K, splits, "hgemm_auto");
    else
        launch_tiled_split<Small64W4Deep, EDGE>(A, B, ws.partial, M, N, K, splits, "hgemm_auto");
    launch_splitk_reduce(ws.partial, reinterpret_cast<half_t *>(C), M, N, splits);
}

template <class Cfg>
void launch_unaligned_plan(const void *A, const void *B, void *C, size_t M, size_t N, size_t K, int splits, const Workspace &ws) {
    HGEMM_CHECK(splits == 1 || (ws.partial != nullptr && ws.partial_bytes >= (size_t)splits * M * partial_ld(N) * sizeof(float)));
    launch_unaligned<Cfg>(A, B, C, M, N, K, splits, ws.partial);
}

// ---- cost model for the tile-aligned shapes.  A candidate is a tile (its kernel), how
// many of its workgroups a CU holds, and three times in microseconds fitted to
// measurements on an MI355X over ~60 shapes (rms error 7 %): `fix` per workgroup
// (prologue, epilogue, scheduling) and the time of one 64-wide K chunk with few (`lo`)
// and with all (`hi`) CUs busy -- the chip is power-limited, so a chunk costs more when
// the whole chip computes.  time = launch + full rounds * (fix + chunks * hi)
//                                 + last partial round * (fix + chunks * between lo and hi)
//                                 + reduction of the fp32 partials when K is split.
struct Candidate {
    int kernel, bm, bn, per_cu, stages;
    double fix, lo, hi;
};
constexpr Candidate CANDIDATES[] = {
    {KERNEL_BIG256, 256, 256, 1, 2, 7.92, 0.841, 1.462},
    {KERNEL_T192, 192, 192, 1, 3, 5.17, 0.495, 0.948},
    {KERNEL_R256x128, 256, 128, 1, 3, 4.25, 0.476, 0.856},
    {KERNEL_MID128, 128, 128, 1, 5, 3.17, 0.266, 0.510},
    {KERNEL_SMALL64, 64, 64, 3, 3, 1.39, 0.294, 0.585},
    // K of at most four chunks only (kept to that below); fitted on 8192^2 ... 16384^2 x 256
    {KERNEL_MID128_S2, 128, 128, 2, 2, 1.77, 0.60, 0.885},
    // whole tiles only, at most one workgroup per CU (larger grids are kept from it below: it is behind there);
    // fitted on 16 to 256 workgroups, K = 256 to 16384, in the forms run_plan picks by the length of a slice
    {KERNEL_SMALL64_W4, 64, 64, 1, 3, 2.40, 0.168, 0.195},
    // the same tile with two workgroups sharing a CU (its 5-stage form takes 80 KB of LDS): grids of one to two
    // tiles per CU, unsliced, fewer than 40 chunks (kept to that below); fitted on 1088^2 ... 1408^2, K = 512 ... 2048,
    // where it is 7-19 % ahead of the 128x128 and one-wave 64x64 tiles; from 2 x CUs + 1 tiles on it is far behind
    {KERNEL_SMALL64_W4, 64, 64, 2, 3, 2.40, 0.10, 0.40},
};
// Tiles between those sizes, run unsliced only.  Fitted on grids of 64 ... 512 tiles, K = 512 ... 4096 (rms 5 %), and
// scaled by the 1.14 by which the figures above exceeded the same measurement of their own tiles (the part's clock under
// load differs from one board to the next; only ratios matter to the choice).  One is taken in place of a plan of whole,
// unsliced tiles where it is predicted BETWEEN_MARGIN ahead, about the error of the fits.  A plan that already fills its
// last round, in K slices or on smaller tiles, stays: there these measured 0.90 ... 1.12x, not what was predicted.
// 600 x 14336 x 4096 83 -> 67 us (160x256; operands that change from call to call), 1.06 ... 1.16x on drawn shapes of 10 ... 35 us.
constexpr Candidate BETWEEN_TILES[] = {
    {KERNEL_T160x128, 160, 128, 1, 4, 3.60, 0.341, 0.547}, {KERNEL_T160x160, 160, 160, 1, 4, 4.89, 0.336, 0.667},
    {KERNEL_T160x256, 160, 256, 1, 3, 4.83, 0.543, 1.018}, {KERNEL_T192x256, 192, 256, 1, 2, 5.57, 0.612, 1.181},
    {KERNEL_T224x256, 224, 256, 1, 2, 6.12, 0.671, 1.359},
};
constexpr double BETWEEN_MARGIN = 0.95;
// launch; reduction kernel: fixed + per slice + fp32 partials written and read back.  Partial sums of a few MB
// come back from the L2s: measured 3.0 us behind the same kernel at 2.4 MB against 4.5-5 us at 4.2 MB, and twice
// the slices cost nothing there.  (Refitted with K-sliced launches dealt slice-major: 2.8-7.4 us for 2-17 MB.)
constexpr double LAUNCH_US = 0.16, REDUCE_US = 3.00, REDUCE_SLICE_US = 0.10, REDUCE_BYTES_PER_US = 8700e3;
constexpr double REDUCE_SMALL_US = 2.40, REDUCE_SMALL_SLICE_US = 0.05, REDUCE_SMALL_BYTES = 3e6;
double reduce_us(int slices, double elems) {
    const double bytes = (double)slices * elems * 4.0;
    const bool small = bytes <= REDUCE_SMALL_BYTES;
    return (small ? REDUCE_SMALL_US : REDUCE_US) + (small ? REDUCE_SMALL_SLICE_US : REDUCE_SLICE_US) * slices +
           2.0 * bytes / REDUCE_BYTES_PER_US;
}
// extra cost of finishing a grid with a separate launch for its last round: in K slices / on smaller tiles
constexpr double TAIL_US = 3.6, TAIL_SUB_US = 4.4;
// K that is no multiple of 64: a 128-byte piece of a row straddles two cache lines, so the copies into LDS ask L2 for twice
// the lines.  Chunk times grow by this factor (5112^3 269 us where 5120^3 takes 208; 1.18 ... 1.30 from 1000^3 to 8184^3), and from
// about 4500^3 on it is cheaper to copy both operands first (5112^3 266 us directly, 196 on copies; 4000^2 x 4040 97, 110).
constexpr double OFF_LINE = 1.27;
// By how much the tiles for unaligned rows may be predicted behind such a product on the four-wave 64x64 tile, or on another, and
// still be ahead: both sides' figures leave out some of what the lines cost.  Their time over that of the plan without them, where
// they are taken: 0.78 ... 0.95 (1400^3 15.7 -> 12.5 us, 1528^2 x 2632 27.5 -> 21.4, 1224^2 x 2056 19.3 -> 16.4; 1000^3, left
// alone, 7.8 us and 7.8).  In K slices it was 0.85 ... 1.15 without a pattern (584^2 x 3000 12.9 us, 14.9 on them): not taken.
constexpr double OFF_LINE_SMALL = 1.25, OFF_LINE_OTHERS = 1.12;
// On tiles of 192x192 and unsliced ones of 256x128, K = 4200 ... 12000 (in slices from 6000), a direct product takes longer than
// that in proportion.  75 shapes where the figures alone prefer it by less than this: 1.15x as long as on copies, 54 of them by more
// than 5 %, 7 shorter (1391 x 4586 x 7592 146 us directly, 102 on copies; 2190 x 3878 x 11528 207, 158; 757 x 14816 x 11168 259,
// 332).  Not on other tiles, where it is ahead as often as behind.
double direct_weight(int kernel, int splits, size_t K) {
    const bool longer = kernel == KERNEL_T192 || (kernel == KERNEL_R256x128 && splits == 1);
    return longer && K >= (splits == 1 ? 4200u : 6000u) && K < 12000 ? 1.18 : 1.0;
}
// that copy: launch and gap, and per byte read and written.  Measured on operands that change 5.0 us for 8 MB, 11.2 for 72, 23.7 for 134
// (4095^2 twice; 19.6 on operands that stay cached) and 87.2 for 536; the rate is lower than those say by the 1.14 by which the tiles' figures exceed measurement, so that the two
// compare (27.9 for 134 MB)
constexpr double COPY_US = 3.5, COPY_BYTES_PER_US = 5500e3;
size_t padded_n(size_t N) { return (N + 7) / 8 * 8; }
size_t padded_k(size_t K) { return (K + 63) / 64 * 64; }
// What a plan with copied operands keeps in the workspace: M + N rows of whole chunks.
size_t copy_bytes(size_t M, size_t N, size_t K) { return (M + N) * padded_k(K) * sizeof(half_t); }
// What hgemm_auto_workspace_bytes reports for it and hgemm_auto_static_workspace holds against its array: where N is no
// multiple of 8 also room for a C' (M x N'), up to the cap of the heap workspace.  C is written in place and nothing is
// kept there; callers have sized reservations by the figure, so it stays, and decides no plan.
size_t reported_copy_bytes(size_t M, size_t N, size_t K) {
    const size_t Np = padded_n(N), Kp = padded_k(K);
    const size_t bytes = ((M + Np) * Kp + (Np != N ? M * Np : 0)) * sizeof(half_t);
    const size_t kept = copy_bytes(M, N, K);
    return bytes <= MAX_PADDED_BYTES ? bytes : kept > MAX_PADDED_BYTES ? kept : MAX_PADDED_BYTES;
}

double predict_us(const Candidate &c, size_t M, size_t N, size_t K, int splits, size_t cus) {
    const size_t wgs = div_ceil(M, (size_t)c.bm) * div_ceil(N, (size_t)c.bn) * (size_t)splits;
    const size_t slots = cus * (size_t)c.per_cu;
    const double chunks = (double)div_ceil(div_ceil(K, (size_t)64), (size_t)splits);  // the longest slice
    const size_t full = wgs / slots, rem = wgs % slots;
    double t = LAUNCH_US + (double)full * (c.fix + chunks * c.hi);
    if (rem) t += c.fix + chunks * (c.lo + (c.hi - c.lo) * (double)rem / (double)slots);
    if (splits > 1) t += reduce_us(splits, (double)M * (double)N);
    return t;
}

// The same grid with its last, partly filled round (`rem` workgroups) run in `ts` K slices
// so that it fills the chip too: whole rounds, then one round of rem * ts shorter
// workgroups, then the reduction of their compact fp32 partial sums.
double predict_tail_us(const Candidate &c, size_t M, size_t N, size_t K, int ts, size_t cus) {
    const size_t wgs = div_ceil(M, (size_t)c.bm) * div_ceil(N, (size_t)c.bn), slots = cus * (size_t)c.per_cu;
    const size_t full = wgs / slots, rem = wgs % slots;
    const double chunks = (double)div_ceil(K, (size_t)64);
    double t = LAUNCH_US + (double)full * (c.fix + chunks * c.hi);
    t += LAUNCH_US + c.fix + (double)div_ceil(div_ceil(K, (size_t)64), (size_t)ts) * (c.lo + (c.hi - c.lo) * (double)(rem * ts) / (double)slots);
    t += reduce_us(ts, (double)rem * c.bm * c.bn) + TAIL_US;
    return t;
}

// A grid of 256x256 tiles whose last round (`rem` workgroups) is handed to a smaller tile
// that divides it: whole rounds of the big tile, then rem * parts workgroups of the small
// one.  No partial sums and no reduction.
double predict_subtile_us(const Candidate &big, const Candidate &small, size_t M, size_t N, size_t K, size_t cus) {
    const size_t wgs = div_ceil(M, (size_t)big.bm) * div_ceil(N, (size_t)big.bn), slots = cus * (size_t)big.per_cu;
    const size_t full = wgs / slots, rem = wgs % slots;
    const size_t parts = (size_t)(big.bm / small.bm) * (big.bn / small.bn);
    const size_t small_slots = cus * (size_t)small.per_cu, small_wgs = rem * parts;
    const double chunks = (double)div_ceil(K, (size_t)64);
    double t = LAUNCH_US + (double)full * (big.fix + chunks * big.hi);
    t += LAUNCH_US + (double)(small_wgs / small_slots) * (small.fix + chunks * small.hi);
    if (small_wgs % small_slots)
        t += small.fix + chunks * (small.lo + (small.hi - small.lo) * (double)(small_wgs % small_slots) / (double)small_slots);
    return t + TAIL_SUB_US;
}

// Number of K slices (1 ... 16) for `tiles` output tiles of a kernel for small M, by a model of its time:
//     t(s) = t_B / balance(s) + [s > 1] (t_B weight s M / K + overhead),    t_B = 2 N K bytes at 5 TB/s,
// balance(s) = w / (ceil(w / CUs) CUs) for w = tiles x s workgroups: the busiest CU runs ceil(w / CUs) of them, whether
// side by side or one after the other, so 144 tiles run better in three slices (432 workgroups, two on most CUs) than
// in two (288: two on a few CUs, one on the rest).  The second term is the traffic of the fp32 partial sums (8 M bytes per
// slice and column of C, out and back) against B's (2 K bytes per column), and the launch that adds them.
//   `weight`, `overhead` (us): 16 and 4 on the tiles up to 64x64, fitted to 140 shapes (M = 9 ... 128, N = 1024 ...
// 64448, K = 1024 ... 16256, operands rotated) timed at ten counts: 1 ... 4 % behind the best count on average.  Partial sums
// scaled by the balance too, 8 and 1 us, which this replaced there, chose too many slices since the tiles' loop is faster
// (6 ... 10 % behind: 12 x 8448 x 1280 in three slices 1.42x the time of one).  The wider and the pipelined tiles keep the older
// form (`scaled`), fitted to 91 shapes.
//   From 48 MB of B on, which 64x64 tiles stream past the caches, partial sums weigh less there: 11.  At 16 a B of 130 ... 170 or 257 ... 290 tiles
// was left in one slice (42 x 8896 x 4864 24.9 us, in three 22.1; 59 x 16576 x 4032 41.8, 38.0); at 8 five slices take the place of three, which are
// ahead (35 x 8770 x 6592 0.89x).  220 shapes whose count changed: geomean 1.069, one more than 5 % slower.
// A slice is a whole number of 64-wide chunks, at least
// two (`min_chunks`: the pipelined tiles need as many as their ring has stages); slices differ by at most one chunk.
// `slice_bytes`: fp32 partial sums of one slice; the slices together stay within `limit`.
struct SliceModel {
    double weight, overhead;
    bool scaled;  // partial sums scaled by the balance
};
constexpr SliceModel SLICES{16.0, 4.0, false}, SLICES_LARGE_B{11.0, 4.0, false}, SLICES_WIDE_TILE{8.0, 1.0, true};
int choose_splits(const SliceModel &model, size_t tiles, size_t M, size_t N, size_t cus, size_t K, size_t slice_bytes, size_t limit,
                  size_t min_chunks = 2) {
    int best = 1;
    double best_us = 0.0;
    const double stream_us = 2.0 * (double)N * (double)K / 5e6;
    for (int s = 1; s <= 16; ++s) {
        if (s > 1 && (K % 8 != 0 || div_ceil(K, (size_t)64) / (size_t)s < min_chunks || (size_t)s * slice_bytes > limit)) break;
        const size_t wgs = tiles * (size_t)s;
        const double balance = (double)wgs / (double)(div_ceil(wgs, cus) * cus);
        const double partials = s > 1 ? stream_us * model.weight * s * (double)M / (double)K : 0.0;
        const double us = stream_us / balance + (model.scaled ? partials / balance : partials) + (s > 1 ? model.overhead : 0.0);
        if (s == 1 || us < best_us - 1e-9) {
            best_us = us;
            best = s;
        }
    }
    return best;
}


// ---- kernels for M <= 128 ("decode-shaped": B is streamed once, the bound is HBM bandwidth).  Which kernel runs
// where was settled by timing the candidates against each other on an MI355X, operands rotated so that every call
// reads HBM: library builds with and without a rule, hgemm_auto on both in one process, over K = 256 ... 28672 x
// N = 256 ... 32768 x M = 1 ... 128.  The outcome is this table: the first row that covers a shape, and whose
// kernel can run it (divisibility), decides.  Rows are boxes in (M, N, K, elements of B); the two conditions that
// are not boxes are flags.
enum SmallMFlags {
    RULE_K_BELOW_4N = 1,        // only where K < 4 N (beyond, K slices across workgroups win)
    RULE_K_NOT_16384S = 2,      // not where K is a multiple of 16384 (the ring kernel's 16 rows of B per workgroup then
                                // lie 32 KB apart: 20-28 % behind)
};
struct SmallMRule {
    int m_lo, m_hi;
    size_t n_lo, n_hi, k_lo, k_hi, b_lo, b_hi;  // inclusive bounds; b = N * K, the elements of B
    int flags, kernel;
};
constexpr size_t ANY = ~(size_t)0;
constexpr size_t LARGE_B = (size_t)48 << 20;  // elements: a B of 96 MB
constexpr SmallMRule SMALL_M_RULES[] = {
    // --- M = 1 ... 8.  Below K = 1024 the streaming kernel (as fast or faster, M = 1 by 6-26 %) where it can run,
    // i.e. N % 32 == 0 and K % 256 == 0; else the ring kernel (2.0x median over what ran such shapes before).
    {1, 8, 1, 8192, 256, 1023, 0, ANY, 0, KERNEL_DECODE_BN16},
    // The ring kernel: 0-60 % ahead (median 18 %); not for K < 2048 against N > 8192 (up to 4 % behind at M = 1).  Its
    // copies of B carry the non-temporal hint from 48 MB of B on, and with the hint it is also ahead against a B of
    // 96 MB or more, where the streaming and split-K kernels used to tie with it: K = 1024 ... 12288 x N = 10240 ...
    // 57344, M = 1: 0.97 ... 1.18x (N = 28672, K = 4096: 39.2 -> 35.9 us, 82 % of 8 TB/s; N = 57344: 87 %), M = 8:
    // 0.95 ... 1.31x from K = 2048 (ties at K = 1024).
    {1, 8, 1, 8192, 256, 2047, 0, ANY, 0, KERNEL_DECODE_RING},
    {1, 8, 1, ANY, 2048, ANY, 0, LARGE_B - 1, 0, KERNEL_DECODE_RING},
    {1, 8, 1, ANY, 8192, ANY, LARGE_B, ANY, RULE_K_NOT_16384S, KERNEL_DECODE_RING},
    {1, 5, 1, ANY, 1024, 8191, LARGE_B, ANY, 0, KERNEL_DECODE_RING},
    {6, 8, 1, ANY, 2048, 8191, LARGE_B, ANY, 0, KERNEL_DECODE_RING},
    // M = 6 ... 8 against a B of 96 MB or more with K < 2048: the split-K kernel (2-16 % ahead of the streaming
    // kernel); below M = 6 and for smaller B the streaming kernel stays ahead.
    {6, 8, 1, ANY, 1, ANY, LARGE_B, ANY, 0, KERNEL_SPLIT_32x64},
    {1, 8, 1, ANY, 1, ANY, 0, ANY, 0, KERNEL_DECODE_BN16},
    // --- M = 9 ... 24 against N >= 14336: the persistent kernel that keeps A in registers, where every wave can hold
    // its slice of A (K = 512 ... 1536 per wave, eight waves; four waves of 1280 at K = 5120).  Against what ran these
    // shapes before, over N = 14336 ... 57344: K = 6144 (split-K before) 1.06 ... 1.30x, K = 10240 and 12288 1.08 ... 1.40x,
    // K = 5120 1.07 ... 1.31x from N = 18432 (0.96 ... 1.08x at 14336), K = 8192 (ring kernel) 1.03 ... 1.14x, K = 4096
    // 1.04 ... 1.06x at M = 16 from N = 18432 (N = 28672: 40.1 -> 37.8 us) and level at M = 9, so from M = 13; M = 17 ... 24
    // (two row tiles, 64x128 pipelined tile before) 1.09 ... 1.13x at N = 18432 and 57344 and 0.93 ... 1.09x at N = 28672
    // depending on the box; M = 25 ... 32 mixed up to N = 32000 (0.88 ... 1.07x) and 1.07 ... 1.24x against N = 40960 ...
    // 151936 (the 64x128 tile's second and later rounds cost it more), so from N = 32768; K <= 3072 mixed (0.68 ... 1.2x),
    // so not taken.
    {9, 16, 18432, ANY, 5120, 5120, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RESIDENT},
    // (of these K the kernel takes 6144, 8192, 10240 and 12288)
    {9, 16, 14336, ANY, 6144, 12288, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RESIDENT},
    {13, 16, 18432, ANY, 4096, 4096, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RESIDENT},
    {17, 24, 18432, ANY, 4096, 4096, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RESIDENT},
    {25, 32, 32768, ANY, 4096, 4096, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RESIDENT},
    // --- M = 9 ... 16: the ring kernel up to N = 8192 while K <= 4096 (K <= 8192 up to N = 4096); beyond, K slices
    // across workgroups are up to 29 % ahead -- except, with the non-temporal copies, against a B of 48 MB or more at
    // K = 2048, 4096 and 8192, where every wave walks 1024 of K (M = 12: 1.05 ... 1.29x, M = 16: 0.97 ... 1.23x over
    // N = 10240 ... 57344); at K = 1024, 3072, 6144 and 12288 the split-K kernel stays ahead (0.84 ... 1.06x).
    {9, 16, 1, 8192, 256, 4096, 0, ANY, RULE_K_BELOW_4N, KERNEL_DECODE_RING},
    // (for K of 4 N and more too: 9 x 1344 x 7936 1.18x, 16 x 1603 x 6848 1.16x)
    {9, 16, 1024, 4096, 4097, 8192, 0, ANY, 0, KERNEL_DECODE_RING},
    {9, 16, 8193, ANY, 2048, 2048, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RING},
    {9, 16, 8193, ANY, 4096, 4096, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RING},
    {9, 16, 8193, ANY, 8192, 8192, (size_t)24 << 20, ANY, 0, KERNEL_DECODE_RING},
    // --- M = 17 ... 64 (two or four row tiles of A per wave): the ring kernel while K is short, where one launch beats
    // the split-K kernel plus the launch that adds its slices: K < 1024 up to N = 8192 (median 1.65x), K <= 2048 up
    // to N = 4096 (median 1.31x); and up to K = 4096 for M <= 24 against N = 3072 ... 4096 (median 1.21x; at
    // N <= 2048 M = 24 is 1-9 % behind).
    {17, 64, 1, 8192, 256, 1023, 0, ANY, RULE_K_BELOW_4N, KERNEL_DECODE_RING},
    {17, 64, 1, 4096, 1024, 2048, 0, ANY, RULE_K_BELOW_4N, KERNEL_DECODE_RING},
    {17, 24, 3072, 4096, 2049, 4096, 0, ANY, RULE_K_BELOW_4N, KERNEL_DECODE_RING},
    // Up to M = 32 also where K is longer or N larger than that, against the split-K family at its best count: N = 1536 ... 4095,
    // K = 2049 ... 5631 1.02 ... 1.64x (24 x 3712 x 4800 1.27x, 32 x 3369 x 5376 1.26x; level at N = 4096, 0.95x beyond: 18 x 4608 x 6656);
    // from there on what eight waves' walk costs more than slices do grows with M and N.  With B from HBM, up to K = 7168: 1.03 ... 1.29x
    // below N = 2304, 0.77 ... 1.05x from there on (32 x 2944 x 6912 11.5 us, 14.0; with B in the Infinity Cache the ring is 1.08 ... 1.28x up to
    // K = 7040), M = 17 ... 24 against N from 3264 on 0.94 ... 1.08x (and 1.0 ... 1.27x: 20 x 3915 x 6400 11.8 -> 9.6): this kernel.
    // N = 4300 ... 8000, K = 1024 ... 1792 1.08 ... 1.34x.
    {17, 32, 1536, 2303, 2049, 7168, 0, ANY, 0, KERNEL_DECODE_RING},
    {17, 32, 2304, 4095, 2049, 6143, 0, ANY, 0, KERNEL_DECODE_RING},
    {17, 24, 3264, 4095, 6144, 7168, 0, ANY, 0, KERNEL_DECODE_RING},
    {17, 32, 4097, 8192, 1024, 1792, 0, ANY, 0, KERNEL_DECODE_RING},
    // --- M = 65 ... 128 (eight row tiles): the ring kernel for K <= 512 up to N = 8192, K <= 1024 up to N = 4096
    // (median 1.45x).
    {65, 128, 1, 8192, 256, 512, 0, ANY, RULE_K_BELOW_4N, KERNEL_DECODE_RING},
    {65, 128, 1, 4096, 513, 1024, 0, ANY, RULE_K_BELOW_4N, KERNEL_DECODE_RING},
    // Against N >= 18432 (at least 144 column tiles, i.e. more than half the CUs busy without K slices): one launch
    // of the hand-scheduled 128x128 tile, B copied with the non-temporal hint.  K = 2048 ... 8192 x N = 18432 ...
    // 32768, M = 65 and 128: 3-50 % ahead of the split-K kernels (N = 28672, K = 4096, M = 128: 53.1 -> 48.6 us,
    // 62.6 % of 8 TB/s), K = 384 ... 768 x N = 28672, 57344: 1.11 ... 1.24x; at N = 16384 mixed (0.84 ... 1.14), below
    // it behind (0.76 ... 0.90).  From K = 320, the shortest K its five-stage ring takes.
    // N = 32769 ... 49152 are 257 ... 384 column tiles of 128, i.e. a second round of workgroups on a part of the chip, but
    // at most 256 tiles of 192: one row of the 192x192 tile (its rows beyond M idle, which an HBM-bound kernel can
    // afford) is 1.11 ... 1.34x up to K = 4096 over N = 34816 ... 49152 (M = 100, N = 36864, K = 1024: 27.1 -> 22.5 us);
    // at K = 8192, where the 128x128 tile finishes its second round in K slices, 0.94 ... 1.03x.
    {65, 128, 32769, 49152, 192, 6144, 0, ANY, 0, KERNEL_T192},
    {65, 128, 18432, ANY, 320, ANY, 0, ANY, 0, KERNEL_MID128},
    // M = 33 ... 64 there: the same kernel on a 64x128 tile, four waves side by side.  K = 384 ... 8192 x N = 18432 ...
    // 57344: 1-4 % ahead of the split-K 64x128 kernel where that ran unsliced (N = 28672, K = 4096, M = 64: 43.3 ->
    // 42.4 us, 70 % of 8 TB/s), 1.35x where it ran in two slices (N = 18432, 20480).
    // (the 192-wide tile here only while the second round of 64x128 tiles would be almost empty: N = 34816: 0.97 ... 1.27x
    // over K = 512 ... 4096; N = 40960: 0.91 ... 1.10x; N = 49152: 0.88 ... 1.03x)
    {33, 64, 32769, 36864, 192, 6144, 0, ANY, 0, KERNEL_T192},
    {33, 64, 18432, ANY, 320, ANY, 0, ANY, 0, KERNEL_ROW64x128},
    // M = 17 ... 32 take that tile too once K is long (half its rows are idle, which an HBM-bound kernel can afford):
    // K = 4096, 8192 x N = 18432 ... 57344: 0.97 ... 1.27x over the split-K 32x64 kernel; K = 2944 ... 3584: 1.00 ... 1.15x;
    // at K <= 2560 that kernel stays ahead or level against N >= 28672 (0.92 ... 1.05x).
    {17, 32, 18432, ANY, 3072, ANY, 0, ANY, 0, KERNEL_ROW64x128},
    // M = 33 ... 128 against N = 6144 ... 18431 with a long K: the same two tiles with K in slices (their copies of B
    // non-temporal too), the slice count by the split-K family's model: over N = 6144 ... 16384, M = 64 and 128,
    // K = 8192 and 16384: 0.99 ... 1.34x of the split-K kernels at their best slice count (median 1.17x; M = 128,
    // N = 10240, K = 16384: 106.9 -> 79.8 us); at K = 4096 mixed (0.92 ... 1.13x), at K = 2048 behind (0.80 ... 1.07x).
    // M = 65 ... 128 already from K = 6144: 1.01 ... 1.30x over N = 6144 ... 14336 at K = 6144 and 7168 (median 1.12x).
    {65, 128, 6144, ANY, 6144, ANY, 0, ANY, 0, KERNEL_MID128},
    // From K = 7168 also against N = 3584 ... 6143 (M > 64; 66 x 4800 x 12928 1.34x, 73 x 4288 x 15680 1.30x, 124 x 5568 x 8000 1.25x) and
    // 4096 ... 6143 (M = 33 ... 64; 53 x 6039 x 7488 1.09x, 61 x 4224 x 16064 1.09x).
    {65, 128, 3584, 6143, 7168, ANY, 0, ANY, 0, KERNEL_MID128},
    {33, 64, 4096, ANY, 7168, ANY, 0, ANY, 0, KERNEL_ROW64x128},
    // --- everything else with N % 64 == 0 and K % 64 == 0: the split-K family, the tile by M; 128-wide tiles where
    // N gives enough of them and is a multiple of 128 (they stream B better).
    {1, 32, 1, ANY, 1, ANY, 0, ANY, 0, KERNEL_SPLIT_32x64},
    {33, 64, 16384, ANY, 1, ANY, 0, ANY, 0, KERNEL_SPLIT_64x128},
    {33, 64, 1, ANY, 1, ANY, 0, ANY, 0, KERNEL_SPLIT_64x64},
    {65, 128, 16384, ANY, 1, ANY, 0, ANY, 0, KERNEL_SPLIT_128x128},
    {65, 128, 1, ANY, 1, ANY, 0, ANY, 0, KERNEL_SPLIT_128x64},
};
constexpr int SMALL_M_RULE_COUNT = (int)(sizeof(SMALL_M_RULES) / sizeof(SMALL_M_RULES[0]));

bool small_m_rule_covers(const SmallMRule &r, size_t M, size_t N, size_t K) {
    const size_t b = N * K;
    if (M < (size_t)r.m_lo || M > (size_t)r.m_hi || N < r.n_lo || N > r.n_hi || K < r.k_lo || K > r.k_hi || b < r.b_lo ||
        b > r.b_hi)
        return false;
    if ((r.flags & RULE_K_BELOW_4N) && K >= 4 * N) return false;
    if ((r.flags & RULE_K_NOT_16384S) && K % 16384 == 0) return false;
    return true;
}

// Kernel that stands in for a row's on sizes its own kernel does not divide, 0 if it cannot run them either.  The ring
// kernel's guarded form also stands in for the two decode kernels that have none.
int small_m_edge_kernel(int kernel, size_t M, size_t N, size_t K) {
    if (K % 8 != 0 || K < 64) return KERNEL_NONE;
    const size_t chunks = div_ceil(K, (size_t)64);
    switch (kernel) {
        case KERNEL_DECODE_RING:
        case KERNEL_DECODE_RESIDENT:
        case KERNEL_DECODE_BN16: return decode_ring_edge_supports(M, N, K) ? (int)KERNEL_DECODE_RING_EDGE : (int)KERNEL_NONE;
        case KERNEL_MID128:
        case KERNEL_ROW64x128: return chunks >= 5 ? kernel : (int)KERNEL_NONE;
        case KERNEL_T192: return chunks >= 3 ? kernel : (int)KERNEL_NONE;
        // below K = 320, where no pipelined row covers N >= 16384: 0.75 ... 1.0x of the time, geomean 0.84 (35 x 52088 x 88 7.5 -> 5.9 us)
        case KERNEL_SPLIT_64x128: return N % 8 == 0 && K < 320 ? (int)KERNEL_SPLIT_64x64 : kernel;
        default: return kernel;  // the split-K family
    }
}

// Whole chunks with aligned rows of C (N % 8 == 0, K % 64 == 0): the pipelined tiles further below run these with guarded
// edges too, so a row's stand-in has to be the faster one.  Timed against them over M = 1 ... 128, N = 8 ... 65536, K = 64 ...
// 32768 (5500 shapes; what they take, then the stand-in):
// * Ring kernel: 1.0 ... 2.3x ahead, but behind where few workgroups walk a long K (N <= 1024 from K of about 16384 on, N <= 1536
//   from 20480: 4 x 96 x 32704 11.6 us, 18.3), where eight waves a workgroup leave a CU no room for a second one and the
//   second or third round fills less than a third of the chip (8 x 4200 x 19008 33.2 us, 43.1), and by 1 ... 12 % for M > 32
//   with more workgroups than CUs up to K = 512.
// * 32x64 and 64x64 split-K tiles: 1.0 ... 1.5x ahead, but 0.86 ... 1.0x beyond K = 16384 at N <= 64, where their 16 slices end
//   (42 x 8 x 29568 10.8 us, 12.7), and the latter 0.69 ... 0.95x at M > 32 from N = 16384 on.
// * 128x64 split-K tile: 1.0 ... 1.1x ahead up to K = 1664, and 0.95 ... 1.15x up to K = 8192 at N <= 4096 and for N = 1536 ... 3072;
//   beyond, 0.73 ... 1.05x (75 x 5808 x 25920 57.8 us, 79.0) until its unsliced tiles fill three quarters of the chip (113 x
//   12496 x 2368 25.8 us, 19.5); 0.6 ... 1.0x at N <= 2048 between K = 128 and 2560, where partial sums of more than 64 rows
//   outweigh so short a K (117 x 8 x 1216 6.4 us, 10.5), except for N up to 256 from K = 12 M on (102 x 40 x 1664 7.0, 5.8).
// * The 128-column split-K tiles: 0.53 ... 1.1x, geomean 0.8 (114 x 50336 x 128 6.2 us, 11.7).  The 128x128 one also where K ends
//   inside a chunk, below K = 320 (N = 16384 ... 65536: 0.49 ... 0.97x of the 2-stage 128x128 tile, geomean 0.72; 65 x 34344 x 120
//   6.9 us, 10.0); not where N % 8 != 0, which costs the pipelined tiles their aligned stores.
bool stand_in_pays(int kernel, size_t M, size_t N, size_t K, size_t cus) {
    if (N % 8) return true;
    if (K % 64) return K >= 320 || kernel != KERNEL_SPLIT_128x128;
    switch (kernel) {
        case KERNEL_DECODE_RING_EDGE: {
            const size_t tiles = div_ceil(N, (size_t)16), last = tiles % cus;
            if ((N <= 1024 && K > 16384) || (N <= 1536 && K > 20480) || (M > 32 && tiles > cus && K <= 512)) return false;
            return decode_ring_edge_waves(M, N, K, cus) < 8 || tiles <= cus || tiles > 3 * cus || last == 0 || last * 3 >= cus;
        }
        case KERNEL_SPLIT_32x64: return N > 64 || K <= 16384;
        case KERNEL_SPLIT_64x64: return N < 16384 && (N > 64 || K <= 16384);
        case KERNEL_SPLIT_128x64:
            if (N >= 16384 || (N <= 2048 && K > 128 && K < 2560 && (N > 256 || K < 896 || K < 12 * M))) return false;
            return K <= 1664 || (N <= 4096 && K <= 8192) || (N >= 1536 && N <= 3072) || div_ceil(N, (size_t)64) * 4 > cus * 3;
        case KERNEL_SPLIT_64x128:
        case KERNEL_SPLIT_128x128: return false;
        default: return true;
    }
}

// Sizes in a row's box at which its stand-in is behind what a later row covers them with: the row is passed over.
// * The persistent kernel's K come as a range in the table and it takes four of them.  At any other K the ring kernel's guarded form in its
//   place takes 1.04 ... 1.47 times as long as the 32x64 split-K tile (30 shapes of M = 9 ... 16, N = 14336 ... 40000, K = 6144 ... 12288, geomean
//   1.13: 16 x 15040 x 10648 66.8 us, 98.4; 10 x 14800 x 7232 37.6, 41.3).
// * The ring kernel's rows for M = 17 ... 32 where K ends inside a chunk, whose rows straddle lines: up to N = 4096 to K = 4608 (1.02 ... 1.37x;
//   beyond 0.67 ... 1.13x, geomean 0.86: 20 x 2624 x 7000 11.4 us, 16.6), beyond that N below K = 1024 (from there on level, 0.90 ... 1.10x).
//   M = 9 ... 16 there with K of 4 N and more: to K = 6144 (1.00 ... 1.26x; beyond 0.91 ... 1.03x).
bool stand_in_covers(const SmallMRule &r, size_t M, size_t N, size_t K) {
    int chunks = 0;
    if (r.kernel == KERNEL_DECODE_RESIDENT) return decode_resident_waves(M, K, &chunks) > 0;
    if (r.kernel != KERNEL_DECODE_RING || K % 64 == 0 || M <= 8 || M > 32) return true;
    if (M <= 16) return K <= 6144 || K < 4 * N;
    return N <= 4096 ? K <= 4608 : K < 1024;
}

// An odd number of whole chunks, which no two waves share evenly: on rows of the ring kernel its guarded form instead of the
// split-K family with its second launch.  M = 1 ... 8, N = 1024 ... 28672, K = 1088 ... 4032: 1.08 ... 1.74x (1 x 1984 x 1344
// 5.9 -> 3.5 us, 8 x 28672 x 3008 32.6 -> 27.7); M = 9 ... 16 up to N = 8192: 1.06 ... 1.30x; M = 17 ... 32, N = 1024 ... 4096, up to
// K = 4032: 1.47 ... 2.15x, M = 33 ... 64 up to K = 1984: 0.99 ... 1.90x (62 x 1792 x 1472 7.2 -> 5.0).  Up to N = 4096 also at K = 4160 ...
// 8192: 1.02 ... 1.27x (21 x 3328 x 6976), M = 1 ... 32 at K = 4160 1.00 ... 1.58x; beyond, eight waves leave a CU one workgroup and the second
// round costs more (1 x 4800 x 6976 13.9 us, 17.0).  On rows of the streaming kernel, which such a K shuts out too, below 48 MB of B
// (17728 x 1088: 1.25 ... 1.35x; 24000 x 1856: 0.96 ... 0.98x).  Below N = 1024 few workgroups share the chip and K slices across them stay.
bool odd_chunks_on_ring(int kernel, size_t N, size_t K) {
    if (N % 16 != 0 || N < 1024 || K % 128 != 64 || K < 1024 || K > (N <= 4096 ? 8192u : 4096u)) return false;
    return kernel == KERNEL_DECODE_RING || (kernel == KERNEL_DECODE_BN16 && N * K < ((size_t)24 << 20));
}

// shapes the kernel of a row can run at all (the row is skipped otherwise)
bool small_m_kernel_supports(int kernel, size_t M, size_t N, size_t K) {
    switch (kernel) {
        case KERNEL_DECODE_RING: return decode_ring_supports(M, N, K);
        case KERNEL_DECODE_RESIDENT: return decode_resident_supports(M, N, K);
        case KERNEL_DECODE_BN16: return decode_supports(M, N, K);
        case KERNEL_MID128:
        case KERNEL_ROW64x128: return N % 8 == 0 && K % 64 == 0 && K >= 64 * 5;
        case KERNEL_T192: return N % 8 == 0 && K % 64 == 0 && K >= 64 * 3;
        case KERNEL_SPLIT_64x128:
        case KERNEL_SPLIT_128x128: return skinny_supports(M, N, K) && N % 128 == 0;
        default: return skinny_supports(M, N, K);
    }
}

// One row of BM x 128 tiles, one workgroup per CU, with more column tiles than CUs: the tiles beyond the whole rounds
// would run as a round of their own on a few CUs, so they are cut into K slices that fill the chip (M = 103,
// N = 34304, K = 6656: 268 tiles, 133 us as two rounds, 80 us this way; hipBLASLt 89 us).  Worth its extra launch and
// reduction when the round it shortens is long, i.e. from K of about 2500 ... 4000 on (M = 76, N = 39552, K = 640:
// 19.8 us as two rounds, 23.7 with the 53 tiles of the second in two slices; K = 1280 ... 1792 with the tail: 78 ... 81 %
// of hipBLASLt, K = 4352 ... 6656: 86 ... 111 %).
void one_row_tail(Plan &p, size_t bm, size_t stages, size_t N, size_t K, size_t cus, size_t partial_limit) {
    const size_t tiles = div_ceil(N, (size_t)128), rem = tiles % cus;
    const size_t tile_bytes = bm * 128 * sizeof(float);
    if (tiles <= cus || rem == 0) return;
    size_t ts = cus / rem < 16 ? cus / rem : 16;
    while (ts >= 2 && (shortest_slice(K, 64, (int)ts) < 64 * stages || ts * rem * tile_bytes > partial_limit)) --ts;
    if (ts >= 2 && (double)(K / 64) * (1.0 - 1.0 / (double)ts) > 32.0) {
        p.tail_tiles = (int)rem;
        p.tail_splits = (int)ts;
        p.partial_bytes = ts * rem * tile_bytes;
    }
}

}  // namespace

bool skinny_supports(size_t M, size_t N, size_t K) {
    return M >= 1 && M <= 128 && N > 0 && N % 64 == 0 && K > 0 && K % 64 == 0;
}

bool same_choice(const Plan &a, const Plan &b) {
    return a.kernel == b.kernel && a.splits == b.splits && a.tail_tiles == b.tail_tiles && a.tail_splits == b.tail_splits &&
           a.tail_kernel == b.tail_kernel;
}
bool left_out(const PlanLimits &limits, const Plan &p) {
    for (int i = 0; i < limits.excluded_count; ++i)
        if (same_choice(limits.excluded[i], p)) return true;
    return false;
}
bool left_out(const PlanLimits &limits, int kernel, int splits, int tail_tiles = 0, int tail_splits = 1,
              int tail_kernel = KERNEL_NONE) {
    Plan p;
    p.kernel = kernel, p.splits = splits, p.tail_tiles = tail_tiles, p.tail_splits = tail_splits, p.tail_kernel = tail_kernel;
    return left_out(limits, p);
}

// What runs products of one chunk of K and a part of the next on ragged sizes instead of the 2-stage 128x128 tile's guarded
// form, or of one chunk instead of the 64x64 split-K tile's; KERNEL_NONE: nothing.
// * Fewer 128x128 tiles than half the CUs: the 64x64 split-K tile, 0.60 ... 0.89x of the time (2308 x 40 x 80 4.4 -> 3.8 us).  N of
//   less than one such tile only with aligned rows of C.
// * Bound by writing C, in lines that rows not a multiple of 32 bytes straddle: the guarded 128x128x32 kernel, whose 8-byte
//   stores merge in L2.  One chunk from C of 3 M elements on 0.64 ... 1.13x (2315 x 55336 x 64 153 us, 99); up to K = 96 from
//   16 rounds of 128x128 tiles on 0.77 ... 0.96x (11111 x 10444 x 72 119 us, 98; 7873 x 56748 x 88 471, 399).
int short_k_kernel(size_t M, size_t N, size_t K, size_t cus) {
    const size_t tiles = div_ceil(M, (size_t)128) * div_ceil(N, (size_t)128);
    if (K > 128 || (N % 8 == 0 && K % 64 == 0 && K > 64)) return KERNEL_NONE;
    if (K == 64) return N % 64 && N % 4 == 0 && M * N >= ((size_t)3 << 20) ? KERNEL_RAGGED : KERNEL_NONE;
    if (M > 128 && tiles * 2 <= cus && (N % 8 == 0 || N >= 64)) return KERNEL_SPLIT_64x64;
    return K <= 96 && N % 4 == 0 && N % 16 && tiles > 16 * cus ? KERNEL_RAGGED : KERNEL_NONE;
}

// One pass that copies A and B with rows of whole 64-wide chunks, then the plan for that K (same products, same result);
// no plan where the copies do not fit.
Plan plan_on_copies(size_t M, size_t N, size_t K, const PlanLimits &limits) {
    if (K < 192 || copy_bytes(M, N, K) > limits.operand_bytes) return Plan();
    PlanLimits inner_limits;
    inner_limits.partial_bytes = limits.partial_bytes;
    inner_limits.operand_bytes = 0;
    Plan p = plan_for(M, N, padded_k(K), inner_limits);
    p.inner_kernel = p.kernel;
    p.kernel = KERNEL_PADDED;
    if (p.est_us > 0.0) p.est_us += COPY_US + 4.0 * (double)((M + N) * padded_k(K)) / COPY_BYTES_PER_US;
    p.operand_bytes = copy_bytes(M, N, K);
    return p;
}

// K % 8 != 0 read where it lies (mfma_unaligned.h).  Times as in CANDIDATES, of a 128-wide chunk, fitted on 80 shapes (M = 2 ... 4863,
// N = 5 ... 19948, K = 215 ... 14927, up to 16 slices; rms 6 ... 11 %) and on the same scale as those.  64x64 twice: one
// workgroup to a CU, and two that share its load path.
constexpr Candidate UNALIGNED_TILES[] = {
    {KERNEL_UNALIGNED64, 64, 64, 1, 1, 3.60, 0.539, 0.709},
    {KERNEL_UNALIGNED64, 64, 64, 2, 1, 3.44, 0.824, 1.361},
    {KERNEL_UNALIGNED96, 96, 96, 1, 1, 4.81, 0.944, 1.007},
    {KERNEL_UNALIGNED128x64, 128, 64, 1, 1, 3.95, 0.935, 0.962},
    {KERNEL_UNALIGNED128, 128, 128, 1, 1, 5.09, 1.206, 1.516},
};
// What a plan on copies is taken to last beside those figures.  Its own estimate says too little for short products (15 ... 20 us of it
// 1.17x: two launches back to back) and too much for long ones (60 us and more 0.90x), where the tiles above are at 0.93x throughout.
// Of 2038 shapes timed both ways (M = 1 ... 5000, N = 16 ... 60000, K = 192 ... 16000) 18 run more than 5 % slower than on copies and the choice
// is 0.27 % behind the better of the two on average; with 4 us more below an estimate of 40 us, and none beyond, 45 and 0.42 %
// (636 x 3819 x 2821 31.8 us on copies, 39.4).  Copies that do not stay in the 256 MB Infinity Cache with what they are made of last
// what they are estimated at (474 x 14498 x 9292 235 us, 193 without).
double copies_us(const Plan &copied) {
    const double more = 9.5 - 0.28 * copied.est_us, least = 2 * copied.operand_bytes > (size_t)256000000 ? 0.0 : -5.0;
    return copied.est_us + (more > 4.0 ? 4.0 : more < least ? least : more);
}
Plan plan_on_unaligned_rows(size_t M, size_t N, size_t K, size_t cus, const PlanLimits &limits) {
    Plan p;
    if (!unaligned_runs(K)) return p;
    const size_t slice_bytes = M * partial_ld(N) * sizeof(float), chunks = div_ceil(K, (size_t)128);
    for (const Candidate &c : UNALIGNED_TILES) {
        const size_t tiles = div_ceil(M, (size_t)c.bm) * div_ceil(N, (size_t)c.bn);
        for (int s = 1; s <= 16 && (size_t)s <= chunks; ++s) {
            const size_t wgs = tiles * (size_t)s, slots = cus * (size_t)c.per_cu;
            if (s > 1 && (wgs > 2 * slots || (size_t)s * slice_bytes > limits.partial_bytes)) break;
            if (wgs >= (size_t)1 << 31 || left_out(limits, c.kernel, s)) continue;
            if (c.kernel == KERNEL_UNALIGNED64 && (c.per_cu == 1) != (wgs <= cus)) continue;
            const double t = predict_us(c, M, N, div_ceil(K, (size_t)128) * 64, s, cus);  // (predict_us counts chunks of 64)
            if (p.kernel != KERNEL_NONE && t >= p.est_us) continue;
            p.kernel = c.kernel;
            p.splits = s;
            p.est_us = t;
            p.partial_bytes = s > 1 ? (size_t)s * slice_bytes : 0;
        }
    }
    return p;
}

// M <= 128: choices come from timing every candidate (tile x slices) on the specification's
// decode shapes on an MI355X, operands rotated so small problems read HBM.  Larger,
// tile-aligned shapes: the cheapest (tile, slices) pair under the cost model above.
Plan plan_for(size_t M, size_t N, size_t K, const PlanLimits &limits) {
    Plan p;
    if (M == 0 || N == 0 || K == 0) return p;
    const size_t cus = (size_t)compute_units();
    const size_t slice_bytes = M * partial_ld(N) * sizeof(float);  // fp32 partial sums of one K slice of the whole product
    // M <= 128: the first row of the table above that covers the shape and whose kernel can run it; where there is none
    // (N or K that nothing divides), the first covering row whose kernel has a form with guarded edges
    for (int at = 0; at < 2 * SMALL_M_RULE_COUNT && M <= 128; ++at) {
        const SmallMRule &r = SMALL_M_RULES[at % SMALL_M_RULE_COUNT];
        const bool edges = at >= SMALL_M_RULE_COUNT;
        if (limits.every_small_m_kernel ? (M < (size_t)r.m_lo || M > (size_t)r.m_hi) : !small_m_rule_covers(r, M, N, K)) continue;
        const bool odd_chunks = !edges && !small_m_kernel_supports(r.kernel, M, N, K) && odd_chunks_on_ring(r.kernel, N, K);
        if (!edges && !odd_chunks && !small_m_kernel_supports(r.kernel, M, N, K)) continue;
        p = Plan();
        p.kernel = edges || odd_chunks ? small_m_edge_kernel(r.kernel, M, N, K) : r.kernel;
        if (p.kernel == KERNEL_NONE) continue;
        if (edges && !limits.every_small_m_kernel && !stand_in_covers(r, M, N, K)) {
            p = Plan();
            continue;
        }
        if (edges && !limits.every_small_m_kernel && !stand_in_pays(p.kernel, M, N, K, cus)) {
            p = Plan();
            break;
        }
        switch (p.kernel) {
            case KERNEL_DECODE_RING: {
                p.splits = decode_ring_waves(M, N, K, cus);
                // Chunks that do not come out even over the waves the rule asks for: dealt unevenly rather than to half as
                // many waves, where those would walk more than 1024 of K each and a CU has one workgroup at most
                // (N = 1216 ... 4096, K = 2176 ... 15744: 0.99 ... 1.68x, median 1.25x; 1 x 1984 x 9600 18.4 -> 11.5 us on
                // eight waves for two; N = 16 ... 1200, K up to 25500: 0.99 ... 2.30x, geomean 1.58).  A shorter walk is latency either way (0.98 ... 1.11x), and with more workgroups
                // they hide the difference and the even form is ahead (N = 5184 ... 46592: 0.84 ... 1.07x).
                const int uneven = decode_ring_edge_waves(M, N, K, cus);
                if (uneven > p.splits && N / 16 <= cus && K > 1024 * (size_t)p.splits) p.kernel = KERNEL_DECODE_RING_EDGE, p.splits = uneven;
                break;
            }
            case KERNEL_DECODE_RING_EDGE: p.splits = decode_ring_edge_waves(M, N, K, cus); break;
            case KERNEL_DECODE_RESIDENT: {
                int chunks = 0;
                p.splits = decode_resident_waves(M, K, &chunks);
                break;
            }
            case KERNEL_DECODE_BN16: {  // the streaming kernel: 16 or 32 columns per workgroup
                int bn = 16, waves = 1;
                decode_plan(M, N, K, cus, &bn, &waves);
                p.kernel = bn == 16 ? KERNEL_DECODE_BN16 : KERNEL_DECODE_BN32;
                p.splits = waves;
                break;
            }
            case KERNEL_T192: p.splits = 1; break;
            case KERNEL_MID128:
            case KERNEL_ROW64x128: {
                // up to one workgroup per CU: K slices by the split-K family's model (the same balance against the
                // same partial sums); more tiles than CUs: whole rounds unsliced, the rest in K slices
                const size_t tiles = div_ceil(N, (size_t)128);
                // (from K = 6144: below, slices were measured level or behind -- M = 96, N = 18432, K = 4096: 40.8 us
                // unsliced, 43.6 in three; at K = 6144 and 7168 against N = 18432 1.00 ... 1.04x)
                p.splits = tiles <= cus && K >= 6144 ? choose_splits(SLICES_WIDE_TILE, tiles, M, N, cus, K, slice_bytes, limits.partial_bytes, 5) : 1;
                if (p.splits > 1) p.partial_bytes = (size_t)p.splits * slice_bytes;
                if (tiles > cus) one_row_tail(p, r.kernel == KERNEL_MID128 ? 128 : 64, 5, N, K, cus, limits.partial_bytes);
                break;
            }
            default: {  // the split-K family: K slices across workgroups, then the ordered reduction
                const size_t bn = (r.kernel == KERNEL_SPLIT_64x128 || r.kernel == KERNEL_SPLIT_128x128) ? 128 : 64;
                // By whole tiles: an N of 8 takes as long as one of 64 (57 x 8 x 1552 unsliced 8.9 us, in 12 slices as at N = 64
                // 5.5; 83 x 17 x 1072 9.5, 6.0).  Below K = 896, and 1280 on the 32-row tile, what N itself asks for, which is
                // no slices at N = 8: the second launch costs more than they return (9 x 24 x 424 3.8 us, in three slices 6.0;
                // 16 x 3 x 1072 6.4, 7.4; 48 x 8 x 944 6.1, 5.9).
                const size_t columns = K >= (p.kernel == KERNEL_SPLIT_32x64 ? 1280u : 896u) ? div_ceil(N, bn) * bn : N;
                size_t tiles = div_ceil(N, bn);
                // M = 65 ... 128 against a B of less than 32 MB: as two rows of 64x64 tiles, whose rings leave a CU room for two
                // workgroups, and half as many slices.  Against the 128x64 tile: up to one of them to a CU, and less than 20 MB of B where K is 2500
                // and more and N 2048, 355 shapes 0.85 ... 1.70x, geomean 1.19 (75 x 1024 x 1664 7.7 -> 6.4 us, 113 x 2560 x 1792 11.2 -> 8.0); more
                // B than that 0.77 ... 1.07x where B comes from HBM, geomean 0.90 (124 x 4160 x 3328 15.2 us, 18.3; from the Infinity Cache the two
                // rows are 4 % ahead), except N of more than a third of the CUs' 128x64 tiles, which leave room for two slices only (90 x
                // 6272 x 2560 15.9 us from HBM and 13.1 from the cache, as two rows 15.2 and 11.0).  Two to a CU where the 128x64 tile has one:
                // ahead below K = 192 and from M = 96 on (1.0 ... 1.16x; below 0.87 ... 1.0x), 0.78 ... 1.0x for longer K (76 x 10048 x 480 6.3, 8.1);
                // ahead again where that tile needs a second round (N > 16384: 1.04 ... 1.32x, 112 x 37824 x 128 11.7 -> 8.9).
                const size_t two_rows = tiles * div_ceil(M, (size_t)64);
                if (p.kernel == KERNEL_SPLIT_128x64 && N * K < ((size_t)1 << 24) &&
                    (two_rows <= cus ? K < 2500 || N < 2048 || N * K < (size_t)10000000 || 3 * tiles > cus : (K < 192 && M >= 96) || tiles > cus))
                    p.kernel = KERNEL_SPLIT_2x64x64, tiles = two_rows;
                const bool wide = p.kernel != KERNEL_SPLIT_32x64 && p.kernel != KERNEL_SPLIT_64x64;
                const SliceModel &model = wide ? SLICES_WIDE_TILE : p.kernel == KERNEL_SPLIT_64x64 && N * K >= ((size_t)24 << 20) ? SLICES_LARGE_B : SLICES;
                p.splits = choose_splits(model, tiles, M, columns, cus, K, slice_bytes, limits.partial_bytes);
                if (p.splits > 1) p.partial_bytes = (size_t)p.splits * slice_bytes;
            }
        }
        if (left_out(limits, p)) continue;
        return p;
    }
    p = Plan();
    // M = 129 ... 192 against many columns: one row of 192x128 tiles, B copied non-temporally, where the last round of
    // workgroups is at least 55 % full (N = 18432 ... 32768, 50688 ... 65536, ...).  Against the cost model's choice
    // (192x192 tiles, 150 of them at N = 28672): N = 28672, K = 2048 ... 8192: 1.17 ... 1.30x (M = 192, K = 2048:
    // 40.3 -> 31.4 us), K = 14336: 0.97 ... 1.12x; N = 57344: 1.01 ... 1.13x up to K = 8192, 0.96 ... 0.98x at 14336;
    // N = 14336 (112 tiles): 0.81 ... 0.86x, N = 34304 (268 tiles): 0.76x.  The ring of four stages keeps three chunks
    // of B in flight per CU where the 192x192 tile's three stages keep two.
    {
        const size_t tiles = div_ceil(N, (size_t)128), last = tiles % cus;
        if (M > 128 && M <= 192 && K % 8 == 0 && K >= 2048 && K <= 12288 && tiles >= 144 &&
            (last == 0 || last * 100 >= cus * 55) && !left_out(limits, KERNEL_ROW192x128, 1)) {
            p.kernel = KERNEL_ROW192x128;
            p.splits = 1;
            return p;
        }
    }
    // Pipelined tiles: M and N may end inside a tile and K inside a chunk (guarded edges; the model charges whole
    // tiles and chunks), as long as rows of A and B stay 16-byte aligned.
    // M and N that 64 does not divide while K does and rows of C are aligned: the one-wave tile keeps M <= 128, a short K in slices
    // (227 x 128 x 1216) and a long K without (555 x 2688 x 4224 21.0 us, 25.9 on the four-wave tile).  Else the four-wave tile is
    // ahead: 1000^2 x 1024 9.9 -> 6.7 us, 504^2 x 512 5.0 -> 4.2, 416^2 x 8192 14.6 -> 11.9.  Not in slices of more than 44 chunks,
    // where 128x128 in slices is (456^2 x 11200, 44 chunks, 14.9 us and 15.3; 480^2 x 14720, 58 chunks, 17.1 and 15.3)
    const bool one_wave = (M % 64 || N % 64) && N % 8 == 0 && K % 64 == 0;
    if (K % 8 == 0 && K >= 64 && limits.excluded_count == 0) {
        p.kernel = short_k_kernel(M, N, K, cus);
        if (p.kernel != KERNEL_NONE) return p;
    }
    double best = 0.0;
    for (Candidate c : CANDIDATES) {
        if (K % 8) break;
        if (K % 64) c.lo *= OFF_LINE, c.hi *= OFF_LINE;
        const bool w4 = c.kernel == KERNEL_SMALL64_W4;
        const int kernel = w4 && (M % 64 || N % 64 || K % 64) ? (int)KERNEL_SMALL64_W4_EDGE : c.kernel;
        for (int s = 1; s <= 32; ++s) {  // K slices: whole chunks, as even as that allows
            if (w4 && one_wave && (M <= 128 || (s > 1 ? K < 2048 || K > 64 * 44 * (size_t)s : K > 2048))) continue;
            if (w4) {
                const size_t wgs = div_ceil(M, (size_t)c.bm) * div_ceil(N, (size_t)c.bn) * (size_t)s;
                if (wgs > cus * (size_t)c.per_cu) break;
                if (c.per_cu == 2 && (wgs <= cus || s > 1 || div_ceil(K, (size_t)64) >= W4_DEEP_MIN_CHUNKS)) break;
                // most CUs busy and a long walk per workgroup: the 128x128 tile in K slices moves half the bytes per
                // flop into LDS and is ahead (1024^2 x 7168: 25.3 us here, 22.2 us in four slices of 128x128 tiles;
                // level at K = 5120, behind at 4096)
                if (wgs * 4 > cus * 3 && shortest_slice(K, 64, s) >= 64 * 96) continue;
            }
            if (c.kernel == KERNEL_MID128_S2 && (s > 1 || K > 256)) break;
            // at most one workgroup of 64x64 tiles per CU: the four-wave tile is ahead of the one-wave tile on
            // every such grid that was measured (the model, fitted on larger grids, flatters the one-wave tile there)
            if (c.kernel == KERNEL_SMALL64 && !one_wave && div_ceil(M, (size_t)64) * div_ceil(N, (size_t)64) * (size_t)s <= cus) continue;
            if (shortest_slice(K, 64, s) < (size_t)64 * c.stages) break;
            if (s > 1 && (size_t)s * slice_bytes > limits.partial_bytes) break;
            if (left_out(limits, kernel, s)) continue;
            const double t = predict_us(c, M, N, K, s, cus);
            if (p.kernel == KERNEL_NONE || t < best) {
                best = t;
                p.kernel = kernel;
                p.splits = s;
                p.est_us = t;
                p.tail_tiles = 0;
                p.tail_splits = 1;
                p.tail_kernel = KERNEL_NONE;
                p.partial_bytes = s > 1 ? (size_t)s * slice_bytes : 0;
            }
        }
        // a grid of whole rounds plus a few workgroups: run those few in K slices
        const size_t wgs = div_ceil(M, (size_t)c.bm) * div_ceil(N, (size_t)c.bn), slots = cus * (size_t)c.per_cu;
        const size_t rem = wgs % slots;
        if (wgs > slots && rem > 0 && !w4 && c.kernel != KERNEL_MID128_S2) {
            for (int ts = 2; ts <= 16; ++ts) {
                if (shortest_slice(K, 64, ts) < (size_t)64 * c.stages || rem * ts > slots) break;
                if ((size_t)ts * rem * c.bm * c.bn * sizeof(float) > limits.partial_bytes) break;
                if (left_out(limits, c.kernel, 1, (int)rem, ts)) continue;
                const double t = predict_tail_us(c, M, N, K, ts, cus);
                if (p.kernel != KERNEL_NONE && t < best) {
                    best = t;
                    p.kernel = c.kernel;
                    p.splits = 1;
                    p.est_us = t;
                    p.tail_tiles = (int)rem;
                    p.tail_splits = ts;
                    p.tail_kernel = KERNEL_NONE;
                    p.partial_bytes = (size_t)ts * rem * c.bm * c.bn * sizeof(float);
                }
            }
            if (c.kernel == KERNEL_BIG256) {  // ... or on smaller tiles that divide this one
                for (Candidate small : CANDIDATES) {
                    if (K % 64) small.lo *= OFF_LINE, small.hi *= OFF_LINE;
                    if (small.kernel == KERNEL_BIG256 || small.kernel == KERNEL_SMALL64_W4 || small.kernel == KERNEL_MID128_S2 ||
                        c.bm % small.bm || c.bn % small.bn)
                        continue;
                    if (div_ceil(K, (size_t)64) < (size_t)small.stages || left_out(limits, c.kernel, 1, (int)rem, 1, small.kernel)) continue;
                    const double t = predict_subtile_us(c, small, M, N, K, cus);
                    if (p.kernel != KERNEL_NONE && t < best) {
                        best = t;
                        p.kernel = c.kernel;
                        p.splits = 1;
                        p.est_us = t;
                        p.tail_tiles = (int)rem;
                        p.tail_splits = 1;
                        p.tail_kernel = small.kernel;
                        p.partial_bytes = 0;
                    }
                }
            }
        }
    }
    const double others = best;
    for (Candidate c : BETWEEN_TILES) {
        if (p.kernel == KERNEL_NONE || p.splits > 1 || p.tail_tiles > 0) break;
        if (div_ceil(K, (size_t)64) < (size_t)c.stages || left_out(limits, c.kernel, 1)) continue;
        if (K % 64) c.lo *= OFF_LINE, c.hi *= OFF_LINE;
        const double t = predict_us(c, M, N, K, 1, cus);
        if (t < BETWEEN_MARGIN * others && t < best) {
            best = t;
            p = Plan();
            p.kernel = c.kernel;
            p.est_us = t;
        }
    }
    if (p.kernel != KERNEL_NONE) {
        if (K % 64) {  // copied to rows of whole lines first?  Not where the model has nothing to say about the copies' plan:
            // M = 129 ... 192 and K = 1992 ... 2040 reach the one-row rule above only with the copies' K, and a copy of all of
            // B before a product that is bound by reading B costs 1.4 ... 3x (160 x 28672 x 2040: 73.0 us, 38.3 without)
            const Plan copied = plan_on_copies(M, N, K, limits);
            if (copied.est_us > 0.0 && copied.est_us < p.est_us * direct_weight(p.kernel, p.splits, K) && !left_out(limits, copied)) return copied;
            // ... or on the tiles for unaligned rows, whose loads through registers lose less by rows that are off the lines (53 bytes
            // a clock and CU of 63, copies direct to LDS 41 of 59)
            if (limits.excluded_count == 0 && M >= 256 && N >= 256) {
                Plan direct = plan_on_unaligned_rows(M, N, K, cus, limits);
                const double weight = p.kernel == KERNEL_SMALL64_W4_EDGE ? OFF_LINE_SMALL : OFF_LINE_OTHERS;
                if (direct.kernel != KERNEL_NONE && direct.splits == 1 && direct.est_us < p.est_us * weight) return direct;
            }
        }
        return p;
    }
    if (K % 8) {
        // Rows of A and B not 16-byte aligned: read where they lie (K from 129 on) or copied first (from 192 on), whichever is
        // predicted faster.  Against copies alone, 206 shapes drawn over the whole range: 0.96 ... 2.5x, geomean 1.35 (929^3 12.0 -> 8.2 us,
        // 439^2 x 7179 21.0 -> 13.4, 16 x 8192 x 4097 39.8 -> 18.2, 147 x 22092 x 1853 46.3 -> 35.9); copies stay ahead for large products
        // (2603^3 46 us, 62 without).  The small-M kernels have no estimate: there B is most of what would be copied, and only where
        // one to eight rows meet a B of less than 2 MB are copies and the ring kernel ahead (2 x 110 x 1083 5.4 us, 6.1).  K below 129,
        // and beyond 2^23 where the copies do not fit: the guarded kernel, which gathers such rows element by element (170 x
        // 214 x 153 23.3 us, 4.6 here).
        Plan copied = plan_on_copies(M, N, K, limits);
        if (copied.kernel != KERNEL_NONE && left_out(limits, copied)) copied = Plan();
        Plan direct = plan_on_unaligned_rows(M, N, K, cus, limits);
        const bool short_b = M <= 8 && N * K < ((size_t)1 << 20);
        const bool copy = copied.est_us > 0.0 ? copies_us(copied) <= direct.est_us : short_b;
        if (direct.kernel != KERNEL_NONE && !(copied.kernel != KERNEL_NONE && copy)) return direct;
        if (copied.kernel != KERNEL_NONE) return copied;
        if (limits.excluded_count == 0) p.kernel = KERNEL_RAGGED;
        return p;
    }
    if (limits.excluded_count > 0) return Plan();  // the tuner's question has no further answer
    if (K >= 64) {  // K of one or two chunks; any M and N: guarded
        p.kernel = KERNEL_SPLIT_64x64;
        p.splits = choose_splits(SLICES_WIDE_TILE, div_ceil(M, 64) * div_ceil(N, 64), M, N, cus, K, slice_bytes, limits.partial_bytes);
        if (p.splits > 1) p.partial_bytes = (size_t)p.splits * slice_bytes;
        return p;
    }
    p.kernel = KERNEL_RAGGED;
    return p;
}

// Rows of A and B that start on 2-byte boundaries (K % 8 != 0), copied so that they start on 128-byte ones: row r of A, then
// row r - M of B, to dst[r][0 .. Kp), zeros from K on.  One wave per row and REALIGN_COLS columns; its loads are 16 bytes per lane
// at the source's own alignment (which this part's vector memory takes at the price of one more cache line per 1 KB),
// all issued before the first store.  Bound by memory: 4095^2 twice, 134 MB there and back.
constexpr int REALIGN_UNROLL = 8, REALIGN_COLS = REALIGN_UNROLL * 64 * 8;
__global__ void __launch_bounds__(256)
    realign_rows_kernel(const half_t *__restrict__ A, const half_t *__restrict__ B, half_t *__restrict__ dst, int M, int rows,
                        int K, int Kp) {
    const int lane = threadIdx.x & 63, row = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= rows) return;
    const half_t *src = row < M ? A + (size_t)row * K : B + (size_t)(row - M) * K;
    half_t *out = dst + (size_t)row * Kp;
    const int block_col = (int)blockIdx.y * REALIGN_COLS, first = block_col + lane * 8;
    // A piece that ends beyond K is loaded as the row's last eight elements and shifted down; one that starts beyond K is
    // zero.  So every lane's loads are one instruction each, inside the row (K >= 8), and none waits for another.
    u32x4 v[REALIGN_UNROLL];
#pragma unroll
    for (int u = 0; u < REALIGN_UNROLL; ++u)
        if (block_col + u * 512 < Kp) {
            const int col = first + u * 512;
            v[u] = *reinterpret_cast<const u32x4_any *>(src + (col + 8 <= K ? col : K - 8));
        }
    const int shift = 16 * (8 - (K & 7)) & 127;  // K % 8 == 0 has no such piece
#pragma unroll
    for (int u = 0; u < REALIGN_UNROLL; ++u)
        if (block_col + u * 512 < Kp) {
            const int col = first + u * 512;
            unsigned __int128 bits = __builtin_bit_cast(unsigned __int128, v[u]);
            bits = col + 8 <= K ? bits : col < K ? bits >> shift : (unsigned __int128)0;
            if (col < Kp) *reinterpret_cast<u32x4 *>(out + col) = __builtin_bit_cast(u32x4, bits);
        }
}

void run_padded(const Plan &p, const Workspace &ws, const void *A, const void *B, void *C, size_t M, size_t N,
                size_t K) {
    const size_t Kp = padded_k(K), rows = M + N;
    HGEMM_CHECK(ws.operands != nullptr && ws.operand_bytes >= rows * Kp * sizeof(half_t));
    HGEMM_CHECK(div_ceil(Kp, (size_t)REALIGN_COLS) <= 65535);
    half_t *copies = reinterpret_cast<half_t *>(ws.operands);
    realign_rows_kernel<<<dim3((unsigned)div_ceil(rows, (size_t)4), (unsigned)div_ceil(Kp, (size_t)REALIGN_COLS)), dim3(256), 0, nullptr>>>(
        reinterpret_cast<const half_t *>(A), reinterpret_cast<const half_t *>(B), copies, (int)M, (int)rows, (int)K, (int)Kp);
    HGEMM_CHECK_HIP_ERROR(hipGetLastError());
    Plan inner = p;
    inner.kernel = p.inner_kernel;
    inner.inner_kernel = KERNEL_NONE;
    inner.operand_bytes = 0;
    HGEMM_CHECK(inner.kernel != KERNEL_PADDED && inner.kernel != KERNEL_RAGGED);
    run_plan(inner, ws, copies, copies + M * Kp, C, M, N, Kp);
}

void run_plan(const Plan &p, const Workspace &ws, const void *A, const void *B, void *C, size_t M, size_t N,
              size_t K) {
    switch (p.kernel) {
        case KERNEL_BIG256: launch_pipelined_plan<Big256>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_T192: launch_pipelined_plan<Tile192>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_R256x128: launch_pipelined_plan<Rect256x128>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_MID128: launch_pipelined_plan<Mid128>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_MID128_S2: launch_pipelined<Mid128S2>(A, B, C, M, N, K, "hgemm_auto"); break;
        case KERNEL_ROW64x128: launch_pipelined_plan<Row64x128>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_ROW192x128: launch_pipelined_plan<Row192x128>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_T160x128: launch_pipelined<Tile160x128>(A, B, C, M, N, K, "hgemm_auto"); break;
        case KERNEL_T160x160: launch_pipelined<Tile160x160>(A, B, C, M, N, K, "hgemm_auto"); break;
        case KERNEL_T160x256: launch_pipelined<Tile160x256>(A, B, C, M, N, K, "hgemm_auto"); break;
        case KERNEL_T192x256: launch_pipelined<Tile192x256>(A, B, C, M, N, K, "hgemm_auto"); break;
        case KERNEL_T224x256: launch_pipelined<Tile224x256>(A, B, C, M, N, K, "hgemm_auto"); break;
        case KERNEL_SMALL64: launch_pipelined_plan<Small64>(A, B, C, M, N, K, p, ws); break;
        case KERNEL_SMALL64_W4: launch_small64_w4<false>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_SMALL64_W4_EDGE: launch_small64_w4<true>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_SPLIT_32x64: launch_splitk_by_length<Split32x64, Split32x64Short>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_SPLIT_2x64x64:
        case KERNEL_SPLIT_64x64: launch_splitk_by_length<Split64x64, Split64x64Short>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_SPLIT_64x128: launch_splitk<Split64x128>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_SPLIT_128x64: launch_splitk<Split128x64>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_SPLIT_128x128: launch_splitk<Split128x128>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_DECODE_BN16: launch_decode(A, B, C, M, N, K, 16, p.splits); break;
        case KERNEL_DECODE_BN32: launch_decode(A, B, C, M, N, K, 32, p.splits); break;
        case KERNEL_DECODE_RING: launch_decode_ring(A, B, C, M, N, K, p.splits); break;
        case KERNEL_DECODE_RING_EDGE: launch_decode_ring_edge(A, B, C, M, N, K, p.splits); break;
        case KERNEL_DECODE_RESIDENT: launch_decode_resident(A, B, C, M, N, K, compute_units()); break;
        case KERNEL_UNALIGNED64: launch_unaligned_plan<Unaligned64>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_UNALIGNED96: launch_unaligned_plan<Unaligned96>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_UNALIGNED128x64: launch_unaligned_plan<Unaligned128x64>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_UNALIGNED128: launch_unaligned_plan<Unaligned128>(A, B, C, M, N, K, p.splits, ws); break;
        case KERNEL_RAGGED: launch_ragged(A, B, C, M, N, K); break;
        case KERNEL_PADDED: run_padded(p, ws, A, B, C, M, N, K); break;
        case KERNEL_SIMT:
            hgemm_simt_naive(reinterpret_cast<const hgemm_half *>(A), reinterpret_cast<const hgemm_half *>(B),
                             reinterpret_cast<hgemm_half *>(C), M, N, K);
            break;
        default: HGEMM_CHECK_MSG(false, "no kernel for M=%zu N=%zu K=%zu", M, N, K);
    }
}

}  // namespace hgemm

using namespace hgemm;

namespace {

// Plans of the shapes this thread saw last: a 5 us launch should not re-run the cost model
// (five tiles x K slices x tails, in doubles) on every call.  Direct-mapped, fixed size,
// per thread: no allocation, no lock.  Two tables: the best plan, and the best plan that
// needs no workspace (what runs when device memory for the workspace cannot be had).
struct CachedPlan {
    size_t M = 0, N = 0, K = 0;
    Plan plan;
};
constexpr int PLAN_CACHE_SLOTS = 64;

// Plans that hgemm_auto_tune measured to be the fastest for a shape: process-wide, consulted before the model.  The
// per-thread tables below are thrown away whenever this one changes (`g_tuned_version`).
struct TunedShape {
    size_t M, N, K;
    bool operator<(const TunedShape &o) const { return M != o.M ? M < o.M : N != o.N ? N < o.N : K < o.K; }
};
std::map<TunedShape, Plan> g_tuned;
std::mutex g_tuned_mutex;
std::atomic<unsigned> g_tuned_version{0};

bool tuned_plan(size_t M, size_t N, size_t K, Plan *out) {
    if (g_tuned_version.load(std::memory_order_acquire) == 0) return false;  // nothing was ever tuned: no lock
    std::lock_guard<std::mutex> lock(g_tuned_mutex);
    const auto it = g_tuned.find(TunedShape{M, N, K});
    if (it == g_tuned.end()) return false;
    *out = it->second;
    return true;
}

// the plan hgemm_auto runs and the hgemm_auto_plan* queries report: the tuned one if there is one, else the model's
Plan current_plan(size_t M, size_t N, size_t K) {
    Plan p;
    return tuned_plan(M, N, K, &p) ? p : plan_for(M, N, K);
}

const Plan &cached_plan(size_t M, size_t N, size_t K, bool without_workspace = false) {
    static thread_local CachedPlan cache[2][PLAN_CACHE_SLOTS];
    static thread_local unsigned seen_version = 0;
    const unsigned version = g_tuned_version.load(std::memory_order_acquire);
    if (version != seen_version) {
        for (auto &table : cache)
            for (CachedPlan &slot : table) slot = CachedPlan();
        seen_version = version;
    }
    const size_t h = (M * 0x9e3779b97f4a7c15ull) ^ (N * 0xc2b2ae3d27d4eb4full) ^ (K * 0x165667b19e3779f9ull);
    CachedPlan &slot = cache[without_workspace ? 1 : 0][(h >> 32) % PLAN_CACHE_SLOTS];
    if (slot.M != M || slot.N != N || slot.K != K) {
        PlanLimits limits;
        if (without_workspace) limits.partial_bytes = limits.operand_bytes = 0;
        if (without_workspace || !tuned_plan(M, N, K, &slot.plan)) slot.plan = plan_for(M, N, K, limits);
        slot.M = M, slot.N = N, slot.K = K;
    }
    return slot.plan;
}

// Runs the cached plan of the shape on the heap workspace; when the workspace does not hold
// what the plan needs and device memory for it cannot be had, the best plan that needs none
// (no K slices, the guarded kernel instead of padded copies).
void run_with_heap_workspace(const void *A, const void *B, void *C, size_t M, size_t N, size_t K) {
    const Plan &p = cached_plan(M, N, K);
    if (p.partial_bytes == 0 && p.operand_bytes == 0) {
        run_plan(p, Workspace(), A, B, C, M, N, K);
        return;
    }
    {
        std::lock_guard<std::mutex> lock(g_heap_mutex);  // held while the plan's launches are enqueued
        Workspace ws;
        if (heap_workspace(p.partial_bytes, p.operand_bytes, &ws, false)) {
            run_plan(p, ws, A, B, C, M, N, K);
            return;
        }
    }
    run_plan(cached_plan(M, N, K, true), Workspace(), A, B, C, M, N, K);
}

}  // namespace

extern "C" void hgemm_skinny(const hgemm_half *A, const hgemm_half *B, hgemm_half *C, size_t M, size_t N, size_t K) {
    check_operands(A, B, C, M, N, K);
    HGEMM_CHECK_MSG(skinny_supports(M, N, K),
                    "hgemm_skinny needs M <= 128, N %% 64 == 0, K %% 64 == 0 (got M=%zu N=%zu K=%zu)", M, N, K);
    run_with_heap_workspace(A, B, C, M, N, K);
}
extern "C" int hgemm_skinny_supports(size_t M, size_t N, size_t K) { return skinny_supports(M, N, K) ? 1 : 0; }

extern "C" void hgemm_auto(const hgemm_half *A, const hgemm_half *B, hgemm_half *C, size_t M, size_t N, size_t K) {
    check_operands(A, B, C, M, N, K);
    run_with_heap_workspace(A, B, C, M, N, K);
}

// The plans hgemm_auto_tune times for a shape, best first by the model: the plan hgemm_auto runs anyway, then the
// best that is none of the earlier.
constexpr int TUNE_MOST_PLANS = 12;
int plans_to_time(size_t M, size_t N, size_t K, int max_plans, Plan *plans) {
    if (max_plans < 1) max_plans = 1;
    if (max_plans > TUNE_MOST_PLANS) max_plans = TUNE_MOST_PLANS;
    int count = 0;
    PlanLimits limits;
    limits.excluded = plans;
    while (count < max_plans) {
        limits.excluded_count = count;
        limits.every_small_m_kernel = count > 0;
        const Plan p = plan_for(M, N, K, limits);
        if (p.kernel == KERNEL_NONE) break;
        plans[count++] = p;
        if (p.kernel == KERNEL_RAGGED || p.kernel == KERNEL_SIMT) break;  // nothing to choose from
    }
    return count;
}

// What hgemm_auto_tune would time, without launching anything: kernel ids and K slices of up to max_plans plans.
extern "C" int hgemm_auto_tune_plans(size_t M, size_t N, size_t K, int max_plans, int *kernels, int *splits) {
    Plan plans[TUNE_MOST_PLANS];
    const int count = plans_to_time(M, N, K, max_plans, plans);
    for (int i = 0; i < count; ++i) {
        if (kernels) kernels[i] = plans[i].kernel;
        if (splits) splits[i] = plans[i].splits;
    }
    return count;
}

// What the calling thread's last hgemm_auto_tune measured, plan by plan in the order they were timed.
struct TuneRecord {
    Plan plan;
    float ms;
};
thread_local TuneRecord t_tune_records[TUNE_MOST_PLANS];
thread_local int t_tune_record_count = 0, t_tune_kept = -1;

// Reads a buffer larger than the caches hold, so that what was cached before is not afterwards.  Reads, not writes:
// the caches are left full of clean lines, as they are in a caller's loop over read-only weights; after a flush that
// writes, the next kernel's loads must first push out dirty lines, which penalises kernels by how they load (the
// streaming decode kernel read 30 us after a writing flush where it takes 13.5 us between other GEMMs).
// `never` is a value no sum of the zero-filled buffer takes, so nothing is stored.
__global__ void __launch_bounds__(256) cache_flush_kernel(floatx4 *buffer, size_t count, float never) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    floatx4 sum = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) sum += buffer[i];
    if (sum[0] + sum[1] + sum[2] + sum[3] == never) buffer[0] = sum;
}

// Times the model's best plans for this shape on the caller's operands and keeps the fastest for every later
// hgemm_auto call of the shape in this process: the first plan is the one hgemm_auto would run anyway, each next
// one the best that is none of the earlier (another tile, another slice count, for M <= 128 another kernel).  Per
// plan three untimed launches, then 5 ... 40 timed ones (about half a millisecond of work) enqueued back to back, each
// between events of its own on the null stream; with HGEMM_TUNE_COLD 512 MiB are read through the device before
// each of them, so that A and B come from HBM as they do for a caller whose weights do not stay cached between
// calls.  About 30 ms of untimed work come first, so that every plan meets a settled clock.  Another plan replaces
// the model's only if it is more than 3 % faster than the better of two timings of the model's.  The call returns when the device is
// idle and C holds the product as the kept plan computes it.
extern "C" int hgemm_auto_tune(const hgemm_half *A, const hgemm_half *B, hgemm_half *C, size_t M, size_t N, size_t K,
                               int max_plans, int flags) {
    check_operands(A, B, C, M, N, K);
    Plan plans[TUNE_MOST_PLANS];
    const int count = plans_to_time(M, N, K, max_plans, plans);
    constexpr size_t FLUSH_BYTES = (size_t)512 << 20;
    floatx4 *flush = nullptr;
    if ((flags & HGEMM_TUNE_COLD) && hipMalloc(reinterpret_cast<void **>(&flush), FLUSH_BYTES) != hipSuccess) {
        (void)hipGetLastError();
        flush = nullptr;  // no memory for it: the plans are timed on whatever the caches hold
    }
    if (flush) HGEMM_CHECK_HIP_ERROR(hipMemsetAsync(flush, 0, FLUSH_BYTES, nullptr));
    constexpr int MOST_LAUNCHES = 40;
    hipEvent_t start[MOST_LAUNCHES], stop[MOST_LAUNCHES];
    for (int i = 0; i < MOST_LAUNCHES; ++i) {
        HGEMM_CHECK_HIP_ERROR(hipEventCreate(&start[i]));
        HGEMM_CHECK_HIP_ERROR(hipEventCreate(&stop[i]));
    }
    auto run = [&](const Plan &p) {  // false: the workspace the plan needs could not be had
        std::lock_guard<std::mutex> lock(g_heap_mutex);
        Workspace ws;
        if ((p.partial_bytes || p.operand_bytes) && !heap_workspace(p.partial_bytes, p.operand_bytes, &ws, false)) return false;
        run_plan(p, ws, A, B, C, M, N, K);
        return true;
    };
    // `launches` launches enqueued back to back (with the flush between them when asked for), each between two events
    // of its own: the device stays busy as in a caller's loop, and the flushes are not in the sum.  Milliseconds per launch.
    auto time_plan = [&](const Plan &p, int launches) {
        for (int i = 0; i < launches; ++i) {
            if (flush) {
                cache_flush_kernel<<<dim3(2048), dim3(256), 0, nullptr>>>(flush, FLUSH_BYTES / sizeof(floatx4), 1.0f);
                HGEMM_CHECK_HIP_ERROR(hipGetLastError());
            }
            HGEMM_CHECK_HIP_ERROR(hipEventRecord(start[i], nullptr));
            run(p);
            HGEMM_CHECK_HIP_ERROR(hipEventRecord(stop[i], nullptr));
        }
        HGEMM_CHECK_HIP_ERROR(hipEventSynchronize(stop[launches - 1]));
        float total = 0.0f;
        for (int i = 0; i < launches; ++i) {
            float ms = 0.0f;
            HGEMM_CHECK_HIP_ERROR(hipEventElapsedTime(&ms, start[i], stop[i]));
            total += ms;
        }
        return total / (float)launches;
    };
    int best = -1, timed = 0;
    float best_ms = 0.0f, first_ms = 0.0f;
    t_tune_record_count = 0;
    // The part is power-managed and takes tens of milliseconds of work to settle from idle: whoever is timed first is
    // timed on a different clock (the model's own plan measured 13-23 % slower than the same kernel a moment later).
    // So the device is kept busy with the first plan for about 30 ms before anything is timed, and that plan is timed
    // once more after all the others; the better of its two timings counts.
    if (count > 0 && run(plans[0])) {
        float spent_ms = 0.0f;
        for (int round = 0; round < 20 && spent_ms < 30.0f; ++round) spent_ms += 5.0f * time_plan(plans[0], 5);
    }
    for (int i = 0; i < count; ++i) {
        if (!run(plans[i])) continue;
        // two untimed launches that also say how many timed ones make about half a millisecond of work (5 ... 40)
        const float rough_ms = time_plan(plans[i], 2);
        int launches = rough_ms > 0.0f ? (int)(0.5f / rough_ms) : MOST_LAUNCHES;
        launches = launches < 5 ? 5 : launches > MOST_LAUNCHES ? MOST_LAUNCHES : launches;
        const float ms = time_plan(plans[i], launches);
        ++timed;
        t_tune_records[t_tune_record_count++] = TuneRecord{plans[i], ms};
        if (i == 0) first_ms = ms;
        // the model's own plan stays unless another is ahead by more than the 3 % that two timings of one plan differ by
        if (best < 0 || ms < (best == 0 ? 0.97f * first_ms : best_ms)) best = i, best_ms = ms, t_tune_kept = t_tune_record_count - 1;
    }
    if (best > 0 && t_tune_record_count > 0 && same_choice(t_tune_records[0].plan, plans[0])) {
        const float rough_ms = time_plan(plans[0], 2);
        int launches = rough_ms > 0.0f ? (int)(0.5f / rough_ms) : MOST_LAUNCHES;
        launches = launches < 5 ? 5 : launches > MOST_LAUNCHES ? MOST_LAUNCHES : launches;
        const float again_ms = time_plan(plans[0], launches);
        if (again_ms < t_tune_records[0].ms) t_tune_records[0].ms = again_ms;
        if (best_ms >= 0.97f * t_tune_records[0].ms) best = 0, best_ms = t_tune_records[0].ms, t_tune_kept = 0;
    }
    for (int i = 0; i < MOST_LAUNCHES; ++i) {
        HGEMM_CHECK_HIP_ERROR(hipEventDestroy(start[i]));
        HGEMM_CHECK_HIP_ERROR(hipEventDestroy(stop[i]));
    }
    HGEMM_CHECK_MSG(best >= 0, "hgemm_auto_tune: no plan for M=%zu N=%zu K=%zu could be run", M, N, K);
    {
        std::lock_guard<std::mutex> lock(g_tuned_mutex);
        g_tuned[TunedShape{M, N, K}] = plans[best];
        g_tuned_version.fetch_add(1, std::memory_order_release);
    }
    run(plans[best]);
    HGEMM_CHECK_HIP_ERROR(hipDeviceSynchronize());
    if (flush) HGEMM_CHECK_HIP_ERROR(hipFree(flush));
    return timed;
}

// The calling thread's last hgemm_auto_tune, plan by plan in the order they were timed: kernel id, K slices,
// milliseconds per launch, whether it is the one that was kept.  Returns 0 past the last plan, else 1.
extern "C" int hgemm_auto_tune_result(int index, int *kernel, int *splits, float *ms, int *kept) {
    if (index < 0 || index >= t_tune_record_count) return 0;
    if (kernel) *kernel = t_tune_records[index].plan.kernel;
    if (splits) *splits = t_tune_records[index].plan.splits;
    if (ms) *ms = t_tune_records[index].ms;
    if (kept) *kept = index == t_tune_kept ? 1 : 0;
    return 1;
}

// Forgets every tuned plan: hgemm_auto goes by the model again.
extern "C" void hgemm_auto_forget_tuning(void) {
    std::lock_guard<std::mutex> lock(g_tuned_mutex);
    g_tuned.clear();
    g_tuned_version.fetch_add(1, std::memory_order_release);
}

// 1 if the shape's plan was set by hgemm_auto_tune.
extern "C" int hgemm_auto_plan_is_tuned(size_t M, size_t N, size_t K) {
    Plan p;
    return tuned_plan(M, N, K, &p) ? 1 : 0;
}

// The tuned kernel by tile, as entry points of their own.  M and N may end inside a tile.
#define HGEMM_DEFINE_PIPELINED_VARIANT(symbol, Cfg, which)                                                   \
    extern "C" void symbol(const hgemm_half *A, const hgemm_half *B, hgemm_half *C, size_t M, size_t N,      \
                           size_t K) {                                                                       \
        check_operands(A, B, C, M, N, K);                                                                    \
        HGEMM_CHECK_MSG(pipelined_supports_edges<Cfg>(M, N, K),                                              \
                        "%s needs N %% 8 == 0, K %% %d == 0, K >= %d (got M=%zu N=%zu K=%zu)", #symbol,      \
                        Cfg::BK, Cfg::BK * Cfg::STAGES, M, N, K);                                            \
        launch_pipelined<Cfg>(A, B, C, M, N, K, #symbol, which);                                             \
    }                                                                                                        \
    extern "C" int symbol##_supports(size_t M, size_t N, size_t K) {                                         \
        return pipelined_supports_edges<Cfg>(M, N, K) ? 1 : 0;                                               \
    }
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_pipelined_64x64, Small64, PipeKernel::Interleaved)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_pipelined_128x128, Mid128, PipeKernel::Interleaved)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_pipelined_192x192, Tile192, PipeKernel::Interleaved)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_pipelined_256x128, Rect256x128, PipeKernel::Interleaved)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_pipelined_256x256, Big256, PipeKernel::Interleaved)
// ... and with each accumulator's MFMAs chained (the tiles that have that kernel)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_chained_192x192, Tile192, PipeKernel::Chained)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_chained_256x128, Rect256x128, PipeKernel::Chained)
HGEMM_DEFINE_PIPELINED_VARIANT(hgemm_mfma_chained_256x256, Big256, PipeKernel::Chained)

extern "C" int hgemm_reserve_workspace(size_t partial_bytes, size_t operand_bytes) {
    std::lock_guard<std::mutex> lock(g_heap_mutex);
    Workspace ws;
    return heap_workspace(partial_bytes, operand_bytes, &ws, true) ? 0 : 1;
}

extern "C" void hgemm_release_workspace(void) {
    const int dev = current_device();
    std::lock_guard<std::mutex> lock(g_heap_mutex);
    Workspace &w = g_heap[dev].ws;
    unsigned char *small = g_heap[dev].small_operands;
    if (w.partial || w.operands || small) HGEMM_CHECK_HIP_ERROR(hipDeviceSynchronize());  // launches may still use them
    if (small) HGEMM_CHECK_HIP_ERROR(hipFree(small));
    if (w.partial) HGEMM_CHECK_HIP_ERROR(hipFree(w.partial));
    if (w.operands) HGEMM_CHECK_HIP_ERROR(hipFree(w.operands));
    g_heap[dev] = HeapState();
}

// Operand bytes reported for a plan: what a caller reserves, and what the static workspace has to hold.
static size_t reported_operand_bytes(const Plan &p, size_t M, size_t N, size_t K) { return p.operand_bytes ? reported_copy_bytes(M, N, K) : 0; }
static size_t padded_partial_bytes(size_t bytes) { return (bytes + 255) / 256 * 256; }
static bool fits_static_workspace(const Plan &p, size_t M, size_t N, size_t K) {
    return padded_partial_bytes(p.partial_bytes) + reported_operand_bytes(p, M, N, K) <= STATIC_WORKSPACE_BYTES;
}

// What hgemm_auto_static_workspace does with a shape whose plan needs more than its array: true, the best plan without a
// workspace; false, it says so and launches nothing.  Products in whole chunks with aligned rows of C are refused (their plan
// is too many K slices of a large C).  Others run a kernel with guarded edges.  Where rows of A and B are not aligned (K % 8 != 0;
// the plan copies them, what is read where it lies fits), which products are run was settled when only the gather kernel could:
// those it took up to twice the time of the copies for, at the rates it was once chosen by (80 TFLOP/s against passes at 3.5 TB/s
// and 4 TB/s for a B that is only streamed): 131 x 67882 x 338, but not 4095^3.  Callers count on what is refused, so it stays.
// Where the reported figure reaches the cap of the heap workspace, all are run.
static bool runs_unaided(size_t M, size_t N, size_t K) {
    if (N % 8 == 0 && K % 64 == 0) return false;
    if ((K % 8 == 0 && cached_plan(M, N, K, true).kernel != KERNEL_RAGGED) || reported_copy_bytes(M, N, K) >= MAX_PADDED_BYTES) return true;
    const size_t Np = padded_n(N), Kp = padded_k(K);
    PlanLimits inner_limits;
    inner_limits.operand_bytes = 0;
    const Plan inner = plan_for(M, Np, Kp, inner_limits);
    const double inner_us = inner.est_us > 0.0 ? inner.est_us : 8.0 + (double)(Np * Kp * 2) / 4e6;
    const double copies_us = 6.0 + 4.0 * (double)((M + Np) * Kp + (Np != N ? M * Np : 0)) / 3.5e6;
    return 5.0 + 2.0 * (double)M * (double)N * (double)K / 80e6 <= 2.0 * (copies_us + inner_us);
}

extern "C" int hgemm_auto_static_workspace(const hgemm_half *A, const hgemm_half *B, hgemm_half *C, size_t M, size_t N,
                                           size_t K) {
    check_operands(A, B, C, M, N, K);
    const Plan *chosen = &cached_plan(M, N, K);  // the plan hgemm_auto runs: same kernels, same order of additions
    if (!fits_static_workspace(*chosen, M, N, K)) {
        if (!runs_unaided(M, N, K)) {
            HLOG("hgemm_auto_static_workspace: the plan for M=%zu N=%zu K=%zu keeps %zu bytes of partial sums and %zu bytes "
                 "of padded operands, the static workspace holds %zu; nothing was launched (hgemm_auto has no such limit)",
                 M, N, K, chosen->partial_bytes, reported_operand_bytes(*chosen, M, N, K), STATIC_WORKSPACE_BYTES);
            return 1;
        }
        chosen = &cached_plan(M, N, K, true);
    }
    const Plan &p = *chosen;
    const size_t partial_bytes = padded_partial_bytes(p.partial_bytes);
    Workspace ws;
    if (partial_bytes + p.operand_bytes > 0) {
        unsigned char *base = static_scratch();
        ws.partial = reinterpret_cast<float *>(base);
        ws.partial_bytes = partial_bytes;
        ws.operands = base + partial_bytes;
        ws.operand_bytes = STATIC_WORKSPACE_BYTES - partial_bytes;
    }
    // Nothing in the array has to start at zero: every kernel that reads partial sums or padded
    // operands reads only what a kernel launched before it in this call has written in full.
    if (partial_bytes + p.operand_bytes > 0) {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);  // one plan's launches at a time into the null stream
        run_plan(p, ws, A, B, C, M, N, K);
    } else {
        run_plan(p, ws, A, B, C, M, N, K);
    }
    return 0;
}

extern "C" size_t hgemm_static_workspace_bytes(void) { return STATIC_WORKSPACE_BYTES; }

extern "C" size_t hgemm_auto_workspace_bytes(size_t M, size_t N, size_t K, size_t *operand_bytes) {
    const Plan p = current_plan(M, N, K);
    if (operand_bytes) *operand_bytes = reported_operand_bytes(p, M, N, K);
    return p.partial_bytes;
}
extern "C" int hgemm_auto_supports(size_t M, size_t N, size_t K) { return M > 0 && N > 0 && K > 0; }

// Which kernel and how many K slices hgemm_auto uses for a shape (for reports and tests).
extern "C" int hgemm_auto_plan(size_t M, size_t N, size_t K, int *splits) {
    const Plan p = current_plan(M, N, K);
    if (splits) *splits = p.splits;
    return p.kernel;
}
// How hgemm_auto treats the last, partly filled round of a large grid: the number of
// workgroups in it that run in K slices (0: none) and, through `splits`, the slice count.
extern "C" int hgemm_auto_plan_tail(size_t M, size_t N, size_t K, int *splits) {
    const Plan p = current_plan(M, N, K);
    if (splits) *splits = p.tail_splits;
    return p.tail_tiles;
}
// Row `index` of the table that decides the kernel for M <= 128 (first covering row whose kernel can run the shape
// wins): bounds = {m_lo, m_hi, n_lo, n_hi, k_lo, k_hi, b_lo, b_hi}, inclusive, b = N * K; flags bit 0: only where
// K < 4 N, bit 1: not where K is a multiple of 16384.  Returns the kernel id, or -1 past the end of the table.
extern "C" int hgemm_small_m_rule(int index, size_t *bounds, int *flags) {
    if (index < 0 || index >= SMALL_M_RULE_COUNT) return -1;
    const SmallMRule &r = SMALL_M_RULES[index];
    if (bounds) {
        const size_t b[8] = {(size_t)r.m_lo, (size_t)r.m_hi, r.n_lo, r.n_hi, r.k_lo, r.k_hi, r.b_lo, r.b_hi};
        for (int i = 0; i < 8; ++i) bounds[i] = b[i];
    }
    if (flags) *flags = r.flags;
    return r.kernel;
}
// Kernel id of the smaller tile that takes over the last round (0: none).
extern "C" int hgemm_auto_plan_tail_kernel(size_t M, size_t N, size_t K) { return current_plan(M, N, K).tail_kernel; }
// 1 if the plan's main launch runs the chained kernel of its tile, 0 for the interleaved one.
extern "C" int hgemm_auto_plan_chained(size_t M, size_t N, size_t K) {
    const Plan p = current_plan(M, N, K);
    if (p.splits < 1) return 0;
    const size_t k_len = shortest_slice(K, 64, p.splits);
    auto workgroups = [&](size_t bm, size_t bn) {  // of the main launch
        return (div_ceil(M, bm) * div_ceil(N, bn) - (size_t)p.tail_tiles) * (size_t)p.splits;
    };
    switch (p.kernel) {
        case KERNEL_BIG256: return use_chained<Big256>(PipeKernel::Auto, workgroups(256, 256), k_len) ? 1 : 0;
        case KERNEL_T192: return use_chained<Tile192>(PipeKernel::Auto, workgroups(192, 192), k_len) ? 1 : 0;
        case KERNEL_R256x128: return use_chained<Rect256x128>(PipeKernel::Auto, workgroups(256, 128), k_len) ? 1 : 0;
        case KERNEL_T160x256: return use_chained<Tile160x256>(PipeKernel::Auto, workgroups(160, 256), k_len) ? 1 : 0;
        case KERNEL_T192x256: return use_chained<Tile192x256>(PipeKernel::Auto, workgroups(192, 256), k_len) ? 1 : 0;
        case KERNEL_T224x256: return use_chained<Tile224x256>(PipeKernel::Auto, workgroups(224, 256), k_len) ? 1 : 0;
        default: return 0;
    }
}
extern "C" const char *hgemm_kernel_name(int kernel) {
    switch (kernel) {
        case KERNEL_BIG256: return "pipelined 256x256x64, 4 waves, LDS ring 3 (A) + 2 (B)";
        case KERNEL_MID128: return "pipelined 128x128x64, 4 waves, 5-stage ring";
        case KERNEL_MID128_S2: return "pipelined 128x128x64, 4 waves, 2-stage ring";
        case KERNEL_ROW64x128: return "pipelined 64x128x64, 4 waves, 5-stage ring";
        case KERNEL_ROW192x128: return "pipelined 192x128x64, 4 waves, 4-stage ring";
        case KERNEL_SMALL64: return "pipelined 64x64x64, 1 wave, 3-stage ring";
        case KERNEL_SMALL64_W4: return "tiled 64x64x64, 4 waves of 32x32, look-ahead ring";
        case KERNEL_SMALL64_W4_EDGE: return "edge-guarded 64x64x64, 4 waves of 32x32, look-ahead ring";
        case KERNEL_T192: return "pipelined 192x192x64, 4 waves, 3-stage ring";
        case KERNEL_R256x128: return "pipelined 256x128x64, 4 waves, 3-stage ring";
        case KERNEL_T160x128: return "160x128x64 pipelined, 4 waves, 4-stage ring";
        case KERNEL_T160x160: return "160x160x64 pipelined, 4 waves, 4-stage ring";
        case KERNEL_T160x256: return "160x256x64 pipelined, 4 waves, 3-stage ring";
        case KERNEL_T192x256: return "192x256x64 pipelined, 4 waves, LDS ring 3 (A) + 2 (B)";
        case KERNEL_T224x256: return "224x256x64 pipelined, 4 waves, LDS ring 3 (A) + 2 (B)";
        case KERNEL_SPLIT_32x64: return "split-K 32x64x64, 2 waves, look-ahead 6-stage or 4-stage ring";
        case KERNEL_SPLIT_64x64: return "split-K 64x64x64, 4 waves, look-ahead 5-stage or 4-stage ring";
        case KERNEL_SPLIT_64x128: return "split-K 64x128x64, 4 waves, 4-stage ring";
        case KERNEL_SPLIT_128x64: return "split-K 128x64x64, 4 waves, 4-stage ring";
        case KERNEL_SPLIT_2x64x64: return "split-K 2x64x64x64, 4 waves a tile, look-ahead 5-stage or 4-stage ring";
        case KERNEL_SPLIT_128x128: return "split-K 128x128x64, 4 waves, 4-stage ring";
        case KERNEL_DECODE_BN16: return "streaming decode, 16 columns per workgroup, one wave per K slice";
        case KERNEL_DECODE_BN32: return "streaming decode, 32 columns per workgroup, one wave per K slice";
        case KERNEL_DECODE_RING: return "streaming decode, 16 columns per workgroup, one wave and one LDS ring per K slice";
        case KERNEL_DECODE_RING_EDGE: return "streaming decode, 16 columns per workgroup, per-wave LDS rings, guarded edges";
        case KERNEL_DECODE_RESIDENT: return "decode with A in registers, persistent workgroups over 16-column tiles, one wave per K slice";
        case KERNEL_RAGGED: return "guarded 128x128x32, 4 waves, any shape";
        case KERNEL_PADDED: return "zero-padded operand copies + kernel of the padded shape";
        case KERNEL_UNALIGNED64: return "rows read where they lie, 64x64x128, 4 waves";
        case KERNEL_UNALIGNED96: return "rows read where they lie, 96x96x128, 4 waves";
        case KERNEL_UNALIGNED128x64: return "rows read where they lie, 128x64x128, 8 waves";
        case KERNEL_UNALIGNED128: return "rows read where they lie, 128x128x128, 8 waves";
        case KERNEL_SIMT: return "scalar fallback";
        default: return "none";
    }
}
