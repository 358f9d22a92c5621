"""hgemm_auto on sizes that end inside a tile and inside a 64-wide K chunk: every kernel with guarded edges, at K one, four
and seven 8-element pieces into its last chunk, N odd, with and without K slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GUARD, POISON = 4096, 0x7E5A   # elements around C (keeps it 16-byte aligned); a NaN no kernel produces

# shape -> start of the kernel's name; together every kernel that has guarded edges, sliced and not
CASES = [
    ((313, 5, 184), "edge-guarded"), ((157, 1, 5104), "edge-guarded"),            # plain ring, alone and in slices
    ((147, 4, 680), "edge-guarded"), ((168, 2, 5120), "edge-guarded"),            # look-ahead ring
    ((2777, 131, 2912), "edge-guarded"), ((2420, 66, 7840), "edge-guarded"),      # its deep form
    ((2358, 397, 360), "edge-guarded"), ((1000, 1000, 1000), "edge-guarded"),     # two workgroups per CU; one
    ((147, 20, 72), "pipelined 128x128"), ((2813, 77, 5520), "pipelined 128x128"),
    ((130, 3768, 6744), "pipelined 192x192"), ((48, 34155, 200), "pipelined 192x192"),
    ((186, 8157, 4984), "pipelined 192x192"), ((131, 19105, 2072), "pipelined 192x128"),
    ((1003, 7001, 616), "pipelined 256x128"), ((2816, 259, 6240), "pipelined 256x128"),
    ((1262, 5671, 1112), "pipelined 256x128"), ((950, 13327, 336), "pipelined 256x256"),
    ((199, 11317, 6312), "pipelined 256x256"), ((2807, 5289, 312), "pipelined 256x256"),
    ((408, 36824, 288), "pipelined 256x256"), ((646, 26708, 616), "pipelined 256x256"),   # last round on smaller tiles
    ((230, 16622, 4152), "pipelined 128x128"), ((258, 25173, 2096), "pipelined 192x192"),  # ... in K slices
    ((463, 9095, 1048), "160x128x64"), ((260, 13347, 1664), "160x128x64"), ((905, 6175, 1128), "160x160x64"),
    ((443, 11908, 768), "160x160x64"), ((2154, 4499, 800), "160x256x64"), ((2233, 4257, 704), "160x256x64"),
    ((517, 16923, 312), "192x256x64"), ((723, 15154, 704), "192x256x64"), ((2911, 4675, 584), "224x256x64"),
    ((2282, 5454, 384), "224x256x64"), ((264, 23283, 4136), "160x256x64"),                 # the last three: chained
    ((655, 13125, 4104), "192x256x64"), ((387, 21799, 4112), "224x256x64"),
    ((36, 19412, 400), "pipelined 64x128"), ((41, 9311, 8208), "pipelined 64x128"), ((17, 35153, 3392), "pipelined 64x128"),
    ((492, 2108, 136), "pipelined 64x64"), ((2574, 1, 3112), "pipelined 64x64"),
    ((7, 20, 72), "split-K 32x64"), ((11, 5, 2792), "split-K 32x64"), ((39, 2, 176), "split-K 64x64"),
    ((34, 2, 7416), "split-K 64x64"), ((38, 18838, 96), "split-K 64x128"), ((38, 17733, 2136), "split-K 64x128"),
    ((67, 1, 216), "split-K 2x64x64x64"), ((76, 2, 6272), "split-K 2x64x64x64"), ((69, 23286, 88), "split-K 128x128"),
    ((74, 17395, 3824), "split-K 128x128"),
    ((66, 10404, 1664), "split-K 128x64"), ((66, 9061, 1968), "split-K 128x64"), ((65, 674, 25472), "split-K 128x64"),
    ((65, 899, 18768), "split-K 128x64"), ((65, 1900, 9048), "split-K 128x64"),
    ((1, 9, 312), "streaming decode"), ((4, 1475, 14528), "streaming decode"), ((18, 220, 288), "streaming decode"),
    ((56, 81, 312), "streaming decode"), ((67, 4295, 272), "streaming decode"), ((67, 146, 280), "streaming decode"),
    ((1, 1984, 9600), "streaming decode, 16 columns per workgroup, per-wave"),             # N and K even, the waves' shares not
    ((18, 4096, 2688), "streaming decode, 16 columns per workgroup, per-wave"),
    ((3, 1984, 1344), "streaming decode, 16 columns per workgroup, per-wave"),             # an odd number of whole chunks
    ((16, 1024, 4032), "streaming decode, 16 columns per workgroup, per-wave"),
    ((8, 17728, 1088), "streaming decode, 16 columns per workgroup, per-wave"),
    ((5, 2048, 4160), "streaming decode, 16 columns per workgroup, per-wave"),
    ((30, 1536, 6976), "streaming decode, 16 columns per workgroup, per-wave"),
    ((511, 511, 511), "rows read where they lie"), ((296, 299, 2113), "rows read where they lie"),
    ((3, 1001, 4099), "rows read where they lie"), ((1027, 520, 193), "rows read where they lie"),
    # operand copies: of a few rows, of short rows, with K slices on them, large ones
    ((1, 1000, 193), "zero-padded operand copies"), ((5, 49, 2585), "zero-padded operand copies"),
    ((3019, 1354, 195), "zero-padded operand copies"), ((1113, 1211, 5707), "zero-padded operand copies"),
    ((2591, 11875, 1833), "zero-padded operand copies"),
]

# Split-K tiles on their look-ahead loop (more than eight chunks to a slice), which ends in a remainder of its steady part that goes by
# the number of chunks: nine to fifteen of them, even and odd, with K ending inside the last one and not, in K slices that differ by
# one chunk, and M one row into the second of two rows of tiles
LOOKAHEAD = [
    ((9, 1, 520), "split-K 32x64", 1), ((10, 1, 640), "split-K 32x64", 1), ((17, 45, 696), "split-K 32x64", 1),
    ((32, 63, 744), "split-K 32x64", 1), ((22, 33, 824), "split-K 32x64", 1), ((31, 46, 888), "split-K 32x64", 1),
    ((30, 46, 920), "split-K 32x64", 1), ((9, 1, 8248), "split-K 32x64", 16), ((21, 250, 9024), "split-K 32x64", 16),
    ((13, 184, 18672), "split-K 32x64", 16), ((23, 98, 19800), "split-K 32x64", 16),
    ((34, 1, 520), "split-K 64x64", 1), ((57, 144, 640), "split-K 64x64", 1), ((35, 87, 696), "split-K 64x64", 1),
    ((48, 85, 760), "split-K 64x64", 1), ((33, 1, 8256), "split-K 64x64", 16), ((57, 181, 11976), "split-K 64x64", 16),
    ((34, 134, 25600), "split-K 64x64", 16), ((52, 88, 27000), "split-K 64x64", 16),
    ((65, 1, 536), "split-K 2x64x64x64", 1), ((122, 75, 600), "split-K 2x64x64x64", 1), ((95, 86, 672), "split-K 2x64x64x64", 1),
    ((84, 81, 832), "split-K 2x64x64x64", 1), ((65, 1, 8560), "split-K 2x64x64x64", 16), ((113, 39, 22016), "split-K 2x64x64x64", 16),
    ((119, 52, 16016), "split-K 2x64x64x64", 16), ((123, 34, 23696), "split-K 2x64x64x64", 16),
]


def _gpu_bits(bits, gpu):
    import torch
    return torch.from_numpy(bits.view(np.int16)).to(gpu).view(torch.float16)


@pytest.mark.parametrize("shape,kernel", CASES)
def test_sizes_inside_tiles_and_chunks(oracle, hgemm_lib, gpu, shape, kernel):
    """Exact on ternary inputs (sums are integers below 2048) inside a guard band; then with an infinity in one row of A, at
    the k that the last chunk and the one before it both read: that row is infinite with B's sign, no other changes."""
    _exact_and_infinite(oracle, hgemm_lib, gpu, shape, kernel)


@pytest.mark.parametrize("shape,kernel,slices", LOOKAHEAD)
def test_look_ahead_split_k_at_its_edges(oracle, hgemm_lib, gpu, shape, kernel, slices):
    M, N, K = shape
    plan = hgemm_lib.auto_plan(M, N, K)
    assert plan["splits"] == slices and -(-K // 64) > 8 * slices, plan
    assert M > 32 or -(-N // 64) * slices <= 512      # (the 32-row tile has the other loop beyond two workgroups to a CU)
    _exact_and_infinite(oracle, hgemm_lib, gpu, shape, kernel)


def _exact_and_infinite(oracle, hgemm_lib, gpu, shape, kernel):
    import torch
    M, N, K = shape
    plan = hgemm_lib.auto_plan(M, N, K)
    assert plan["kernel"].startswith(kernel), plan
    A, B = oracle.fill((M, K), 31, 1, oracle.TERNARY, 0, 1), oracle.fill((N, K), 31, 2, oracle.TERNARY, 0, 1)
    expect = oracle.hgemm(A, B)
    assert np.abs(expect.view(np.float16).astype(np.float32)).max() < 2048
    buf = torch.full((GUARD + M * N + GUARD,), POISON, dtype=torch.int16, device=gpu)
    C = buf[GUARD:GUARD + M * N].view(torch.float16).view(M, N)
    Ad, Bd = _gpu_bits(A, gpu), _gpu_bits(B, gpu)
    print(f"[gpu] hgemm_auto M={M} N={N} K={K} {plan['kernel']} x{plan['splits']} tail {plan['tail_tiles']}", flush=True)
    hgemm_lib.call("hgemm_auto", Ad, Bd, C, M, N, K)
    host = buf.cpu().numpy().view(np.uint16)
    assert np.all(host[:GUARD] == POISON) and np.all(host[GUARD + M * N:] == POISON)
    assert np.array_equal(host[GUARD:GUARD + M * N].reshape(M, N), expect)
    row, k = M - 1, K - 60 if K >= 64 else 0
    Bd[:, k] = torch.where(torch.arange(N, device=gpu) % 2 == 0, 1.0, -1.0).half()
    Ad[row, k] = float("inf")
    hgemm_lib.call("hgemm_auto", Ad, Bd, C, M, N, K)
    assert torch.equal(C[row], torch.where(torch.arange(N, device=gpu) % 2 == 0, float("inf"), float("-inf")).half())
    assert M == 1 or bool(torch.isfinite(C[:row]).all())


# The tiles between 128x128 and 256x256 on whole chunks with aligned rows of C: M and N whole tiles, or ending inside one, each a
# form of its own, and on the interleaved or (K of 4096 on; three of the tiles have it) the chained kernel, with stores of its own
FORMS = [
    ((160, 16640, 320), "160x128x64", False), ((131, 17008, 320), "160x128x64", False),
    ((320, 19840, 320), "160x160x64", False), ((139, 33016, 320), "160x160x64", False),
    ((320, 24832, 256), "160x256x64", False), ((259, 22120, 256), "160x256x64", False),
    ((640, 11776, 4096), "160x256x64", True), ((277, 24016, 4160), "160x256x64", True), ((600, 14336, 4096), "160x256x64", True),
    ((384, 25600, 320), "192x256x64", False), ((486, 16608, 320), "192x256x64", False),
    ((1344, 7424, 4160), "192x256x64", True), ((652, 13080, 4288), "192x256x64", True),
    ((224, 33280, 320), "224x256x64", False), ((408, 22168, 320), "224x256x64", False),
    ((448, 22272, 4096), "224x256x64", True), ((389, 22560, 4096), "224x256x64", True),
]


@pytest.mark.parametrize("shape,tile,chained", FORMS)
def test_every_form_of_the_tiles_between(oracle, hgemm_lib, gpu, shape, tile, chained):
    """Exact on ternary inputs inside a guard band, C starting as NaN: eight rows from every 61 (so every row of tiles, wave and
    register group of one) against the checker, the rest written and finite."""
    import torch
    M, N, K = shape
    plan = hgemm_lib.auto_plan(M, N, K)
    assert plan["kernel"].startswith(tile) and plan["chained"] == chained and plan["splits"] == 1 and plan["tail_tiles"] == 0, plan
    A, B = oracle.fill((M, K), 33, 1, oracle.TERNARY, 0, 1), oracle.fill((N, K), 33, 2, oracle.TERNARY, 0, 1)
    buf = torch.full((GUARD + M * N + GUARD,), POISON, dtype=torch.int16, device=gpu)
    C = buf[GUARD:GUARD + M * N].view(torch.float16).view(M, N)
    print(f"[gpu] hgemm_auto M={M} N={N} K={K} {plan['kernel']} chained {chained}", flush=True)
    hgemm_lib.call("hgemm_auto", _gpu_bits(A, gpu), _gpu_bits(B, gpu), C, M, N, K)
    host = buf.cpu().numpy().view(np.uint16)
    assert np.all(host[:GUARD] == POISON) and np.all(host[GUARD + M * N:] == POISON)
    got = host[GUARD:GUARD + M * N].reshape(M, N)
    assert not np.any((got & 0x7C00) == 0x7C00), "outputs left unwritten or non-finite"
    rows = np.unique(np.concatenate([np.arange(m0, min(M, m0 + 8)) for m0 in range(0, M, 61)] + [np.arange(M - 8, M)]))
    assert np.array_equal(got[rows], oracle.hgemm(np.ascontiguousarray(A[rows]), B))


def test_call_refuses_what_it_refused_before_on_every_call(hgemm_lib, gpu):
    """Operands pass the binding's one-expression check or are told why not, also after calls that were in order."""
    import torch
    A, B = torch.ones((48, 64), dtype=torch.float16, device=gpu), torch.ones((40, 64), dtype=torch.float16, device=gpu)
    C = torch.empty((48, 40), dtype=torch.float16, device=gpu)
    for _ in range(2):
        hgemm_lib.call("hgemm_auto", torch.nn.Parameter(A, requires_grad=False), B, C, 48, 40, 64)  # a Tensor's subclass
        assert bool((C == 64).all())
        shifted = torch.ones(48 * 64 + 1, dtype=torch.float16, device=gpu)[1:].view(48, 64)
        for bad, error, needle in [(A.float(), TypeError, "float16"), (A.cpu(), ValueError, "GPU"), (A[:, :32], ValueError, "shape"),
                                   (A.t().contiguous().t(), ValueError, "contiguous"), (shifted, ValueError, "16-byte"),
                                   (A.bfloat16(), TypeError, "float16"), ([1.0], TypeError, "list")]:
            with pytest.raises(error, match=needle):
                hgemm_lib.call("hgemm_auto", bad, B, C, 48, 40, 64)
        with pytest.raises(ValueError, match="cannot run"):
            hgemm_lib.call("hgemm_mfma_base", A, B, C, 48, 40, 64)
        with pytest.raises(KeyError, match="no such"):
            hgemm_lib.call("no such", A, B, C, 48, 40, 64)


def test_the_longest_k(hgemm_lib, gpu):
    """K within one chunk of 2^31: chunk counts round up without leaving 32 bits."""
    import torch
    K = (1 << 31) - 56
    A, B = torch.zeros((1, K), dtype=torch.float16, device=gpu), torch.zeros((1, K), dtype=torch.float16, device=gpu)
    at = torch.tensor([0, 7, 63, 64, K // 2, K - 65, K - 64, K - 57, K - 56, K - 9, K - 8, K - 1], device=gpu)
    A[0, at], B[0, at] = 1.0, 3.0
    C = torch.empty((1, 1), dtype=torch.float16, device=gpu)
    print(f"[gpu] hgemm_auto M=1 N=1 K={K}", flush=True)
    hgemm_lib.call("hgemm_auto", A, B, C, 1, 1, K)
    assert C.item() == 3.0 * len(at)
