"""Rows of A and B that start on 2-byte boundaries (K % 8 != 0), read where they lie: every tile, with and without K slices,
at the edges of tiles and of the 128-wide chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GUARD, POISON = 4096, 0x7E5A   # elements around C (keeps it 16-byte aligned); a NaN no kernel produces

# shape -> tile, sliced or not.  K: one element into the second chunk, one short of a whole one, four (even) and odd in between
CASES = [
    ((1, 1, 129), "64x64x128", False), ((64, 64, 255), "64x64x128", False), ((65, 63, 257), "64x64x128", False),
    ((129, 130, 191), "64x64x128", False), ((9, 1100, 1531), "64x64x128", True), ((70, 70, 2047), "64x64x128", True),
    ((929, 929, 929), "64x64x128", False), ((265, 265, 3735), "64x64x128", True), ((3, 1001, 4099), "64x64x128", True),
    ((1435, 1435, 1435), "96x96x128", False), ((147, 22092, 1853), "96x96x128", False), ((795, 795, 3639), "96x96x128", True),
    ((535, 535, 14563), "96x96x128", True),
    ((1119, 1119, 1119), "128x64x128", False), ((1664, 996, 275), "128x64x128", False), ((537, 537, 3121), "128x64x128", True),
    ((1681, 1681, 537), "128x128x128", False), ((393, 5106, 647), "128x128x128", False), ((825, 6292, 130), "128x128x128", False),
    ((779, 779, 11221), "128x128x128", True), ((1009, 1009, 7364), "128x128x128", True),
]

# 64 does not divide K though 8 does: the same tiles, unsliced, for products that they are ahead on; 64 divides K but not M or N:
# the four-wave tile of 64x64 on whole chunks, unsliced up to K = 2048 and in slices from there on
ALIGNED_CASES = [
    ((1264, 1264, 1264), "where they lie, 128x64x128", False), ((1403, 1318, 1416), "where they lie, 128x64x128", False),
    ((1193, 1591, 1848), "where they lie, 128x64x128", False), ((377, 5817, 1240), "where they lie, 96x96x128", False),
    ((1416, 1416, 3096), "where they lie, 96x96x128", False), ((462, 4128, 3912), "where they lie, 96x96x128", False),
    ((129, 1000, 640), "edge-guarded 64x64x64", False), ((1000, 1000, 1024), "edge-guarded 64x64x64", False),
    ((1000, 1000, 2048), "edge-guarded 64x64x64", False), ((376, 376, 2048), "edge-guarded 64x64x64", True),
    ((177, 1088, 2432), "edge-guarded 64x64x64", True), ((264, 264, 6784), "edge-guarded 64x64x64", True),
]


def _gpu_bits(bits, gpu):
    import torch
    return torch.from_numpy(bits.view(np.int16)).to(gpu).view(torch.float16)


@pytest.mark.parametrize("shape,tile,sliced", CASES)
def test_unaligned_rows(oracle, hgemm_lib, gpu, shape, tile, sliced):
    """Exact on ternary inputs (sums are integers below 2048) inside a guard band; then with an infinity in one row of A, at a
    k that the last chunk and the one before it both read: that row is infinite with B's sign, no other changes."""
    _exact_and_infinite(oracle, hgemm_lib, gpu, shape, f"where they lie, {tile}", sliced)


@pytest.mark.parametrize("shape,kernel,sliced", ALIGNED_CASES)
def test_aligned_rows_off_the_lines(oracle, hgemm_lib, gpu, shape, kernel, sliced):
    """The same for products whose rows are 16-byte aligned and whose K, M or N no tile divides."""
    _exact_and_infinite(oracle, hgemm_lib, gpu, shape, kernel, sliced)


def _exact_and_infinite(oracle, hgemm_lib, gpu, shape, kernel, sliced):
    import torch
    M, N, K = shape
    plan = hgemm_lib.auto_plan(M, N, K)
    assert kernel in plan["kernel"] and (plan["splits"] > 1) == sliced, plan
    A, B = oracle.fill((M, K), 41, 1, oracle.TERNARY, 0, 1), oracle.fill((N, K), 41, 2, oracle.TERNARY, 0, 1)
    expect = oracle.hgemm(A, B)
    assert np.abs(expect.view(np.float16).astype(np.float32)).max() < 2048
    buf = torch.full((GUARD + M * N + GUARD,), POISON, dtype=torch.int16, device=gpu)
    C = buf[GUARD:GUARD + M * N].view(torch.float16).view(M, N)
    Ad, Bd = _gpu_bits(A, gpu), _gpu_bits(B, gpu)
    print(f"[gpu] hgemm_auto M={M} N={N} K={K} {plan['kernel']} x{plan['splits']}", flush=True)
    hgemm_lib.call("hgemm_auto", Ad, Bd, C, M, N, K)
    host = buf.cpu().numpy().view(np.uint16)
    assert np.all(host[:GUARD] == POISON) and np.all(host[GUARD + M * N:] == POISON)
    assert np.array_equal(host[GUARD:GUARD + M * N].reshape(M, N), expect)
    row, k = M - 1, K - 128
    Bd[:, k] = torch.where(torch.arange(N, device=gpu) % 2 == 0, 1.0, -1.0).half()
    Ad[row, k] = float("inf")
    hgemm_lib.call("hgemm_auto", Ad, Bd, C, M, N, K)
    assert torch.equal(C[row], torch.where(torch.arange(N, device=gpu) % 2 == 0, float("inf"), float("-inf")).half())
    assert M == 1 or bool(torch.isfinite(C[:row]).all())


def test_static_workspace_takes_what_it_took(hgemm_lib, gpu):
    """Rows read where they lie keep partial sums at most, which fit the array; copies beyond it are refused."""
    import torch
    limit = hgemm_lib.static_workspace_bytes()
    for (M, N, K), taken in [((1111, 1111, 5565), True), ((16, 8192, 4097), True), ((4095, 4095, 4095), False)]:
        need = hgemm_lib.auto_workspace_bytes(M, N, K)
        assert need["operands"] == 0 if taken else need["operands"] >= 2 * (M + N) * K
        assert (need["partial"] + need["operands"] <= limit) == taken
        gen = torch.Generator(device=gpu).manual_seed(7)
        A, B = (torch.randint(-1, 2, (rows, K), generator=gen, device=gpu, dtype=torch.int8).half() for rows in (M, N))
        C, D = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu), torch.empty((M, N), dtype=torch.float16, device=gpu)
        rc = hgemm_lib.dll.hgemm_auto_static_workspace(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K)
        assert (rc == 0) == taken
        if taken:
            hgemm_lib.call("hgemm_auto", A, B, D, M, N, K)
            assert torch.equal(C, D)      # whole numbers: the same in any order of additions
