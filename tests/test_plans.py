"""What hgemm_auto plans at sizes where two routes meet (no launch, no GPU)."""
import pytest


@pytest.mark.parametrize("M", [129, 150, 192])
@pytest.mark.parametrize("N", [18432, 28672, 57344])
def test_no_copies_below_the_one_row_rule(hgemm_lib, M, N):
    """K just short of 2048: the copies' padded K would be the first the 192x128 one-row rule covers."""
    for K in range(1992, 2048, 8):
        assert hgemm_lib.auto_workspace_bytes(M, N, K)["operands"] == 0, K


@pytest.mark.parametrize("size", [4600, 5112, 6200])
def test_tuner_times_direct_plans_beside_copies(hgemm_lib, size):
    """K a multiple of 8 and not of 64: copied operands are one plan of several, wherever they come in the order."""
    plans = hgemm_lib.tune_plans(size, size, size, 8)
    on_copies = [p["kernel"].startswith("zero-padded") for p in plans]
    assert len(plans) >= 4 and sum(on_copies) == 1, plans


@pytest.mark.parametrize("shape", [(2603, 2603, 2603), (4095, 4095, 4095), (600, 14336, 4095), (3, 100, 1001), (1111, 1111, 5565)])
def test_tuner_times_rows_read_where_they_lie_beside_copies(hgemm_lib, shape):
    """K % 8 != 0: copies are one plan of several, wherever they come in the order."""
    plans = hgemm_lib.tune_plans(*shape, 12)
    assert len({(p["kernel"], p["splits"]) for p in plans}) == len(plans) >= 5, plans
    assert sum(p["kernel"].startswith("zero-padded operand copies") for p in plans) == 1, plans
    assert all(p["kernel"].startswith(("zero-padded operand copies", "rows read where they lie")) for p in plans), plans


@pytest.mark.parametrize("M,N,K", [(24001, 24001, 1001), (16385, 16385, 8191), (20001, 20001, 4001)])
def test_copies_are_planned_by_what_is_copied(hgemm_lib, M, N, K):
    """(M + N) rows of whole chunks within the workspace's 1 GiB, whatever a C of that size would take."""
    assert 2 * (M + N) * ((K + 63) // 64 * 64) <= 1 << 30
    assert hgemm_lib.auto_plan(M, N, K)["kernel"].startswith("zero-padded")
    assert hgemm_lib.auto_workspace_bytes(M, N, K)["operands"] <= 1 << 30


@pytest.mark.parametrize("shape,sliced", [
    ((58, 8, 1664), True), ((58, 17, 1664), True), ((83, 17, 1072), True), ((121, 17, 2304), True), ((20, 9, 1608), True),
    ((13, 8, 512), False), ((13, 17, 512), False), ((26, 8, 544), False), ((13, 8, 904), False), ((16, 3, 1072), False)])
def test_slice_counts_below_one_tile_of_columns(hgemm_lib, shape, sliced):
    """The split-K family goes by whole tiles, N = 3 ... 17 as N = 64, but for a K of less than 896 (1280 up to M = 32)."""
    M, N, K = shape
    plan = hgemm_lib.auto_plan(M, N, K)
    assert plan["kernel"].startswith("split-K")
    assert plan["splits"] == (hgemm_lib.auto_plan(M, 64, (K + 63) // 64 * 64)["splits"] if sliced else 1), plan


# shape -> what runs it, on whole chunks with aligned rows of C that no row of the small-M table divides: the faster of a
# pipelined tile and a table kernel's guarded form (microseconds of the two when they were compared)
@pytest.mark.parametrize("shape,kernel", [
    ((114, 50336, 128), "pipelined 128x128x64, 4 waves, 2"),   # 6.2, 11.7 on 128x128 split-K
    ((40, 57864, 128), "pipelined 128x128x64, 4 waves, 2"),    # 6.1, 8.3 on 64x128 split-K
    ((117, 8, 1216), "pipelined 64x64"),                       # 6.4, 10.5 on 128x64 split-K
    ((75, 5808, 25920), "pipelined 128x128"),                  # 57.8, 79.0
    ((42, 8, 29568), "pipelined 64x64"),                       # 10.8, 12.7 on 64x64 split-K
    ((4, 96, 32704), "pipelined 64x64"),                       # 11.6, 18.3 on the ring kernel
    ((8, 4200, 19008), "pipelined 64x64"),                     # 33.2, 43.1
    ((50, 8072, 320), "pipelined 64x64"),                      # 4.6, 5.3
    ((1, 3544, 25216), "streaming decode"),                    # 37.1 on the 64x64 tile, 29.0
    ((6, 640, 640), "streaming decode"),
    ((113, 12496, 2368), "split-K 128x64"),                    # 25.8, 19.5
    ((102, 40, 1664), "split-K 2x64x64x64"),                   # 7.0, 5.8 on 128x64 split-K
    ((28, 7968, 21952), "split-K 32x64"),                      # 65.1, 57.1
    ((59, 3240, 24896), "split-K 64x64"),                      # 37.5, 33.4
    ((84, 11736, 832), "split-K 128x64"),                      # 9.2, 8.4
])
def test_small_m_on_whole_chunks_of_ragged_columns(hgemm_lib, shape, kernel):
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith(kernel)


# K ends inside one of its first five chunks, N = 16384 ... 65536 with aligned rows of C (microseconds before and after)
@pytest.mark.parametrize("shape,kernel", [
    ((65, 34344, 120), "pipelined 128x128x64, 4 waves, 2"),    # 10.0, 6.9 (128x128 split-K before)
    ((117, 40784, 104), "pipelined 128x128x64, 4 waves, 2"),
    ((35, 52088, 88), "split-K 64x64"),                        # 7.5, 5.9 (64x128 split-K before)
    ((69, 23286, 88), "split-K 128x128"),                      # rows of C not aligned
])
def test_small_m_on_short_k(hgemm_lib, shape, kernel):
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith(kernel)


# K of one chunk, or one and a part, on ragged sizes (microseconds on the tile that ran them before, now)
@pytest.mark.parametrize("shape,kernel", [
    ((2308, 40, 80), "split-K 64x64"),                         # 4.4, 3.8
    ((163, 991, 128), "split-K 64x64"),                        # 4.8, 3.5
    ((147, 20, 72), "pipelined 128x128"),                      # less than one 64-column tile, rows of C not aligned
    ((428, 10574, 96), "pipelined 128x128"),                   # too many tiles
    ((11111, 10444, 72), "guarded"),                           # 119, 98
    ((7873, 56748, 88), "guarded"),                            # 471, 399
    ((8077, 37696, 72), "pipelined 128x128"),                  # whole lines of C
    ((2315, 55336, 64), "guarded"),                            # 153, 99
    ((2315, 55296, 64), "split-K 64x64"),                      # whole tiles of columns
    ((300, 1000, 64), "split-K 64x64"),                        # small C
])
def test_ragged_sizes_on_one_or_two_chunks(hgemm_lib, shape, kernel):
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith(kernel)


@pytest.mark.parametrize("shape,copied", [
    ((1391, 4586, 7592), True),      # 146 us directly, 102
    ((2190, 3878, 11528), True),     # 207, 158
    ((5112, 5112, 5112), True),      # 266, 196
    ((1198, 9512, 11240), False),    # 210, 286
    ((4000, 4000, 4000), False),     # 81.5, 98.0
    ((3296, 3584, 3488), False),     # 54.6, 64.8
    ((1000, 1000, 1000), False),
])
def test_copies_of_aligned_rows_where_they_pay(hgemm_lib, shape, copied):
    """K a multiple of 8 and not of 64 runs on guarded kernels or on copies with rows of whole cache lines."""
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith("zero-padded") == copied


# M = 9 ... 16 against N from 14336 on (microseconds on the ring kernel's guarded form, on the split-K tile)
@pytest.mark.parametrize("shape,kernel", [
    ((16, 15040, 10648), "split-K 32x64"),                     # 98.4, 66.8
    ((10, 14800, 7232), "split-K 32x64"),                      # 41.3, 37.6
    ((16, 15257, 8320), "split-K 32x64"),                      # 51.3, 39.8
    ((12, 28672, 6152), "split-K 32x64"),
    ((12, 20001, 8192), "streaming decode"),                   # a K of the persistent kernel's: its row's stand-in
    ((12, 20000, 8192), "decode with A in registers"),
])
def test_rows_of_the_persistent_kernel_hold_at_its_k_only(hgemm_lib, shape, kernel):
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith(kernel)


# M = 9 ... 32 against N up to 8192 (microseconds on the split-K tile, on the ring kernel)
@pytest.mark.parametrize("shape,kernel", [
    ((32, 2944, 6912), "split-K 32x64"),                       # 11.5, 14.0
    ((20, 3915, 6400), "streaming decode"),                    # 13.4, 12.8; 11.8, 9.6 with B in the Infinity Cache
    ((24, 3648, 6144), "streaming decode"),                    # 13.0, 13.5; 11.1, 9.2
    ((30, 1536, 6976), "streaming decode"),                    # the longer K below N = 2304
    ((24, 2560, 6080), "streaming decode"),
    ((20, 2624, 7000), "split-K 32x64"),                       # 11.4, 16.6: K ends inside a chunk
    ((29, 2511, 7024), "split-K 32x64"),                       # 11.7, 17.6
    ((24, 2560, 4600), "streaming decode"),
    ((24, 4400, 1672), "split-K 32x64"),
    ((24, 6400, 1664), "streaming decode"),
    ((14, 1504, 7080), "split-K 32x64"),                       # 8.8, 9.9
    ((14, 2048, 7080), "streaming decode"),
])
def test_ring_kernel_for_few_rows_and_a_long_k(hgemm_lib, shape, kernel):
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith(kernel)


# K % 8 != 0 read where it lies: sizes whose copies would not fit the array of the static workspace, and others
@pytest.mark.parametrize("shape", [(520, 520, 14561), (1000, 1000, 8001), (3330, 656, 6006), (453, 4600, 6178), (16, 8192, 4097),
                                   (5, 35434, 1547), (1111, 1111, 1111), (515, 1032, 1100)])
def test_workspace_reported_is_what_the_plan_keeps(hgemm_lib, shape):
    """No copies are reported where none are made, and the static workspace refuses nothing that fits it as reported."""
    plan, need = hgemm_lib.auto_plan(*shape), hgemm_lib.auto_workspace_bytes(*shape)
    assert "read where they lie" in plan["kernel"] and need["operands"] == 0
    assert (need["partial"] > 0) == (plan["splits"] > 1) and need["partial"] <= hgemm_lib.static_workspace_bytes()


def test_static_workspace_refuses_what_does_not_fit(hgemm_lib, capfd):
    """Before any device call: so also without a GPU."""
    import ctypes
    need = hgemm_lib.auto_workspace_bytes(4095, 4095, 4095)
    assert need["operands"] > hgemm_lib.static_workspace_bytes()
    address = ctypes.c_void_p(1 << 20)
    assert hgemm_lib.dll.hgemm_auto_static_workspace(address, address, address, 4095, 4095, 4095) == 1
    assert str(need["operands"]) in capfd.readouterr().err


# K % 8 != 0, M > 8 (microseconds on copies, read where they lie)
@pytest.mark.parametrize("shape,copied", [
    ((636, 3819, 2821), True),       # 31.8, 39.4
    ((2794, 693, 9069), True),       # 64.8, 87.1
    ((264, 10926, 1455), True),      # 27.2, 34.2
    ((1395, 1439, 8649), True),      # 62.0, 79.8
    ((2603, 2603, 2603), True),      # 46, 62
    ((929, 929, 929), False),        # 12.0, 8.2
    ((2400, 414, 1458), False),      # 17.5, 12.4
    ((339, 18066, 8334), False),     # 230, 172: copies beyond the Infinity Cache
])
def test_copies_of_unaligned_rows_where_they_pay(hgemm_lib, shape, copied):
    kernel = hgemm_lib.auto_plan(*shape)["kernel"]
    assert kernel.startswith("zero-padded operand copies" if copied else "rows read where they lie"), kernel


# M = 65 ... 128 against a B of less than 32 MB (microseconds on the 128x64 tile, as two rows of 64x64 tiles)
@pytest.mark.parametrize("shape,two_rows", [
    ((75, 1024, 1664), True),        # 7.7, 6.4
    ((113, 2560, 1792), True),       # 11.2, 8.0
    ((80, 8192, 576), True),
    ((80, 8256, 576), False),        # more than one 64x64 tile to a CU
    ((121, 10470, 152), True),       # 5.5, 4.8: below K = 192 from M = 96 on
    ((77, 13632, 128), False),       # 3.9, 4.3
    ((67, 14126, 64), False),        # 3.5, 3.9
    ((112, 37824, 128), True),       # 11.7, 8.9: more than one 128x64 tile too
    ((80, 22592, 256), True),        # 8.5, 7.7
    ((76, 10048, 480), False),       # 6.3, 8.1
    ((125, 8832, 904), False),       # 13.3, 16.1
    ((124, 4160, 3328), False),      # 15.0, 17.9
    ((65, 4529, 3328), False),       # 13.9, 16.5
    ((100, 1984, 8192), True),
    ((65, 6493, 2416), True),        # 16.6, 15.3
    ((90, 6272, 2560), True),        # 15.9, 15.2; 13.1, 11.0 with B in the Infinity Cache
    ((100, 5696, 2752), True),       # 16.0, 15.5; 14.0, 11.2
    ((83, 5056, 2624), False),       # 13.1, 14.1
])
def test_two_rows_of_split_k_tiles_where_they_pay(hgemm_lib, shape, two_rows):
    assert hgemm_lib.auto_plan(*shape)["kernel"].startswith("split-K 2x64x64x64" if two_rows else "split-K 128x64")


# 64x64 split-K tiles against a B of 48 MB and more
@pytest.mark.parametrize("shape,splits", [
    ((64, 10432, 6528), 3),          # 1.14x of one slice
    ((56, 10335, 5440), 3),          # 1.17
    ((59, 16576, 4032), 3),          # 1.09
    ((43, 8832, 5824), 3),           # five slices 0.92 of three
    ((46, 11328, 6848), 1),          # four slices 0.97 of one
])
def test_slice_counts_for_a_large_b(hgemm_lib, shape, splits):
    plan = hgemm_lib.auto_plan(*shape)
    assert plan["kernel"].startswith("split-K 64x64") and plan["splits"] == splits, plan
