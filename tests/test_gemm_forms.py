"""Which form of a GEMM kernel a launch takes.  The rules are host code and run here without a GPU, on 256 units and
on fewer; the forms' results are compared in the test_gpu_gemm_* files."""
import ctypes

import pytest

from helpers import bench_lib

LDS_OF_A_UNIT = 160 * 1024
TILES = ((8, 8), (6, 8), (8, 6), (5, 8), (6, 6), (4, 8), (3, 8), (4, 6), (3, 6), (4, 4), (3, 4), (2, 4))
WIDTHS = (4, 32, 36, 256, 1028, 6144, 8192, 8452, 28672)


@pytest.fixture(scope="module")
def few_rows():
    lib = bench_lib()
    lib.twb_gemm_ksplit_form.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 3 + [ctypes.POINTER(ctypes.c_int64)]

    def form(M, N, K, count=1, cap=0, cus=256):
        f = (ctypes.c_int64 * 6)()
        assert lib.twb_gemm_ksplit_form(M, N, K, count, cap, cus, f) == 1, (M, N, K, count, cap, cus)
        return dict(zip(("rows", "cols", "stages", "stream", "lds", "groups"), f))

    return form


@pytest.mark.parametrize("cus", [256, 80])
@pytest.mark.parametrize("K", [8, 64, 200, 1024, 3584, 3696, 7168])
def test_every_launch_of_few_rows_has_a_kernel(few_rows, K, cus):
    for M in (*range(1, 130), 1000):
        for N in WIDTHS:
            for count, cap in ((1, 0), (8, 0), (1, 7), (3, 160)):
                f = few_rows(M, N, K, count, cap, cus)
                assert f["lds"] <= LDS_OF_A_UNIT and f["cols"] % 4 == 0 and f["rows"] * -(-M // f["rows"]) >= M
                assert not cap or f["groups"] <= cap


@pytest.mark.parametrize("cus", [256, 80])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32])
def test_units_with_several_tiles_hold_two_workgroups(few_rows, M, cus):
    """Up to 32 rows: a third slab in LDS only where no unit has a second tile to fill its waits with, and past 16
    rows only where rows of b are whole lines."""
    for K in (128, 1024, 3584, 3696):
        for N in WIDTHS:
            for count, cap in ((1, 0), (4, 0), (8, 0), (1, 16), (2, 200)):
                f = few_rows(M, N, K, count, cap, cus)
                tiles = count * -(-N // f["cols"])
                if tiles > (min(cap, cus) if cap else cus):
                    assert 2 * f["lds"] <= LDS_OF_A_UNIT, (N, K, count, cap)
                else:
                    whole_lines = K % 64 == 0
                    assert f["stages"] == (3 if whole_lines or M <= 16 else 2), (N, K, count, cap)


@pytest.mark.parametrize("M,rows", [(65, 40), (80, 40), (88, 48), (96, 48), (97, 64)])
def test_even_shares_of_two_row_tiles(few_rows, M, rows):
    """Not where a grid cap makes workgroups of long inner dimensions walk several tiles."""
    for N, K in ((4096, 2048), (6144, 2048), (4096, 2112), (1024, 3584)):
        for cap in (0, 16, 160, 255, 256, 1000):
            f = few_rows(M, N, K, 1, cap)
            assert f["rows"] == (64 if K > 2048 and 0 < cap < 256 else rows), (N, K, cap)


@pytest.mark.parametrize("K", [16, 80, 208, 336, 528, 544, 784, 1040, 1056, 1264, 1312, 1952, 2016, 72, 328, 1000, 7384])
def test_short_rows_are_fetched_by_slabs(K):
    """Whole lines cost a tile more than they give there; rows that are no multiple of 16 never take them."""
    assert [bench_lib().twb_gemm_tile_rows(*s, ctypes.c_int64(K)) for s in TILES] == [1] * len(TILES)


@pytest.mark.parametrize("K,lines", [(1296, 7), (3696, 7), (2080, 5), (7392, 5), (64, 0), (1024, 0), (3584, 0)])
def test_long_rows_are_fetched_by_lines_where_the_ring_has_room(K, lines):
    kinds = [bench_lib().twb_gemm_tile_rows(*s, ctypes.c_int64(K)) for s in TILES]
    assert kinds.count(2) == lines and kinds.count(0 if K % 64 == 0 else 1) == len(TILES) - lines


@pytest.mark.parametrize("M,most_mib", [(65, 64), (72, 64), (73, 56), (80, 56), (81, 31), (96, 31)])
def test_large_weights_keep_tiles_of_64_rows(few_rows, M, most_mib):
    for mib in (8, 16, 31, 33, 40, 56, 57, 64, 65, 112):
        f = few_rows(M, 8192, 64 * mib)           # 8192 columns: a MiB per 64 of K
        assert (f["rows"] < 64) == (mib <= most_mib), mib


@pytest.mark.parametrize("M", [8, 32, 64, 96, 128])
def test_tiles_of_a_batch_are_no_narrower_than_its_rounds_need(few_rows, M):
    for N in (264, 1024, 2048, 4096, 6144, 8192):
        for count in (1, 2, 3, 8, 16):
            f = few_rows(M, N, 1024, count)
            row_tiles, widest = count * -(-M // f["rows"]), 64 if M > 64 else 32
            full_width = row_tiles * -(-N // widest)
            rounds = -(-full_width // 256)
            assert f["groups"] <= max(full_width, 256 * rounds), (N, count)
