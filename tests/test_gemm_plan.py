"""The GEMM's launch plan (host code, no device needed): what it names can be launched."""
import pytest

from gpu_util import Q4K, Q6K, Q8_0, ROWS, SMALL, WAVES, gemm_converts_itself, gemm_pair_plan, gemm_plan, gemm_small_lds, gemm_workspace_bytes

Q5K, Q3K, Q2K = 13, 11, 10
TYPES = [Q4K, Q6K, Q8_0, Q5K, Q3K, Q2K]
GRID_YZ = 65535  # workgroups a launch may have along y and along z


def tall(limit):
    """Weight row counts around every power of two from 2^14 up, and the most the entry point takes."""
    return [n for e in range(14, 31) for n in ((1 << e) - 1, (1 << e) + 1, 3 << (e - 1)) if n <= limit] + [limit]


# The tile kernel's grid counts eighths of its 32- or 64-row tiles along z.
@pytest.mark.parametrize("t", TYPES)
def test_tall_weights_stay_within_the_grid(t):
    for n in tall(0x7FFFFF00):
        for m in (1, 2, 16, 17, 24, 32, 33, 64, 200, 4096):
            for k in (256, 2304, 5120):
                p = gemm_plan(t, m, n, k)
                if p.kernel == WAVES:
                    assert (-(-n // (32 * p.nr)) + 7) // 8 <= GRID_YZ, (m, n, k, p)
    for n0, n1 in ((16776000, 16776000), (16776704, 1), (16776001, 701), (8388609, 8388609)):
        for m in (17, 32):
            p = gemm_pair_plan(t, m, n0, n1, 256)
            if p is not None and p.kernel == WAVES:
                assert (-(-n0 // (32 * p.nr)) - (-n1 // (32 * p.nr)) + 7) // 8 <= GRID_YZ, (m, n0, n1, p)


# What the kernels keep there: the pre-pass's items (16 bytes per row, operand group and half super-block: 16 groups, and one or
# two per half for sums of sub-blocks of 32 or 16 elements where the type has mins), the row scales, the partial tiles of a K
# split, and what the tile kernel requests past the last item.
@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("m,n,k", [(5, 700, 256), (16, 4096, 4096), (24, 1000, 14336), (64, 4096, 2304), (300, 96, 5120), (512, 14336, 4096),
                                   (1800, 64, 7168), (2048, 1024, 4096)])
def test_workspace_holds_what_is_written(t, m, n, k):
    p = gemm_plan(t, m, n, k)
    groups = {Q6K: 16, Q8_0: 16, Q3K: 20, Q2K: 20}.get(t, 18)
    up = lambda v: -(-v // 256) * 256
    need = up(k // 256 * 2 * groups * p.mp * 16) + up(4 * p.mp) + (up(4 * p.splits * p.mp * n) if p.splits > 1 else 0)
    assert gemm_workspace_bytes(t, m, n, k) == need + (256 * p.mp if p.kernel == WAVES else 0)


# Calls of the entry point that allocates nothing: what its 32 MiB of scratch hold with activations padded to whole tiles fits, also where the
# padding to 128 rows that a batch's weights share would not.
@pytest.mark.parametrize("t,m,n,k", [(Q6K, 1040, 125, 13568), (Q4K, 814, 67, 16128), (Q3K, 677, 68, 17920), (Q8_0, 1040, 125, 13568), (Q5K, 814, 67, 16128)])
def test_scratch_that_whole_tiles_fit(t, m, n, k):
    p = gemm_plan(t, m, n, k)
    assert p.kernel == WAVES and p.mp % 128 == 64, p
    assert gemm_workspace_bytes(t, m, n, k) <= 32 << 20


# Two weights of one batch of which one has tiles of four waves and the other of eight: one launch where that is faster (us: apart, together).
@pytest.mark.parametrize("t,m,n0,n1,k,share", [
    (Q4K, 100, 4096, 1024, 4096, True),    # 20.9, 17.6: q and k of a grouped-query attention
    (Q4K, 128, 3072, 1024, 3072, True),    # 17.6, 12.9
    (Q6K, 96, 4096, 1024, 4096, True),     # 28.0, 20.1
    (Q8_0, 160, 2048, 512, 2048, True),    # 16.2, 11.3
    (Q5K, 160, 2048, 512, 2048, True),     # 16.2, 11.1
    (Q2K, 46, 504, 6528, 1280, True),      # 13.2, 8.8
    (Q3K, 141, 1763, 348, 256, True),      # 12.9, 8.4: a row of one super-block has one wave either way
    (Q4K, 790, 1095, 273, 7680, True),     # 58.8, 44.2
    (Q8_0, 300, 2560, 1280, 2560, False),  # 26.9, 30.6
    (Q4K, 720, 1008, 504, 5888, False),    # 39.3, 51.1: of 288 workgroups 48 on each of four dies
    (Q8_0, 311, 5917, 463, 1280, False),   # 24.7, 31.6: 65 on one die
    (Q2K, 560, 6724, 374, 1280, False),    # 34.3, 38.7
    (Q8_0, 454, 318, 3869, 4096, False)])  # 46.2, 52.9
def test_pairs_of_four_and_eight_waves(t, m, n0, n1, k, share):
    a, b = gemm_plan(t, m, n0, k), gemm_plan(t, m, n1, k)
    assert (a.kernel, b.kernel) == (WAVES, WAVES) and a.nw != b.nw
    assert (gemm_pair_plan(t, m, n0, n1, k) is not None) == share


# Two weights whose tiles alone let the dies share the activations, and together do not: apart where each die would then read more of them than it
# can hold, and that takes longer (us: together, apart).
@pytest.mark.parametrize("t,m,n0,n1,k,share", [
    (Q4K, 2048, 4600, 4600, 4096, False),  # 390, 232
    (Q4K, 1487, 3322, 3322, 4864, False),  # 206, 155
    (Q4K, 1081, 2352, 2352, 5888, True),   # 111, 139
    (Q2K, 1709, 5502, 5502, 9216, False),  # 927, 533
    (Q3K, 1848, 5305, 5305, 6400, False),  # 673, 430
    (Q5K, 1456, 3032, 1694, 7168, False),  # 224, 193
    (Q8_0, 2004, 2932, 2932, 6912, False), # 373, 329
    (Q8_0, 1540, 1891, 1891, 7936, True),  # 216, 226
    (Q6K, 2362, 3366, 3366, 4608, True)])  # 370, 380
def test_pairs_of_many_activation_rows(t, m, n0, n1, k, share):
    assert gemm_plan(t, m, n0, k).kernel == WAVES and gemm_plan(t, m, n1, k).kernel == WAVES
    assert (gemm_pair_plan(t, m, n0, n1, k) is not None) == share


# Tiles of which one die has twice the others' share, or a few more than it has compute units: the row kernels (1.28 and 1.33 times as fast).
@pytest.mark.parametrize("t,m,n,k", [(Q4K, 615, 1276, 8704), (Q6K, 153, 5344, 9472)])
def test_uneven_dies_take_the_rows(t, m, n, k):
    assert gemm_plan(t, m, n, k).kernel == ROWS


# Few activation rows: the kernel that measured faster (us with the short-batch kernel, with the tile kernel), clear cases of either.
@pytest.mark.parametrize("t,m,n,k,kernel", [
    (Q5K, 19, 17096, 19712, SMALL),  # 84, 135: long rows in three rounds of tiles
    (Q5K, 30, 4355, 26112, SMALL),   # 45, 63: long rows that half fill one round
    (Q4K, 26, 16541, 18944, SMALL),  # 71, 100
    (Q4K, 19, 17542, 14848, SMALL),  # 59, 80
    (Q8_0, 19, 37321, 2048, SMALL),  # 27, 36
    (Q4K, 24, 4096, 4096, WAVES),    # 12.8, 10.4
    (Q4K, 17, 8192, 5120, WAVES),    # 20, 15
    (Q5K, 20, 4096, 3072, WAVES),    # 13.4, 10.4
    (Q8_0, 32, 6144, 3072, WAVES),   # 16, 13
    (Q8_0, 20, 1024, 20480, WAVES),  # 37, 19 (row kernel: longer than eight runs)
    (Q4K, 12, 8192, 5120, WAVES),    # 15.9, 13.6
    (Q5K, 12, 14336, 4352, WAVES)])  # 27, 24
def test_few_rows_take_the_faster_kernel(t, m, n, k, kernel):
    assert gemm_plan(t, m, n, k).kernel == kernel, gemm_plan(t, m, n, k)


# A row of one or two super-blocks has as many waves: tiles of 64 weight rows for them only where 32 would be several rounds.
@pytest.mark.parametrize("t,m,n,k", [(Q8_0, 20, 10275, 256), (Q2K, 21, 9389, 256), (Q5K, 28, 9202, 256), (Q2K, 22, 18800, 512)])
def test_short_rows_take_the_small_tile(t, m, n, k):
    p = gemm_plan(t, m, n, k)
    assert (p.kernel, p.nr) == (WAVES, 1), p  # (8.5 us, 11 with 64 rows)


# A launch of rows of one to four super-blocks counts on 8, 4 or 2 workgroups a compute unit (160 KiB of LDS, 128 bytes a workgroup of which are
# the row scales'), up to sixteen row tiles each (four of one super-block): all of them fit, whoever converts the activations.
@pytest.mark.parametrize("xf32", [False, True])
@pytest.mark.parametrize("t", TYPES)
def test_short_batch_workgroups_fit_together(t, xf32):
    for spr in range(1, 5):
        for tiles in (1, 2, 4, 8, 9, 16)[:6 if spr > 1 else 3]:
            assert (gemm_small_lds(t, 16, 256 * spr, tiles, True, xf32) + 128) * (8 // spr) <= 160 * 1024, (spr, tiles)
    for tiles in (1, 8, 9, 64):
        for m, k, own in ((16, 2048, True), (16, 4096, True), (16, 4096, False), (32, 2048, False), (32, 4096, False)):
            if m == 16 or (t in (Q4K, Q5K, Q8_0) and tiles < 64):
                assert gemm_small_lds(t, m, k, tiles, own, xf32) + 128 <= 160 * 1024, (m, k, own, tiles)


# Who converts bf16 activations of a row of more than eight super-blocks, single weights (us by a pre-pass, by the waves themselves).
@pytest.mark.parametrize("t,m,n,k,own", [
    (Q3K, 4, 16908, 5120, False),    # 36.2, 38.6
    (Q3K, 12, 47394, 2304, False),   # 36.5, 40.5
    (Q3K, 16, 28582, 10496, False),  # 68.6, 75.1
    (Q8_0, 6, 36966, 5376, False),   # 66.0, 67.1
    (Q3K, 10, 18833, 4096, True),    # 23.1, 22.9
    (Q3K, 6, 946, 14592, True),      # 16.2, 15.4
    (Q4K, 5, 14336, 4096, True),
    (Q6K, 10, 18136, 5888, True),    # 43.3, 42.9
    (Q2K, 9, 17631, 8192, True)])    # 35.6, 30.1
def test_who_converts(t, m, n, k, own):
    assert gemm_plan(t, m, n, k).kernel == SMALL
    assert gemm_converts_itself(t, m, n, k, 1) == own
    assert not gemm_converts_itself(t, m, n, k, 1, shared=True)
    assert gemm_converts_itself(t, m, n, 2048, 1, shared=True)
