"""GPU parity of the tile GEMM (gemm_kw.hip): a workgroup owns a tile of Y and its waves split K."""
import numpy as np
import pytest

import pmetal_amd as pm
from pmetal_amd import _lib
from gpu_util import Q4K, Q6K, Q8_0, ROWS, SMALL, WAVES, gemm_pair_plan, gemm_plan
from test_gpu_gemm import gpu_qgemm, reference

pytestmark = pytest.mark.gpu

BLOCK = {Q4K: 144, Q6K: 210, Q8_0: 34, 13: 176, 11: 110, 10: 84}


@pytest.fixture(scope="module", autouse=True)
def _device():
    pm.init(0)


def random_blocks(rng, t, n, k):
    """Every scale, min and quant pattern; d (and dmin) of ordinary size and, where the format allows it, of both signs."""
    raw = rng.integers(0, 256, size=(n * (k // (32 if t == Q8_0 else 256)), BLOCK[t]), dtype=np.uint8)
    d = (rng.uniform(0.5, 2.0, (raw.shape[0], 2)) * 0.01 * rng.choice([-1.0, 1.0], (raw.shape[0], 2))).astype(np.float16).view(np.uint8)
    at = {Q4K: 0, 13: 0, Q6K: 208, Q8_0: 0, 11: 108, 10: 80}[t]
    width = 4 if t in (Q4K, 13, 10) else 2
    raw[:, at:at + width] = d[:, :width]
    return raw.reshape(-1)


# (m, n, k): one weight row, one super-block; row counts around 32 and 64 on both sides (all in 32 x 32 tiles: test_each_tile has the
# others); rows of 7, 8, 9 and 17 super-blocks (waves of equal and of different length); a narrow weight with long rows (K split over
# workgroups, the last split shorter than the others); (200, 4100, 768): the row kernels for all types but Q8_0
@pytest.mark.parametrize("m,n,k", [(17, 1, 256), (32, 31, 1792), (33, 33, 2048), (64, 64, 2304), (65, 65, 4352), (63, 97, 512),
                                   (48, 40, 18688), (29, 70, 33024), (130, 1000, 1024), (200, 4100, 768)])
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_tiles_match_dequantize_then_matmul(oracle, t, m, n, k):
    rng = np.random.default_rng(7 * t + m + n + k)
    raw = random_blocks(rng, t, n, k)
    bits = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32)).reshape(m, k)
    x = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    for order in (0, 1) if t in (Q4K, 13) else (0,):
        want = reference(oracle, t, raw, n, k, x, order)
        got = gpu_qgemm(t, raw, n, k, bits, m, order=order)
        # bf16 activations and the integer weight tiles are exact; what is left are at most k / 16 + 16 additions in f32 on
        # partial sums within four times the largest result
        bound = (k / 16 + 16) * 2.0 ** -24 * 4
        assert np.max(np.abs(got - want)) <= bound * np.max(np.abs(want)), order
        got16 = gpu_qgemm(t, raw, n, k, bits, m, y_dtype=pm.DTYPE_BF16, order=order)
        assert np.max(np.abs(got16 - want)) <= (2.0 ** -8 + bound) * np.max(np.abs(want)), order


# Up to 16 activation rows: both sides of each line between this kernel and the short-batch kernels (9, 12, 13, 17, 20, 21, 24, 25,
# 33, 36 and 37 super-blocks a row; 4096 and 7168 weight rows), one and sixteen activation rows, a weight row count off every tile
@pytest.mark.parametrize("m,n,k", [(1, 33, 2304), (16, 1, 2304), (5, 7168, 2304), (4, 7169, 2304), (16, 70, 3072), (16, 4097, 2560), (3, 65, 3328), (2, 97, 4352),
                                   (16, 31, 5120), (7, 4129, 5376), (16, 40, 6144), (9, 33, 6400), (16, 4100, 8448), (1, 64, 9216), (6, 30, 9472)])
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_short_batches_match_dequantize_then_matmul(oracle, t, m, n, k):
    test_tiles_match_dequantize_then_matmul(oracle, t, m, n, k)


# Two weights of a batch on either side of the line share their prepared activations and take a kernel each; two on one side a launch.
@pytest.mark.parametrize("m,k,ns", [(16, 2560, (33, 4097)), (5, 3072, (4100, 70)), (12, 2304, (97, 64)), (16, 5376, (4129, 40))])
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_short_batch_pairs_match_separate_calls(oracle, t, m, k, ns):
    test_pairs_match_separate_calls(oracle, t, m, k, ns)


# The pre-pass holds 1, 2, 3, 4, 6 or 8 items per thread, or reads a longer row twice; one, two (from 384 rows on) or four rows (from
# 1024 on) per workgroup.  Rows of activations that end inside a workgroup, row lengths on both sides of each step.
@pytest.mark.parametrize("m,k", [(3, 4096), (18, 4352), (17, 16384), (20, 16640), (33, 32768), (2, 33024), (385, 4096), (390, 4352), (385, 33024),
                                 (1025, 2048), (1026, 2304), (1025, 8192), (1027, 8448), (1025, 16640),
                                 (18, 8448), (3, 12288), (17, 12544), (33, 24576), (2, 24832), (385, 12288), (390, 12544), (385, 24576),
                                 (1026, 4352), (1025, 6144), (1025, 6400), (1025, 12288), (1027, 12544)])
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 10])
def test_prepared_activations(oracle, t, m, k):
    n = 5
    rng = np.random.default_rng(t + m + k)
    raw = random_blocks(rng, t, n, k)
    bits = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32)).reshape(m, k)
    x = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    for order in (0, 1) if t in (Q4K, 13) else (0,):
        want = reference(oracle, t, raw, n, k, x, order)
        for given in (bits, x):  # the same values in either type: exact operands for both, the bound of the test above
            got = gpu_qgemm(t, raw, n, k, given, m, order=order, x_dtype=pm.DTYPE_BF16 if given is bits else pm.DTYPE_F32)
            assert np.max(np.abs(got - want)) <= (k / 16 + 16) * 2.0 ** -24 * 4 * np.max(np.abs(want)), (order, given.dtype)


# Two weights that share their activations, against a call each: short batches and wave tiles, which go in one launch, row counts off
# every tile, the seam between the two inside a round; row kernels, which at these sizes do not share a launch (test_pairs_in_one_launch
# has sizes that do); three weights of which two are neighbours of one kind.
@pytest.mark.parametrize("m,k,ns", [(3, 512, (17, 130)), (16, 4096, (1, 1000)), (16, 2304, (4600, 33)), (17, 1024, (31, 65)), (64, 1792, (97, 64)),
                                    (100, 768, (300, 129)), (600, 512, (7000, 6300)), (1030, 256, (3900, 4111)), (40, 512, (70, 50, 20))])
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_pairs_match_separate_calls(oracle, t, m, k, ns):
    rng = np.random.default_rng(t + m + k)
    raws = [random_blocks(rng, t, n, k) for n in ns]
    bits = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32)).reshape(m, k)
    x = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    lib = _lib.load()
    dx, dws = pm.DeviceBuffer.from_host(bits), [pm.DeviceBuffer.from_host(raw) for raw in raws]
    for order in (0, 1) if t in (Q4K, 13) else (0,):
        dys = [pm.DeviceBuffer(m * n * 4 + 256) for n in ns]
        for dy in dys:
            pm.check(lib.pmetal_hip_memset(dy.ptr, 0xFF, dy.nbytes, None))
        descs = (_lib.GemmDesc * len(ns))(*[_lib.GemmDesc(t, pm.DTYPE_F32, order, 0, n, w.ptr, y.ptr) for n, w, y in zip(ns, dws, dys)])
        pm.check(lib.pmetal_hip_qgemm_batch(descs, len(ns), k, dx.ptr, pm.DTYPE_BF16, m, None))
        pm.check(lib.pmetal_hip_sync(None))
        for n, raw, dy in zip(ns, raws, dys):
            out = dy.to_host(np.uint8)
            assert np.all(out[m * n * 4:] == 0xFF)
            got, want = out[:m * n * 4].view(np.float32).reshape(m, n), reference(oracle, t, raw, n, k, x, order)
            assert np.max(np.abs(got - want)) <= (k / 16 + 16) * 2.0 ** -24 * 4 * np.max(np.abs(want)), order
            assert np.array_equal(got, gpu_qgemm(t, raw, n, k, bits, m, order=order)), order


# ... of which one has tiles of four waves and the other of eight (or the five of a short row), in one launch.  Of each tile: the weight of four
# waves in front and behind, its tiles one to a workgroup beside four waves that wait (the first two cases), two to a workgroup, an odd and an
# even number of them, where that saves a round of workgroups.  The last seven: the dies share the blocks of activation rows.
MIXED = [(1, 1, 193, 2048, (174, 1980)), (1, 1, 135, 1280, (2656, 68)), (1, 1, 213, 1280, (1665, 654)), (1, 1, 155, 2048, (35, 3227)), (1, 1, 130, 1280, (2210, 1048)),
         (2, 1, 163, 2048, (177, 2310)), (2, 1, 161, 1280, (2386, 71)), (2, 1, 182, 1280, (2049, 656)), (2, 1, 190, 2048, (520, 2193)), (2, 1, 177, 2304, (49, 2661)),
         (2, 2, 162, 2048, (551, 2193)), (2, 2, 231, 1280, (1695, 367)), (2, 2, 272, 1280, (1040, 2221)), (2, 2, 384, 2304, (1483, 1177)), (2, 2, 234, 1792, (1872, 2188)),
         (1, 1, 531, 1280, (778, 132)), (1, 1, 544, 1792, (223, 720)), (2, 1, 620, 2048, (591, 125)), (2, 1, 551, 1536, (159, 654)),
         (2, 2, 581, 1792, (687, 343)), (2, 2, 585, 1280, (225, 820)), (2, 2, 545, 1536, (416, 525))]
MIXED = [(t, *c) for c in MIXED for t in (Q4K, Q6K, Q8_0, 13, 11, 10)] + [(Q6K, 1, 2, 31, 2304, (1003, 9001)), (Q8_0, 1, 2, 31, 1280, (8500, 6000))]


@pytest.mark.parametrize("t,mb,nr,m,k,ns", MIXED)
def test_pairs_of_four_and_eight_waves(oracle, t, mb, nr, m, k, ns):
    p = gemm_pair_plan(t, m, *ns, k)
    assert p is not None and (p.kernel, p.mb, p.nr) == (WAVES, mb, nr), p
    assert {gemm_plan(t, m, n, k).nw for n in ns} == {4, 8}
    test_pairs_match_separate_calls(oracle, t, m, k, ns)


def test_results_in_one_place_are_not_paired(oracle):
    m, n, k = 64, 300, 512
    rng = np.random.default_rng(5)
    raws = [random_blocks(rng, Q4K, n, k) for _ in range(2)]
    bits = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32)).reshape(m, k)
    lib = _lib.load()
    dx, dws, dy = pm.DeviceBuffer.from_host(bits), [pm.DeviceBuffer.from_host(raw) for raw in raws], pm.DeviceBuffer(m * n * 4)
    descs = (_lib.GemmDesc * 2)(*[_lib.GemmDesc(Q4K, pm.DTYPE_F32, 0, 0, n, w.ptr, dy.ptr) for w in dws])
    pm.check(lib.pmetal_hip_qgemm_batch(descs, 2, k, dx.ptr, pm.DTYPE_BF16, m, None))
    pm.check(lib.pmetal_hip_sync(None))
    want = gpu_qgemm(Q4K, raws[1], n, k, bits, m)  # the last one's
    assert np.array_equal(dy.to_host(np.float32).reshape(m, n), want)


# ---- every kernel that the plan names, at shapes for which it is asserted to name it -------------------------------
TYPES = [Q4K, Q6K, Q8_0, 13, 11, 10]


def orders(t):
    return (0, 1) if t in (Q4K, 13) else (0,)


def bf16_rows(oracle, rng, m, k):
    bits = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32)).reshape(m, k)
    return bits, oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)


def bound(k):  # as above: at most k / 16 + 16 additions in f32 on partial sums within four times the largest result
    return (k / 16 + 16) * 2.0 ** -24 * 4


# The four tiles of the tile kernel: 32 or 64 activation rows by 32 or 64 weight rows.  Rows just past a tile on either side, rows of
# 2, 3, 7, 9 and 10 super-blocks (2, 3, 7 and 5 waves; 9: the last wave has one where the others have two); 700 activation rows: the dies
# share out the activations and not the weights, over more than one tile of these.
@pytest.mark.parametrize("mb,nr,m,n,k", [(1, 1, 33, 4000, 512), (1, 1, 600, 100, 512), (1, 1, 600, 130, 2304),
                                         (1, 2, 17, 12289, 2304), (1, 2, 32, 10049, 2560), (1, 2, 17, 10049, 4352),
                                         (2, 1, 33, 8129, 768), (2, 1, 161, 2561, 512), (2, 1, 300, 1473, 1792), (2, 1, 700, 705, 512),
                                         (2, 2, 33, 8257, 2304), (2, 2, 97, 4097, 1792), (2, 2, 700, 1000, 1024)])
@pytest.mark.parametrize("t", TYPES)
def test_each_tile(oracle, t, mb, nr, m, n, k):
    p = gemm_plan(t, m, n, k)
    assert (p.kernel, p.mb, p.nr, p.splits) == (WAVES, mb, nr, 1), p
    test_tiles_match_dequantize_then_matmul(oracle, t, m, n, k)


# ... with four and with eight waves, which decide how many columns a thread takes where the tiles are added: odd weight row counts (rows of
# results that begin at any of them, a last piece of one to three columns), rows of 3, 4, 5, 6 and 8 super-blocks (fewer than the waves, as
# many, and a wave with one more than the others), the last activation row of a tile alone in its block; and two weights in
# one launch, to the bit what each is alone.
@pytest.mark.parametrize("mb,nr,nw,m,n,k", [(1, 1, 4, 81, 9837, 1280), (1, 1, 8, 47, 3529, 2048), (1, 1, 4, 20, 17001, 768), (2, 1, 4, 35, 7427, 1024),
                                            (2, 1, 4, 304, 1591, 1536), (2, 2, 4, 97, 14829, 1024), (2, 2, 4, 399, 3967, 1280), (2, 2, 8, 49, 12359, 1024)])
@pytest.mark.parametrize("t", TYPES)
def test_each_tile_with_either_wave_count(oracle, t, mb, nr, nw, m, n, k):
    p = gemm_plan(t, m, n, k)
    assert (p.kernel, p.mb, p.nr, p.splits, p.nw) == (WAVES, mb, nr, 1, nw), p
    test_tiles_match_dequantize_then_matmul(oracle, t, m, n, k)
    if (mb, nr) == (2, 2):
        assert gemm_pair_plan(t, m, n, n - 128, k).nw == nw
        test_pairs_match_separate_calls(oracle, t, m, k, (n, n - 128))


# ... and with K split over workgroups, which the plan does for long rows; the last split is shorter than the others (69, 73 and 17
# super-blocks in four, 73 in two)
@pytest.mark.parametrize("t,mb,nr,splits,m,n,k", [(Q4K, 2, 1, 4, 161, 321, 18688), (Q6K, 2, 1, 4, 33, 1025, 4352), (Q8_0, 2, 1, 4, 33, 1025, 4352),
                                                  (13, 2, 1, 4, 33, 1025, 4352), (Q6K, 2, 2, 2, 97, 2561, 18688), (Q8_0, 2, 2, 4, 33, 2049, 18688),
                                                  (13, 2, 2, 4, 193, 577, 18688), (11, 2, 2, 4, 63, 2561, 18688), (10, 2, 2, 4, 33, 2561, 18688),
                                                  (Q4K, 2, 2, 4, 513, 321, 18688), (Q4K, 2, 1, 2, 700, 321, 18688)])
def test_each_tile_with_a_k_split(oracle, t, mb, nr, splits, m, n, k):
    p = gemm_plan(t, m, n, k)
    assert (p.kernel, p.mb, p.nr, p.splits) == (WAVES, mb, nr, splits), p
    test_tiles_match_dequantize_then_matmul(oracle, t, m, n, k)


# Weights so tall that the plan keeps the short-batch kernels with two blocks of activations (Q4_K, Q5_K, Q8_0) and the row kernels with
# 32 and with 64 activation rows; a sample of rows at both ends and in the middle against the oracle.  Rows of 1, 2, 9 and 16 super-blocks
# and, in runs with partial tiles, of 32 and (Q8_0) 9 and 16; 136: longer than the short-batch kernels take.  The first two: rows of 20 and
# 17 super-blocks where the tile kernel ends, whose second run of the short-batch kernels leaves waves without a super-block.
TWO_BLOCKS = {Q4K: SMALL, 13: SMALL, Q8_0: SMALL, Q6K: ROWS, 11: ROWS, 10: WAVES}
ALL_ROWS, ALL_SMALL = dict.fromkeys(TYPES, ROWS), dict.fromkeys(TYPES, SMALL)


@pytest.mark.parametrize("m,n,k,kernel", [(9, 14401, 5120, ALL_SMALL), (16, 14401, 4352, ALL_SMALL), (17, 24577, 4096, TWO_BLOCKS), (32, 24577, 4096, TWO_BLOCKS), (17, 12289, 8192, TWO_BLOCKS), (32, 12289, 8192, TWO_BLOCKS),
                                          (29, 50001, 2304, TWO_BLOCKS), (24, 400001, 256, TWO_BLOCKS), (25, 200001, 512, TWO_BLOCKS), (24, 3100, 34816, {**ALL_ROWS, 10: WAVES}),
                                          (33, 70001, 512, ALL_ROWS), (64, 40001, 512, ALL_ROWS), (192, 40001, 256, ALL_ROWS), (33, 60001, 2304, ALL_ROWS)])
@pytest.mark.parametrize("t", TYPES)
def test_tall_weights(oracle, t, m, n, k, kernel):
    p = gemm_plan(t, m, n, k)
    assert p.kernel == kernel[t] and (p.kernel != ROWS or p.mb == (1 if m <= 32 else 2)), p
    rng = np.random.default_rng(t + m + n + k)
    raw = random_blocks(rng, t, n, k)
    bits, x = bf16_rows(oracle, rng, m, k)
    rows = np.r_[0:300, n // 2 - 100:n // 2 + 100, n - 300:n]
    sample = raw.reshape(n, -1)[rows].reshape(-1)
    for order in orders(t):
        want = reference(oracle, t, sample, len(rows), k, x, order)
        got = gpu_qgemm(t, raw, n, k, bits, m, order=order)
        assert np.all(np.isfinite(got))
        assert np.max(np.abs(got[:, rows] - want)) <= bound(k) * np.max(np.abs(want)), order
        got16 = gpu_qgemm(t, raw, n, k, bits, m, y_dtype=pm.DTYPE_BF16, order=order)
        assert np.max(np.abs(got16[:, rows] - want)) <= (2.0 ** -8 + bound(k)) * np.max(np.abs(want)), order


# Two weights in one launch, for each kernel that takes them: the plan is asked that it is one launch.  Row kernels with 128, 64 and 32
# activation rows, short batches with two blocks of activations, tiles whose plan for the pair is a larger tile than each weight's own.
@pytest.mark.parametrize("m,k,ns,kernel", [(300, 512, (8200, 8201), ALL_ROWS), (200, 512, (9000, 9401), ALL_ROWS), (1030, 512, (8200, 8301), ALL_ROWS),
                                           (40, 256, (76801, 76900), ALL_ROWS), (24, 256, (400001, 400100), TWO_BLOCKS), (24, 4096, (24577, 24600), {Q4K: SMALL, 13: SMALL, 10: WAVES}),
                                           (20, 512, (4100, 4201), dict.fromkeys(TYPES, WAVES)), (64, 512, (4100, 4201), dict.fromkeys(TYPES, WAVES))])
@pytest.mark.parametrize("t", TYPES)
def test_pairs_in_one_launch(oracle, t, m, k, ns, kernel):
    if t not in kernel:
        assert gemm_pair_plan(t, m, *ns, k) is None  # (a K split: each on its own)
        return
    p, alone = gemm_pair_plan(t, m, *ns, k), gemm_plan(t, m, ns[0], k)
    assert p is not None and p.kernel == kernel[t], p
    if kernel[t] == WAVES and m == 64:
        assert (p.mb, p.nr) != (alone.mb, alone.nr), (p, alone)
    rng = np.random.default_rng(t + m + k)
    raws = [random_blocks(rng, t, n, k) for n in ns]
    bits, x = bf16_rows(oracle, rng, m, k)
    lib = _lib.load()
    dx, dws = pm.DeviceBuffer.from_host(bits), [pm.DeviceBuffer.from_host(raw) for raw in raws]
    for order in orders(t):
        for y_dtype, size in ((pm.DTYPE_F32, 4), (pm.DTYPE_BF16, 2)):
            dys = [pm.DeviceBuffer(m * n * size + 256) for n in ns]
            alone = [pm.DeviceBuffer(m * n * size) for n in ns]
            for dy in dys:
                pm.check(lib.pmetal_hip_memset(dy.ptr, 0xFF, dy.nbytes, None))
            descs = (_lib.GemmDesc * 2)(*[_lib.GemmDesc(t, y_dtype, order, 0, n, w.ptr, y.ptr) for n, w, y in zip(ns, dws, dys)])
            pm.check(lib.pmetal_hip_qgemm_batch(descs, 2, k, dx.ptr, pm.DTYPE_BF16, m, None))
            for n, w, y in zip(ns, dws, alone):
                pm.check(lib.pmetal_hip_qgemm(t, w.ptr, n, k, dx.ptr, pm.DTYPE_BF16, m, y.ptr, y_dtype, order, None))
            pm.check(lib.pmetal_hip_sync(None))
            for n, raw, dy, one in zip(ns, raws, dys, alone):
                out = dy.to_host(np.uint8)
                assert np.all(out[m * n * size:] == 0xFF)
                assert np.array_equal(out[:m * n * size], one.to_host(np.uint8)), (order, y_dtype)
                if y_dtype == pm.DTYPE_F32:
                    rows = np.r_[0:200, n - 200:n]
                    want = reference(oracle, t, raw.reshape(n, -1)[rows].reshape(-1), len(rows), k, x, order)
                    got = out[:m * n * 4].view(np.float32).reshape(m, n)[:, rows]
                    assert np.max(np.abs(got - want)) <= bound(k) * np.max(np.abs(want)), order


# Two weights that the plan would put in one launch, but one's results lie over what the other reads or writes.  In one launch the order
# of the workgroups makes each of these wrong for certain: the launch takes three rounds of workgroups, its nine blocks of 128
# activation rows one after the other, both weights in each.  (a) The second weight's first blocks of results lie over the last blocks
# of the first one's.  (b) The first one's results lie over the second one's blocks, (c) the other way round: the first 72 rows of
# results replace a weight that eight more blocks of rows read.
@pytest.mark.parametrize("over", ["results", "second weight", "first weight"])
def test_results_over_the_neighbour_are_not_paired(oracle, over):
    t, m, n, k = Q4K, 1030, 8200, 512
    p = gemm_pair_plan(t, m, n, n, k)
    assert p is not None and p.kernel == ROWS and p.mb == 4, p
    rng = np.random.default_rng(11)
    raws = [random_blocks(rng, t, n, k) for _ in range(2)]
    bits, _ = bf16_rows(oracle, rng, m, k)
    lib = _lib.load()
    dx = pm.DeviceBuffer.from_host(bits)
    y_bytes = m * n * 4

    def outputs(batch):
        buf = pm.DeviceBuffer(2 * y_bytes)
        pm.check(lib.pmetal_hip_memset(buf.ptr, 0, buf.nbytes, None))
        dws = [pm.DeviceBuffer.from_host(raw) for raw in raws]
        ys, ws = [buf.ptr, buf.ptr + y_bytes], [w.ptr for w in dws]
        if over == "results":
            ys[1] = buf.ptr + 900 * n * 4
        else:
            at = 1 if over == "second weight" else 0
            ws[at] = ys[1 - at]
            pm.check(lib.pmetal_hip_h2d(ws[at], raws[at].ctypes.data, raws[at].size))
        if batch:
            descs = (_lib.GemmDesc * 2)(*[_lib.GemmDesc(t, pm.DTYPE_F32, 0, 0, n, w, y) for w, y in zip(ws, ys)])
            pm.check(lib.pmetal_hip_qgemm_batch(descs, 2, k, dx.ptr, pm.DTYPE_BF16, m, None))
        else:
            for w, y in zip(ws, ys):
                pm.check(lib.pmetal_hip_qgemm(t, w, n, k, dx.ptr, pm.DTYPE_BF16, m, y, pm.DTYPE_F32, 0, None))
        pm.check(lib.pmetal_hip_sync(None))
        return buf.to_host(np.uint8)

    assert np.array_equal(outputs(True), outputs(False))


# Up to 16 rows the short-batch kernels' waves convert the activations they multiply, one or two super-blocks of each row with a scale of
# their own.  Magnitudes that change from super-block to super-block, rows of zeros and of denormals, sizes below and above two
# super-blocks a wave, whole and partial last runs, 1 to 16 rows, both activation types and orders.
@pytest.mark.parametrize("m,n,k", [(1, 40, 256), (16, 33, 768), (5, 50, 2048), (15, 20, 3328), (16, 70, 4096), (9, 130, 7168), (2, 35, 11008)])
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_short_batches_convert_rows_of_any_scale(oracle, t, m, n, k):
    rng = np.random.default_rng(31 * t + m + k)
    raw = random_blocks(rng, t, n, k)
    x = rng.standard_normal((m, k // 256, 256)) * np.exp2(rng.integers(-30, 30, (m, k // 256, 1)))
    x[rng.random((m, k // 256)) < 0.1] = 0.0
    x = x.reshape(m, k).astype(np.float32)
    if m > 4:
        x[1], x[3] = 0.0, x[3] * np.float32(1e-38)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xb = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    for order in (0, 1) if t in (Q4K, 13) else (0,):
        w = np.abs(oracle.dequantize(t, raw, [n, k], order=order).reshape(n, k).astype(np.float64))
        # against the sum of the products' magnitudes: f32 sums of integer tiles up to four times it (the min terms), and, for f32
        # activations, their rounding to eleven bits; below the smallest normal f16, 2^-14 of 2^9, a step of 2^-25
        for values, dtype, rounding in ((bits, pm.DTYPE_BF16, 0.0), (x, pm.DTYPE_F32, 2.0 ** -12)):
            xv = xb if dtype == pm.DTYPE_BF16 else x
            got = gpu_qgemm(t, raw, n, k, values, m, order=order, x_dtype=dtype)
            want = reference(oracle, t, raw, n, k, xv, order)
            size = np.abs(xv.astype(np.float64)) @ w.T
            assert np.all(np.abs(got - want) <= ((k / 16 + 16) * 2.0 ** -24 * 4 + 2 * rounding) * size + k * 2.0 ** -149), (order, dtype)


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_short_batches_write_over_their_activations(oracle, t):
    rng = np.random.default_rng(t)
    lib = _lib.load()
    for m, n, k, dtype, size in ((16, 2048, 2048, pm.DTYPE_F32, 4), (7, 4096, 2048, pm.DTYPE_BF16, 2), (16, 500, 7168, pm.DTYPE_F32, 4)):
        raw = random_blocks(rng, t, n, k)
        x = rng.standard_normal((m, k)).astype(np.float32)
        values = x if dtype == pm.DTYPE_F32 else oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
        want = gpu_qgemm(t, raw, n, k, values, m, x_dtype=dtype)
        dw, both = pm.DeviceBuffer.from_host(raw), pm.DeviceBuffer(max(m * k * size, m * n * 4) + 512)
        for at in (0, 256):  # results from the activations' start, and from a little behind it
            pm.check(lib.pmetal_hip_h2d(both.ptr, np.ascontiguousarray(values).ctypes.data, m * k * size))
            pm.check(lib.pmetal_hip_qgemm(t, dw.ptr, n, k, both.ptr, dtype, m, both.ptr + at, pm.DTYPE_F32, 0, None))
            pm.check(lib.pmetal_hip_sync(None))
            got = both.to_host(np.uint8)[at:at + m * n * 4].view(np.float32).reshape(m, n)
            assert np.array_equal(got, want), (m, n, k, at)


@pytest.mark.parametrize("x_dtype", [pm.DTYPE_BF16, pm.DTYPE_F32])
def test_batches_of_kernels_with_and_without_a_pre_pass(oracle, x_dtype):
    """Weights of one call whose plans differ in who converts the activations, and in where the workspace keeps what."""
    rng = np.random.default_rng(3)
    lib = _lib.load()
    for m, k, specs in ((12, 2304, [(Q4K, 300), (Q4K, 9000), (Q4K, 400), (Q8_0, 9000), (Q4K, 300)]),
                        (12, 14336, [(Q6K, 300), (Q4K, 300), (Q6K, 400), (11, 300), (Q4K, 500)]),
                        (9, 5120, [(Q4K, 300), (Q6K, 14400), (Q4K, 300), (Q8_0, 300), (Q6K, 14400), (Q8_0, 300)]),
                        # launches that convert for themselves between others of one layout; the partial tiles of the first one's K split
                        # lie over the last converted activations, those of the second one behind them
                        (9, 5120, [(Q4K, 300), (Q6K, 14500), (Q4K, 300), (Q4K, 14500), (Q4K, 400)]),
                        (7, 3840, [(t, 272) for t in (Q4K, Q6K, Q8_0, 10, 11, 13)] * 2)):  # a pre-pass per pair of super-blocks, the last half a pair
        x = rng.standard_normal((m, k)).astype(np.float32)
        dx = pm.DeviceBuffer.from_host(x if x_dtype == pm.DTYPE_F32 else oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k))
        ws = [pm.DeviceBuffer.from_host(random_blocks(rng, t, n, k)) for t, n in specs]
        ys, ones = ([pm.DeviceBuffer(m * n * 4) for _, n in specs] for _ in range(2))
        descs = (_lib.GemmDesc * len(specs))(*[_lib.GemmDesc(t, pm.DTYPE_F32, 0, 0, n, w.ptr, y.ptr) for (t, n), w, y in zip(specs, ws, ys)])
        pm.check(lib.pmetal_hip_qgemm_batch(descs, len(specs), k, dx.ptr, x_dtype, m, None))
        for (t, n), w, y in zip(specs, ws, ones):
            pm.check(lib.pmetal_hip_qgemm(t, w.ptr, n, k, dx.ptr, x_dtype, m, y.ptr, pm.DTYPE_F32, 0, None))
        pm.check(lib.pmetal_hip_sync(None))
        for i, (a, b) in enumerate(zip(ys, ones)):
            assert np.array_equal(a.to_host(np.uint8), b.to_host(np.uint8)), (m, k, i)


# A batch whose first results lie over its activations: weights that follow one another in one layout are all multiplied by the activations
# as they were before the first of them, whoever converts them (rows of at most eight super-blocks: every launch; longer: one
# launch for all of a form, or two forms of one layout), the next layout by what is there then.  Bit for bit as calls of their own over copies.
@pytest.mark.parametrize("m,k,specs", [(16, 2048, [(Q4K, 300), (Q4K, 500), (Q4K, 70)]), (5, 512, [(Q8_0, 33), (Q8_0, 33), (Q8_0, 100), (Q8_0, 4)]),
                                       (9, 1280, [(Q6K, 200), (Q6K, 40), (11, 50), (10, 60), (Q6K, 70)]), (16, 4096, [(Q4K, 300), (Q4K, 500), (Q4K, 70), (13, 90)]),
                                       (7, 3840, [(11, 40), (11, 50), (10, 60)]), (12, 2304, [(Q4K, 300), (Q4K, 9000), (Q4K, 400), (Q8_0, 9000), (Q8_0, 300)]),
                                       (3, 5120, [(Q6K, 14400), (Q6K, 300), (Q6K, 14500)]), (20, 1024, [(Q4K, 300), (Q4K, 500), (Q4K, 70)])])
@pytest.mark.parametrize("dtype,size", [(pm.DTYPE_F32, 4), (pm.DTYPE_BF16, 2)])
def test_batches_write_over_their_activations(oracle, m, k, specs, dtype, size):
    rng = np.random.default_rng(m + k)
    lib = _lib.load()
    x = rng.standard_normal((m, k)).astype(np.float32)
    values = np.ascontiguousarray(x if dtype == pm.DTYPE_F32 else oracle.f32_to_bf16_bits(x.reshape(-1)))
    ws = [pm.DeviceBuffer.from_host(random_blocks(rng, t, n, k)) for t, n in specs]
    layouts = [10 if t == 11 else t for t, _ in specs]  # (in the order of the reference Q4_K and Q5_K have layouts of their own)
    x_bytes = m * k * size
    for at in (0, 256):
        both = [pm.DeviceBuffer(max(x_bytes, at + m * specs[0][1] * size)) for _ in range(2)]
        for b in both:
            pm.check(lib.pmetal_hip_h2d(b.ptr, values.ctypes.data, x_bytes))
        outs = [[pm.DeviceBuffer(m * n * size) for _, n in specs[1:]] for _ in range(2)]
        descs = [_lib.GemmDesc(t, dtype, 0, 0, n, w.ptr, both[0].ptr + at if i == 0 else outs[0][i - 1].ptr) for i, ((t, n), w) in enumerate(zip(specs, ws))]
        pm.check(lib.pmetal_hip_qgemm_batch((_lib.GemmDesc * len(specs))(*descs), len(specs), k, both[0].ptr, dtype, m, None))
        for i, ((t, n), w) in enumerate(zip(specs, ws)):
            if i == 0 or layouts[i] != layouts[i - 1]:
                pm.check(lib.pmetal_hip_sync(None))
                given = pm.DeviceBuffer.from_host(both[1].to_host(np.uint8)[:x_bytes])
            pm.check(lib.pmetal_hip_qgemm(t, w.ptr, n, k, given.ptr, dtype, m, both[1].ptr + at if i == 0 else outs[1][i - 1].ptr, dtype, 0, None))
        pm.check(lib.pmetal_hip_sync(None))
        for i, (a, b) in enumerate(zip([both[0]] + outs[0], [both[1]] + outs[1])):
            assert np.array_equal(a.to_host(np.uint8), b.to_host(np.uint8)), (at, i)


# A re-blocked weight of two parts multiplies twice; its f32 results over the activations are those that lie apart from them.
@pytest.mark.parametrize("m,n,k", [(16, 2048, 2048), (3, 40, 256), (7, 500, 1280), (16, 600, 2304), (9, 300, 4096), (20, 300, 1024)])
@pytest.mark.parametrize("t", [13, 11, 10])
@pytest.mark.parametrize("dtype,size", [(pm.DTYPE_F32, 4), (pm.DTYPE_BF16, 2)])
def test_reblocked_weights_write_over_their_activations(oracle, t, m, n, k, dtype, size):
    rng = np.random.default_rng(t + m + k)
    lib = _lib.load()
    x = rng.standard_normal((m, k)).astype(np.float32)
    values = np.ascontiguousarray(x if dtype == pm.DTYPE_F32 else oracle.f32_to_bf16_bits(x.reshape(-1)))
    dw, parts = pm.DeviceBuffer.from_host(random_blocks(rng, t, n, k)), lib.pmetal_hip_reblock_size(t, n, k)
    dr, dx, dy = pm.DeviceBuffer(parts), pm.DeviceBuffer.from_host(values), pm.DeviceBuffer(m * n * 4)
    pm.check(lib.pmetal_hip_reblock_dev(t, dw.ptr, n, k, 0, dr.ptr, parts, None))
    pm.check(lib.pmetal_hip_qgemm_reblocked(t, dr.ptr, parts, n, k, dx.ptr, dtype, m, dy.ptr, pm.DTYPE_F32, None))
    both = pm.DeviceBuffer(max(m * k * size, m * n * 4) + 256)
    for at in (0, 256):
        pm.check(lib.pmetal_hip_h2d(both.ptr, values.ctypes.data, m * k * size))
        pm.check(lib.pmetal_hip_qgemm_reblocked(t, dr.ptr, parts, n, k, both.ptr, dtype, m, both.ptr + at, pm.DTYPE_F32, None))
        pm.check(lib.pmetal_hip_sync(None))
        assert np.array_equal(both.to_host(np.uint8)[at:at + m * n * 4], dy.to_host(np.uint8)), at


# An infinity among ordinary activations of up to 16 rows: the results of its row are infinite, with the sign of its weight (a weight of 0:
# NaN), and the others as ever.  It shares a word with an element far larger than the others, in the upper half of it or in the lower:
# that one may not be overlooked for the row's largest magnitude, or it would overflow to the other infinity.  (Types without a
# min term: the sums that those multiply are NaN.)
@pytest.mark.parametrize("k", [256, 2048, 3328])
@pytest.mark.parametrize("t", [Q8_0, Q6K])
@pytest.mark.parametrize("dtype", [pm.DTYPE_BF16, pm.DTYPE_F32])
def test_short_batches_with_infinities(oracle, t, k, dtype):
    m, n = 16, 24
    assert gemm_plan(t, m, n, k).kernel == SMALL
    rng = np.random.default_rng(t + k)
    raw = random_blocks(rng, t, n, k)
    x = (rng.standard_normal((m, k)) * 1e-3).astype(np.float32)
    for r in range(15):  # (the last row has none)
        at = 2 * rng.integers(k // 2)
        x[r, at + r % 2], x[r, at + 1 - r % 2] = -3e4 * (-1.0) ** (r // 2), np.inf * (-1.0) ** (r // 2)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    x = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    got = gpu_qgemm(t, raw, n, k, bits if dtype == pm.DTYPE_BF16 else x, m, x_dtype=dtype)
    w = oracle.dequantize(t, raw, [n, k]).reshape(n, k).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.T
    assert np.isfinite(want[15]).all() and np.isinf(want[:15]).sum() > 100
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    assert np.max(np.abs(got[15] - want[15])) <= bound(k) * np.max(np.abs(want[15]))


# Splits of K of a tile, added by the workgroup that comes last (a call of its own, the first weight of a batch) or by a launch behind (the
# other weights, whose call has no pre-pass to clear the counters): the same bits.  (weight rows, tile, splits) of each weight: two and four
# splits, the last one shorter (17 super-blocks in fives: two, six of its waves without work; no plan has a split without any); one row and column past a
# tile and short of it; 32 x 32, 64 x 32 and 64 x 64 tiles, up to 128 of them.
SPLIT_CASES = [(17, 4352, ((64, 1, 1, 4), (70, 1, 1, 4))), (17, 8448, ((1, 1, 1, 4), (33, 1, 1, 4))), (31, 8192, ((70, 1, 1, 4), (4096, 1, 1, 2))),
               (32, 9728, ((2560, 1, 1, 2), (31, 1, 1, 4))), (64, 8192, ((97, 1, 1, 4), (1000, 1, 1, 4))), (63, 14336, ((65, 1, 1, 4), (2048, 2, 1, 4))),
               (100, 8192, ((1023, 2, 1, 4), (130, 1, 1, 4))), (200, 14336, ((1000, 2, 2, 4), (64, 1, 1, 4))), (500, 8192, ((700, 2, 2, 2), (129, 2, 1, 4)))]


@pytest.mark.parametrize("m,k,weights", SPLIT_CASES)
@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
def test_splits_of_a_tile(oracle, t, m, k, weights):
    for n, mb, nr, splits in weights:
        p = gemm_plan(t, m, n, k)
        if (t, m, n) != (Q8_0, 31, 4096):  # (the short-batch kernel)
            assert (p.kernel, p.mb, p.nr, p.splits) == (WAVES, mb, nr, splits), p
    test_pairs_match_separate_calls(oracle, t, m, k, [w[0] for w in weights])


@pytest.mark.parametrize("m,n,k,y_dtype", [(27, 4096, 14336, pm.DTYPE_F32), (100, 1001, 8192, pm.DTYPE_BF16)])
def test_splits_of_a_tile_replayed(m, n, k, y_dtype):
    p = gemm_plan(Q6K, m, n, k)
    assert p.kernel == WAVES and p.splits > 1
    lib, size = _lib.load(), m * n * (4 if y_dtype == pm.DTYPE_F32 else 2)
    rng = np.random.default_rng(m)
    dw, dx, dy = pm.DeviceBuffer.from_host(random_blocks(rng, Q6K, n, k)), pm.DeviceBuffer.from_host(rng.standard_normal((m, k)).astype(np.float32)), pm.DeviceBuffer(size)
    stream = lib.pmetal_hip_stream_create()

    def call():
        pm.check(lib.pmetal_hip_qgemm(Q6K, dw.ptr, n, k, dx.ptr, pm.DTYPE_F32, m, dy.ptr, y_dtype, 0, stream))

    try:
        call()
        pm.check(lib.pmetal_hip_sync(stream))
        want = dy.to_host(np.uint8)
        pm.check(lib.pmetal_hip_record_begin(stream))
        for _ in range(2):
            call()
        rec = lib.pmetal_hip_record_end(stream)
        assert rec, lib.pmetal_hip_last_error_message()
        for rep in range(4):
            pm.check(lib.pmetal_hip_memset(dy.ptr, 0xFF, size, None))
            pm.check(lib.pmetal_hip_sync(None))
            pm.check(lib.pmetal_hip_replay(rec, stream))
            pm.check(lib.pmetal_hip_sync(stream))
            assert np.array_equal(dy.to_host(np.uint8), want), rep
        lib.pmetal_hip_recording_destroy(rec)
    finally:
        lib.pmetal_hip_stream_destroy(stream)


# So many activation rows that a wave's way from one of its super-blocks to the next is more than 4 GiB of items (1920 bytes a row for Q2_K, 1728
# for Q4_K, with four waves): rows from every part of them, the last one among them.
@pytest.mark.parametrize("t,m", [(10, 2300001), (Q4K, 2560001)])
def test_millions_of_activation_rows(oracle, t, m):
    n, k, chunk = 64, 1280, 100000
    p = gemm_plan(t, m, n, k)
    assert (p.kernel, p.nw) == (WAVES, 4) and 3 * {10: 640, Q4K: 576}[t] * p.mp > 1 << 32
    lib, stream = _lib.load(), _lib.load().pmetal_hip_stream_create()  # (its workspace goes with it)
    rng = np.random.default_rng(m)
    raw = random_blocks(rng, t, n, k)
    dw, dx, df, dy = pm.DeviceBuffer.from_host(raw), pm.DeviceBuffer(2 * m * k), pm.DeviceBuffer(4 * chunk * k), pm.DeviceBuffer(4 * m * n)
    try:
        for r in range(0, m, chunk):
            elems = min(chunk, m - r) * k
            pm.check(lib.pmetal_hip_fill_normal_f32(df.ptr, elems, r + 1, 1.0, 0.0, 0.0, stream))
            pm.check(lib.pmetal_hip_f32_to_bf16_dev(df.ptr, dx.ptr + 2 * r * k, elems, stream))
        pm.check(lib.pmetal_hip_memset(dy.ptr, 0xFF, 4 * m * n, stream))
        pm.check(lib.pmetal_hip_qgemm(t, dw.ptr, n, k, dx.ptr, pm.DTYPE_BF16, m, dy.ptr, pm.DTYPE_F32, 0, stream))
        pm.check(lib.pmetal_hip_sync(stream))
        rows = np.concatenate([np.arange(4), rng.integers(0, m, 40), np.arange(m - 4, m)])
        x, got = np.empty((rows.size, k), np.uint16), np.empty((rows.size, n), np.float32)
        for i, r in enumerate(rows):
            pm.check(lib.pmetal_hip_d2h(x[i].ctypes.data, dx.ptr + 2 * int(r) * k, 2 * k))
            pm.check(lib.pmetal_hip_d2h(got[i].ctypes.data, dy.ptr + 4 * int(r) * n, 4 * n))
    finally:
        pm.check(lib.pmetal_hip_stream_destroy(stream))
    want = reference(oracle, t, raw, n, k, oracle.bf16_bits_to_f32(x.reshape(-1)).reshape(rows.size, k), 0)
    assert np.max(np.abs(got - want)) <= (k / 16 + 16) * 2.0 ** -24 * 4 * np.max(np.abs(want))  # (the bound of the other tiles)
