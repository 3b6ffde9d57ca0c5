"""GPU parity of the tile GEMM (gemm_kw.hip): a workgroup owns a tile of Y and its waves split K."""
import numpy as np
import pytest

import pmetal_amd as pm
from pmetal_amd import _lib
from gpu_util import Q4K, Q6K, Q8_0
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


# (m, n, k): one weight row, one super-block; edges of the 32- and 64-row blocks of both sides; rows of 7, 8, 9 and 17
# super-blocks (waves of equal and of different length); a narrow weight with long rows (K split over workgroups, the last
# split shorter than the others); enough tiles for more than one round of workgroups
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


# The pre-pass holds 1, 2, 4 or 8 items per thread, or reads a longer row twice; one, two (from 384 rows on) or four rows (from
# 1024 on) per workgroup.  Rows of activations that end inside a workgroup, row lengths on both sides of each step.
@pytest.mark.parametrize("m,k", [(3, 4096), (18, 4352), (17, 16384), (20, 16640), (33, 32768), (2, 33024), (385, 4096), (390, 4352), (385, 33024),
                                 (1025, 2048), (1026, 2304), (1025, 8192), (1027, 8448), (1025, 16640)])
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


# Two weights that share their activations go in one launch: every kernel that takes such a pair (short batches, the wave tiles,
# the rows, whose rounds of workgroups neither weight fills), row counts off every tile, the seam between the two inside a
# round; three weights of which two are neighbours of one kind; results of one in place of the other's stay calls of their own.
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
