"""GPU parity: dequant-fused Q4_K GEMM against dequantize-then-matmul (f64 accumulation).

Tolerance: max relative error <= 1e-3, element-wise over outputs with
|y| > 1e-3 * max|y| and normwise (max|dy| / max|y|), as for the GEMV."""
import numpy as np
import pytest

import pmetal_amd as pm
from gpu_util import Q4K, Q6K, Q8_0, rel_errors, weights
from pmetal_amd import _lib

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.fixture(scope="module", autouse=True)
def _device():
    pm.init(0)


def gpu_qgemm(t, wq, n, k, x_bits, m, y_dtype=pm.DTYPE_F32, order=0, x_dtype=pm.DTYPE_BF16):
    lib = _lib.load()
    dw = pm.DeviceBuffer.from_host(np.ascontiguousarray(wq, dtype=np.uint8))
    dx = pm.DeviceBuffer.from_host(x_bits)
    ysz = 4 if y_dtype == pm.DTYPE_F32 else 2
    dy = pm.DeviceBuffer(m * n * ysz)
    pm.check(lib.pmetal_hip_memset(dy.ptr, 0xFF, m * n * ysz, None))
    pm.check(lib.pmetal_hip_qgemm(t, dw.ptr, n, k, dx.ptr, x_dtype, m, dy.ptr, y_dtype, order, None))
    pm.check(lib.pmetal_hip_sync(None))
    if y_dtype == pm.DTYPE_F32:
        return dy.to_host(np.float32).reshape(m, n)
    return (dy.to_host(np.uint16).astype(np.uint32) << 16).view(np.float32).reshape(m, n)


def reference(oracle, t, wq, n, k, x_f32, order):
    w = oracle.dequantize(t, wq, [n, k], order=order).reshape(n, k).astype(np.float64)
    return (x_f32.astype(np.float64) @ w.T).astype(np.float32)


@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (16, 128, 512), (64, 256, 1024), (128, 384, 4096), (33, 200, 768),
                                   (130, 129, 256), (512, 512, 2048), (257, 160, 512), (300, 100, 768)])
def test_qgemm_q4k_matches_dequantize_then_matmul(oracle, m, n, k):
    wq = oracle.quantize(Q4K, weights(m + n + k, n * k, outliers=1e-3))
    x = np.random.default_rng(m * 7 + k).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    for order in (0, 1):
        want = reference(oracle, Q4K, wq, n, k, xr, order)
        got = gpu_qgemm(Q4K, wq, n, k, bits, m, order=order)
        elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
        print(f"Q4_K GEMM m={m} n={n} k={k} order={order}: elem {elem:.2e} norm {norm:.2e}")
        assert elem <= TOL and norm <= TOL


def test_qgemm_bf16_output_and_large_activations(oracle):
    m, n, k = 64, 256, 1024
    wq = oracle.quantize(Q4K, weights(5, n * k))
    x = np.random.default_rng(6).standard_normal((m, k)).astype(np.float32)
    x[3] *= 1e6   # a row far outside the f16 range: handled by the per-row power-of-two scale
    x[5] *= 1e-6
    x[7] = 0.0
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    want = reference(oracle, Q4K, wq, n, k, xr, 0)
    got = gpu_qgemm(Q4K, wq, n, k, bits, m)
    for row in range(m):  # per row: the rows have wildly different magnitudes
        elem, norm = rel_errors(got[row], want[row])
        assert elem <= TOL and norm <= TOL, (row, elem, norm)
    got16 = gpu_qgemm(Q4K, wq, n, k, bits, m, y_dtype=pm.DTYPE_BF16)
    for row in (0, 3, 5, 63):
        scale = np.max(np.abs(want[row])) or 1.0
        assert np.max(np.abs(got16[row] - want[row])) / scale <= 2.0 ** -8  # bf16 rounding of the output


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0])
@pytest.mark.parametrize("m", [24, 150, 192, 200, 300])
def test_qgemm_f32_activations(oracle, t, m):
    """f32 activations are rounded once to f16 at the row's power-of-two scale (11 significant bits; a bf16 cast
    would keep 8): against the unrounded reference the result holds the 1e-3 bound norm-wise, and element-wise
    against the reference fed the same rounded activations."""
    n, k = 320, 1024
    wq = oracle.quantize(t, weights(90 + m, n * k))
    x = np.random.default_rng(91 + m).standard_normal((m, k)).astype(np.float32)
    x[1] *= 3e4
    got = gpu_qgemm(t, wq, n, k, x, m, x_dtype=pm.DTYPE_F32)
    want = reference(oracle, t, wq, n, k, x, 0)
    # the kernel's rounding: x * 2^-e to f16 with the row maximum in [2^9, 2^10), then back
    e = np.floor(np.log2(np.max(np.abs(x), axis=1, keepdims=True))) - 9
    xr = (np.ldexp(x, (-e).astype(np.int32)).astype(np.float16).astype(np.float32) * np.exp2(e)).astype(np.float32)
    want_r = reference(oracle, t, wq, n, k, xr, 0)
    for row in range(m):
        _, norm = rel_errors(got[row], want[row])
        elem_r, norm_r = rel_errors(got[row], want_r[row])
        assert norm <= TOL and elem_r <= TOL and norm_r <= TOL, (row, norm, elem_r, norm_r)


@pytest.fixture(scope="module")
def config2_weights(oracle):
    """The 14336 x 4096 Q4_K weight of the GEMM configuration: quantized on the device, and every byte compared with the
    oracle's quantizer (run on all host threads) before any product is taken."""
    n, k = 14336, 4096
    w = weights(31, n * k)
    wq = pm.quantize(w, Q4K)
    want = oracle.quantize(Q4K, w, threads=min(oracle.host_threads(), 16))
    assert np.array_equal(wq, want)
    return wq


@pytest.mark.parametrize("m", [16, 64, 128, 512, 2048])
def test_qgemm_config2_full_size(oracle, config2_weights, m):
    """M = 512 and the sweep 16 / 64 / 128 / 2048 at K = 4096, N = 14336, bf16 activations ~ N(0, 1).  The f64 reference covers
    every activation row against 1152 weight rows (the first and last 64 and 1024 drawn at random): all of the kernel's
    code paths for the shape (K split and partial-tile reduction for few rows, 128-row workgroups and the four-row
    pre-pass for many) contribute to every output column alike."""
    n, k = 14336, 4096
    wq = config2_weights
    x = np.random.default_rng(32 + m).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    got = gpu_qgemm(Q4K, wq, n, k, bits, m)
    assert np.isfinite(got).all()
    rows = np.unique(np.concatenate([np.arange(64), np.arange(n - 64, n),
                                     np.random.default_rng(m).choice(n, 1024, replace=False)]))
    row_bytes = k // 256 * 144
    sub = wq.reshape(n, row_bytes)[rows].reshape(-1)
    want = oracle.qmatmul(Q4K, sub, rows.size, k, xr, threads=min(oracle.host_threads(), 16))
    elem, norm = rel_errors(got[:, rows].reshape(-1), want.reshape(-1))
    print(f"Q4_K GEMM {m}x14336x4096: elem {elem:.2e} norm {norm:.2e} over {rows.size} weight rows")
    assert elem <= TOL and norm <= TOL
    # every column, cheaply: row 0 of the product is the GEMV of activation row 0 (itself checked against the oracle at
    # this shape in the GEMV tests)
    from gpu_util import gpu_qgemv
    y0 = gpu_qgemv(Q4K, wq, n, k, bits[0], pm.DTYPE_BF16)
    e0, n0 = rel_errors(got[0], y0)
    assert n0 <= 1e-4, (e0, n0)


def test_qgemm_agrees_with_qgemv_and_qlinear_dispatch(oracle):
    from gpu_util import gpu_qgemv
    lib = _lib.load()
    n, k = 512, 2048
    wq = oracle.quantize(Q4K, weights(41, n * k))
    bits = oracle.f32_to_bf16_bits(np.random.default_rng(42).standard_normal(k).astype(np.float32))
    y_gemv = gpu_qgemv(Q4K, wq, n, k, bits, pm.DTYPE_BF16)
    y_gemm = gpu_qgemm(Q4K, wq, n, k, bits.reshape(1, k), 1).reshape(-1)
    elem, norm = rel_errors(y_gemm, y_gemv)
    assert norm <= 1e-5
    lin = pm.GgufLinear(Q4K, n, k, wq)
    y1 = lin.forward(pm.DeviceBuffer.from_host(bits), m=1).to_host(np.float32)
    assert np.array_equal(y1, y_gemv)  # m == 1 dispatches to the GEMV
    xb = np.tile(bits, (4, 1))
    y4 = lin.forward(pm.DeviceBuffer.from_host(xb), m=4).to_host(np.float32).reshape(4, n)
    assert np.allclose(y4[2], y_gemv, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("m,n,k", [(2, 96, 512), (5, 1000, 1024), (40, 260, 2048), (96, 700, 1024), (384, 1024, 1024)])
def test_qgemm_q4k_k_split_is_deterministic_and_ragged_rows(oracle, m, n, k):
    """Short batches split K over several workgroups and add fp32 partial tiles in a fixed order: two runs give the
    same bits; n is not a multiple of the 32 rows a wave owns."""
    wq = oracle.quantize(Q4K, weights(300 + m, n * k))
    x = np.random.default_rng(301 + m).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    want = reference(oracle, Q4K, wq, n, k, xr, 1)
    got = gpu_qgemm(Q4K, wq, n, k, bits, m, order=1)
    again = gpu_qgemm(Q4K, wq, n, k, bits, m, order=1)
    assert np.array_equal(got, again)
    elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
    assert elem <= TOL and norm <= TOL


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0])
def test_qgemm_long_rows_with_k_split_above_128_rows(oracle, t):
    """A down-projection-like shape (few weight rows, long k): more than 128 activation rows and a K split."""
    m, n, k = 192, 512, 14336
    wq = oracle.quantize(t, weights(800 + t, n * k))
    x = np.random.default_rng(801 + t).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    want = reference(oracle, t, wq, n, k, xr, 0)
    got = gpu_qgemm(t, wq, n, k, bits, m)
    elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
    print(f"type {t} GEMM {m}x{n}x{k}: elem {elem:.2e} norm {norm:.2e}")
    assert elem <= TOL and norm <= TOL
    assert np.array_equal(got, gpu_qgemm(t, wq, n, k, bits, m))


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0])
@pytest.mark.parametrize("xf32", [False, True])
def test_qgemm_more_than_1024_activation_rows(oracle, t, xf32):
    """1100 rows (not a multiple of 128): the activation pre-pass handles four rows per workgroup from 1024 rows on."""
    m, n, k = 1100, 256, 768
    wq = oracle.quantize(t, weights(900 + t, n * k, outliers=1e-3))
    x = np.random.default_rng(901 + t).standard_normal((m, k)).astype(np.float32)
    x[7] *= 3e4
    x[1099] *= 2e-5
    if xf32:  # the kernel rounds f32 activations to f16 at the row's power-of-two scale
        e = np.floor(np.log2(np.max(np.abs(x), axis=1, keepdims=True))) - 9
        xr = (np.ldexp(x, (-e).astype(np.int32)).astype(np.float16).astype(np.float32) * np.exp2(e)).astype(np.float32)
        xin, xd = x, pm.DTYPE_F32
    else:
        xin = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
        xr, xd = oracle.bf16_bits_to_f32(xin.reshape(-1)).reshape(m, k), pm.DTYPE_BF16
    for order in ((0, 1) if t == Q4K else (0,)):
        want = reference(oracle, t, wq, n, k, xr, order)
        got = gpu_qgemm(t, wq, n, k, xin, m, order=order, x_dtype=xd)
        # per activation row: rows differ by nine orders of magnitude
        for rows in (slice(0, 7), slice(7, 8), slice(8, 1099), slice(1099, 1100)):
            elem, norm = rel_errors(got[rows].reshape(-1), want[rows].reshape(-1))
            assert elem <= TOL and norm <= TOL, (t, order, rows, elem, norm)


def test_qgemm_argument_errors():
    lib = _lib.load()
    buf = pm.DeviceBuffer(1 << 16)
    assert lib.pmetal_hip_qgemm(Q4K, buf.ptr, 4, 256, buf.ptr, 1, 0, buf.ptr, 0, 0, None) == 6   # m == 0
    assert lib.pmetal_hip_qgemm(Q4K, buf.ptr, 4, 100, buf.ptr, 1, 4, buf.ptr, 0, 0, None) == 6   # k % 256
    assert lib.pmetal_hip_qgemm(Q8_0, buf.ptr, 4, 96, buf.ptr, 1, 4, buf.ptr, 0, 0, None) == 6   # k % 256 (a valid Q8_0 row)
    assert lib.pmetal_hip_qgemm(Q4K, buf.ptr, 4, 256, buf.ptr, 1, 4, buf.ptr, 7, 0, None) == 1   # y_dtype


@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (16, 128, 512), (64, 256, 1024), (128, 384, 4096), (33, 200, 768),
                                   (130, 129, 256), (300, 512, 2048), (512, 1024, 2048)])
def test_qgemm_q6k_matches_dequantize_then_matmul(oracle, m, n, k):
    wq = oracle.quantize(Q6K, weights(60 + m, n * k))
    x = np.random.default_rng(61 + m).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xb = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    want = reference(oracle, Q6K, wq, n, k, xb, 0)
    got = gpu_qgemm(Q6K, wq, n, k, bits, m)
    elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
    print(f"Q6_K GEMM m={m} n={n} k={k}: elem {elem:.2e} norm {norm:.2e}")
    assert elem <= TOL and norm <= TOL
    if m == 16:  # extreme scales: every |sc| = 128 sub-block and the all-zero super-block (d = -0)
        w = weights(62, n * k)
        w[: 256] = 0.0
        w[256:512] = np.where(np.arange(256) % 2 == 0, 1.0, -1.0).astype(np.float32)
        wq = oracle.quantize(Q6K, w)
        want = reference(oracle, Q6K, wq, n, k, xb, 0)
        got = gpu_qgemm(Q6K, wq, n, k, bits, m)
        elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
        assert elem <= TOL and norm <= TOL


@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (16, 128, 512), (64, 256, 1024), (128, 384, 4096), (33, 200, 768),
                                   (130, 129, 256), (512, 512, 2048), (257, 160, 512), (300, 100, 768)])
def test_qgemm_q8_0_matches_dequantize_then_matmul(oracle, m, n, k):
    wq = oracle.quantize(Q8_0, weights(700 + m + n, n * k, outliers=1e-3))
    x = np.random.default_rng(m * 5 + k).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    want = reference(oracle, Q8_0, wq, n, k, xr, 0)
    got = gpu_qgemm(Q8_0, wq, n, k, bits, m)
    elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
    print(f"Q8_0 GEMM m={m} n={n} k={k}: elem {elem:.2e} norm {norm:.2e}")
    assert elem <= TOL and norm <= TOL
    got16 = gpu_qgemm(Q8_0, wq, n, k, bits, m, y_dtype=pm.DTYPE_BF16)
    assert np.max(np.abs(got16 - want)) / np.max(np.abs(want)) <= 2.0 ** -8


def test_qlinear_q8_0_rows_that_are_not_a_multiple_of_256(oracle):
    """Q8_0 rows may be any multiple of 32; the fused GEMM needs 256: qlinear then runs one GEMV per activation row."""
    n, k, m = 96, 480, 3
    wq = oracle.quantize(Q8_0, weights(51, n * k))
    x = np.random.default_rng(52).standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    lin = pm.GgufLinear(Q8_0, n, k, wq)
    y = lin.forward(pm.DeviceBuffer.from_host(bits), m=m).to_host(np.float32).reshape(m, n)
    want = reference(oracle, Q8_0, wq, n, k, oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k), 0)
    elem, norm = rel_errors(y.reshape(-1), want.reshape(-1))
    assert elem <= TOL and norm <= TOL


def test_qgemm_on_two_streams_of_one_thread_keep_separate_scratch(oracle):
    """Two GEMMs in flight on two streams of the same thread: each stream has its own scratch inside the library, so
    neither the converted activations nor the partial tiles of one can be overwritten by the other; a later, larger
    shape on the first stream makes that stream's scratch grow."""
    lib = _lib.load()
    s1, s2 = lib.pmetal_hip_stream_create(), lib.pmetal_hip_stream_create()
    assert s1 and s2
    try:
        jobs = []
        for i, (m, n, k, s) in enumerate([(96, 512, 8192, s1), (200, 768, 1024, s2), (40, 256, 4096, s1), (700, 1024, 2048, s1),
                                          (17, 300, 2048, s2)]):
            wq = oracle.quantize(Q4K, weights(950 + i, n * k))
            x = np.random.default_rng(960 + i).standard_normal((m, k)).astype(np.float32)
            bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
            xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
            dw, dx, dy = pm.DeviceBuffer.from_host(wq), pm.DeviceBuffer.from_host(bits), pm.DeviceBuffer(4 * m * n)
            jobs.append((m, n, k, s, dw, dx, dy, reference(oracle, Q4K, wq, n, k, xr, 0)))
        for rep in range(3):  # launched back to back, nothing waits in between
            for m, n, k, s, dw, dx, dy, _ in jobs:
                pm.check(lib.pmetal_hip_qgemm(Q4K, dw.ptr, n, k, dx.ptr, pm.DTYPE_BF16, m, dy.ptr, pm.DTYPE_F32, 0, s))
        pm.check(lib.pmetal_hip_sync(s1))
        pm.check(lib.pmetal_hip_sync(s2))
        for m, n, k, s, dw, dx, dy, want in jobs:
            got = dy.to_host(np.float32).reshape(m, n)
            elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
            assert elem <= TOL and norm <= TOL, (m, n, k, elem, norm)
    finally:
        lib.pmetal_hip_stream_destroy(s1)
        lib.pmetal_hip_stream_destroy(s2)


# Q5_K, Q3_K and Q2_K: matrix kernels of their own (and, for weights prepared that way, an exact re-blocking into Q6_K
# super-blocks: one tensor, or two for the formats with mins).  d / dmin offsets inside a block, for random block bytes with
# finite scales:
REBLOCKED = {13: (176, (0, 2)), 11: (110, (108,)), 10: (84, (80, 82))}


@pytest.mark.parametrize("t", sorted(REBLOCKED))
@pytest.mark.parametrize("m,n,k", [(9, 128, 256), (16, 128, 512), (33, 200, 768), (130, 129, 256), (300, 512, 2048)])
def test_qgemm_q5k_q3k_q2k_matches_dequantize_then_matmul(oracle, t, m, n, k):
    """Random block bytes (every scale, min and quant value; negative Q3_K scales) and quantized weights, both element
    orders for Q5_K, f32 and bf16 results, against the oracle's dequantize-then-matmul in f64."""
    size, d_at = REBLOCKED[t]
    rng = np.random.default_rng(1000 * t + m + n + k)
    raw = rng.integers(0, 256, size=(n * (k // 256), size), dtype=np.uint8)
    for j, off in enumerate(d_at):
        raw[:, off:off + 2] = np.frombuffer(np.array([0.01 * (j + 1)], np.float16).tobytes(), np.uint8)
    raw[3, d_at[0]:d_at[0] + 2] = np.frombuffer(np.array([-0.03], np.float16).tobytes(), np.uint8)  # a negative d
    x = rng.standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xb = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    for wq in (raw.reshape(-1), oracle.quantize(t, weights(t + m, n * k, outliers=1e-3))):
        for order in ((0, 1) if t == 13 else (0,)):
            want = reference(oracle, t, wq, n, k, xb, order)
            got = gpu_qgemm(t, wq, n, k, bits, m, order=order)
            elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
            print(f"type {t} GEMM m={m} n={n} k={k} order={order}: elem {elem:.2e} norm {norm:.2e}")
            assert elem <= TOL and norm <= TOL
            got16 = gpu_qgemm(t, wq, n, k, bits, m, y_dtype=pm.DTYPE_BF16, order=order)
            assert np.allclose(got16, got, rtol=2.0 ** -8, atol=1e-30)
    # f32 activations: the GEMM rounds them to f16 at the row's power-of-two scale (test_qgemm_f32_activations); both
    # parts of a re-blocked tensor see the same rounded values
    got = gpu_qgemm(t, raw.reshape(-1), n, k, x, m, x_dtype=pm.DTYPE_F32)
    want = reference(oracle, t, raw.reshape(-1), n, k, x, 0)
    e = np.floor(np.log2(np.max(np.abs(x), axis=1, keepdims=True))) - 9
    xr = (np.ldexp(x, (-e).astype(np.int32)).astype(np.float16).astype(np.float32) * np.exp2(e)).astype(np.float32)
    want_r = reference(oracle, t, raw.reshape(-1), n, k, xr, 0)
    for row in range(m):
        _, norm = rel_errors(got[row], want[row])
        elem_r, norm_r = rel_errors(got[row], want_r[row])
        assert norm <= 2 * TOL and elem_r <= TOL and norm_r <= TOL, (row, norm, elem_r, norm_r)


@pytest.mark.parametrize("t,order", [(13, 0), (13, 1), (11, 0), (10, 0)])
@pytest.mark.parametrize("m,n,k", [(7, 96, 512), (23, 200, 2048), (40, 300, 1024), (130, 257, 768), (300, 64, 2048)])
def test_qgemm_q5k_q3k_q2k_unit_activations_pick_single_weights(oracle, t, order, m, n, k):
    """The matrix kernels of Q5_K (the Q4_K kernel with the fifth bits from qh) and of Q3_K / Q2_K (sixteen 16-element
    sub-blocks): with unit activations row r of the result is column c_r of the dequantized weight, bit for bit -- every
    quant value, scale and min, both element orders of Q5_K, every k-step and lane position over the rows, rows that start
    at 2- and 4-byte aligned addresses -- and the re-blocked form of the same weight gives the same numbers to the f32
    summation order."""
    lib = _lib.load()
    size, d_at = REBLOCKED[t]
    rng = np.random.default_rng(77 * m + n + k + order + t)
    raw = rng.integers(0, 256, size=(n * (k // 256), size), dtype=np.uint8)
    for j, off in enumerate(d_at):
        raw[:, off:off + 2] = np.frombuffer(np.array([0.01 * (j + 1)], np.float16).tobytes(), np.uint8)
    raw = raw.reshape(-1)
    w = oracle.dequantize(t, raw, [n, k], order=order).reshape(n, k)
    for rep in range(3):
        cols = (np.arange(m) * (29 + 2 * rep) + 31 * rep + 3) % k
        xu = np.zeros((m, k), np.float32)
        xu[np.arange(m), cols] = 1.0
        got = gpu_qgemm(t, raw, n, k, oracle.f32_to_bf16_bits(xu.reshape(-1)).reshape(m, k), m, order=order)
        for r, c in enumerate(cols):
            assert np.array_equal(got[r], w[:, c]), (rep, r, c)
    # against the re-blocked form (two Q6_K tensors) on random activations
    x = rng.standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    got = gpu_qgemm(t, raw, n, k, bits, m, order=order)
    dw = pm.DeviceBuffer.from_host(raw)
    size = lib.pmetal_hip_reblock_size(t, n, k)
    dr, dx, dy = pm.DeviceBuffer(size), pm.DeviceBuffer.from_host(bits), pm.DeviceBuffer(4 * m * n)
    pm.check(lib.pmetal_hip_reblock_dev(t, dw.ptr, n, k, order, dr.ptr, size, None))
    pm.check(lib.pmetal_hip_qgemm_reblocked(t, dr.ptr, size, n, k, dx.ptr, pm.DTYPE_BF16, m, dy.ptr, pm.DTYPE_F32, None))
    pm.check(lib.pmetal_hip_sync(None))
    other = dy.to_host(np.float32).reshape(m, n)
    assert np.max(np.abs(got - other)) <= 1e-5 * np.max(np.abs(other))


@pytest.mark.parametrize("t", sorted(REBLOCKED))
def test_qlinear_q5k_q3k_q2k_dispatch(oracle, t):
    """qlinear: two activation rows one fused GEMV each on a weight of at most 2^23 elements (a larger one takes its
    short-batch GEMM), above that the GEMM; both agree with the oracle; a second, smaller call reuses the scratch
    buffer."""
    lib = _lib.load()
    if True:
        n, k = 2080, 4096  # above 2^23 elements: two rows are one GEMM
        wq = oracle.quantize(t, weights(t, n * k, outliers=1e-3))
        dw = pm.DeviceBuffer.from_host(wq)
        x = np.random.default_rng(2).standard_normal((2, k)).astype(np.float32)
        x = oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(x.reshape(-1))).reshape(2, k)
        dx, dy = pm.DeviceBuffer.from_host(x), pm.DeviceBuffer(4 * 2 * n)
        pm.check(lib.pmetal_hip_qlinear(t, dw.ptr, n, k, dx.ptr, pm.DTYPE_F32, 2, dy.ptr, pm.DTYPE_F32, 0, None))
        pm.check(lib.pmetal_hip_sync(None))
        elem, norm = rel_errors(dy.to_host(np.float32), reference(oracle, t, wq, n, k, x, 0).reshape(-1))
        assert elem <= TOL and norm <= TOL, (elem, norm)
    n, k = 320, 1024
    wq = oracle.quantize(t, weights(t, n * k, outliers=1e-3))
    dw = pm.DeviceBuffer.from_host(wq)
    for m in (8, 9, 64, 3, 2):
        x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
        x = oracle.bf16_bits_to_f32(oracle.f32_to_bf16_bits(x.reshape(-1))).reshape(m, k)  # survives the GEMM's f16 rounding
        dx, dy = pm.DeviceBuffer.from_host(x), pm.DeviceBuffer(4 * m * n)
        pm.check(lib.pmetal_hip_qlinear(t, dw.ptr, n, k, dx.ptr, pm.DTYPE_F32, m, dy.ptr, pm.DTYPE_F32, 0, None))
        pm.check(lib.pmetal_hip_sync(None))
        want = reference(oracle, t, wq, n, k, x, 0)
        elem, norm = rel_errors(dy.to_host(np.float32), want.reshape(-1))
        assert elem <= TOL and norm <= TOL, (t, m, elem, norm)
    # the GEMM's own argument checks
    assert lib.pmetal_hip_qgemm(t, dw.ptr, n, k, dx.ptr, pm.DTYPE_F32, 0, dy.ptr, pm.DTYPE_F32, 0, None) == 6
    assert lib.pmetal_hip_qgemm(t, dw.ptr, n, k, dx.ptr, pm.DTYPE_F32, 3, dy.ptr + 4, pm.DTYPE_F32, 0, None) == 1
    assert lib.pmetal_hip_qgemm(t, dw.ptr, n, k, dx.ptr, pm.DTYPE_F32, 3, dy.ptr, 7, 0, None) == 1
    lib.pmetal_hip_clear_error()


def test_qlinear_falls_back_to_the_gemm_when_the_gemv_refuses_the_row_length(oracle):
    """Q5_K rows longer than the GEMV's activation staging (k > 32768): one activation row still has the GEMM.
    A Q8_0 row that is not a multiple of 256 with a bf16 output has no kernel and says so."""
    lib = _lib.load()
    n, k = 64, 33024
    rng = np.random.default_rng(77)
    wq = oracle.quantize(13, (rng.standard_normal(n * k) * 0.02).astype(np.float32))
    x = rng.standard_normal(k).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x)
    xr = oracle.bf16_bits_to_f32(bits)
    dw, dx, dy = pm.DeviceBuffer.from_host(wq), pm.DeviceBuffer.from_host(bits), pm.DeviceBuffer(4 * n)
    assert lib.pmetal_hip_qgemv(13, dw.ptr, n, k, dx.ptr, pm.DTYPE_BF16, dy.ptr, 0, None) == 7
    msg = lib.pmetal_hip_last_error_message()
    assert b"n=64" in msg and b"k=33024" in msg
    pm.check(lib.pmetal_hip_qlinear(13, dw.ptr, n, k, dx.ptr, pm.DTYPE_BF16, 1, dy.ptr, pm.DTYPE_F32, 0, None))
    pm.check(lib.pmetal_hip_sync(None))
    want = oracle.qmatvec(13, wq, n, k, xr)
    elem, norm = rel_errors(dy.to_host(np.float32), want)
    assert elem <= TOL and norm <= TOL, (elem, norm)
    w8 = pm.DeviceBuffer.from_host(oracle.quantize(Q8_0, (rng.standard_normal(64 * 96) * 0.02).astype(np.float32)))
    y16 = pm.DeviceBuffer(2 * 4 * 64)
    x8 = pm.DeviceBuffer.from_host(bits[:4 * 96].copy())
    assert lib.pmetal_hip_qlinear(Q8_0, w8.ptr, 64, 96, x8.ptr, pm.DTYPE_BF16, 4, y16.ptr, pm.DTYPE_BF16, 0, None) == 6
    assert b"f32 only" in lib.pmetal_hip_last_error_message()
    lib.pmetal_hip_clear_error()


def test_qgemm_batch_equals_separate_calls(oracle):
    """Weights that share their activations: pmetal_hip_qgemm_batch gives the bits of one pmetal_hip_qgemm per weight
    (mixed types, element orders, output types, with and without a K split)."""
    lib = _lib.load()
    k = 2048
    rng = np.random.default_rng(5150)
    # (Q5_K behind Q4_K in the GGML order shares its converted activations; in the REF order it has a layout of its own; Q3_K and
    # Q2_K share theirs)
    specs = [(Q4K, 768, 0, pm.DTYPE_F32), (Q4K, 512, 0, pm.DTYPE_BF16), (Q4K, 256, 1, pm.DTYPE_F32), (13, 512, 1, pm.DTYPE_F32),
             (13, 384, 0, pm.DTYPE_BF16), (11, 300, 0, pm.DTYPE_F32), (10, 520, 0, pm.DTYPE_BF16), (Q6K, 640, 0, pm.DTYPE_F32),
             (Q6K, 320, 0, pm.DTYPE_BF16), (Q8_0, 384, 0, pm.DTYPE_F32), (Q4K, 1024, 0, pm.DTYPE_F32), (13, 256, 0, pm.DTYPE_F32)]
    ws = [pm.DeviceBuffer.from_host(oracle.quantize(t, weights(800 + i, n * k))) for i, (t, n, _, _) in enumerate(specs)]
    for m in (3, 48, 300):
        xb = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32))
        dx = pm.DeviceBuffer.from_host(xb)
        sizes = [m * n * (4 if yd == pm.DTYPE_F32 else 2) for (_, n, _, yd) in specs]
        y_one = [pm.DeviceBuffer(sz) for sz in sizes]
        y_bat = [pm.DeviceBuffer(sz) for sz in sizes]
        descs = (_lib.GemmDesc * len(specs))()
        for i, (t, n, order, yd) in enumerate(specs):
            pm.check(lib.pmetal_hip_memset(y_bat[i].ptr, 0xFF, sizes[i], None))
            pm.check(lib.pmetal_hip_qgemm(t, ws[i].ptr, n, k, dx.ptr, pm.DTYPE_BF16, m, y_one[i].ptr, yd, order, None))
            descs[i] = _lib.GemmDesc(t, yd, order, 0, n, ws[i].ptr, y_bat[i].ptr)
        pm.check(lib.pmetal_hip_qgemm_batch(descs, len(specs), k, dx.ptr, pm.DTYPE_BF16, m, None))
        pm.check(lib.pmetal_hip_sync(None))
        for i in range(len(specs)):
            assert np.array_equal(y_one[i].to_host(np.uint8), y_bat[i].to_host(np.uint8)), (m, specs[i])
    bad = (_lib.GemmDesc * 1)(_lib.GemmDesc(15, 0, 0, 0, 256, ws[0].ptr, y_bat[0].ptr))  # Q8_K: activations only
    assert lib.pmetal_hip_qgemm_batch(bad, 1, k, dx.ptr, pm.DTYPE_BF16, 3, None) == 2
    lib.pmetal_hip_clear_error()


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0])
@pytest.mark.parametrize("m", [300, 200, 516])
def test_qgemm_batch_wide_and_narrow_weights_share_x(oracle, t, m):
    """A wide and a narrow weight of one type and element order behind each other (q_proj / k_proj of a prefill): the launch plan
    pads the activation rows differently for the two (m = 300: 384 rows for n = 4096, 320 for n = 1024), so the converted
    activations of the first must not serve the second.  Both orders of the descriptors, bit for bit against separate calls."""
    lib = _lib.load()
    k = 4096
    rng = np.random.default_rng(977 + m + t)
    ns = (4096, 1024)
    ws = [pm.DeviceBuffer.from_host(oracle.quantize(t, weights(4100 + n, n * k))) for n in ns]
    xb = oracle.f32_to_bf16_bits(rng.standard_normal(m * k).astype(np.float32))
    dx = pm.DeviceBuffer.from_host(xb)
    y_one = []
    for w, n in zip(ws, ns):
        y = pm.DeviceBuffer(m * n * 4)
        pm.check(lib.pmetal_hip_qgemm(t, w.ptr, n, k, dx.ptr, pm.DTYPE_BF16, m, y.ptr, pm.DTYPE_F32, 0, None))
        pm.check(lib.pmetal_hip_sync(None))
        y_one.append(y.to_host(np.uint8))
    for first in (0, 1):
        idx = (first, 1 - first)
        y_bat = [pm.DeviceBuffer(m * ns[i] * 4) for i in idx]
        descs = (_lib.GemmDesc * 2)()
        for j, i in enumerate(idx):
            pm.check(lib.pmetal_hip_memset(y_bat[j].ptr, 0xFF, m * ns[i] * 4, None))
            descs[j] = _lib.GemmDesc(t, pm.DTYPE_F32, 0, 0, ns[i], ws[i].ptr, y_bat[j].ptr)
        pm.check(lib.pmetal_hip_qgemm_batch(descs, 2, k, dx.ptr, pm.DTYPE_BF16, m, None))
        pm.check(lib.pmetal_hip_sync(None))
        for j, i in enumerate(idx):
            assert np.array_equal(y_one[i], y_bat[j].to_host(np.uint8)), (m, first, ns[i])


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
@pytest.mark.parametrize("m", [1, 2, 5, 9, 16, 17, 25, 32])
@pytest.mark.parametrize("n,k", [(700, 2048), (333, 4096), (16, 2048), (4099, 4096), (40, 1024),
                                 # rows of more than 16 super-blocks: runs of 16, partial tiles added in a second kernel
                                 (500, 14336), (130, 6144), (77, 11008), (64, 32768),
                                 # rows of 11, 1, 3, 20 and 13 super-blocks: Q6_K rows then start at any even address, the last
                                 # waves own one super-block where the others own two (13)
                                 (333, 2816), (1001, 256), (250, 768), (123, 5120), (47, 3328),
                                 # rows of 72 and 136 super-blocks; 136 are more runs than the fused kernels take (eight of 16): the
                                 # row kernels with a K split of their own at up to 16 activation rows
                                 (40, 18432), (24, 34816)])
def test_qgemm_short_batches(oracle, t, m, n, k):
    """Few activation rows.  Up to 16: the fused kernels that read the weights once (rows of up to 16 super-blocks whole, longer ones in
    runs of 16), or, for the rows of 11 and of 20 super-blocks, the tile kernel; 17 to 32: the tile kernel (the weights are too small
    here for the fused kernels' two-block form, which the tall weights of test_gpu_gemm_tiles.py take).  Random block bytes (every
    scale, min and quant pattern), row counts that are no multiple of the 16-row tiles, one full tile, more tiles than workgroups take
    in one round; bf16 and f32 activations, f32 and bf16 outputs;
    unit activations that pick single weights out of the matrix."""
    rng = np.random.default_rng(1000 * t + 31 * m + n + k)
    block = {Q4K: 144, Q6K: 210, Q8_0: 34, 13: 176, 11: 110, 10: 84}[t]
    per = 32 if t == Q8_0 else 256
    raw = rng.integers(0, 256, size=(n * (k // per), block), dtype=np.uint8)
    half = np.frombuffer(np.array([0.01, 0.02], np.float16).tobytes(), np.uint8)
    if t in (Q4K, 13):
        raw[:, 0:4] = half
    elif t == Q6K:
        raw[:, 208:210] = half[:2]
    elif t == 11:
        raw[:, 108:110] = half[:2]
    elif t == 10:
        raw[:, 80:84] = half
    else:
        raw[:, 0:2] = (rng.uniform(0.5, 2.0, raw.shape[0]) * 0.01 * rng.choice([-1.0, 1.0], raw.shape[0])).astype(np.float16).view(np.uint8).reshape(-1, 2)
    raw = raw.reshape(-1)
    x = rng.standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    want = reference(oracle, t, raw, n, k, xr, 0)
    got = gpu_qgemm(t, raw, n, k, bits, m)
    elem, norm = rel_errors(got.reshape(-1), want.reshape(-1))
    assert elem <= TOL and norm <= TOL, (elem, norm)
    got16 = gpu_qgemm(t, raw, n, k, bits, m, y_dtype=pm.DTYPE_BF16)
    assert np.max(np.abs(got16 - want)) / np.max(np.abs(want)) <= 2.0 ** -8
    # f32 activations that are exact in f16 at the row's scale: small integers
    xi = rng.integers(-8, 9, size=(m, k)).astype(np.float32)
    got = gpu_qgemm(t, raw, n, k, xi, m, x_dtype=pm.DTYPE_F32)
    elem, norm = rel_errors(got.reshape(-1), reference(oracle, t, raw, n, k, xi, 0).reshape(-1))
    assert elem <= TOL and norm <= TOL, (elem, norm)
    # unit vectors: row r of the activations picks column (r * 97 + 5) % k of the dequantized weight, bit for bit where
    # the weight is exact in the output
    xu = np.zeros((m, k), np.float32)
    cols = [(r * 97 + 5 + 13 * m) % k for r in range(m)]
    for r, c in enumerate(cols):
        xu[r, c] = 1.0
    got = gpu_qgemm(t, raw, n, k, oracle.f32_to_bf16_bits(xu.reshape(-1)).reshape(m, k), m)
    w = oracle.dequantize(t, raw, [n, k]).reshape(n, k)
    for r, c in enumerate(cols):
        assert np.allclose(got[r], w[:, c], rtol=1e-6, atol=0), (r, c)


@pytest.mark.parametrize("t", [Q4K, Q6K, Q8_0, 13, 11, 10])
@pytest.mark.parametrize("m", [9, 29])
def test_qgemm_short_batch_very_tall_weight(oracle, t, m):
    """300 000 weight rows against 9 (29) activation rows: more row tiles per workgroup than its LDS holds finished tiles for,
    so the grid has more workgroups than compute units.  The first 2000 and the last 3000 rows against the oracle."""
    n, k = 300000, 2048
    rng = np.random.default_rng(t + m)
    block = {Q4K: 144, Q6K: 210, Q8_0: 34, 13: 176, 11: 110, 10: 84}[t]
    per = 32 if t == Q8_0 else 256
    raw = rng.integers(0, 256, size=(n * (k // per), block), dtype=np.uint8)
    half = np.frombuffer(np.array([0.01, 0.02], np.float16).tobytes(), np.uint8)
    if t in (Q4K, 13):
        raw[:, 0:4] = half
    elif t == Q6K:
        raw[:, 208:210] = half[:2]
    elif t == 11:
        raw[:, 108:110] = half[:2]
    elif t == 10:
        raw[:, 80:84] = half
    else:
        raw[:, 0:2] = half[:2]
    x = rng.standard_normal((m, k)).astype(np.float32)
    bits = oracle.f32_to_bf16_bits(x.reshape(-1)).reshape(m, k)
    xr = oracle.bf16_bits_to_f32(bits.reshape(-1)).reshape(m, k)
    got = gpu_qgemm(t, raw.reshape(-1), n, k, bits, m)
    rows = np.r_[0:2000, n - 3000:n]
    sub = raw.reshape(n, -1)[rows].reshape(-1)
    want = reference(oracle, t, sub, len(rows), k, xr, 0)
    elem, norm = rel_errors(got[:, rows].reshape(-1), want.reshape(-1))
    assert elem <= TOL and norm <= TOL, (elem, norm)
