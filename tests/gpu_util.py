"""Helpers shared by the GPU parity tests (everything goes through the C ABI of libpmetal_hip.so)."""
import ctypes as C

import numpy as np

import pmetal_amd as pm
from pmetal_amd import _lib

Q8_0, Q4K, Q6K = 8, 12, 14


def weights(seed, n, std=0.02, outliers=0.0):
    """N(0, std^2) with an optional fraction of +-0.5 outliers (the quantizer benchmark's distribution)."""
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal(n) * std).astype(np.float32)
    if outliers:
        idx = rng.random(n) < outliers
        w[idx] = np.where(rng.random(int(idx.sum())) < 0.5, np.float32(0.5), np.float32(-0.5))
    return w


def gpu_quantize_dev(t, x):
    """Device-resident entry point: upload f32, quantize on the stream, download the bytes."""
    lib = _lib.load()
    x = np.ascontiguousarray(x, dtype=np.float32)
    nbytes = lib.pmetal_hip_tensor_size(t, x.size)
    dx = pm.DeviceBuffer.from_host(x) if x.size else pm.DeviceBuffer(16)
    dq = pm.DeviceBuffer(max(nbytes, 16))
    pm.check(lib.pmetal_hip_memset(dq.ptr, 0xA5, max(nbytes, 16), None))  # poison: every byte must be written
    pm.check(lib.pmetal_hip_quantize_dev(t, dx.ptr, x.size, dq.ptr, nbytes, None), "quantize")
    pm.check(lib.pmetal_hip_sync(None))
    return dq.to_host(np.uint8, nbytes)


def gpu_dequantize_dev(t, raw, n, order=0):
    lib = _lib.load()
    raw = np.ascontiguousarray(raw, dtype=np.uint8)
    dq = pm.DeviceBuffer.from_host(raw) if raw.size else pm.DeviceBuffer(16)
    dy = pm.DeviceBuffer(max(4 * n, 16))
    pm.check(lib.pmetal_hip_memset(dy.ptr, 0xA5, max(4 * n, 16), None))
    pm.check(lib.pmetal_hip_dequantize_dev(t, dq.ptr, raw.size, dy.ptr, n, order, None))
    pm.check(lib.pmetal_hip_sync(None))
    return dy.to_host(np.float32, n)


def gpu_qgemv(t, wq, n, k, x, x_dtype, order=0):
    """x: float32 array (x_dtype 0) or uint16 bf16 bit patterns (x_dtype 1)."""
    lib = _lib.load()
    dw = pm.DeviceBuffer.from_host(np.ascontiguousarray(wq, dtype=np.uint8))
    dx = pm.DeviceBuffer.from_host(x)
    dy = pm.DeviceBuffer(4 * n)
    pm.check(lib.pmetal_hip_memset(dy.ptr, 0xFF, 4 * n, None))  # NaN poison
    pm.check(lib.pmetal_hip_qgemv(t, dw.ptr, n, k, dx.ptr, x_dtype, dy.ptr, order, None))
    pm.check(lib.pmetal_hip_sync(None))
    return dy.to_host(np.float32, n)


def rel_errors(got, want):
    """(element-wise max relative error over |want| > 1e-3*max|want|, normwise max error)."""
    got = got.astype(np.float64)
    want = want.astype(np.float64)
    scale = np.max(np.abs(want))
    diff = np.abs(got - want)
    big = np.abs(want) > 1e-3 * scale
    elem = float(np.max(diff[big] / np.abs(want[big]))) if big.any() else 0.0
    return elem, float(np.max(diff) / scale) if scale > 0 else float(np.max(diff))


def first_mismatch(a, b, block):
    bad = np.nonzero(a != b)[0]
    if bad.size == 0:
        return "identical"
    i = int(bad[0])
    return (f"{bad.size} differing bytes in {np.unique(bad // block).size} blocks; first at byte {i} "
            f"(block {i // block}, offset {i % block}): got {a[i]} want {b[i]}")


# ---- the GEMM's launch plan, so that a test can say which kernel its shape takes ---------------------------------
# (qgemm_pair_plan and qgemm_workspace_bytes by their C++ names, as _lib.gemm_plan finds qgemm_plan)
Plan, gemm_plan = _lib.GemmPlan, _lib.gemm_plan
SMALL, WAVES, ROWS = _lib.GEMM_SMALL, _lib.GEMM_WAVES, _lib.GEMM_ROWS


def gemm_pair_plan(t, m, n0, n1, k):
    """The plan of two weights in one launch, or None where each goes on its own."""
    fn = _lib.load()._ZN3pmh15qgemm_pair_planElllljPNS_8GemmPlanE
    fn.restype, fn.argtypes = C.c_bool, [C.c_int64, C.c_int64, C.c_int64, C.c_int64, C.c_uint32, C.POINTER(Plan)]
    p = Plan()
    return p if fn(m, n0, n1, k, t, C.byref(p)) else None


def gemm_workspace_bytes(t, m, n, k):
    fn = _lib.load()._ZN3pmh21qgemm_workspace_bytesEjlll
    fn.restype, fn.argtypes = C.c_size_t, [C.c_uint32, C.c_int64, C.c_int64, C.c_int64]
    return fn(t, m, n, k)


def codec_chunk(n):
    """Elements of a staging chunk of the host codec."""
    fn = _lib.load()._ZN3pmh11codec_chunkEm
    fn.restype, fn.argtypes = C.c_size_t, [C.c_size_t]
    return fn(n)


def gemm_small_lds(t, m, k, tiles_per_wg, own, xf32):
    fn = _lib.load()._ZN3pmh15qgemm_small_ldsEjllibb
    fn.restype, fn.argtypes = C.c_size_t, [C.c_uint32, C.c_int64, C.c_int64, C.c_int, C.c_bool, C.c_bool]
    return fn(t, m, k, tiles_per_wg, own, xf32)


def gemm_converts_itself(t, m, n, k, x_dtype, second_n=0, shared=False):
    """Whether a launch's waves convert the activations they multiply."""
    fn = _lib.load()._ZN3pmh21qgemm_converts_itselfERKNS_8GemmPlanEjlllljb
    fn.restype, fn.argtypes = C.c_bool, [C.POINTER(Plan), C.c_uint32, C.c_int64, C.c_int64, C.c_int64, C.c_int64, C.c_uint32, C.c_bool]
    return fn(C.byref(gemm_plan(t, m, n, k)), t, m, n, second_n, k, x_dtype, shared)
