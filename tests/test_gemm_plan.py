"""The GEMM's launch plan (host code, no device needed): what it names can be launched."""
import pytest

from gpu_util import Q4K, Q6K, Q8_0, WAVES, gemm_pair_plan, gemm_plan

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
