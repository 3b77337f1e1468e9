"""Which products esep_gemm takes from the vendor BLAS (esep_gemm_pays) and how it launches them, on the
CPU: the ranges where it measured faster, and not the ones around them (microseconds of the library / of
the kernel on an MI355X, operands warm, fp16; the rule's comment in csrc/gemm.hip has the whole table)."""

import pytest

from solution.body import _hip

# (M, N, K, B given as [K, N], library, here)
MEASURED = [
    (4096, 256, 1536, 0, 9.2, 22.5), (512, 2048, 1536, 0, 9.1, 18.1), (512, 1536, 1536, 0, 8.9, 15.5),
    (700, 2048, 2048, 0, 13.2, 19.8), (300, 151936, 1536, 0, 185.1, 240.7),
    (350, 152064, 3584, 0, 448.5, 511.6), (128, 11008, 2048, 0, 15.3, 20.4), (512, 512, 3584, 0, 9.3, 14.5),
    (1031, 1536, 8960, 0, 48.9, 54.2), (4096, 151936, 1536, 0, 1623.0, 1779.1),
    (512, 1536, 1536, 1, 11.2, 15.6), (512, 896, 1152, 1, 8.4, 10.2), (16, 896, 896, 1, 4.6, 7.2),
    (2300, 1536, 8960, 1, 79.7, 91.5), (1500, 11008, 2048, 1, 76.2, 88.5), (3001, 2048, 11008, 1, 134.6, 151.9),
    (4096, 1536, 151936, 1, 1721.4, 1763.8), (180, 13824, 5120, 1, 44.0, 51.1),
    (1031, 1536, 17920, 1, 199.4, 73.7), (16, 1536, 151936, 1, 288.2, 113.4), (3750, 1536, 151936, 1, 2496.1, 1717.0),
    (1031, 1536, 8960, 1, 63.3, 53.0), (3001, 1536, 8960, 1, 95.8, 89.4), (1285, 896, 9728, 1, 73.5, 41.8),
    (128, 3584, 3584, 1, 27.7, 16.4), (1500, 896, 4864, 1, 39.7, 27.2), (3001, 1536, 1536, 1, 29.4, 24.1),
    (3750, 8960, 1536, 1, 108.8, 119.4), (3001, 8960, 1536, 1, 86.5, 82.8), (4096, 11008, 2048, 1, 174.4, 168.2),
    (1500, 896, 896, 1, 12.0, 8.1), (400, 3584, 18944, 0, 167.0, 72.0), (400, 1536, 8960, 0, 33.7, 26.2),
    (400, 151936, 1536, 0, 254.7, 231.3), (16, 151936, 1536, 0, 160.5, 90.3),
]


@pytest.mark.parametrize("M,N,K,b_kn,library,here", MEASURED)
def test_the_faster_one_is_taken(M, N, K, b_kn, library, here):
    assert _hip.lib().esep_gemm_pays(M, N, K, b_kn) == int(here < library)


def test_the_gpu_tests_cover_the_plans():
    """The sizes of test_gpu_gemm.py reach every tile shape, with one split of the contraction and with
    several (the plan's prices decide, so a retuned figure could drop one)."""
    from test_gpu_gemm import SIZES

    plans = [_hip.lib().esep_gemm_plan(*size) for size in SIZES]
    assert {(p & 15, p >> 4 > 1) for p in plans} == {(s, m) for s in range(5) for m in (False, True)}
