"""What the float32 products of few tokens choose, asked on the host."""
import ctypes

import pytest

from sprout_lm_amd import ops


@pytest.fixture(scope="module")
def lib():
    try:
        return ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")


def test_parts_are_counted_on_the_fullest_xcd(lib):
    """Parts that fill the chip once fill no XCD more than once: a 33rd block on one of them is a round for all."""
    taken = 0
    for T in (17, 48, 64, 65, 100, 128, 129, 160, 200, 255):
        for N, K in ((896, 4864), (1536, 8960), (2048, 2048), (3584, 3584), (3584, 18944), (5120, 5120), (1000, 4096)):
            plan = (ctypes.c_int * 3)()
            if lib.sp_gemm_f32_parts_plan(T, N, K, plan):
                continue
            rows, columns, parts = plan
            t, n = -(-T // rows), -(-N // columns)
            fullest = (n // 8 * t + -(-(n % 8) * t // 8)) * parts
            assert t * n * parts > 256 or fullest <= 32, (T, N, K, rows, columns, parts)
            taken += 1
    assert taken > 40


def test_eight_waves_share_a_k_that_four_do_not_ask_for_at_once(lib):
    for N, K in ((896, 4864), (896, 896), (1152, 896), (2560, 2560), (151936, 896), (9728, 512), (896, 192)):
        assert lib.sp_gemm_f32_waves(N, K) == 8, (N, K)
    # few steps a wave as it is, and matrices that are bound by what is on its way
    for N, K in ((30000, 256), (32000, 64), (32000, 128), (15000, 256), (896, 128), (64, 64), (151936, 64), (1536, 8960), (5120, 5120), (65536, 2052)):
        assert lib.sp_gemm_f32_waves(N, K) == 4, (N, K)
