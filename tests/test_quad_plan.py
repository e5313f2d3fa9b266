"""The choice of block shape of the product on four waves a block, asked of the library without running a kernel (no GPU)."""
import itertools
import random

import pytest

from sprout_lm_amd import ops
from tests.test_gpu_quad_products import ROTATING_SIZES, SIZES

SHAPES = {(64, 64, 4), (96, 128, 2), (128, 64, 4), (128, 128, 2), (128, 128, 4), (128, 192, 2), (160, 192, 2), (192, 128, 2), (192, 192, 2),
          (256, 128, 3), (128, 256, 2), (160, 256, 2), (320, 128, 2), (192, 256, 2), (256, 192, 2), (288, 192, 2), (256, 256, 2)}
KINDS = [ops.PLAN_STORE, ops.PLAN_ACCUMULATE, ops.PLAN_GATED]


@pytest.fixture(autouse=True, scope="module")
def built_library():
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")


@pytest.mark.parametrize("kind", KINDS)
def test_plan_invariants(kind):
    for T, N, K in itertools.product([1, 64, 65, 100, 264, 777, 2048, 8192], [8, 16, 130, 900, 1152, 37888, 151936], [64, 70, 192, 3584, 27648]):
        plan = ops.quad_plan(kind, T, N, K)
        if T <= 16 or K % 64 or N % (16 if kind == ops.PLAN_GATED else 8) or N * K * 2 >= 1 << 32:
            assert plan is None, (T, N, K)          # other kernels' products
            continue
        if T <= 64 and plan is None:
            continue
        rows, cols, splits, buffers = plan
        assert (rows, cols, buffers) in SHAPES, (T, N, K, plan)
        assert buffers * rows * 128 + (buffers + 1) * cols * 128 <= 160 * 1024
        # only float atomics join partial sums; every split has a step
        assert splits == 1 or (kind == ops.PLAN_ACCUMULATE and K // 64 // splits >= 4), (T, N, K, plan)


def test_no_product_is_cut_that_the_other_kernels_leave_whole():
    """Parts of K meet in float atomics, whose order no two runs share: sums that the eight-wave kernel gives the same bits in every
    run (the down product of a prompt of 2,048 tokens at 7B sizes, the output product of 65 to 512 at 0.5B sizes) stay so."""
    rng = random.Random(3)
    sizes = list(itertools.product([65, 200, 512, 1500, 2048, 4096], [896, 1536, 3584, 5120], [896, 3584, 4864, 8960, 18944, 27648]))
    sizes += [(round(17 * 2 ** rng.uniform(0, 7)), 8 * rng.randint(1, 2000), 64 * rng.randint(1, 400)) for _ in range(4000)]
    cut = 0
    for T, N, K in sizes:
        plan = ops.quad_plan(ops.PLAN_ACCUMULATE, T, N, K)
        if plan is None or plan[2] == 1:
            continue
        cut += 1
        if T > 64 or N * K >= 6 << 20:          # the eight-wave kernel's, otherwise
            assert ops.pipe_plan(ops.PLAN_ACCUMULATE, T, N, K)[2] > 1, (T, N, K, plan)
    assert cut > 500
    for T, N, K in [(58, 4992, 1024), (42, 6648, 640), (34, 4760, 1216)]:      # the kernel for few tokens takes these in one part
        assert ops.quad_plan(ops.PLAN_ACCUMULATE, T, N, K)[2] == 1


def test_few_tokens_are_taken_where_measurements_say_so():
    taken = lambda kind, T, N, K: ops.quad_plan(kind, T, N, K) is not None
    assert taken(ops.PLAN_GATED, 17, 9728, 896) and not taken(ops.PLAN_GATED, 16, 9728, 896) and not taken(ops.PLAN_GATED, 64, 37888, 3584)
    assert taken(ops.PLAN_ACCUMULATE, 45, 896, 4864) and not taken(ops.PLAN_ACCUMULATE, 24, 896, 4864)
    assert taken(ops.PLAN_ACCUMULATE, 17, 3584, 3584) and not taken(ops.PLAN_ACCUMULATE, 64, 896, 896)
    assert taken(ops.PLAN_STORE, 17, 151936, 896) and not taken(ops.PLAN_STORE, 64, 152064, 3584)
    assert not taken(ops.PLAN_STORE, 32, 7168, 5120) and taken(ops.PLAN_STORE, 33, 7168, 5120)
    # on either side of lines that are no preset's: gated products of many rows and a long K are 7 to 33 % longer on four waves
    for T in (17, 33, 64):
        assert not any(taken(ops.PLAN_GATED, T, n, k) for n in (18432, 22528, 28672) for k in (2048, 2560, 3072))
        assert all(taken(ops.PLAN_GATED, T, n, k) for n in (2048, 8192, 16384) for k in (512, 2048, 3072))
    assert taken(ops.PLAN_GATED, 40, 28672, 1024) and not taken(ops.PLAN_GATED, 48, 28672, 1024)
    # stored products of up to 32 tokens and few rows are 2 to 16 % longer there
    assert not any(taken(ops.PLAN_STORE, 24, n, k) for n in (1152, 3072, 4608) for k in (2048, 4096, 5120))
    assert taken(ops.PLAN_STORE, 24, 6144, 4096) and taken(ops.PLAN_STORE, 24, 8192, 5120) and taken(ops.PLAN_STORE, 48, 12288, 8192)


def test_outputs_of_few_columns_are_cut_rather_than_read_by_every_xcd():
    """With less than 8 weight tiles an XCD reads its run of the tokens alone: 512 rows of w on blocks of 128 columns and in two parts
    of K (48 us at 4,096 tokens, K = 8,192; 128 x 64 in one part, which every XCD reads all tokens for, 80)."""
    for T, K, most in [(2048, 8192, 4), (3000, 4864, 3), (4096, 4864, 2), (4096, 8192, 2)]:
        rows, cols, splits, _ = ops.quad_plan(ops.PLAN_ACCUMULATE, T, 512, K)
        assert cols == 128 and 2 <= splits <= most, (T, K, rows, cols, splits)


def test_rotation_takes_heads_of_whole_sixty_fours():
    for T, (nq, nkv, hd, K) in itertools.product([64, 65, 264, 2048], [(14, 2, 64, 896), (28, 4, 128, 3584), (3, 1, 48, 896), (2, 2, 192, 64)]):
        plan = ops.quad_plan(ops.PLAN_ROTATING, T, (nq + 2 * nkv) * hd, K, hd)
        assert (plan is None) == (T <= 64 or hd % 64 != 0), (T, nq, nkv, hd, K, plan)
        assert plan is None or (plan[:2] + plan[3:] in SHAPES and plan[1] != 192 and plan[2] == 1)
        # a caller asks the library once for the folded call, by sizes
        assert T <= 64 or ops.fused_supported(ops.FUSED_ROPE, T, (nq + 2 * nkv) * hd, K, hd, hd) == (plan is not None)


def test_kernel_tests_reach_every_block_shape():
    for kind in KINDS:
        seen = {}
        for T, N, K in SIZES[kind]:
            plan = ops.quad_plan(kind, T, N, K)
            seen.setdefault((plan[0], plan[1], plan[3]), set()).add(plan[2] > 1)
        assert set(seen) == SHAPES, SHAPES - set(seen)
        assert kind != ops.PLAN_ACCUMULATE or sum(True in s for s in seen.values()) >= 8
    rotating = {p[:2] + p[3:] for p in (ops.quad_plan(ops.PLAN_ROTATING, T, (nq + 2 * nkv) * hd, K, hd) for T, nq, nkv, hd, K in ROTATING_SIZES)}
    assert rotating == {s for s in SHAPES if s[1] != 192}
