"""The choice of block shape and split of the tiled product on up to eight waves a block, asked of the library without running a
kernel (no GPU): invariants over a sweep of sizes, and the decisions that measurements on the GPU settled.  Where results are whole
eights that start at 16 bytes another kernel has these products (tests/test_quad_plan.py)."""
import itertools

import pytest

from sprout_lm_amd import ops



@pytest.fixture(autouse=True, scope="module")
def built_library():
    """The plan is asked of the compiled library, which needs hipcc where it is not built yet, but no GPU."""
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")


SHAPES = {(256, 256), (256, 128), (128, 128), (64, 64), (64, 256), (64, 128), (384, 256), (256, 160)}
PAIRED = {(256, 256), (256, 128), (128, 128), (64, 256), (64, 128), (384, 256)}    # an even number of tile columns a wave


def sizes():
    tokens = [1, 5, 16, 17, 64, 65, 128, 200, 256, 264, 512, 777, 1024, 1100, 2048, 4096, 8192]
    rows = [64, 130, 896, 1152, 3584, 4608, 5120, 9728, 37888, 151936]
    depth = [64, 192, 896, 1088, 3584, 4864, 5120, 18944, 27648]
    return itertools.product(tokens, rows, depth)


@pytest.mark.parametrize("kind", [ops.PLAN_STORE, ops.PLAN_ACCUMULATE, ops.PLAN_GATED])
def test_plan_invariants(kind):
    for T, N, K in sizes():
        plan = ops.pipe_plan(kind, T, N, K)
        if N * K * 2 >= 1 << 32:      # a tile's offset into the weights has 32 bits: another kernel's product
            assert plan is None, (T, N, K)
            continue
        assert plan is not None, (T, N, K)          # K is a multiple of 64 everywhere here
        rows, cols, splits, waves = plan
        assert (rows, cols) in SHAPES and splits >= 1
        if kind == ops.PLAN_GATED:
            # gate and up rows alternate between a wave's tile columns (64 x 64 for up to 64 tokens is two waves with
            # two tile columns each; for more tokens it is four waves with one)
            assert (rows, cols) in PAIRED or T <= 64, (T, N, K, plan)
        if kind != ops.PLAN_ACCUMULATE:
            assert splits == 1, (T, N, K, plan)                  # only float atomics can join partial sums
        assert splits == 1 or K // 64 // splits >= 8, (T, N, K, plan)
        if T > 64:   # few tokens have shapes of their own
            assert (rows, cols) != (64, 256)


def test_products_the_kernel_does_not_take():
    assert ops.pipe_plan(ops.PLAN_STORE, 300, 100, 70) is None          # K is no multiple of 64
    assert ops.pipe_plan(ops.PLAN_STORE, 300, 100, 0) is None
    assert ops.pipe_plan(7, 300, 128, 128) is None
    assert ops.pipe_plan(ops.PLAN_ROTATING, 300, 1152, 896) is None     # the four-wave product rotates, and the decode kernels


def test_decisions_that_measurements_settled():
    """(kind, T, N, K) -> plan: each of these was timed against the other shapes with operands from memory.  They hold where a
    result does not start at 16 bytes, and at sizes beside these that are no whole eights."""
    settled = {
        (ops.PLAN_STORE, 2048, 37888, 3584): (256, 256, 1),       # fills the chip: the largest blocks
        (ops.PLAN_STORE, 2048, 4608, 3584): (256, 160, 1),        # 232 blocks where 256 x 256 make 144
        (ops.PLAN_ACCUMULATE, 2048, 5120, 27648): (256, 160, 1),  # 256 blocks where 256 x 256 make 160
        (ops.PLAN_ACCUMULATE, 2048, 3584, 3584): (256, 128, 1),
        (ops.PLAN_ACCUMULATE, 2048, 896, 4864): (128, 128, 2),
        (ops.PLAN_ACCUMULATE, 2048, 896, 896): (64, 64, 1),
        (ops.PLAN_GATED, 2048, 9728, 896): (384, 256, 1),
        (ops.PLAN_GATED, 256, 9728, 896): (128, 128, 1),
    }
    for args, want in settled.items():
        got = ops.pipe_plan(*args)
        assert (got[:3] if got else None) == want, (args, got, want)


def test_kernel_tests_reach_every_block_shape():
    """The sizes that tests/test_gpu_kernels.py runs on the GPU, asked here for their plans: every block shape of the
    plain and the gated product is reached by at least one of them."""
    import importlib
    kernels = importlib.import_module("tests.test_gpu_kernels")
    plain = {(rows, cols, waves, split) for rows, cols, waves, split in kernels.BLOCK_SHAPE_SIZES.values()}
    assert {(r, c) for r, c, _, _ in plain} == SHAPES - {(64, 256)} and {s for _, _, _, s in plain} == {False, True}
    for (accumulate, T, N, K), (rows, cols, waves, split) in kernels.BLOCK_SHAPE_SIZES.items():
        kind = ops.PLAN_ACCUMULATE if accumulate else ops.PLAN_STORE
        got = ops.pipe_plan(kind, T, N, K)
        assert (got[0], got[1], got[3], got[2] > 1) == (rows, cols, waves, split), (T, N, K, got)
        assert ops.quad_plan(kind, T, N, K) is None, (T, N, K)          # it is this kernel that runs
    assert all(ops.quad_plan(ops.PLAN_GATED, T, 2 * I, K) is None for T, I, K in kernels.EIGHT_WAVE_GATED_SIZES)
    gated = {ops.pipe_plan(ops.PLAN_GATED, T, 2 * I, K)[:2] for T, I, K in kernels.EIGHT_WAVE_GATED_SIZES}
    assert gated == {(64, 128), (128, 128), (256, 128), (256, 256), (384, 256)}, gated


def test_blocks_are_numbered_so_that_every_tile_runs_once_and_the_xcds_share_them():
    """The tiled product's numbering of its blocks (block b runs on XCD b % 8): every (token tile, weight tile) is
    some block's, once; a weight tile of the whole eights lies on one XCD with all its token tiles (nobody else
    fetches it); and no XCD holds more blocks than its even share of the left-over tiles, rounded up."""
    for tiles_t in list(range(1, 20)) + [33, 64]:
        for tiles_n in list(range(1, 41)) + [148, 149, 593]:
            blocks = ops.pipe_tiles(tiles_t, tiles_n)
            assert len(blocks) % 8 == 0
            seen, per_xcd, home = {}, [0] * 8, {}
            for b, tile in enumerate(blocks):
                if tile is None:
                    continue
                t, n = tile
                assert 0 <= t < tiles_t and 0 <= n < tiles_n and tile not in seen, (tiles_t, tiles_n, b, tile)
                seen[tile] = b
                per_xcd[b % 8] += 1
                if n < tiles_n // 8 * 8:
                    assert home.setdefault(n, b % 8) == b % 8 == n % 8, (tiles_t, tiles_n, b, tile)
            assert len(seen) == tiles_t * tiles_n
            left = tiles_n % 8
            assert max(per_xcd) == tiles_n // 8 * tiles_t + -(-left * tiles_t // 8), (tiles_t, tiles_n, per_xcd)
    with pytest.raises(ops.KernelError):
        ops.pipe_tiles(0, 5)



def test_parts_of_prompts_lie_at_whole_sixteen_bytes_of_a_mixed_step_s_workspace():
    """They come behind the one-query sequences' parts and are read and written sixteen bytes at a time; those in turn are as many
    floats as heads, sequences and chunks give, 1,386 here."""
    lib = ops.library()
    for nq, nkv, hd, n_decode, ctx in [(7, 1, 64, 1, 700), (5, 5, 16, 3, 257), (14, 2, 64, 8, 4096), (3, 1, 80, 5, 1100)]:
        decode = lib.sp_attention_workspace_floats(1, hd, 16, nq, nkv, 0, n_decode, ctx, 0, 0)
        assert decode % 4 == 0 and 0 <= decode - n_decode * nq * -(-ctx // 256) * (hd + 2) < 4


def test_rows_go_through_lds_where_there_are_several_of_a_long_k():
    """Up to 768 numbers a row they gain nothing, and at 33 to 64 tokens lose up to a fifth; past 1,024 they have no room."""
    pays = ops.library().sp_staged_rows_pay
    assert all(pays(T, K) for T in (4, 8, 33, 45, 64) for K in (776, 896, 1016, 1024))
    assert not any(pays(T, K) for T in (1, 3, 4, 8, 9, 16, 32, 33, 64) for K in (8, 256, 512, 576, 768, 1032, 3584))
    assert not any(pays(T, 896) for T in (1, 2, 3, 9, 32))
