"""How many parts a prompt's keys are cut into, asked on the host: the walk's length decides, and the work beside it, not the blocks alone."""
import pytest

from sprout_lm_amd import ops


@pytest.fixture(scope="module")
def lib():
    try:
        return ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")


def _parts(floats, tiles, nq, hd):
    assert floats % (tiles * 32 * nq * (hd + 2)) == 0
    return max(1, floats // (tiles * 32 * nq * (hd + 2)))


def _asked(lib, nq, nkv, hd, queries, behind, answers=0, context=0):
    """Parts of a step of one prompt, beside `answers` one-query sequences: without hints (`sp_attention_workspace_floats`) and with them."""
    tiles = -(-queries // 32)
    args = (1, hd, 16, nq, nkv, 0, answers, context if answers else 0, tiles, behind + queries)
    beside = (answers * nq * -(-context // 256) * (hd + 2) + 3) // 4 * 4 if answers and context > 256 else 0
    walk = ops.mean_tile_walk([queries], [behind + queries])
    return [_parts(n - beside, tiles, nq, hd)
            for n in (lib.sp_attention_workspace_floats(*args), lib.sp_attention_workspace_hinted(*args, walk, answers * context))]


# us with one part and with the parts at least that are asked for: 608 and 219; 605 and 333; 604 and 425; 586 and 376 (8); 173 and 79; 168 and 104
@pytest.mark.parametrize("nq,nkv,hd,queries,behind,answers,least", [
    (28, 4, 128, 257, 30720, 8, 3), (28, 4, 128, 512, 30720, 8, 2), (28, 4, 128, 640, 30720, 0, 3), (40, 8, 128, 257, 30720, 0, 3),
    (28, 4, 128, 257, 8192, 8, 3), (28, 4, 128, 256, 30720, 1, 3), (28, 4, 128, 512, 8192, 1, 2), (40, 8, 128, 320, 8192, 8, 3),
    (14, 2, 64, 640, 8192, 1, 2)])
def test_long_walks_are_cut_beside_answers_too(lib, nq, nkv, hd, queries, behind, answers, least):
    for parts in _asked(lib, nq, nkv, hd, queries, behind, answers, 63 if answers == 1 else 2048):
        assert parts >= least


def test_short_walks_and_full_chips_are_not_cut(lib):
    for queries, behind, answers in ((512, 0, 0), (640, 0, 8), (960, 1024, 8), (960, 8192, 0), (2048, 30720, 8)):
        assert _asked(lib, 28, 4, 128, queries, behind, answers, 2048)[1] == 1
    # beside 45 answers, whose own work fills the chip, a walk of 1,344 keys is left whole: 51 us, in three parts 58
    assert _asked(lib, 28, 4, 128, 320, 1024, 45, 2000)[1] == 1


def test_a_part_holds_two_stages_or_one_of_wide_heads_and_there_are_32_at_most(lib):
    for nq, nkv, hd in ((28, 4, 128), (12, 4, 64), (8, 1, 256), (16, 1, 192), (3, 3, 80), (1, 1, 16)):
        for queries in (2, 33, 128, 500, 1000):
            for behind in (0, 300, 600, 1100, 5000, 32000, 130000):
                for parts in _asked(lib, nq, nkv, hd, queries, behind, 3, 700):
                    assert parts <= 32 and (parts == 1 or parts * (128 if hd > 128 else 256) <= behind + queries + 127)


def test_prompts_and_many_answers_have_launches_of_their_own(lib):
    """Few one-query blocks go with the prompts' blocks, many do not: either side of the lines."""
    pays = lambda hd, nq, nkv, tiles, answers, longest, keys: bool(lib.sp_attention_mixed_pays(hd, nq, nkv, tiles, answers, longest, keys))
    assert pays(128, 28, 4, 4, 1, 63, 63) and pays(64, 14, 2, 4, 1, 256, 1)                       # one answer that has just begun
    assert pays(64, 14, 2, 8, 5, 1500, 4000) and pays(128, 28, 4, 8, 8, 4096, 18000)            # the steps that gain
    assert pays(64, 16, 8, 2, 16, 4096, 16 * 3400) and not pays(64, 16, 8, 2, 24, 4096, 24 * 3500)      # eight waves, heads of 64
    assert not pays(64, 16, 8, 2, 128, 4096, 128 * 1300)
    assert pays(128, 28, 4, 2, 8, 8192, 8 * 8000) and not pays(128, 28, 4, 2, 24, 16384, 24 * 7000)     # many chunks a sequence
    assert pays(128, 28, 4, 2, 8, 32768, 8 * 2000)        # known as a bucket, though few of its chunks hold keys
    assert pays(64, 32, 8, 2, 32, 4096, 32 * 1300) and not pays(64, 32, 8, 2, 128, 4096, 128 * 1300)    # four waves
    assert not pays(64, 16, 8, 2, 128, 4096, 0)           # keys not known: all of them as long as the longest


def test_walks_count_in_fractions_for_the_kernel_of_two_heads_a_wave(lib):
    """144 blocks that walk 3,768 keys fill the chip as 256 of 2,048 do (62 us against 123): three parts of 1,024 keys at least, which only that
    kernel has here; 2,600 keys do not."""
    assert _asked(lib, 48, 6, 64, 768, 3000) == [3, 3]
    assert _asked(lib, 48, 6, 64, 768, 1832) == [1, 1]


def test_short_walks_of_wide_heads_are_cut_into_single_stages(lib):
    assert _asked(lib, 8, 1, 256, 48, 512) == [5, 5] and _asked(lib, 4, 4, 256, 48, 512, 8, 2048) == [5, 5]
