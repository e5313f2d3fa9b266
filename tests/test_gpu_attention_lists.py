"""Prompt attention of heads of 64 in steps of many prompts: lists of tiles that a wave holds, that the waves of a block read into LDS in one trip and
in several, and whose sums over 64 entries are more than 64 themselves; and on the host which kernel such steps take."""
import pytest

from sprout_lm_amd import ops
from tests.attention_rows_helpers import OTHER, OWN, PARTS, SHARED, against_the_general_kernel, choice, choice_of, form

# (heads, groups, [(context, queries)], form, order of the list): 65 to 256 entries, up to 1,024, more, and more than 4,096; without entries
# that have no rows (eight heads a set), and with most of them so (one)
CASES = [(32, 8, [(300, 300)] * 20, OWN, None), (32, 8, [(301, 300)] * 30, OWN, "shuffled"), (8, 2, [(2, 2)] * 4200, OWN, None),
         (64, 8, [(100, 100)] * 40, OWN, None), (16, 2, [(400, 2)] * 4200, OWN, "backwards"), (6, 1, [(40000, 300)] + [(64, 64)] * 150, PARTS, None),
         (6, 1, [(64, 64)] * 60 + [(40000, 300)], PARTS, "shuffled"), (16, 2, [(100, 100)] * 40, SHARED, None), (12, 4, [(6000, 40)] + [(64, 63)] * 150, SHARED, "shuffled"),
         (8, 8, [(512, 512)] * 20, SHARED, None), (8, 8, [(1024, 1000)] * 33, SHARED, None), (8, 8, [(400, 2)] * 4200, SHARED, None)]


def test_which_steps():
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")
    assert all(form(*case[:3]) == case[3] for case in CASES)
    # one head a group, several rounds of blocks and short walks: shared rows took 1.25, 1.35 and 1.2 of the other kernels' time; 0.98 and 0.9
    assert form(8, 8, [(64, 64)] * 256) == form(16, 16, [(64, 64)] * 256) == form(16, 16, [(100, 100)] * 100) == OTHER
    assert form(8, 8, [(512, 512)] * 32) == form(8, 8, [(1024, 1024)] * 16) == SHARED
    # 78 prompts of 2 to 207, one walk of 4,037 keys among them: in three parts 144 us, on shared rows 116
    assert choice_of(64, 8, 150, 4037, 435)[2:] == (1, 1)
    # a list whose blocks an entry do not fit where they are put
    assert choice(14, 2, [(2, 2)] * 60000) and choice(14, 2, [(2, 2)] * 62000) is None


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_long_lists(case):
    nq, nkv, seqs, expected, listed = CASES[case]
    assert form(nq, nkv, seqs) == expected
    against_the_general_kernel(nq, nkv, seqs, listed, seed=case, same_pages=len(seqs) > 1000)
