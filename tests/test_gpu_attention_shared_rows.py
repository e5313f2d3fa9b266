"""Prompt attention whose blocks of four waves share 64 rows and take 32 keys of a stage each: groups and lengths that end anywhere in a block, in
a stage and in a wave's keys, lists of more than a wave's entries and in any order, page tables that LDS does not hold, pools beyond 4 GB; and on
the host which steps take it."""
import pytest

from sprout_lm_amd import ops
from tests.attention_rows_helpers import SHARED, against_the_general_kernel, choice, form


def test_which_steps():
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")
    shared = lambda *a: (choice(*a) or (0, 0, 0, 0))[3] == 1
    # times of this one over what else would run: 0.77, 0.82, 0.75, 0.81, 0.81
    assert shared(14, 2, [(2048, 2048)]) and shared(14, 2, [(47, 47), (89, 89), (169, 169), (322, 322), (611, 611)])
    assert shared(8, 8, [(2048, 2048)]) and shared(32, 8, [(1024, 1024)]) and shared(14, 2, [(2048, 2048)] * 2)
    # 1.21, 1.35, 1.4 (one head a group and little work), 1.4 and 1.2 (rows of their own)
    assert not any(shared(*a) for a in ((14, 2, [(512, 512)]), (14, 2, [(2304, 256)]), (8, 8, [(300, 300)] * 6)))
    assert choice(32, 8, [(2048, 2048)] * 2) == (4, 8, 1, 0) and choice(14, 2, [(32768, 2048)])[3] == 0
    # beside answers
    assert shared(14, 2, [(2040, 2040)], 40) and not shared(14, 2, [(300, 300)] * 4, 40)
    for heads in ((14, 2), (12, 4), (64, 8), (16, 8), (8, 8)):
        for behind in range(0, 33000, 1100):
            for n in (2, 250, 2048):
                p = choice(*heads, [(behind + n, n)])
                assert p is None or (p[0] * p[1] >= heads[0] and (not p[3] or p[2] == 1))


# (heads, groups, [(context, queries)], order of the tile list, tokens a page, pages of the pool)
CASES = [(14, 2, [(2048, 2048)], None, 16, 0), (14, 2, [(47, 47), (89, 89), (169, 169), (322, 322), (611, 611)], None, 16, 0),
         (14, 2, [(2, 2)] * 70 + [(33, 33)] * 9 + [(129, 129), (700, 1), (1163, 1100)], "shuffled", 16, 0), (32, 8, [(128, 127), (257, 255), (640, 513)], None, 8, 0),
         (8, 8, [(1000, 999), (1100, 1000)], None, 64, 0), (26, 2, [(1280, 1025)], "backwards", 16, 0), (8, 8, [(20000, 2048)], None, 8, 0),
         (12, 4, [(2100, 2048), (2300, 2011)], None, 16, 0), (32, 8, [(1500, 1024), (700, 613), (65, 65)], None, 16, 0), (64, 8, [(385, 385)], None, 32, 0), (14, 2, [(2050, 1999)], None, 16, (1 << 32) // (2 * 16 * 128) + 700)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_shared_rows(case):
    nq, nkv, seqs, listed, page, pool = CASES[case]
    assert form(nq, nkv, seqs, page=page) == SHARED
    against_the_general_kernel(nq, nkv, seqs, listed, page, pool, seed=case)
