"""Prompt attention whose blocks hold runs of rows of all heads of a key/value head: groups and lengths that end anywhere in a wave, a
block and a tile of the list, whole walks and parts, lists in any order, pools beyond 4 GB; and on the host which steps would take it, were there not the
blocks whose waves share their rows."""
import ctypes

import pytest

from sprout_lm_amd import ops
from tests.attention_rows_helpers import OWN, PARTS, against_the_general_kernel, form


def plan(nq, nkv, seqs, beside=0):
    """The launch on rows of their own, None where the kernels of other heads are the faster ones.  Whether it runs says `form`."""
    tiles, walk = sum(-(-n // 32) for _, n in seqs if n > 1), ops.mean_tile_walk([n for _, n in seqs], [c for c, _ in seqs])
    out = (ctypes.c_int * 3)()
    longest = max(c for c, n in seqs if n > 1)
    return None if ops.library().sp_attention_rows_plan(64, 16, nq, nkv, tiles, longest, walk, beside, out) else tuple(out)


def test_which_steps():
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")
    # either side of the lines: 0.70 and 1.20 of the other kernel's time; 0.86 and 1.13 with two heads a group
    assert plan(14, 2, [(8192, 640)]) == (7, 2, 8) and plan(14, 2, [(2048, 2048)]) is None
    assert plan(16, 8, [(10240, 2048)]) and plan(16, 8, [(4096, 2048)]) is None and plan(12, 12, [(32768, 2048)]) is None
    # beside answers a longer walk is asked for
    assert plan(14, 2, [(4096, 1000)]) and plan(14, 2, [(4096, 1000)], 40) is None and plan(14, 2, [(32768, 2048)], 40)
    # walks of less than 3,000 keys stay whole, and many of them are needed: 0.48, 0.97 and 1.43
    assert plan(32, 8, [(2048, 2048)] * 2) == (4, 8, 1) and plan(24, 2, [(2048, 2048)]) == (6, 4, 1) and plan(7, 1, [(2048, 2048)] * 2) is None
    assert all(form(*case[:3]) == case[3] for case in CASES)
    # few long walks among many short ones are what is cut; more than eight heads are sets of one size
    assert plan(64, 8, [(30000, 300)] + [(256, 256)] * 2)[2] > 4 and plan(26, 2, [(10240, 2048)])[:2] == (7, 4)
    for heads in ((14, 2), (12, 4), (64, 8), (16, 8)):
        for behind in range(0, 33000, 1100):
            for n in (2, 250, 2048):
                p = plan(*heads, [(behind + n, n)])
                assert p is None or (1 <= p[2] <= 32 and (p[2] == 1 or p[2] * 1024 <= behind + n + 127))


# (heads, groups, [(context, queries)], form, order of the tile list, pages of the pool): rows that end within a tile of 32, in a wave's first and
# in its last row, in a block's last; a head too many in the last set; one query a sequence between prompts; whole walks with three to eight heads a set
CASES = [(14, 2, [(6000, 1097)], PARTS, None, 0), (14, 2, [(9000, 293), (2500, 37), (300, 1), (4100, 256)], PARTS, None, 0),
         (6, 1, [(16500, 555), (16500, 171)], PARTS, None, 0), (26, 2, [(5000, 523)], PARTS, None, 0), (16, 8, [(9000, 1029)], PARTS, None, 0),
         (64, 8, [(800, 800), (801, 289)], OWN, None, 0), (14, 2, [(12000, 300), (7000, 301)], PARTS, "backwards", 0),
         (14, 2, [(12000, 300), (7000, 301)], PARTS, "shuffled", 0), (14, 2, [(9001, 600)], PARTS, None, (1 << 32) // (2 * 16 * 128) + 700),
         (32, 8, [(2047, 2011), (2048, 2048)], OWN, None, 0), (12, 4, [(2048, 2047), (2300, 2011), (2049, 2048)], OWN, "shuffled", 0),
         (40, 8, [(2041, 2041)], OWN, None, 0), (24, 2, [(2048, 2048), (2100, 1999)], OWN, None, 0), (14, 2, [(2500, 2489), (2048, 2011), (2222, 2221)], OWN, "backwards", 0),
         (24, 8, [(2300, 2011), (2100, 2048)], OWN, None, (1 << 32) // (8 * 16 * 128) + 700)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_runs_of_rows(case):
    nq, nkv, seqs, expected, listed, pool = CASES[case]
    assert plan(nq, nkv, seqs) is not None and form(nq, nkv, seqs) == expected
    against_the_general_kernel(nq, nkv, seqs, listed, pool=pool, seed=case)
