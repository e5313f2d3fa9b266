"""Prompt attention whose blocks hold runs of rows of all heads of a key/value head: groups and lengths that end anywhere in a wave, a
block and a tile of the list, parts of the walk, lists in any order, pools beyond 4 GB; and on the host which steps take it."""
import ctypes

import pytest
import torch

from sprout_lm_amd import ops

DEV = "cuda"


def plan(nq, nkv, seqs, beside=0):
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
    # few long walks among many short ones are what is cut; more than eight heads are sets of one size
    assert plan(64, 8, [(30000, 300)] + [(256, 256)] * 2)[2] > 4 and plan(26, 2, [(10240, 2048)])[:2] == (7, 4)
    for heads in ((14, 2), (12, 4), (64, 8), (16, 8)):
        for behind in range(0, 33000, 1100):
            for n in (2, 250, 2048):
                p = plan(*heads, [(behind + n, n)])
                assert p is None or (1 <= p[2] <= 32 and (p[2] == 1 or p[2] * 1024 <= behind + n + 127))


# (heads, groups, [(context, queries)], order of the tile list, pages of the pool): rows that end within a tile of 32, in a wave's first and
# in its last row, in a block's last; a head too many in the last set; one query a sequence between prompts
CASES = [(14, 2, [(6000, 1097)], None, 0), (14, 2, [(9000, 293), (2500, 37), (300, 1), (4100, 256)], None, 0), (6, 1, [(16500, 555), (16500, 171)], None, 0),
         (26, 2, [(5000, 523)], None, 0), (12, 4, [(2100, 2048), (2300, 2011)], None, 0), (32, 8, [(1500, 1024), (700, 613), (65, 65)], None, 0),
         (16, 8, [(9000, 1029)], None, 0), (64, 8, [(800, 800), (801, 289)], None, 0), (14, 2, [(12000, 300), (7000, 301)], "backwards", 0),
         (14, 2, [(12000, 300), (7000, 301)], "shuffled", 0), (14, 2, [(9001, 600)], None, (1 << 32) // (2 * 16 * 128) + 700)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_runs_of_rows(case):
    nq, nkv, seqs, listed, pool = CASES[case]
    assert plan(nq, nkv, seqs) is not None
    page = 16
    g = torch.Generator(device=DEV).manual_seed(case)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = [-(-c // page) for c, _ in seqs]
    T, total = sum(n for _, n in seqs), sum(pages) + 3
    order = torch.randperm(total, device=DEV, generator=g).int() + max(0, pool - total)
    tables = torch.full((len(seqs), max(pages) + 1), -1, dtype=torch.int32, device=DEV)
    for i, n in enumerate(pages):
        tables[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    k, v = (torch.empty(max(pool, total), *shape, device=DEV, dtype=torch.bfloat16) for shape in ((nkv, page, 64), (nkv, 64, page)))
    # keys that stand far out, so that running maxima are moved late in a walk
    far = torch.where(torch.rand(total, 1, page, 1, device=DEV, generator=g) < 0.002, 8.0, 1.0)
    k[-total:], v[-total:] = (rand(total, nkv, page, 64) * far).bfloat16(), rand(total, nkv, 64, page).bfloat16()
    q = rand(T, nq * 64).bfloat16()

    def attention(kind, values):
        out = torch.full_like(q, float("nan"))
        batch = ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
        tiles, n = batch.lists["tiles_multi_32"]
        if kind == 0 and listed:
            by = torch.arange(n - 1, -1, -1) if listed == "backwards" else torch.randperm(n, generator=torch.Generator().manual_seed(7))
            batch.lists["tiles_multi_32"] = (tiles[by.to(DEV)].contiguous(), n)
        ops.attention(q, nq * 64, k, values, tables, batch, out, nq, nkv, 64, None, 0.125, kind=kind)
        return out.double()

    got, want, size = attention(0, v), attention(1, v), attention(1, v.abs() if not pool else v.clone().abs_())
    # weights rounded to bfloat16 (2^-9 of each, on both sides of the quotient's numerator only) and both results rounded
    assert ((got - want).abs() <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6).all()
