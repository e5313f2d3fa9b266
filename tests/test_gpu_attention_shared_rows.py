"""Prompt attention whose blocks of four waves share 64 rows and take 32 keys of a stage each: groups and lengths that end anywhere in a block, in
a stage and in a wave's keys, lists of more than a wave's entries and in any order, page tables that LDS does not hold, pools beyond 4 GB; and on
the host which steps take it."""
import ctypes

import pytest
import torch

from sprout_lm_amd import ops

DEV = "cuda"


def choice(nq, nkv, seqs, beside=0, page=16):
    tiles, walk = sum(-(-n // 32) for _, n in seqs if n > 1), ops.mean_tile_walk([n for _, n in seqs], [c for c, _ in seqs])
    out = (ctypes.c_int * 4)()
    longest = max(c for c, n in seqs if n > 1)
    return None if ops.library().sp_attention_rows_choice(64, page, nq, nkv, tiles, longest, walk, beside, out) else tuple(out)


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
         (64, 8, [(385, 385)], None, 32, 0), (14, 2, [(2050, 1999)], None, 16, (1 << 32) // (2 * 16 * 128) + 700)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_shared_rows(case):
    nq, nkv, seqs, listed, page, pool = CASES[case]
    assert (choice(nq, nkv, seqs, page=page) or (0, 0, 0, 0))[3] == 1
    g = torch.Generator(device=DEV).manual_seed(case)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = [-(-c // page) for c, _ in seqs]
    T, total = sum(n for _, n in seqs), sum(pages) + 3
    order = torch.randperm(total, device=DEV, generator=g).int() + max(0, pool - total)
    tables = torch.full((len(seqs), max(pages) + 1), -1, dtype=torch.int32, device=DEV)
    for i, n in enumerate(pages):
        tables[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    k, v = (torch.empty(max(pool, total), *shape, device=DEV, dtype=torch.bfloat16) for shape in ((nkv, page, 64), (nkv, 64, page)))
    # keys that stand far out, so that running maxima are moved late in a walk and waves' maxima lie far apart
    far = torch.where(torch.rand(total, 1, page, 1, device=DEV, generator=g) < 0.002, 8.0, 1.0)
    k[-total:], v[-total:] = (rand(total, nkv, page, 64) * far).bfloat16(), rand(total, nkv, 64, page).bfloat16()
    q = rand(T, nq * 64).bfloat16()

    def attention(kind, values):
        out = torch.full((T + 1, nq * 64), 7.0, dtype=torch.bfloat16, device=DEV)      # a row behind the last stays as it is
        batch = ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
        tiles, n = batch.lists["tiles_multi_32"]
        if kind == 0 and listed:
            by = torch.arange(n - 1, -1, -1) if listed == "backwards" else torch.randperm(n, generator=torch.Generator().manual_seed(7))
            batch.lists["tiles_multi_32"] = (tiles[by.to(DEV)].contiguous(), n)
        ops.attention(q, nq * 64, k, values, tables, batch, out[:T], nq, nkv, 64, None, 0.125, kind=kind)
        assert (out[T] == 7).all()
        return out[:T].double()

    got, want, size = attention(0, v), attention(1, v), attention(1, v.abs() if not pool else v.clone().abs_())
    # weights rounded to bfloat16 (2^-9 of each, on both sides of the quotient's numerator only) and both results rounded
    assert ((got - want).abs() <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6).all()
