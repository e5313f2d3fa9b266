"""What the tests of prompt attention for heads of 64 share: which kernel a step takes, and its result against the general kernel's."""
import ctypes

import torch

DEV = "cuda"
# forms of a launch: a wave's rows are its own (whole walks, or parts that a merge joins), a block's waves share theirs, the other kernels
OWN, PARTS, SHARED, OTHER = "own rows", "own rows, walks in parts", "shared rows", "other kernels"


def choice(nq, nkv, seqs, beside=0, page=16):
    """What sp_attention does with the prompts of [(context, queries)]: (heads of a set, sets, parts, whether waves share rows), or None."""
    from sprout_lm_amd import ops
    tiles, walk = sum(-(-n // 32) for _, n in seqs if n > 1), ops.mean_tile_walk([n for _, n in seqs], [c for c, _ in seqs])
    return choice_of(nq, nkv, tiles, max(c for c, n in seqs if n > 1), walk, beside, page)


def choice_of(nq, nkv, tiles, longest, walk, beside=0, page=16):
    """... with a list of `tiles` entries, the longest walk and the mean one."""
    from sprout_lm_amd import ops
    out = (ctypes.c_int * 4)()
    return None if ops.library().sp_attention_rows_choice(64, page, nq, nkv, tiles, longest, walk, beside, out) else tuple(out)


def form(*args, **kw):
    plan = choice(*args, **kw)
    return OTHER if plan is None else SHARED if plan[3] else PARTS if plan[2] > 1 else OWN


def against_the_general_kernel(nq, nkv, seqs, listed=None, page=16, pool=0, seed=0, same_pages=False):
    """Every row within what the roundings allow.  `listed`: the tile list backwards or shuffled; `pool`: pages of the pools at least, the used ones
    last; `same_pages`: sequences read the same pages."""
    from sprout_lm_amd import ops
    g = torch.Generator(device=DEV).manual_seed(seed)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = [-(-c // page) for c, _ in seqs]
    T, total = sum(n for _, n in seqs), (max(pages) if same_pages else sum(pages)) + 3
    order = (torch.randperm(total, device=DEV, generator=g).int() + max(0, pool - total)).cpu()
    tables = torch.full((len(seqs), max(pages) + 1), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        tables[i, :n] = order[at:at + n]
        at += 0 if same_pages else n
    tables = tables.to(DEV)
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
