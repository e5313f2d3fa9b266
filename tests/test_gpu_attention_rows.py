"""Prompt attention of heads of 64 against the general kernel, in each form that its launch takes; keys, values and queries that are not finite."""
import pytest
import torch

from tests.attention_rows_helpers import OWN, PARTS, SHARED, form

pytestmark = pytest.mark.gpu
DEV = "cuda"


def attention(kind, q, k, v, tables, batch, nq, nkv, **options):
    from sprout_lm_amd import ops
    out = torch.full_like(q, float("nan"))
    ops.attention(q, nq * 64, k, v, tables, batch, out, nq, nkv, 64, None, 0.125, kind=kind, **options)
    return out.double()


# (heads, groups, tokens a page, [(context, queries)], form): whole walks and 14 to 32 parts of the keys, a part of which lies beyond some
# rows; groups of 4 to 8 and of 12 heads (two sets); queries in no whole tiles; walks that end
# in the first and in the last of a stage's steps; more page numbers than LDS holds
CASES = [(64, 8, 8, [(1024, 1024)], OWN), (48, 8, 32, [(700, 700), (331, 300), (33, 33), (9, 1)], SHARED), (24, 2, 64, [(2049, 2049)], SHARED),
         (14, 2, 16, [(4129, 2048)], SHARED), (14, 2, 16, [(4224, 2017), (2100, 31)], SHARED), (14, 2, 16, [(33001, 250)], PARTS),
         (7, 1, 8, [(16384, 1000), (200, 200)], PARTS), (64, 8, 8, [(33000, 2048)], OWN), (56, 8, 16, [(4096, 4096 - 2048), (130, 130)], OWN),
         # a one-query sequence whose parts are no whole number of sixteen bytes, before the prompt's in the workspace
         (7, 1, 16, [(700, 1), (16384, 1000)], PARTS),
         # whole walks with sizes like those that run on shared rows above
         (48, 8, 32, [(1700, 1700), (1331, 1300), (33, 33), (9, 1)], OWN), (24, 2, 64, [(2049, 2049), (2081, 2017)], OWN), (32, 8, 16, [(2129, 2048), (2100, 1931)], OWN)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_rows_attention(case):
    from sprout_lm_amd import ops
    nq, nkv, page, seqs, expected = CASES[case]
    assert form(nq, nkv, seqs, page=page) == expected
    g = torch.Generator(device=DEV).manual_seed(case)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = [-(-c // page) for c, _ in seqs]
    T, total = sum(n for _, n in seqs), sum(pages) + 3
    order = torch.randperm(total, device=DEV, generator=g).int()
    tables = torch.full((len(seqs), max(pages) + 1), -1, dtype=torch.int32, device=DEV)
    for i, n in enumerate(pages):
        tables[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    k, v = rand(total, nkv, page, 64), rand(total, nkv, 64, page)
    # keys that stand far out, so that running maxima are moved late in a walk
    k *= torch.where(torch.rand(total, 1, page, 1, device=DEV, generator=g) < 0.002, 8.0, 1.0)
    q, k, v = rand(T, nq * 64).bfloat16(), k.bfloat16(), v.bfloat16()
    batch = ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
    got = attention(0, q, k, v, tables, batch, nq, nkv)
    args = (q, k, v, tables, ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV), nq, nkv)
    want = attention(1, *args)
    size = attention(1, q, k, v.abs(), *args[3:])
    # weights rounded to bfloat16 (2^-9 of each, on both sides of the quotient's numerator only) and both results rounded
    assert ((got - want).abs() <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("nq,nkv,ctx,n,expected", [(14, 2, 4129, 2048, SHARED), (64, 8, 3340, 1100, OWN), (14, 2, 6000, 1097, PARTS)])
def test_keys_and_values_that_are_not_finite(nq, nkv, ctx, n, expected):
    """As the general kernel has it: a key whose score is minus infinity weighs nothing, an infinite value is one for every row that
    sees it, NaN stays with the rows and dimensions it reaches.  All before the first query, so that every row sees them."""
    from sprout_lm_amd import ops
    assert form(nq, nkv, [(ctx, n)]) == expected
    page, G = 16, nq // nkv
    inf = float("inf")
    g = torch.Generator(device=DEV).manual_seed(5)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = -(-ctx // page)
    k, v, q = rand(pages, nkv, page, 64), rand(pages, nkv, 64, page), rand(n, nq, 64)
    tables = torch.arange(pages, device=DEV, dtype=torch.int32)[None].contiguous()
    q[..., 3] = q[..., 3].abs() + 0.1
    k[5, :, 7, 3], k[40, 0, 0, 3] = -inf, -inf                  # scores of minus infinity
    v[9, 0, 11, 2], v[60, 1, 12, 15], v[61, 1, 12, 0] = inf, inf, -inf
    v[80, 1, 40, 8] = float("nan")
    q[100, 3, 9] = float("nan")
    q, k, v = q.view(n, -1).bfloat16(), k.bfloat16(), v.bfloat16()
    results = [attention(kind, q, k, v, tables, ops.AttentionBatch.build([n], [ctx], DEV), nq, nkv) for kind in (0, 1)]
    got, want = (x.view(n, nq, 64) for x in results)
    assert got[100, 3].isnan().all()      # (the general kernel's row of a query that is NaN has zeros)
    got[100, 3] = want[100, 3] = 0.0
    assert torch.equal(got.isnan(), want.isnan()) and want.isinf().sum() == G * n - 1
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    good = want.isfinite()
    assert good.float().mean() > 0.95
    # as above, of values of unit size
    assert ((got - want)[good].abs() <= 2.0 ** -8 * 4 + 2.0 ** -8 * want[good].abs()).all()


@pytest.mark.parametrize("nq,nkv,ctx,n,expected", [(14, 2, 4129, 2048, SHARED), (64, 8, 3340, 1100, OWN), (14, 2, 6000, 1097, PARTS)])
def test_a_key_with_most_of_the_weight(nq, nkv, ctx, n, expected):
    """A key behind the first 32 whose weight against their maximum is between 2^8 and 2^12, and lies between two numbers that bfloat16 holds: the running
    maximum has to follow it, so that it weighs 1."""
    assert form(nq, nkv, [(ctx, n)]) == expected
    page, first, at = 16, 32, 128 + 5
    bits = torch.arange(0x4000, 0x4200, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)      # 2 to 32
    scores = bits[(bits.double() > 5.6) & (bits.double() < 8.2)]
    weights = scores.double().exp()
    worst = ((weights.float().bfloat16().double() - weights) / weights).abs().argmax()
    b, weight = scores[worst], weights[worst]
    assert abs(float(weight.float().bfloat16()) - weight) > 0.0035 * weight
    g = torch.Generator(device=DEV).manual_seed(3)
    pages = -(-ctx // page)
    k, v = (torch.zeros(pages, nkv, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((page, 64), (64, page)))
    k[..., 0] = -30.0
    k[:first // page, ..., 0] = 0.0
    k[at // page, :, at % page, 0] = b.to(DEV)
    late = (1 + torch.rand(nkv, 64, device=DEV, generator=g)).bfloat16()
    v[at // page, :, :, at % page] = late
    q = torch.zeros(n, nq, 64, dtype=torch.bfloat16, device=DEV)
    q[..., 0] = 8.0                                   # times 0.125: a key's first number is its score
    tables = torch.arange(pages, device=DEV, dtype=torch.int32)[None].contiguous()
    from sprout_lm_amd import ops
    got = attention(0, q.view(n, -1), k, v, tables, ops.AttentionBatch.build([n], [ctx], DEV), nq, nkv).view(n, nkv, nq // nkv, 64)
    want = late.double() * float(weight) / (float(weight) + first)
    # the result is rounded to bfloat16 (2^-8 of it); the other keys' values are 0, their weights sum up in float32, or are e^-30
    assert ((got - want[None, :, None]).abs() <= 2.0 ** -8 * want[None, :, None] * 1.001).all()
