"""Prompt attention of heads of 64 over pages that hold more keys than the kernel fetches at a time, and as few as it takes,
against the general kernel: walks that end within a run of 64 keys, in its first and in its last key, parts that begin within a page; on shared rows, on
rows of their own and on those with walks in parts."""
import pytest
import torch

from tests.attention_rows_helpers import OWN, PARTS, SHARED, form

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("page", [8, 64, 128, 256, 1024])
@pytest.mark.parametrize("seqs,expected", [([(4160, 2048)], SHARED), ([(4161, 2047)], SHARED), ([(16447, 1000), (300, 300)], PARTS), ([(33025, 513)], PARTS),
                                           ([(2305, 2048), (2111, 2047), (2240, 2001)], OWN)])
def test_rows_attention_over_pages(page, seqs, expected):
    from sprout_lm_amd import ops
    nq, nkv = 14, 2
    assert form(nq, nkv, seqs, page=page) == expected
    g = torch.Generator(device=DEV).manual_seed(page + seqs[0][0])
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = [-(-c // page) for c, _ in seqs]
    T, total = sum(n for _, n in seqs), sum(pages) + 2
    order = torch.randperm(total, device=DEV, generator=g).int()
    tables = torch.full((len(seqs), max(pages) + 1), -1, dtype=torch.int32, device=DEV)
    for i, n in enumerate(pages):
        tables[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    q, k, v = rand(T, nq * 64).bfloat16(), rand(total, nkv, page, 64).bfloat16(), rand(total, nkv, 64, page).bfloat16()

    def run(kind, values):
        out = torch.full_like(q, float("nan"))
        batch = ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
        ops.attention(q, nq * 64, k, values, tables, batch, out, nq, nkv, 64, None, 0.125, kind=kind)
        return out.double()

    got, want, size = run(0, v), run(1, v), run(1, v.abs())
    # weights rounded to bfloat16 (2^-9 of each, on both sides of the quotient's numerator only) and both results rounded
    assert ((got - want).abs() <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6).all()
