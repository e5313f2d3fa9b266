"""One-query attention of many sequences of different lengths: whichever block takes a chunk of the keys, each is taken once."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (sequences, longest context, heads, groups, head size, tokens a page): chunks that are a power of two and not, one chunk,
# sequences of one token beside the longest
@pytest.mark.parametrize("n,top,nq,nkv,hd,page", [(45, 4096, 14, 2, 64, 16), (20, 2900, 14, 2, 64, 16), (9, 900, 8, 2, 128, 12),
                                                  (33, 500, 28, 4, 128, 16), (70, 200, 4, 4, 64, 8), (3, 30000, 14, 2, 64, 16)])
def test_chunks_of_ragged_sequences(n, top, nq, nkv, hd, page):
    from sprout_lm_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n + top)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    lengths = [max(1, round(top ** (i / (n - 1)))) for i in range(n)]
    pages = [-(-c // page) for c in lengths]
    total = sum(pages) + 1
    order = torch.randperm(total, device=DEV, generator=g).int()
    tables = torch.full((n, max(pages)), -1, dtype=torch.int32, device=DEV)
    for i, c in enumerate(pages):
        tables[i, :c] = order[sum(pages[:i]):sum(pages[:i]) + c]
    k, v, q = (x.bfloat16() for x in (rand(total, nkv, page, hd), rand(total, nkv, hd, page), rand(n, nq * hd)))
    out = torch.full_like(q, float("nan"))
    ops.attention(q, nq * hd, k, v, tables, ops.AttentionBatch.build([1] * n, lengths, DEV), out, nq, nkv, hd, None, hd ** -0.5, kind=0)
    for i, c in enumerate(lengths):
        idx = tables[i, :pages[i]].long()
        keys = k[idx].permute(1, 0, 2, 3).reshape(nkv, -1, hd)[:, :c].double().repeat_interleave(nq // nkv, 0)
        values = v[idx].permute(1, 2, 0, 3).reshape(nkv, hd, -1)[:, :, :c].double().repeat_interleave(nq // nkv, 0)
        weights = ((keys * q[i].double().view(nq, 1, hd)).sum(-1) * hd ** -0.5).softmax(-1)[:, None]
        want, size = (weights * values).sum(-1), (weights * values.abs()).sum(-1)
        # the weights and the result rounded to bfloat16 (2^-9 of each), the rest float32
        assert ((out[i].double().view(nq, hd) - want).abs() <= 2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6).all(), i
