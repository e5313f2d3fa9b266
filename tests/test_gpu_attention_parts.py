"""Prompts whose keys are cut into parts, alone and beside one-query sequences, in one launch and in two, against the softmax in 64 bits.  Values at both
ends of every stage of 128 keys are eight times as large: one that a part's end leaves out or takes twice moves a row by a tenth of itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (query heads, key/value heads, head size, page): blocks of one, two and four heads on four and on eight waves
SHAPES = [(14, 2, 64, 16), (7, 1, 128, 16), (4, 2, 128, 32), (3, 3, 80, 8), (5, 1, 256, 16), (6, 1, 192, 16), (8, 4, 64, 8)]
# (context, queries): few tiles far behind, two prompts of different walks, walks of parts that no stage's end meets, many answers beside
BATCHES = [[(9000, 40)], [(4097, 70), (300, 1)], [(2500, 257), (33, 33), (700, 1), (1, 1)], [(6100, 2), (5000, 100)], [(1409, 129)] + [(640 + i, 1) for i in range(40)]]


@pytest.mark.parametrize("nq,nkv,hd,page", SHAPES)
@pytest.mark.parametrize("seqs", BATCHES)
@pytest.mark.parametrize("window", [None, 900])
def test_against_64_bits(nq, nkv, hd, page, seqs, window):
    from sprout_lm_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(nq * hd + len(seqs))
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    pages = [-(-c // page) for c, _ in seqs]
    width, total = max(pages), sum(pages)
    k, v = torch.zeros(total, nkv, page, hd, device=DEV, dtype=torch.bfloat16), torch.zeros(total, nkv, hd, page, device=DEV, dtype=torch.bfloat16)
    tables = torch.full((len(seqs), width), -1, dtype=torch.int32, device=DEV)
    order = torch.randperm(total, device=DEV, generator=gen)
    plain, used = [], 0
    for i, (c, _) in enumerate(seqs):
        mine = order[used:used + pages[i]]
        used += pages[i]
        tables[i, :pages[i]] = mine.to(torch.int32)
        keys, values = rand(pages[i] * page, nkv, hd).bfloat16(), rand(pages[i] * page, nkv, hd)
        place = torch.arange(len(values), device=DEV) % 128
        values[(place == 0) | (place == 127)] *= 8
        values = values.bfloat16()
        k[mine] = keys.view(-1, page, nkv, hd).transpose(1, 2)
        v[mine] = values.view(-1, page, nkv, hd).permute(0, 2, 3, 1)
        plain.append((keys[:c].double(), values[:c].double()))
    rows = sum(n for _, n in seqs)
    q = rand(rows, nq * hd).bfloat16()
    batch = ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
    out = torch.full((rows + 1, nq * hd), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.attention(q, nq * hd, k, v, tables, batch, out[:rows], nq, nkv, hd, window, hd ** -0.5)
    assert (out[rows] == 7).all()
    at = 0
    for (c, n), (keys, values) in zip(seqs, plain):
        position = torch.arange(c - n, c, device=DEV)[:, None]
        key = torch.arange(c, device=DEV)[None, :]
        hidden = (key > position) | (key <= position - window if window else torch.zeros_like(key, dtype=torch.bool))
        for h in range(nq):
            mine = q[at:at + n, h * hd:(h + 1) * hd].double()
            scores = (mine @ keys[:, h // (nq // nkv)].t().contiguous()) * hd ** -0.5
            want = scores.masked_fill(hidden, float("-inf")).softmax(-1) @ values[:, h // (nq // nkv)]
            got = out[at:at + n, h * hd:(h + 1) * hd].double()
            # weights and results are rounded to bfloat16: 2^-9 of each at most, of random sign over keys and columns
            assert ((got - want).norm(dim=-1) <= 2 ** -7 * want.norm(dim=-1)).all(), (c, n, h)
        at += n
