"""Steps that hold prompts and one-query sequences: one launch takes the blocks of both kinds and one their merges.  One-query sequences
have the same keys in the same order as in a step of their own, and the same results bit for bit; a prompt's keys may lie in fewer parts."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (query heads, key/value heads, head size, page): the blocks of one, two and four heads of a group
SHAPES = [(14, 2, 64, 16), (28, 4, 128, 16), (8, 4, 128, 32), (3, 3, 80, 8), (16, 16, 64, 16), (20, 1, 16, 8)]
# (context, queries): chunks of the one-query kernel from one to eighteen, an odd number of its blocks; prompts of one tile, of parts of the
# keys, of tiles in pairs
BATCHES = [[(1, 1), (1, 1), (1, 1), (2, 2)], [(300, 1), (33, 33), (4500, 1)], [(700, 1), (1500, 250), (257, 1), (129, 128)],
           [(90, 40), (4097, 70), (4096, 1)], [(2048, 2048), (513, 1), (31, 1)], [(1100, 1050), (255, 1)]]


def _run(q, k, v, tables, seqs, rows, nq, nkv, hd, options):
    from sprout_lm_amd import ops
    batch = ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
    out = torch.full((len(rows), nq * hd), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.attention(q[rows].contiguous(), nq * hd, k, v, tables, batch, out, nq, nkv, hd, options.get("window"), hd ** -0.5,
                  scores="capped" if "softcap" in options else "scaled_dot", softcap=options.get("softcap", 0.0))
    return out


@pytest.mark.parametrize("nq,nkv,hd,page", SHAPES)
@pytest.mark.parametrize("seqs", BATCHES)
@pytest.mark.parametrize("options", [{}, {"window": 200}, {"softcap": 3.0}])
def test_both_kinds_in_one_launch(nq, nkv, hd, page, seqs, options):
    gen = torch.Generator(device=DEV).manual_seed(nq * hd + len(seqs))
    pages = [-(-c // page) for c, _ in seqs]
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=gen).to(torch.bfloat16)
    k, v = rand(sum(pages), nkv, page, hd), rand(sum(pages), nkv, hd, page)
    order = torch.randperm(sum(pages), device=DEV, generator=gen).to(torch.int32)
    tables = torch.full((len(seqs), max(pages)), -1, dtype=torch.int32, device=DEV)
    starts, used = [], 0
    for i, n in enumerate(pages):
        tables[i, :n] = order[used:used + n]
        used += n
        starts.append(sum(m for _, m in seqs[:i]))
    q = rand(sum(n for _, n in seqs), nq * hd)
    got = _run(q, k, v, tables, seqs, list(range(len(q))), nq, nkv, hd, options)
    assert torch.isfinite(got.float()).all()
    for one in (True, False):
        mine = [i for i, (_, n) in enumerate(seqs) if (n == 1) == one]
        rows = [starts[i] + j for i in mine for j in range(seqs[i][1])]
        alone = _run(q, k, v, tables[mine].contiguous(), [seqs[i] for i in mine], rows, nq, nkv, hd, options)
        if one:
            assert torch.equal(got[rows], alone)
            continue
        # other parts, other maxima under the weights' rounding to bfloat16: a weight is off by 2^-9 of itself at most, the sum over keys of
        # random values by 2^-9 / sqrt(3) of its size, the result by its own rounding, on either side; one of 2,048 keys missing is 0.022
        a, b = (x.float().view(len(rows), nq, hd) for x in (got[rows], alone))
        assert ((a - b).norm(dim=-1) <= 2 ** -6 * b.norm(dim=-1)).all()
