"""Attention of short contexts and the output projection in one launch: one to eight waves' keys, ragged batches, one key, pages of every kind,
groups of one and of sixteen heads, widths that end within a block's rows; windows, sinks, capped scores, blocks of positions; and which steps take it:
none that launches of its own give the same bits every time."""
import pytest
import torch

from sprout_lm_amd import ops
from tests.test_gpu_kernels import run_attention

DEV = "cuda"
SIZES = [(14, 2, 64, 16, 896), (3, 1, 32, 8, 100), (32, 32, 16, 16, 120), (8, 1, 64, 4, 17), (12, 4, 48, 12, 300), (32, 2, 16, 32, 65)]
# several sets of heads and a K that no product cuts: contexts of one chunk have launches of their own
WHOLE = [(4, 4, 16, 16, 264), (6, 2, 48, 12, 300), (4, 2, 64, 16, 896), (4, 2, 32, 16, 8192)]
CONTEXTS = [[1], [64], [65], [256], [79, 256, 1, 33], [257], [512], [511, 3, 300]]


def takes(hd, page, nq, nkv, contexts, hidden):
    return bool(ops.library().sp_attention_decode_project_takes(hd, page, nq, nkv, len(contexts), max(contexts), hidden))


def project_waves(hd, nq, nkv, contexts, hidden):
    """Waves of a block that takes attention and projection (0: launches of their own, or the merge that projects)."""
    return ops.library().sp_attention_project_waves(hd, nq, nkv, len(contexts), max(contexts), hidden)


def test_which_steps():
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")
    assert all(takes(hd, page, nq, nkv, c, hidden) for nq, nkv, hd, page, hidden in SIZES for c in CONTEXTS)
    # as many blocks as CUs, a set's columns, a head's size: beyond them contexts of one chunk have launches of their own
    assert takes(64, 16, 14, 2, [79] * 8, 896) and not takes(64, 16, 14, 2, [79] * 16, 896)
    for nq in range(1, 32):
        for nkv in [n for n in range(2, nq + 1) if nq % n == 0]:
            for hd in (16, 32, 48, 64):
                # (a part of K holds 256 numbers at least)
                assert nq * hd >= 512 or not any(takes(hd, 16, nq, nkv, [c] * n, w) for c in (1, 79, 256) for n in (1, 3, 8) for w in (16, 300, 896, 8192))
    assert all(takes(hd, page, nq, nkv, c, hidden) == (max(c) > 256 and hidden <= 2048) for nq, nkv, hd, page, hidden in WHOLE for c in CONTEXTS)
    # on eight waves, narrow models and many blocks: launches of their own took 0.92, 0.91, 0.92 and 0.84 of the time; 1.04, 1.05 and 1.15 of it
    assert not any(project_waves(*a) for a in ((64, 8, 8, [500] * 4, 512), (64, 8, 2, [500] * 16, 512), (64, 8, 4, [500] * 8, 512), (64, 8, 1, [500] * 32, 512)))
    assert all(project_waves(*a) == 8 for a in ((64, 12, 4, [500] * 5, 768), (64, 8, 8, [500] * 2, 512), (64, 8, 8, [300], 512), (32, 16, 2, [500] * 8, 256)))
    assert project_waves(64, 8, 8, [256] * 4, 512) == 4
    assert not takes(64, 16, 16, 1, [79], 896) and not takes(128, 16, 4, 2, [79], 896) and not takes(128, 16, 28, 4, [79], 3584)


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nkv,hd,page,hidden", SIZES)
@pytest.mark.parametrize("contexts", CONTEXTS)
@pytest.mark.parametrize("window", [None, 70])
def test_short_contexts(nq, nkv, hd, page, hidden, contexts, window):
    got, want = run_attention(torch.bfloat16, nq, nkv, hd, page, [(c, 1) for c in contexts], window=window, kind=0, seed=hidden, hidden=hidden)
    assert not (got != got).any()
    # weights and outputs of unit size rounded to bfloat16, a row of w_o of unit norm: as the steps of several chunks are tested
    assert abs(got - want).max() <= 2e-2 * (1 + abs(want).max())


@pytest.mark.gpu
@pytest.mark.parametrize("options", [{"sinks": True}, {"scores": "capped", "softcap": 3.0}, {"mask_chunk": 48}, {"sinks": True, "window": 50}])
@pytest.mark.parametrize("contexts", [[90, 7], [400]])
def test_score_stages(options, contexts):
    nq, nkv, hd, page, hidden = 14, 2, 64, 16, 896
    g = torch.Generator(device=DEV).manual_seed(len(contexts))
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    options = dict(options)
    window = options.pop("window", None)
    if options.get("sinks"):
        options["sinks"] = rand(nq)
    T, pages = len(contexts), [-(-c // page) for c in contexts]
    tables = torch.zeros(T, max(pages), dtype=torch.int32, device=DEV)
    for i, n in enumerate(pages):
        tables[i, :n] = torch.arange(sum(pages[:i]), sum(pages[:i]) + n, device=DEV)
    q, k, v = rand(T, nq * hd).bfloat16(), rand(sum(pages), nkv, page, hd).bfloat16(), rand(sum(pages), nkv, hd, page).bfloat16()
    w_o, before = (rand(hidden, nq * hd) * (nq * hd) ** -0.5).bfloat16(), rand(T, hidden)
    batch = lambda: ops.AttentionBatch.build([1] * T, contexts, DEV)
    residual, out = before.clone(), torch.full_like(q, float("nan"))
    assert ops.attention(q, nq * hd, k, v, tables, batch(), out, nq, nkv, hd, window, 0.125, project=(w_o, residual), **options)
    assert ops.attention(q, nq * hd, k, v, tables, batch(), out, nq, nkv, hd, window, 0.125, kind=1, **options) is False
    want = out.float() @ w_o.float().T
    # each of the 896 outputs is off by a rounding of at most 2^-8 of its size on either side, weighed by rows of w_o of unit norm
    assert ((residual - before) - want).abs().max() <= 2 * 2.0 ** -8 * (out.float().abs() @ w_o.float().abs().T).max()


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nkv,hd,page,hidden", WHOLE)
def test_steps_that_repeat_bit_for_bit(nq, nkv, hd, page, hidden):
    g = torch.Generator(device=DEV).manual_seed(hidden)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    contexts = [79, 256, 1]
    T, pages = len(contexts), -(-256 // page)
    q, k, v = rand(T, nq * hd).bfloat16(), rand(T * pages, nkv, page, hd).bfloat16(), rand(T * pages, nkv, hd, page).bfloat16()
    w_o, before = (rand(hidden, nq * hd) * (nq * hd) ** -0.5).bfloat16(), rand(T, hidden)
    tables = torch.arange(T * pages, device=DEV, dtype=torch.int32).view(T, pages)
    batch = ops.AttentionBatch.build([1] * T, contexts, DEV)

    def step():
        residual, out = before.clone(), torch.full_like(q, float("nan"))
        if not ops.attention(q, nq * hd, k, v, tables, batch, out, nq, nkv, hd, None, hd ** -0.5, project=(w_o, residual)):
            ops.gemm(out, w_o, residual, accumulate=True)
        return residual

    first = step()
    assert all(torch.equal(step(), first) for _ in range(40))


@pytest.mark.gpu
@pytest.mark.parametrize("contexts", [[79, 256, 200], [400, 300, 512]])
def test_keys_and_values_that_are_not_finite(contexts):
    """As attention and product in launches of their own have it: a key whose score is minus infinity weighs nothing, an infinite or undefined value is in
    every column of the rows that see it, and in no other sequence's."""
    nq, nkv, hd, page, hidden = 14, 2, 64, 16, 896
    inf = float("inf")
    g = torch.Generator(device=DEV).manual_seed(contexts[0])
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    T, pages = len(contexts), 32
    q, k, v = rand(T, nq, hd), rand(T * pages, nkv, page, hd), rand(T * pages, nkv, hd, page)
    q[..., 3] = q[..., 3].abs() + 0.1
    k[0, :, 0, 3], k[2, 0, 5, 3], k[pages + 15, 1, 15, 3] = -inf, -inf, -inf
    v[pages + 1, 0, 11, 2], v[pages + 12, 1, 12, 0] = inf, -inf         # the second sequence alone
    v[2 * pages + 3, 1, 40, 8] = float("nan")                           # the third
    q, k, v = q.view(T, -1).bfloat16(), k.bfloat16(), v.bfloat16()
    w_o, before = (rand(hidden, nq * hd) * (nq * hd) ** -0.5).bfloat16(), rand(T, hidden)
    tables = torch.arange(T * pages, device=DEV, dtype=torch.int32).view(T, pages)
    batch = lambda: ops.AttentionBatch.build([1] * T, contexts, DEV)
    folded, apart, out = before.clone(), before.clone(), torch.full_like(q, float("nan"))
    assert project_waves(hd, nq, nkv, contexts, hidden) == (4 if max(contexts) <= 256 else 8)
    assert ops.attention(q, nq * hd, k, v, tables, batch(), out, nq, nkv, hd, None, 0.125, project=(w_o, folded))
    assert ops.attention(q, nq * hd, k, v, tables, batch(), out, nq, nkv, hd, None, 0.125) is False
    ops.gemm(out, w_o, apart, accumulate=True)
    assert apart[0].isfinite().all() and not apart[1].isfinite().any() and apart[2].isnan().all()
    assert torch.equal(folded.isnan(), apart.isnan()) and torch.equal(folded[apart.isinf()], apart[apart.isinf()])
    # outputs of attention off by a rounding of at most 2^-8 of their size on either side, weighed by rows of w_o of unit norm
    assert (folded[0] - apart[0]).abs().max() <= 2 * 2.0 ** -8 * (out[0].float().abs() @ w_o.float().abs().T).max()
