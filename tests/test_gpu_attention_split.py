"""float32 prompt attention on numbers in three bfloat16 parts (heads of 64), against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (heads, groups, tokens a page, [(context, queries)]): one part of the keys and several, some beyond a row's keys; groups of 1 to 8
# heads (waves without one, two sets); tiles and stages that end early; one-query sequences beside prompts; more page
# numbers than LDS holds
CASES = [(4, 4, 4, [(1, 1), (17, 17)]), (2, 1, 16, [(64, 64), (65, 1), (700, 33)]), (14, 2, 16, [(1000, 700), (40, 40), (4000, 1)]),
         (9, 3, 8, [(513, 513)]), (8, 1, 64, [(129, 129), (2047, 31)]), (5, 1, 32, [(300, 299)]),
         (2, 1, 4, [(9000, 40)]), (64, 16, 4, [(8700, 520)]), (14, 2, 16, [(2048, 2048)])]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_split_attention(case):
    from sprout_lm_amd import ops
    nq, nkv, page, seqs = CASES[case]
    g = torch.Generator(device=DEV).manual_seed(case)
    rand = lambda *shape: torch.randn(*shape, device=DEV, generator=g)
    pages = [-(-c // page) for c, _ in seqs]
    T, total = sum(n for _, n in seqs), sum(pages) + 3
    order = torch.randperm(total, device=DEV, generator=g).int()
    tables = torch.full((len(seqs), max(pages) + 1), -1, dtype=torch.int32, device=DEV)
    k, v, q = rand(total, nkv, page, 64), rand(total, nkv, 64, page), rand(T, nq * 64)
    k *= torch.where(torch.rand(total, 1, page, 1, device=DEV, generator=g) < 0.01, 8.0, 1.0)      # maxima that move late
    v *= torch.exp2(torch.randint(-20, 20, (1, nkv, 64, 1), device=DEV, generator=g).float())
    batch = lambda: ops.AttentionBatch.build([n for _, n in seqs], [c for c, _ in seqs], DEV)
    for i, n in enumerate(pages):
        tables[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    out = torch.full_like(q, float("nan"))
    ops.attention(q, nq * 64, k, v, tables, batch(), out, nq, nkv, 64, None, 0.125, kind=0)
    plain = torch.full_like(q, float("nan"))      # and the kernel on the vector units
    ops.attention(q, nq * 64, k, v, tables, batch(), plain, nq, nkv, 64, None, 0.125, kind=2)
    row, squares = 0, [0.0, 0.0]
    for i, (ctx, n) in enumerate(seqs):
        idx = tables[i, :pages[i]].long()
        keys = k[idx].permute(1, 0, 2, 3).reshape(nkv, -1, 64)[:, :ctx].double()
        values = v[idx].permute(1, 2, 0, 3).reshape(nkv, 64, -1)[:, :, :ctx].double()
        hidden = torch.arange(ctx, device=DEV)[None, :] > torch.arange(ctx - n, ctx, device=DEV)[:, None]
        for h in range(nq):
            x, kk, vv = q[row:row + n, 64 * h:64 * h + 64].double(), keys[h * nkv // nq], values[h * nkv // nq]
            s = (x @ kk.t() * 0.125).masked_fill(hidden, float("-inf"))
            weights = s.softmax(-1)
            want, size = weights @ vv.t(), weights @ vv.abs().t()
            # a score: three products of 2^-22 left out or unrepresented, 24 sums of sixteen products each, of the products' magnitudes;
            # it moves a weight twice (itself and the denominator); exponentials, weights and sums a few units of 2^-23, a chain of
            # ctx / 64 sums among them
            reach = (x.abs() @ kk.abs().t() * 0.125).masked_fill(hidden, 0.0).amax(-1, keepdim=True)
            limit = (2 * (3 * 2.0 ** -22 + 24 * 2.0 ** -24) * reach + 2.0 ** -19 + ctx / 64 * 2.0 ** -24) * size
            for j, got in enumerate((out, plain)):
                error = got[row:row + n, 64 * h:64 * h + 64].double() - want
                assert (error.abs() <= limit).all(), (case, i, h)
                squares[j] += float((error / size).square().sum())
        row += n
    # Those limits add every rounding up at its largest; over many numbers the parts' error is smaller than that of sums in float32
    # (0.44 to 0.95 of it here), a kernel that leaves the third parts out has 18 times as much: no more than the other kernel's, with
    # a quarter for the few hundred numbers of the smallest case's rows.
    assert squares[0] <= 1.25 ** 2 * squares[1], [(x / T / nq / 64) ** 0.5 for x in squares]


def test_the_error_of_the_sums_over_values_has_no_side():
    """The instruction's sums end below the true ones; odd rows' other sign takes that out of every mean over rows."""
    from sprout_lm_amd import ops
    nq, nkv, page, ctx, n = 4, 1, 16, 4096, 2048
    g = torch.Generator(device=DEV).manual_seed(3)
    q = 0.2 * torch.randn(n, nq * 64, device=DEV, generator=g)      # weights of one size: the values' sums carry the error
    k, v = (torch.randn(ctx // page, nkv, *s, device=DEV, generator=g) for s in ((page, 64), (64, page)))
    v += 2.0
    tables = torch.arange(ctx // page, device=DEV, dtype=torch.int32)[None].contiguous()
    out = torch.full_like(q, float("nan"))
    ops.attention(q, nq * 64, k, v, tables, ops.AttentionBatch.build([n], [ctx], DEV), out, nq, nkv, 64, None, 0.125)
    keys, values = k[:, 0].reshape(ctx, 64).double(), v[:, 0].permute(1, 0, 2).reshape(64, ctx).double()
    hidden = torch.arange(ctx, device=DEV)[None] > torch.arange(ctx - n, ctx, device=DEV)[:, None]
    s = (q.view(n, nq, 64).double() @ keys.t() * 0.125).masked_fill(hidden[:, None], float("-inf"))
    want = s.softmax(-1) @ values.t()
    error = (out.view(n, nq, 64).double() - want) / want
    even, odd = float(error[::2].mean()), float(error[1::2].mean())
    # Both kinds of rows share what the denominators' sums and the quotient are off by (5e-9 here); what the instruction drops, 1.1e-8,
    # lies on either side of it, so that the means have different signs.  With one sign for all rows they would agree within 7
    # deviations of a mean of as many independent errors.
    noise = 7 * float(error.square().mean().sqrt()) / (error.numel() / 2) ** 0.5
    assert abs(even - odd) > 2 * noise and abs(even + odd) < abs(even - odd), (even, odd, noise)


def prompt(seed, nq=4, nkv=2, ctx=600, n=40, page=16):
    """Queries, pools, tables and batch of one prompt's last n tokens; the rows of keys [nkv, ctx, 64] and values [nkv, 64, ctx] that
    `fill` writes into the pools."""
    from sprout_lm_amd import ops
    g = torch.Generator(device=DEV).manual_seed(seed)
    q, keys, values = (torch.randn(*s, device=DEV, generator=g) for s in ((n, nq * 64), (nkv, ctx, 64), (nkv, 64, ctx)))
    pages = -(-ctx // page)
    tables = torch.randperm(pages, device=DEV, generator=g).int()[None]

    def run(scale=0.125):
        k, v = torch.zeros(pages, nkv, page, 64, device=DEV), torch.zeros(pages, nkv, 64, page, device=DEV)
        pad = torch.zeros(nkv, pages * page - ctx, 64, device=DEV)
        k[tables[0].long()] = torch.cat([keys, pad], 1).view(nkv, pages, page, 64).permute(1, 0, 2, 3)
        v[tables[0].long()] = torch.cat([values, pad.transpose(1, 2)], 2).view(nkv, 64, pages, page).permute(2, 0, 1, 3)
        out = torch.full_like(q, float("nan"))
        ops.attention(q, nq * 64, k, v, tables, ops.AttentionBatch.build([n], [ctx], DEV), out, nq, nkv, 64, None, scale)
        return out.view(n, nq, 64).double()

    def want(scale=0.125):
        x, kk, vv = q.view(n, nq, 64).double(), keys.double().repeat_interleave(nq // nkv, 0), values.double().repeat_interleave(nq // nkv, 0)
        hidden = torch.arange(ctx, device=DEV)[None] > torch.arange(ctx - n, ctx, device=DEV)[:, None]
        # (a sum of products, number by number: an infinity times a zero is NaN here as there)
        scores = torch.stack([(x[i, :, None] * kk).sum(-1) for i in range(n)]) * scale
        weights = scores.masked_fill(hidden[:, None], float("-inf")).softmax(-1)
        return torch.stack([(weights[i, :, None] * vv).sum(-1) for i in range(n)])

    return q.view(n, nq, 64), keys, values, run, want


@pytest.mark.parametrize("scale", [0.0, -0.125, -2.0, 0.7])
def test_scales_that_are_not_positive(scale):
    q, keys, values, run, want = prompt(1)
    # a few units of 2^-23 of sums of unit numbers, of scores up to |scale| 64
    assert (run(scale) - want(scale)).abs().max() <= 1e-5 * max(1.0, abs(scale) * 8)


def test_numbers_that_are_not_finite_and_at_the_ends_of_the_range():
    inf = float("inf")
    top = 3.4e38      # more than bfloat16's largest number

    def check(change, seed, rel=1e-5):
        q, keys, values, run, want = prompt(seed)
        change(q, keys, values)
        got, ref = run(), want()
        assert torch.equal(got.isnan(), ref.isnan()), (change, (got.isnan() != ref.isnan()).nonzero()[:8])
        good = ref.isfinite()
        assert torch.equal(got[~good & ~ref.isnan()], ref[~good & ~ref.isnan()])
        # a few units of 2^-23 of sums of numbers of one size: against the largest result of the head's dimension
        error, size = ((x.where(good, torch.zeros(()).to(x))).abs().amax(0) for x in (got - ref, ref))
        assert (error <= rel * size).all(), (change, (error > rel * size).nonzero()[:8])
        return ref

    def keys_of_minus_infinity(q, keys, values):      # every score of them is minus infinity: they weigh nothing
        q[..., 3] = q[..., 3].abs() + 0.1
        keys[:, 5:300:7, 3] = -inf

    def one_infinite_key(q, keys, values):            # scores of both signs
        keys[1, 100, 9] = inf

    def infinite_values(q, keys, values):
        values[0, 7, 33], values[0, 8, 34], values[0, 8, 35], values[1, 9, 36] = inf, inf, -inf, -inf

    def queries(q, keys, values):
        q[3, 1, 5], q[7, 2, 0], q[9, 3, 63] = inf, float("nan"), -inf

    def nan_value(q, keys, values):
        values[1, 4, 400] = float("nan")

    def near_the_top(q, keys, values):
        values[:, 2] *= top / 2000      # (the sums before they are divided by the weights' have to stay in the range themselves)
        values[0, 2, 17] = top
        q[..., 4] *= 1e-38
        keys[:, 20:90, 4] = top

    def tiny(q, keys, values):
        values[:, 2] *= 2.0 ** -112
        values[0, 3] *= 2.0 ** -120

    def large_queries(q, keys, values):      # the keys' last bits are beyond their third parts
        q[..., 4] *= 2.0 ** 121
        keys[..., 4] *= 2.0 ** -124

    def tiny_queries(q, keys, values):
        q[..., 4] *= 2.0 ** -124
        keys[..., 4] *= 2.0 ** 121

    assert check(keys_of_minus_infinity, 2).isfinite().all()
    assert check(one_infinite_key, 3).isnan().any()
    assert check(infinite_values, 4).isinf().any()
    check(queries, 5)
    check(nan_value, 6)
    check(near_the_top, 7)
    check(tiny, 8)
    check(large_queries, 9)
    check(tiny_queries, 10)
