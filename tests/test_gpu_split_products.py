"""float32 products of many tokens as products of bfloat16 parts, against float64 products of the same numbers."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

# What the parts, the six products and the float32 sums may lose of a sum of K products, against the sum of their magnitudes: the
# products that are left out are 2^-25 together, the K / 16 sums of sixteen first parts' products round to 2^-24 of the running sum
# each (their errors add up in the worst case only), the sums of the others to 2^-32, and two more where they meet and pieces add.
def bound(K):
    return 2.0 ** -25 + (K / 16 + 2) * 2.0 ** -24 + 5 * K / 16 * 2.0 ** -32


def rows(T, K, seed, span=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(T, K, device=DEV, generator=g)
    if span:      # rows of very different sizes, and numbers of very different sizes within a row
        x *= torch.exp2(torch.randint(-span, span + 1, (T, 1), device=DEV, generator=g).float())
        x *= torch.exp2(torch.randint(-12, 1, (T, K), device=DEV, generator=g).float())
    return x.contiguous()


def scratch(n):
    return torch.empty(n, dtype=torch.uint8, device=DEV)


# one and several tiles of every block shape with remainders, one step and an odd number of steps of K, rows that a wave and that a
# block splits, K in one piece and in several (the last of them shorter), weights of more than a chunk
@pytest.mark.parametrize("T,N,K", [(256, 64, 64), (257, 1, 96), (300, 129, 896), (513, 4865, 160), (260, 896, 4864),
                                   (2048, 1152, 896), (1025, 2432, 2080), (2048, 9728, 96), (256, 70, 8256), (256, 9001, 8192), (2048, 5000, 5120)])
@pytest.mark.parametrize("kind", ["rows", "norm", "gate"])
def test_split_products(T, N, K, kind):
    from sprout_lm_amd import ops
    span = 40 if kind == "rows" else 0
    a, w = rows(T, 2 * K if kind == "gate" else K, T + N, span), rows(N, K, K, span)
    bias = torch.randn(N, device=DEV) if N != 1 else None
    weight = 1 + 0.1 * torch.randn(K, device=DEV)
    x = a.double()
    if kind == "norm":
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * weight.double()
    elif kind == "gate":
        x = torch.nn.functional.silu(x[:, :K]) * x[:, K:]
    want, size = x @ w.double().t(), x.abs() @ w.double().abs().t()
    # a norm's scale and a gate are float32 numbers themselves: a few units of their last place, of every product
    limit = (bound(K) + (0 if kind == "rows" else 2.0 ** -20)) * size + 2.0 ** -22 * (0 if bias is None else bias.double().abs())
    options = {"norm": {"norm": (weight, 1e-6)}, "gate": {"activation": "silu"}, "rows": {}}[kind]
    out = torch.full((T, N), float("nan"), device=DEV)
    assert ops.gemm_f32_split(a, w, out, scratch, bias=bias, **options)
    ref = want + (0 if bias is None else bias.double())
    assert ((out.double() - ref).abs() <= limit).all()
    if kind == "rows":
        base = torch.randn(T, N, device=DEV)
        acc = base.clone()
        assert ops.gemm_f32_split(a, w, acc, scratch, bias=None if bias is None else bias.bfloat16(), accumulate=True)
        ref = base.double() + want + (0 if bias is None else bias.bfloat16().double())
        assert ((acc.double() - ref).abs() <= limit + 2.0 ** -23 * (base.double().abs() + want.abs())).all()


def test_rows_of_zeros_and_numbers_that_are_not_finite():
    from sprout_lm_amd import ops
    a, w = rows(256, 96, 1), rows(70, 96, 2)
    a[3] = 0
    a[5, 7], a[9, 0], w[4, 95] = float("inf"), float("nan"), float("-inf")
    a[11] *= 2.0 ** 120
    a[12] *= 2.0 ** -120
    out, plain = torch.empty(256, 70, device=DEV), torch.empty(256, 70, device=DEV)
    assert ops.gemm_f32_split(a, w, out, scratch)
    ops.gemm(a, w, plain)
    assert torch.equal(out.isfinite(), plain.isfinite()) and not out[5].isfinite().any() and not out[9].isfinite().any()
    good = out.isfinite()
    assert (out[3][good[3]] == 0).all()
    size = (a.double().abs() @ w.double().abs().t())[good]
    assert ((out.double() - a.double() @ w.double().t())[good].abs() <= bound(96) * size).all()


def test_what_the_split_product_does_not_take():
    from sprout_lm_amd import ops
    out = lambda T, N: torch.empty(T, N, device=DEV)
    assert not ops.gemm_f32_split(rows(255, 96, 1), rows(8, 96, 2), out(255, 8), scratch)      # few tokens
    assert not ops.gemm_f32_split(rows(256, 100, 1), rows(8, 100, 2), out(256, 8), scratch)    # K in no whole steps of 32
    assert not ops.gemm_f32_split(rows(256, 96, 1).bfloat16(), rows(8, 96, 2), out(256, 8), scratch)
    shifted = torch.empty(256 * 96 + 1, device=DEV)[1:].view(256, 96)                          # operands off 16 bytes
    assert not ops.gemm_f32_split(shifted, rows(8, 96, 2), out(256, 8), scratch)


@pytest.mark.parametrize("K", [896, 4864])
def test_the_error_has_no_side(K):
    """The instruction's sums end below the true ones; odd rows' other sign takes that out of every mean."""
    from sprout_lm_amd import ops
    a, w, out = rows(2048, K, 3), rows(896, K, 4), torch.empty(2048, 896, device=DEV)
    assert ops.gemm_f32_split(a, w, out, scratch)
    want = a.double() @ w.double().t()
    error = (out.double() - want) / want.square().mean().sqrt()
    spread = float(error.square().mean().sqrt())
    # means of independent errors: 7 deviations over all, over the rows' and over the columns' means together
    assert abs(float(error.mean())) <= 7 * spread / (2048 * 896) ** 0.5
    assert float(error.mean(0).square().mean().sqrt()) <= 2 * spread / 2048 ** 0.5
    assert float(error.mean(1).square().mean().sqrt()) <= 2 * spread / 896 ** 0.5


def spread(x, w, out):
    """2-norm of the error over the 2-norm of the result, against 64 bits."""
    want = x.double() @ w.double().t()
    return float((out.double() - want).norm() / want.norm())


def both(x, w):
    """Errors of this product and of the float32 instruction's."""
    from sprout_lm_amd import ops
    out, plain = (torch.empty(x.shape[0], w.shape[0], device=DEV) for _ in range(2))
    assert ops.gemm_f32_split(x, w, out, scratch)
    ops.gemm(x, w, plain)
    return spread(x, w, out), spread(x, w, plain)


@pytest.mark.parametrize("power", [0, 18, 24, 40, 100])
@pytest.mark.parametrize("against", ["its inverse", "zero"])
def test_a_number_that_stands_far_out_of_its_row(power, against):
    """It meets a weight that takes it back, or none: the others must keep all their bits beside it."""
    x, w = rows(300, 896, 11), rows(200, 896, 12)
    x[:, 5] *= 2.0 ** power
    w[:, 5] *= 0.0 if against == "zero" else 2.0 ** -power
    got, plain = both(x, w)
    assert got <= plain
    x, w = rows(200, 896, 12), rows(300, 896, 11)      # and among the weights
    w[:, 5] *= 2.0 ** power
    x[:, 5] *= 0.0 if against == "zero" else 2.0 ** -power
    got, plain = both(x.repeat(2, 1), w)
    assert got <= plain


@pytest.mark.parametrize("count", [1, 2, 4, 8, 64])
def test_few_products_carry_the_result(count):
    """Weights with `count` numbers a row that are not zero: no worse than the float32 instruction, a quarter more for the spread of
    so few roundings."""
    x, w = rows(512, 896, 21), torch.zeros(1024, 896, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(22)
    at = torch.rand(1024, 896, device=DEV, generator=g).argsort(-1)[:, :count]
    w.scatter_(1, at, torch.randn(1024, count, device=DEV, generator=g))
    got, plain = both(x, w)
    assert got <= 1.25 * plain


@pytest.mark.parametrize("mode", ["store", "add"])
def test_infinities_stay_infinities(mode):
    from sprout_lm_amd import ops
    x, w = rows(300, 160, 31), rows(190, 160, 32)
    inf = float("inf")
    x[5, 7], x[9, 0], x[11, 3], x[11, 4], x[299, 159] = inf, float("nan"), inf, inf, -inf
    w[4, 95], w[189, 7], w[60, 30], w[61] = -inf, inf, float("nan"), 0.0
    out, plain = torch.ones(300, 190, device=DEV), torch.ones(300, 190, device=DEV)
    bias = torch.randn(190, device=DEV)
    assert ops.gemm_f32_split(x, w, out, scratch, bias=bias, accumulate=mode == "add")
    ops.gemm(x, w, plain, bias=bias, accumulate=mode == "add")
    assert torch.equal(out.isnan(), plain.isnan()), (out.isnan() != plain.isnan()).nonzero()[:8]
    assert plain.isinf().sum() > 300
    assert torch.equal(out[out.isinf()], plain[out.isinf()]) and torch.equal(out.isinf(), plain.isinf())


@pytest.mark.parametrize("T,N,K", [(300, 190, 160), (512, 512, 4864), (260, 130, 8256)])
def test_rows_with_a_nan_are_not_walked(T, N, K):
    """NaN whatever they meet, infinities beside them too, on either side and in any piece of K; and in the time of finite rows, where
    rows with an infinity are taken number by number (of all rows that would be 80 times the product itself)."""
    from sprout_lm_amd import ops
    x, w = rows(T, K, 41), rows(N, K, 42)
    out, plain = torch.empty(T, N, device=DEV), torch.empty(T, N, device=DEV)

    def best():
        times = []
        for _ in range(5):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            assert ops.gemm_f32_split(x, w, out, lambda n: kept)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    kept = scratch(ops.gemm_f32_split_bytes(T, N, K))
    finite = best()
    x[:, K - 1] = float("nan")
    x[7] = float("nan")
    x[9], w[3, 5] = 1.0, float("nan")
    with_nan = best()
    x[11, 0], w[4, 6] = float("inf"), float("-inf")
    assert ops.gemm_f32_split(x, w, out, scratch)
    ops.gemm(x, w, plain)
    assert torch.equal(out.isnan(), plain.isnan()) and plain.isnan().sum() == (T - 1) * N + 1
    good = ~plain.isnan()
    assert torch.equal(out[good].isinf(), plain[good].isinf())
    assert with_nan < 4 * finite + 0.2, (with_nan, finite)



def test_the_step_takes_no_tensor_that_it_does_not_use():
    """A gated feed-forward of 2,048 tokens at 0.5B sizes: the norm and the gate are folded, so that neither the normed rows nor the
    gated ones have a tensor; and what the whole of it takes is less than half as much again as rows and gate took before the parts."""
    from sprout_lm_amd import ops
    from sprout_lm_amd.engine.batch import StepContext, Workspace
    from sprout_lm_amd.parts.mlp import GatedMLP
    from sprout_lm_amd.parts.norm import RMSNorm
    T, H, I = 2048, 896, 4864
    assert ops.gemm_f32_split_pays(T, 2 * I, H) and ops.gemm_f32_split_pays(T, H, I)
    mlp, norm = GatedMLP(H, I), RMSNorm(H, 1e-6)
    gate, up, down = rows(I, H, 1), rows(I, H, 2), rows(H, I, 3)
    mlp.bind(dict(zip(mlp.names, (gate, up, down))))
    norm.bind({"weight": torch.ones(H, device=DEV)})
    ctx = StepContext(Workspace(torch.device(DEV)), torch.float32)
    residual = rows(T, H, 4)
    x = torch.nn.functional.rms_norm(residual.double(), (H,), eps=1e-6)
    want = residual.double() + (torch.nn.functional.silu(x @ gate.double().t()) * (x @ up.double().t())) @ down.double().t()
    assert mlp.forward_from_residual(ctx, norm, residual)
    assert float((residual.double() - want).norm() / want.norm()) < 2e-6
    held = {name for name, _ in ctx.workspace._flat}
    assert held == {"gate_up", "f32_split"}
    assert sum(t.numel() * t.element_size() for t in ctx.workspace._flat.values()) <= 1.5 * 4 * T * (3 * I + H)


@pytest.mark.parametrize("H,I,kv", [(896, 4864, 128), (3584, 18944, 512), (5120, 27648, 1024)])
def test_workspace_of_the_largest_steps(H, I, kv):
    """Split operands of a step of 2,048 tokens: 200 MB at most, whatever the sizes."""
    from sprout_lm_amd import ops
    assert max(ops.gemm_f32_split_bytes(2048, n, k) for n, k in ((2 * I, H), (H, I), (H + 2 * kv, H), (H, H))) <= 200e6


# a product for every block shape of the four-wave kernel, with tiles of tokens and rows that are not whole
@pytest.mark.parametrize("T,N,K", [(1025, 6001, 1920), (1300, 4098, 288), (321, 4098, 1920), (450, 4098, 64), (450, 2050, 96),
                                   (256, 33, 64), (513, 4097, 384)])
def test_every_block_shape(T, N, K):
    from sprout_lm_amd import ops
    a, w, bias = rows(T, K, T), rows(N, K, N), torch.randn(N, device=DEV)
    size = a.double().abs() @ w.double().abs().t()
    want = a.double() @ w.double().t() + bias.double()
    limit = bound(K) * size + 2.0 ** -22 * bias.double().abs()
    out = torch.full((T + 1, N), 7.0, device=DEV)
    assert ops.gemm_f32_split(a, w, out[:T], scratch, bias=bias)
    assert ((out[:T].double() - want).abs() <= limit).all() and (out[T] == 7).all()
    acc = torch.ones(T + 1, N, device=DEV)
    assert ops.gemm_f32_split(a, w, acc[:T], scratch, bias=bias, accumulate=True)
    assert ((acc[:T].double() - 1 - want).abs() <= limit + 2.0 ** -23 * (1 + want.abs())).all() and (acc[T] == 1).all()


# tiles with remainders of every pair of sixteen, every block shape's ends, weights of more than a chunk; sums that are not finite
# on either side of a gate
@pytest.mark.parametrize("T,N,K", [(256, 32, 64), (257, 96, 96), (300, 160, 896), (2048, 9728, 96), (1025, 2464, 2080), (321, 4128, 1920), (450, 2080, 96),
                                   (1300, 4128, 288), (600, 16384, 5120)])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "relu", "clamped_swish"])
def test_gates_in_the_product(T, N, K, activation):
    """The product of both halves is the plain one's, number by number, and so is what the gate makes of it."""
    from sprout_lm_amd import ops
    a, w, weight = rows(T, K, T + 1), (rows(N, K, N + 1) * K ** -0.5), 1 + 0.1 * torch.randn(K, device=DEV)
    both, want = torch.empty(T, N, device=DEV), torch.empty(T, N // 2, device=DEV)
    for options in ({"norm": (weight, 1e-6)}, {}):
        assert ops.gemm_f32_split(a, w, both, scratch, **options)
        ops.silu_mul(both, want, activation=activation, limit=7.0)
        out = torch.full((T + 1, N // 2), 7.0, device=DEV)
        assert ops.gemm_f32_split(a, w, out[:T], scratch, activation=activation, limit=7.0, gates=True, **options)
        # the gate's exponential and division, two float32 functions of a few units each, may be contracted differently
        assert ((out[:T] - want).abs() <= 2.0 ** -20 * want.abs()).all() and (out[T] == 7).all()


def test_gates_of_numbers_that_are_not_finite():
    from sprout_lm_amd import ops
    a, w = rows(300, 96, 1), rows(160, 96, 2)
    a[5, 7], a[9, 0], a[11, 3] = float("inf"), float("nan"), float("-inf")
    w[4, 95], w[80 + 4, 1], w[17, 2], w[80 + 40, 5], w[79, 0] = float("-inf"), float("inf"), float("nan"), float("inf"), float("inf")
    both, want, out = torch.empty(300, 160, device=DEV), torch.empty(300, 80, device=DEV), torch.empty(300, 80, device=DEV)
    for activation in ("silu", "relu", "clamped_swish"):
        assert ops.gemm_f32_split(a, w, both, scratch)
        ops.silu_mul(both, want, activation=activation, limit=7.0)
        assert ops.gemm_f32_split(a, w, out, scratch, activation=activation, limit=7.0, gates=True)
        good = want.isfinite()
        assert torch.equal(out.nan_to_num(nan=3.5, posinf=2.5, neginf=1.5)[~good], want.nan_to_num(nan=3.5, posinf=2.5, neginf=1.5)[~good])
        # a finite half that meets one that is not is summed again, in 64 bits
        assert ((out - want)[good].abs() <= 2.0 ** -18 * (1 + want[good].abs())).all()


@pytest.mark.parametrize("T,N,K,why", [(300, 48, 96, "a gate of no whole sixteens"), (300, 160, 5152, "K in two pieces"), (255, 160, 96, "few tokens")])
def test_gates_that_the_product_does_not_take(T, N, K, why):
    from sprout_lm_amd import ops
    a, w, out = rows(T, K, 1), rows(N, K, 2), torch.full((T, N // 2), 7.0, device=DEV)
    assert not ops.gemm_f32_split_gates(T, N, K), why
    assert not ops.gemm_f32_split(a, w, out, scratch, activation="silu", gates=True) and (out == 7).all()
    a, w, out = rows(300, 96, 1), rows(160, 96, 2), torch.full((300, 80), 7.0, device=DEV)
    assert not ops.gemm_f32_split(a, w, out, scratch, gates=True) and not ops.gemm_f32_split(a, w, out, scratch, activation="silu", gates=True, accumulate=True)
