"""Products whose sum the next norm joins from parts of K: the parts, the joining norm, and steps of a model that take this way."""
import math

import pytest
import torch

from sprout_lm_amd import ops

DEV = "cuda"


@pytest.fixture(scope="module")
def built_library():
    try:
        return ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")


@pytest.mark.parametrize("tiles_t,tiles_n,parts", [(1, 1, 2), (2, 7, 3), (16, 7, 2), (10, 7, 4), (3, 19, 6), (1, 28, 12), (5, 5, 16)])
def test_every_block_has_a_tile_and_a_part_of_its_own(built_library, tiles_t, tiles_n, parts):
    import ctypes
    blocks = tiles_t * tiles_n * parts
    out = (ctypes.c_int * (3 * blocks))()
    assert built_library.sp_quad_part_tiles(tiles_t, tiles_n, parts, out) == 0
    triples = [tuple(out[3 * b:3 * b + 3]) for b in range(blocks)]
    assert sorted(triples) == [(t, n, p) for t in range(tiles_t) for n in range(tiles_n) for p in range(parts)]


def test_plan(built_library):
    """Parts only where they are taken and pay: more than 64 tokens (float32: 17 to 255), every part with steps of its own."""
    for dtype, step in ((torch.bfloat16, 64), (torch.float32, 32)):
        for T in (1, 16, 17, 64, 65, 100, 255, 256, 264, 1238, 2048, 8192):
            for N in (8, 12, 896, 1536, 3584, 5120, 8192, 8200):
                for K in (48, 64, 896, 3584, 4864, 18944):
                    parts = ops.gemm_parts_plan(dtype, T, N, K)
                    assert parts == 0 or (parts > 1 and K // step // parts >= 3 and N % 8 == 0 and N <= 8192), (dtype, T, N, K, parts)
                    assert parts == 0 or parts * T * N <= 1 << 25
                    assert parts == 0 or (64 < T if dtype == torch.bfloat16 else 16 < T < 256)
    assert ops.gemm_parts_plan(torch.bfloat16, 1238, 896, 4864) and ops.gemm_parts_plan(torch.bfloat16, 264, 3584, 18944)
    assert ops.gemm_parts_plan(torch.float32, 160, 896, 4864)


# edges of token tiles and weight tiles, few and many parts, K that its parts do not divide
SIZES = [(65, 896, 4864), (100, 896, 896), (129, 904, 4864), (160, 3584, 18944), (264, 3584, 3584), (511, 1536, 8960), (1238, 896, 4864),
         (2047, 888, 4864), (70, 8192, 5120), (200, 2056, 6080)]
F32_SIZES = [(17, 896, 4864), (64, 896, 896), (65, 904, 4864), (160, 896, 4864), (255, 3584, 3616)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,T,N,K", [(torch.bfloat16, *s) for s in SIZES] + [(torch.float32, *s) for s in F32_SIZES])
def test_parts_add_up(dtype, T, N, K):
    parts = ops.gemm_parts_plan(dtype, T, N, K)
    assert parts > 1
    gen = torch.Generator(device=DEV).manual_seed(T + N)
    x = torch.randn(T, K, device=DEV, generator=gen).to(dtype)
    w = (torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).to(dtype)
    room = torch.full((parts + 1, T, N), 7.0, device=DEV)
    ops.gemm_parts(x, w, room[:parts])
    want = x.double() @ w.double().T
    got = room[:parts].double().sum(0)
    # float32 sums of K products of unit variance in all, in parts: an error of a rounding of the running sum a step of the sum
    assert (got - want).abs().max().item() <= 2e-5 * max(1.0, math.sqrt(K) / 8) * (1 + want.abs().max().item())
    assert (room[parts] == 7).all()
    again = torch.empty_like(room[:parts])
    ops.gemm_parts(x, w, again)
    assert torch.equal(again, room[:parts])                       # nobody adds to another's sum


@pytest.mark.gpu
@pytest.mark.parametrize("H", [8, 896, 1024, 1032, 2056, 3584, 8192])
@pytest.mark.parametrize("parts,T", [(1, 1), (2, 5), (3, 300), (4, 64), (9, 33)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_joining_norm(H, parts, T, dtype):
    gen = torch.Generator(device=DEV).manual_seed(H + T)
    x = torch.randn(T, H, device=DEV, generator=gen)
    owed = torch.randn(parts, T, H, device=DEV, generator=gen)
    weight = (1 + 0.1 * torch.randn(H, device=DEV, generator=gen)).to(dtype)
    total = owed[0].clone()
    for p in owed[1:]:
        total += p
    want = x + total                                              # the same roundings in the same order
    norm = torch.empty(T, H, dtype=dtype, device=DEV)
    ops.rmsnorm(want, weight, 1e-6, norm)
    rows = torch.tensor([T - 1, 0], dtype=torch.int32, device=DEV)
    picked, kept = torch.empty(2, H, dtype=dtype, device=DEV), x.clone()
    ops.rmsnorm_join(kept, owed, weight, 1e-6, picked, rows)
    assert torch.equal(kept, x) and torch.equal(picked, norm[rows.long()])
    joined, out = x.clone(), torch.empty_like(norm)
    ops.rmsnorm_join(joined, owed, weight, 1e-6, out)
    assert torch.equal(joined, want) and torch.equal(out, norm)
    ops.join(x, owed)
    assert torch.equal(x, want)


def test_a_subclass_does_not_inherit_the_claim():
    """A class derived from a part that leaves its sums to the next norm may read the residual after them: it is not taken that way."""
    from sprout_lm_amd.parts.base import claims
    from sprout_lm_amd.parts.attention import Attention
    from sprout_lm_amd.parts.block import PreNormBlock
    from sprout_lm_amd.parts.mlp import GatedMLP
    for base, name in ((Attention, "adds_last"), (GatedMLP, "adds_last"), (PreNormBlock, "settles")):
        derived = type("Derived", (base,), {})
        claimed = type("Claimed", (base,), {name: True})
        assert [claims(c.__new__(c), name) for c in (base, derived, claimed)] == [True, False, True]


@pytest.mark.gpu
def test_a_norm_with_numbers_of_its_own_joins_first():
    from sprout_lm_amd.engine.batch import StepContext, Workspace
    from sprout_lm_amd.parts.norm import RMSNorm

    class OnePlus(RMSNorm):
        def forward(self, ctx, x, out, rows=None):
            ops.rmsnorm(x, 1 + self.weight, self.eps, out, rows)
            return out

    x, owed, weight = torch.randn(5, 64, device=DEV), torch.randn(2, 5, 64, device=DEV), torch.randn(64, device=DEV)
    want, out = torch.empty(5, 64, device=DEV), torch.empty(5, 64, device=DEV)
    ops.rmsnorm(x + (owed[0] + owed[1]), 1 + weight, 1e-6, want)
    norm, ctx = OnePlus(64, 1e-6), StepContext(Workspace(torch.device(DEV)), torch.float32)
    norm.bind({"weight": weight})
    ctx.owed = owed
    norm.forward_joining(ctx, x, out)
    assert torch.equal(out, want) and ctx.owed is None


# A step of a model whose accumulating products are left in parts for the next norm, against the same step where every product is added at once.
# Between the layers stand a block that does not settle what is owed, a layer without a feed-forward, norms of another kind and a last norm of chosen rows.
H, HEADS, KV, HD, INNER, VOCAB = 512, 8, 2, 64, 1536, 320


def _toy_plan():
    from sprout_lm_amd.models.plan import LayerCall, LayerPlan, ModelPlan, PartPlan

    def layer(i, block, norm, ffn=True):
        base = f"l{i}."
        norms = lambda name: PartPlan("norm", norm, {"size": H, "eps": 1e-6}, f"{base}{name}.")
        parts = {"mixer_norm": norms("na"),
                 "mixer": PartPlan("mixer", "attention", {"hidden": H, "heads": HEADS, "kv_heads": KV, "head_dim": HD, "qkv_bias": False,
                                                          "position": PartPlan("position", "rotary_neox", {"head_dim": HD, "theta": 1e4})}, base)}
        if ffn:
            parts["ffn_norm"] = norms("nb")
            parts["ffn"] = PartPlan("feed_forward", "gated_mlp", {"hidden": H, "inner": INNER}, base)
        return LayerPlan(block, parts)

    layers = [layer(0, "pre_norm", "rmsnorm"), layer(1, "pre_norm", "rmsnorm", ffn=False), layer(2, "parallel", "rmsnorm"),
              layer(3, "pre_norm", "layernorm"), layer(4, "pre_norm", "rmsnorm", ffn=False), layer(5, "parallel", "layernorm"),
              layer(6, "pre_norm", "rmsnorm")]
    return lambda last: ModelPlan("ToyOwedForCausalLM", None, H, VOCAB, 4096, (0,), PartPlan("embedding", "token_embedding", {"vocab": VOCAB, "hidden": H}, "e."),
                                  layers, [LayerCall(i, i) for i in range(len(layers))], PartPlan("norm", last, {"size": H, "eps": 1e-6}, "n."),
                                  PartPlan("head", "linear_head", {"vocab": VOCAB, "hidden": H, "tied": False}, "h."))


@pytest.mark.gpu
@pytest.mark.parametrize("last", ["rmsnorm", "layernorm"])
@pytest.mark.parametrize("dtype,tokens,bound", [(torch.bfloat16, (100,), 2e-2), (torch.bfloat16, (33, 60), 2e-2), (torch.float32, (64,), 1e-5),
                                                (torch.float32, (1, 100, 2), 1e-5)])
def test_a_step_with_products_in_parts(monkeypatch, last, dtype, tokens, bound):
    from sprout_lm_amd.engine.batch import StepEntry
    from sprout_lm_amd.engine.runner import ModelRunner
    from sprout_lm_amd.weights.random_init import random_tensors
    T, device = sum(tokens), torch.device("cuda", torch.cuda.current_device())
    taken = {"gemm_parts": 0, "rmsnorm_join": 0, "join": 0}
    for name in taken:
        def counted(*args, _inner=getattr(ops, name), _name=name, **kw):
            taken[_name] += 1
            return _inner(*args, **kw)
        monkeypatch.setattr(ops, name, counted)
    sure = {k: ops.gemm_parts_plan(dtype, T, H, k) > 1 for k in (H, INNER)}
    assert sure[INNER], "sizes at which nothing is left in parts"
    plan = _toy_plan()(last)
    ids = [[(7 * i + 3 * s) % VOCAB for i in range(n)] for s, n in enumerate(tokens)]

    def logits():
        runner = ModelRunner(plan, random_tensors(plan.expected_tensors(), 5, dtype=dtype, device=device), dtype, device, block_size=16, num_blocks=32,
                             max_sequences=len(tokens), use_graphs=False)
        out = []
        for _ in range(2):
            entries = []
            for row in ids:
                seq = runner.cache.create()
                assert runner.cache.reserve(seq, len(row))
                entries.append(StepEntry(seq, row, sorted({0, len(row) // 2, len(row) - 1})))
            out.append(runner.step(entries).clone())
            for e in entries:
                runner.cache.release(e.seq)
        return out

    with_parts = logits()
    # the gated layers' last products at least, each joined once: before a block that does not settle and by norms of other kinds as a sum
    # alone, by the others on their way
    assert taken["gemm_parts"] >= 2 * 3 and taken["rmsnorm_join"] + taken["join"] == taken["gemm_parts"] and taken["join"] >= 2 and taken["rmsnorm_join"] >= 2
    before = dict(taken)
    monkeypatch.setattr(ops, "gemm_parts_plan", lambda *a: 0)
    at_once = logits()
    assert taken == before
    for got in with_parts:
        assert (got - at_once[0]).norm() <= bound * at_once[0].norm()      # roundings; one part of one product left out changes it by 7 to 97 %
