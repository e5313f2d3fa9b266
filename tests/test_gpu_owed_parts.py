"""Steps of a model whose accumulating products are left in parts for the next norm: the same step where every product is added at once.  Between
the layers stand a block that does not settle what is owed, a layer without a feed-forward, norms of another kind and a last norm of chosen rows."""
import pytest
import torch

from sprout_lm_amd import ops

pytestmark = pytest.mark.gpu
H, HEADS, KV, HD, INNER, VOCAB = 512, 8, 2, 64, 1536, 320


def _plan():
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
    plan = _plan()(last)
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
