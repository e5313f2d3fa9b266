"""The steps that a server of this engine runs, one case a kind of step.

A case is one step of a model with the weights and requests a server has at that moment: requests that have
answered for a while and bring one token each, prompts (whole, or a portion behind what is computed already) and
mixtures of both.  Sizes are those of the command line's presets, all layers; weights and tokens are random.
`run` takes the step through the model runner as the engine and the trace replay do: steps of one token a request
with `launch_decode`, the tokens of the step before read while this one computes, other steps with `step_recorded`
where it takes them and `step` where it does not.  Before each pass the step's own tokens are taken back
(`CacheManager.commit` with the earlier length), so that every pass computes the same step.  Its output is the
step's logits, which depend on every key and value that the step writes, in every layer.

Fields of a case: `preset`, `dtype`; `answers`: requests that bring one token, with contexts (that token counted)
from `low` to `high`, evenly spread over the logarithm; `prompts`: requests that bring `short` to `long` tokens
each, spread likewise, behind `behind` tokens computed before; the last token's logits are wanted of each.
"""
from __future__ import annotations

import math
import random

import torch

PAGE = 16                # tokens in a page of the cache
STEP = 2048              # most prompt tokens of one step


# ---------------------------------------------------------------------------------------------- the cases
def _case(preset, dtype="bfloat16", answers=0, low=0, high=0, prompts=0, short=0, long=0, behind=0):
    return {"preset": preset, "dtype": dtype, "answers": answers, "low": low, "high": high, "prompts": prompts,
            "short": short, "long": long, "behind": behind}


def listed() -> list[dict]:
    cases = {
        # one user's short question to the smallest model: launches and latency
        "answer 0.5b b1": _case("qwen2.5-0.5b", answers=1, low=79, high=79),
        # a small batch deep in its conversations: the benchmark's decode step
        "answer 0.5b b8": _case("qwen2.5-0.5b", answers=8, low=4096, high=4096),
        # a full server: many requests, no two as far as each other, a number that fills no power of two
        "answer 0.5b b45 ragged": _case("qwen2.5-0.5b", answers=45, low=190, high=4096),
        # the batch at a model of ordinary size
        "answer 7b b8": _case("qwen2.5-7b", answers=8, low=4096, high=4096),
        # one user of the largest model, the workload the reference publishes its figures for
        "answer 32b b1": _case("qwen2.5-32b", answers=1, low=63, high=63),
        # a prompt as the benchmark reads it, small and ordinary model
        "prompt 0.5b 2048": _case("qwen2.5-0.5b", prompts=1, short=2048, long=2048),
        "prompt 7b 2048": _case("qwen2.5-7b", prompts=1, short=2048, long=2048),
        # several chat prompts that arrived together, odd lengths
        "prompts 0.5b ragged": _case("qwen2.5-0.5b", prompts=5, short=47, long=611),
        # the end of a document of 32,768 tokens: attention over all that was read before
        "prompt 0.5b far": _case("qwen2.5-0.5b", prompts=1, short=2048, long=2048, behind=30720),
        # a batch that goes on answering while a new prompt is read beside it
        "answers and prompt 7b": _case("qwen2.5-7b", answers=8, low=1024, high=4096, prompts=1, short=256, long=256,
                                       behind=1024),
        # the float32 path, for users who need exact numbers: both directions
        "answer 0.5b b8 float32": _case("qwen2.5-0.5b", "float32", answers=8, low=4096, high=4096),
        "prompt 0.5b 2048 float32": _case("qwen2.5-0.5b", "float32", prompts=1, short=2048, long=2048),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1)) - 0.5 / high))))


def draw(rng) -> dict:
    """Another step of the same ranges: 1 to 64 answering requests (16 at 7B sizes and in float32) at contexts of 32
    to 4,096, up to 6 prompts of 24 to 2,048 tokens together, up to 30,720 tokens behind them, or both."""
    preset, dtype = rng.choice([("qwen2.5-0.5b", "bfloat16")] * 3 + [("qwen2.5-7b", "bfloat16")] * 2
                               + [("qwen2.5-0.5b", "float32")])
    small = preset == "qwen2.5-0.5b" and dtype == "bfloat16"
    kind = rng.choice(["answers", "prompts", "both"])
    answers = low = high = prompts = short = long = behind = 0
    if kind != "prompts":
        answers = _log_int(rng, 1, (64 if small else 16) if kind == "answers" else 16)
        high = _log_int(rng, 32, 4096)
        low = _log_int(rng, 16, high)
    if kind != "answers":
        prompts = rng.randint(1, 6) if kind == "prompts" else 1
        long = _log_int(rng, 24, (STEP if kind == "prompts" else 512) // prompts)
        short = _log_int(rng, min(24, long), long)
        behind = rng.choice([0, 0, _log_int(rng, 16, 30720 if small and prompts == 1 and kind == "prompts" else 2048)])
    return _case(preset, dtype, answers, low, high, prompts, short, long, behind)


def _spread(n, low, high):
    return [high] if n == 1 else [round(low * (high / low) ** (i / (n - 1))) for i in range(n)]


def _requests(case) -> list[tuple[int, int]]:
    """(tokens computed before the step, tokens of the step) of every request, in the order of the step."""
    return ([(n - 1, 1) for n in _spread(case["answers"], case["low"], case["high"])] if case["answers"] else []) \
        + ([(case["behind"], n) for n in _spread(case["prompts"], case["short"], case["long"])] if case["prompts"] else [])


# ---------------------------------------------------------------------------------------------- inputs
def _config(case) -> dict:
    from sprout_lm_amd.cli import PRESETS
    return dict(PRESETS[case["preset"]])


def _shapes(c) -> dict:
    """Tensor name -> (shape, mean, deviation): rows of unit size through every product, scores of a deviation of
    about 1.7, norm weights around 1."""
    H, I = c["hidden_size"], c["intermediate_size"]
    d = H // c["num_attention_heads"]
    q, kv = H, c["num_key_value_heads"] * d
    out = {"model.embed_tokens.weight": ((c["vocab_size"], H), 0.0, H ** -0.5)}
    for i in range(c["num_hidden_layers"]):
        b = f"model.layers.{i}."
        out[b + "input_layernorm.weight"] = ((H,), 1.0, 0.1)
        for name, rows, scale in (("q", q, 1.2), ("k", kv, 1.2), ("v", kv, 1.0)):
            out[f"{b}self_attn.{name}_proj.weight"] = ((rows, H), 0.0, scale * H ** -0.5)
            out[f"{b}self_attn.{name}_proj.bias"] = ((rows,), 0.0, 0.5)
        out[b + "self_attn.o_proj.weight"] = ((H, q), 0.0, q ** -0.5)
        out[b + "post_attention_layernorm.weight"] = ((H,), 1.0, 0.1)
        out[b + "mlp.gate_proj.weight"] = ((I, H), 0.0, H ** -0.5)
        out[b + "mlp.up_proj.weight"] = ((I, H), 0.0, H ** -0.5)
        out[b + "mlp.down_proj.weight"] = ((H, I), 0.0, I ** -0.5)
    out["model.norm.weight"] = ((H,), 1.0, 0.1)
    if not c["tie_word_embeddings"]:
        out["lm_head.weight"] = ((c["vocab_size"], H), 0.0, H ** -0.5)
    return out


def _weights(case, seed) -> dict:
    generator = torch.Generator(device="cuda").manual_seed(2 * seed)
    dtype = getattr(torch, case["dtype"])
    return {name: torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=generator)
            for name, (shape, mean, std) in _shapes(_config(case)).items()}


def _tokens(case, seed) -> list[list[int]]:
    """All tokens of every request, those of the step last."""
    rng, vocab = random.Random(2 * seed + 1), _config(case)["vocab_size"]
    return [[rng.randrange(vocab) for _ in range(before + new)] for before, new in _requests(case)]


def prepare(case, seed):
    """The model on the device, its cache pool, and the requests with everything before the step computed."""
    from sprout_lm_amd.engine.batch import StepEntry
    from sprout_lm_amd.engine.runner import ModelRunner
    from sprout_lm_amd.registry import build_model_plan, config_from_dict
    from sprout_lm_amd.sampling.params import SamplingParams
    plan = build_model_plan(config_from_dict(_config(case)))
    histories, sizes = _tokens(case, seed), _requests(case)
    runner = ModelRunner(plan, _weights(case, seed), getattr(torch, case["dtype"]), torch.device("cuda", torch.cuda.current_device()),
                         block_size=PAGE, num_blocks=sum(-(-(a + b) // PAGE) for a, b in sizes), max_sequences=len(sizes))
    requests = []
    for (before, new), tokens in zip(sizes, histories):
        seq = runner.cache.create()
        if not runner.cache.reserve(seq, before + new):
            raise RuntimeError("The pool is too small for the case's requests.")
        for start in range(0, before, STEP):
            runner.step([StepEntry(seq, tokens[start:min(before, start + STEP)], [])])
        requests.append((before, StepEntry(seq, tokens[before:], [new - 1])))
    greedy = SamplingParams(temperature=0.0, ignore_eos=True)
    return {"runner": runner, "requests": requests, "entries": [e for _, e in requests], "answering": case["prompts"] == 0,
            "params": [greedy] * len(requests), "counters": [before for before, _ in requests], "earlier": None}


def run(state):
    """One step; its float32 logits at the wanted places."""
    runner, entries = state["runner"], state["entries"]
    for before, entry in state["requests"]:
        runner.cache.commit(entry.seq, before)
    if state["answering"]:
        pending = runner.launch_decode(entries, state["params"], state["counters"])
        earlier, state["earlier"] = state["earlier"], pending
        if earlier is not None:
            runner.finish_decode(earlier)
        return pending.logits[:len(entries)]
    logits = runner.step_recorded(entries)
    return runner.step(entries) if logits is None else logits


# ---------------------------------------------------------------------------------------------- cost, bounds, truth
def work(case) -> dict:
    """Every weight the step uses read once (of the embedding only the step's rows, and all of it where it is the
    output matrix too), the earlier keys and values read once, the step's written, the logits written."""
    c, sizes = _config(case), _requests(case)
    element = 2 if case["dtype"] == "bfloat16" else 4
    H, I, V, L = c["hidden_size"], c["intermediate_size"], c["vocab_size"], c["num_hidden_layers"]
    kv = c["num_key_value_heads"] * (H // c["num_attention_heads"])
    layer = 2 * H * H + 2 * H * kv + 3 * H * I
    tokens, before = sum(n for _, n in sizes), sum(b for b, _ in sizes)
    pairs = sum(b * n + n * (n + 1) // 2 for b, n in sizes)
    elements = L * (layer + 2 * kv * (before + tokens)) + V * H + tokens * H
    return {"bytes": element * elements + 4 * len(sizes) * V,
            "flops": 2 * L * layer * tokens + 4 * L * H * pairs + 2 * len(sizes) * V * H}


def tolerance(case) -> dict:
    """About four times what was measured against `exact` and between two runs whose sums come in another order:
    bfloat16 0.3 to 0.6 % of the norm, no logit off by more than 2.6 % of their deviation; float32 0.7 to 1.5e-6."""
    return {"rel": 2e-2, "max": 1e-1} if case["dtype"] == "bfloat16" else {"rel": 1e-5, "max": 1e-4}


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight


def _turn(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend(q, k, v):
    """Causal attention of one request: q [tokens, heads, d], k and v [tokens, kv heads, d]."""
    n, heads, d = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    for h in range(k.shape[1]):
        keys, values = k[:, h].t().contiguous(), v[:, h].contiguous()
        for a in range(0, n, 512):
            b = min(n, a + 512)
            rows = q[a:b, h * group:(h + 1) * group].reshape(-1, d)            # token by token, the group's heads together
            scores = (rows @ keys[:, :b]).view(b - a, group, b) * d ** -0.5
            later = torch.arange(b, device=q.device)[None, :] > torch.arange(a, b, device=q.device)[:, None]
            scores.masked_fill_(later[:, None, :], -math.inf)
            out[a:b, h * group:(h + 1) * group] = (scores.softmax(-1).view(-1, b) @ values[:b]).view(b - a, group, d)
    return out


def exact(case, seed):
    """The logits of the same weights and tokens in 64 bits: every request's whole sequence, without a cache.  None
    where that is too much to compute."""
    c = _config(case)
    layer = 2 * c["hidden_size"] ** 2 + 3 * c["hidden_size"] * c["intermediate_size"]
    if 2 * c["num_hidden_layers"] * layer * sum(b + n for b, n in _requests(case)) > 5e14:
        return None
    heads, kv_heads, H = c["num_attention_heads"], c["num_key_value_heads"], c["hidden_size"]
    d, eps = H // heads, c["rms_norm_eps"]
    w = _weights(case, seed)
    get = lambda name: w[name].double()
    ids = [torch.tensor(t, device="cuda") for t in _tokens(case, seed)]
    ends = [0]
    for t in ids:
        ends.append(ends[-1] + len(t))
    x = w["model.embed_tokens.weight"][torch.cat(ids)].double()
    position = torch.cat([torch.arange(len(t), device="cuda", dtype=torch.float64) for t in ids])
    angle = position[:, None] * c["rope_theta"] ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    for i in range(c["num_hidden_layers"]):
        b = f"model.layers.{i}."
        normed = _rms(x, get(b + "input_layernorm.weight"), eps)
        q, k, v = (torch.addmm(get(f"{b}self_attn.{n}_proj.bias"), normed, get(f"{b}self_attn.{n}_proj.weight").t())
                   for n in "qkv")
        q, k = _turn(q.view(-1, heads, d), cos, sin), _turn(k.view(-1, kv_heads, d), cos, sin)
        v = v.view(-1, kv_heads, d)
        mixed = torch.cat([_attend(q[a:e], k[a:e], v[a:e]) for a, e in zip(ends, ends[1:])])
        x += mixed.view(-1, H) @ get(b + "self_attn.o_proj.weight").t()
        gate, up, down = (get(f"{b}mlp.{n}_proj.weight").t() for n in ("gate", "up", "down"))
        weight = get(b + "post_attention_layernorm.weight")
        for a in range(0, len(x), 4096):
            normed = _rms(x[a:a + 4096], weight, eps)
            x[a:a + 4096] += (torch.nn.functional.silu(normed @ gate) * (normed @ up)) @ down
    last = torch.tensor([e - 1 for e in ends[1:]], device="cuda")
    rows = _rms(x[last], get("model.norm.weight"), eps)
    head = w["model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"]
    return torch.cat([rows @ part.double().t() for part in head.split(16384)], -1)
