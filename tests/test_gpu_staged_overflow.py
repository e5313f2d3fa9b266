"""Products that normalise their rows into LDS, where the last normed number of a row overflows: results are infinite, as the sums are, and no
zero past the end of K meets it."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _want(x, nw, w, dtype):
    """The sums in 64 bits of normed rows rounded to `dtype` (to infinity where they overflow)."""
    normed = (x * (x.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * nw.float()).to(dtype)
    assert torch.isinf(normed[:, -1].float()).all() and normed[:, :-1].isfinite().all()
    return normed.double() @ w.double().T


def _operands(T, N, K, dtype):
    gen = torch.Generator(device=DEV).manual_seed(T + K)
    x = torch.rand(T, K, device=DEV, generator=gen) + 0.5
    w = ((torch.rand(N, K, device=DEV, generator=gen) + 0.5) / K).to(dtype)      # positive: no infinity meets its opposite
    nw = torch.ones(K, device=DEV)
    x[:, -1], nw[-1] = 4.0, 3e38                                                 # 4 / 1.1 * 3e38 is beyond float32 and bfloat16
    return x, nw.to(dtype), w


@pytest.mark.parametrize("T", [4, 8, 40])
@pytest.mark.parametrize("K", [832, 896, 904, 1016])      # whole steps of 64 that four waves do not share evenly, and none
def test_rotated(T, K):
    from sprout_lm_amd import ops
    nq, nkv, hd = 4, 2, 64
    x, nw, w = _operands(T, (nq + 2 * nkv) * hd, K, torch.bfloat16)
    q = torch.empty(T, nq * hd, dtype=torch.bfloat16, device=DEV)
    k, v = (torch.zeros(4, nkv, *s, dtype=torch.bfloat16, device=DEV) for s in ((16, hd), (hd, 16)))
    slots = torch.arange(T, dtype=torch.int32, device=DEV)
    inv = torch.zeros(hd // 2, device=DEV)                                       # nothing is turned
    ops.qkv_rope_cache(w, None, q, torch.zeros(T, dtype=torch.int32, device=DEV), inv, hd, slots, k, v, nq, nkv, hd, residual=x, norm_weight=nw, eps=1e-6)
    want = _want(x, nw, w, torch.bfloat16)
    assert torch.isposinf(want).all()
    values = torch.stack([v[t // 16, :, :, t % 16] for t in range(T)])
    assert torch.isposinf(values.float()).all()


@pytest.mark.parametrize("T", [1, 8])
@pytest.mark.parametrize("K", [132, 900, 1020])
def test_float32(T, K):
    from sprout_lm_amd import ops
    I = 24
    x, nw, w = _operands(T, 2 * I, K, torch.float32)
    assert torch.isposinf(_want(x, nw, w, torch.float32)).all()
    out = torch.empty(T, I, device=DEV)
    assert ops.gate_up_silu_f32(w, x, out, activation="relu", norm_weight=nw, eps=1e-6)
    assert torch.isposinf(out).all()
