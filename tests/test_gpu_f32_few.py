"""The float32 products of a decode step on either side of the rules that choose a block: rows normalised once into LDS (up to 8 tokens of K up to
1,024), eight waves on K, and what is left to the others; against float64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
# tokens at both ends of the staged rows and past them; K at the ends, in no whole sixteens, and past them
SIZES = [(T, K) for T in (1, 7, 8, 9) for K in (64, 132, 900, 1020, 1024, 1028)]


def _operands(T, N, K):
    gen = torch.Generator(device=DEV).manual_seed(T * 31 + N + K)
    x = 3 * torch.randn(T, K, device=DEV, generator=gen)
    w = torch.randn(N, K, device=DEV, generator=gen) * 2 / math.sqrt(K)
    nw = 0.5 + torch.rand(K, device=DEV, generator=gen)
    normed = x.double() / (x.double().square().mean(-1, keepdim=True) + 1e-6).sqrt() * nw.double()
    return x, w, nw, normed


def _close(got, want, K):      # float32 sums of K products, and a few roundings of the norm and the activation
    assert (got.double() - want).abs().max().item() <= 1e-5 * max(1, math.sqrt(K) / 8) * (1 + want.abs().max().item())


@pytest.mark.parametrize("T,K", SIZES)
@pytest.mark.parametrize("I", [5, 264])
def test_gated_with_norm(T, K, I):
    from sprout_lm_amd import ops
    x, w, nw, normed = _operands(T, 2 * I, K)
    out = torch.full((T + 1, I), 7.0, device=DEV)
    assert ops.gate_up_silu_f32(w, x, out[:T], norm_weight=nw, eps=1e-6)
    gate, up = normed @ w[:I].double().T, normed @ w[I:].double().T
    _close(out[:T], gate / (1 + (-gate).exp()) * up, K)
    assert (out[T] == 7).all()


@pytest.mark.parametrize("T,K", SIZES)
@pytest.mark.parametrize("nq,nkv,hd", [(3, 1, 32), (14, 2, 64)])      # blocks of eight waves where K is long enough, and many blocks
def test_rotated_with_norm(T, K, nq, nkv, hd):
    from sprout_lm_amd import ops
    N = (nq + 2 * nkv) * hd
    x, w, nw, normed = _operands(T, N, K)
    q = torch.full((T + 1, nq * hd), 7.0, device=DEV)
    k, v = torch.zeros(2, nkv, 8, hd, device=DEV), torch.zeros(2, nkv, hd, 8, device=DEV)
    positions = torch.arange(5, 5 + T, device=DEV, dtype=torch.int32)
    slots = torch.arange(T, device=DEV, dtype=torch.int32)
    inv = (1e4 ** (-torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)).float()
    assert ops.qkv_rope_cache_f32(w, None, x, q[:T], positions, inv, torch.zeros_like(inv), hd, slots, k, v, nq, nkv, hd, norm_weight=nw, eps=1e-6)
    want = (normed @ w.double().T).view(T, nq + 2 * nkv, hd)
    angle = positions.double()[:, None, None] * inv.double()
    a, b = want[..., :hd // 2], want[..., hd // 2:]
    turned = torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)
    _close(q[:T].view(T, nq, hd), turned[:, :nq], K)
    assert (q[T] == 7).all()
    for t in range(T):
        _close(k[t // 8, :, t % 8], turned[t, nq:nq + nkv], K)
        _close(v[t // 8, :, :, t % 8], want[t, nq + nkv:], K)


# up to 8 M weights eight waves, more of them four; heads of 65,536 rows and a short K eight; K of less steps than there are waves
@pytest.mark.parametrize("T", [1, 8, 16])
@pytest.mark.parametrize("N,K", [(20, 64), (896, 896), (904, 4864), (2504, 3200), (1000, 8004), (65540, 196), (65540, 2052)])
def test_plain(T, N, K):
    from sprout_lm_amd import ops
    x, w, _, _ = _operands(T, N, K)
    want = x.double() @ w.double().T
    out = torch.full((T + 1, N), 7.0, device=DEV)
    ops.gemm(x, w, out[:T])
    _close(out[:T], want, K)
    ops.gemm(x, w, out[:T], accumulate=True)
    _close(out[:T], 2 * want, K)
    assert (out[T] == 7).all()
