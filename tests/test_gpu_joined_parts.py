"""Products whose sum the next norm joins from parts of K: the parts and the joining norm (tests/test_gpu_owed_parts.py has steps of a model)."""
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
