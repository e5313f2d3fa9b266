"""The tiled product on four waves a block: a size for every block shape and epilogue, edges of tiles of tokens and of rows, as few
steps along K as the ring has buffers and fewer, K split over blocks; against float32 products of the same bfloat16 operands."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

STORE, ACCUMULATE, GATED = 0, 1, 2          # the kinds of sp_quad_plan
_STORED = [(65, 8, 64), (65, 72, 128), (66, 264, 192), (97, 131 * 8, 256), (65, 20000, 64), (65, 13608, 1920), (193, 26664, 64), (97, 26664, 192),
           (193, 20000, 1920), (321, 20000, 1920), (777, 9736, 64), (777, 20000, 896), (130, 20000, 1920), (513, 13608, 192), (513, 20000, 384),
           (193, 26664, 1920), (2047, 4904, 384), (641, 20000, 896), (1300, 9736, 576), (289, 26664, 192)]
_STORED_FEW = [(17, 6152, 2048), (33, 2056, 1536), (64, 40000, 896), (45, 4104, 896)]
# a split of K in two and more on every shape but the largest
_SPLIT = [(65, 8, 576), (65, 9736, 1920), (65, 4904, 4864), (97, 9736, 3584), (193, 9736, 4864), (130, 20000, 3584), (777, 4904, 4864),
          (130, 9736, 4864), (161, 20000, 4864), (257, 13608, 4864), (17, 3592, 3584), (45, 904, 4864), (64, 2568, 5120),
          (835, 2312, 5696), (434, 2592, 7680), (769, 2592, 7488), (1366, 3280, 7168), (1490, 1440, 5824), (1385, 3080, 6528)]
_GATED = [(65, 16, 64), (66, 528, 128), (65, 19472, 64), (65, 14400, 1920), (97, 40000, 64), (97, 19472, 256), (193, 19472, 1920), (321, 19472, 1920),
          (130, 40000, 64), (130, 53328, 192), (130, 19472, 1920), (161, 40000, 192), (321, 27216, 384), (193, 27216, 1920), (193, 40000, 384),
          (193, 53328, 896), (777, 14400, 576), (289, 27216, 192), (17, 9728, 896), (45, 9760, 896), (64, 17920, 1536)]
SIZES = {STORE: _STORED + _STORED_FEW, ACCUMULATE: _STORED + _SPLIT, GATED: _GATED}
ROTATING_SIZES = [(65, 1, 1, 64, 64), (193, 56, 8, 128, 64), (321, 56, 8, 64, 1920), (2047, 8, 8, 128, 64), (289, 64, 8, 128, 320),
                  (777, 56, 8, 128, 1920), (777, 64, 8, 128, 256), (513, 64, 8, 128, 1088), (2047, 64, 8, 64, 384), (2047, 8, 8, 128, 1920),
                  (1238, 64, 8, 128, 896), (2047, 28, 4, 128, 320), (70, 2, 1, 192, 128)]


def _operands(T, N, K):
    gen = torch.Generator(device=DEV).manual_seed(T * 7 + N)
    x = torch.randn(T, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).to(torch.bfloat16)
    return x, w, torch.randn(N, device=DEV, generator=gen), x.float() @ w.float().T


@pytest.mark.parametrize("T,N,K", _STORED + _STORED_FEW)
def test_store(T, N, K):
    from sprout_lm_amd import ops
    x, w, bias, want = _operands(T, N, K)
    for b in (None, bias, bias.to(torch.bfloat16)):
        full = want if b is None else want + b.float()
        out = torch.full((T + 1, N), 7.0, dtype=torch.bfloat16, device=DEV)        # a row behind the last stays as it is
        ops.gemm(x, w, out[:T], bias=b)
        # rounding to bfloat16 is half a unit of eight bits
        assert (out[:T].float() - full).abs().max().item() <= 2 ** -8 * (1 + full.abs().max().item())
        assert (out[T] == 7).all()
        out32 = torch.full((T + 1, N), 7.0, device=DEV)
        ops.gemm(x, w, out32[:T], bias=b)
        assert (out32[:T] - full).abs().max().item() <= 2e-5 * max(1.0, math.sqrt(K) / 8) * (1 + full.abs().max().item())
        assert (out32[T] == 7).all()


@pytest.mark.parametrize("T,N,K", _STORED + _SPLIT)
def test_accumulate(T, N, K):
    from sprout_lm_amd import ops
    x, w, bias, want = _operands(T, N, K)
    for b in (None, bias, bias.to(torch.bfloat16)):
        before = torch.randn(T + 1, N, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3))
        out = before.clone()
        ops.gemm(x, w, out[:T], bias=b, accumulate=True)
        full = before[:T] + (want if b is None else want + b.float())
        assert (out[:T] - full).abs().max().item() <= 2e-5 * max(1.0, math.sqrt(K) / 8) * (1 + full.abs().max().item())
        assert torch.equal(out[T], before[T])


@pytest.mark.parametrize("T,N,K", [(2048, 3584, 18944), (2048, 1536, 8960), (200, 896, 896), (512, 3584, 3584)])
def test_sums_in_one_part_repeat_bit_for_bit(T, N, K):
    from sprout_lm_amd import ops
    assert ops.quad_plan(ops.PLAN_ACCUMULATE, T, N, K)[2] == 1
    x, w, _, _ = _operands(T, N, K)
    before = torch.randn(T, N, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3))
    runs = [before.clone() for _ in range(4)]
    for out in runs:
        ops.gemm(x, w, out, accumulate=True)
    assert all(torch.equal(runs[0], out) for out in runs[1:])


@pytest.mark.parametrize("T,N,K", _GATED)
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gated(T, N, K, activation):
    from sprout_lm_amd import ops
    x, w, _, want = _operands(T, N, K)
    I = N // 2
    g, u = want.to(torch.bfloat16).float().split(I, 1)
    full = (torch.nn.functional.silu(g) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")) * u
    out = torch.full((T + 1, I), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.gate_up_silu(w, out[:T], x=x, activation=activation)
    # gate and up are rounded to bfloat16 where float32 sums in another order may round to the other side: a unit of eight bits of
    # either factor, and half of one of the result
    assert (out[:T].float() - full).abs().max().item() <= 2 ** -6 * (1 + full.abs().max().item())
    assert ((out[:T].float() - full).norm() / full.norm()).item() <= 4e-3
    assert (out[T] == 7).all()


@pytest.mark.parametrize("T,nq,nkv,hd,K", ROTATING_SIZES)
def test_rotating(T, nq, nkv, hd, K):
    from tests.test_gpu_kernels import check_fused_qkv_rope_cache
    check_fused_qkv_rope_cache(T, nq, nkv, hd, K, 16, False)


def test_outputs_that_do_not_start_at_sixteen_bytes():
    """The four-wave kernel stores sixteen bytes at a time; such an output is another kernel's, with the same result."""
    from sprout_lm_amd import ops
    x, w, bias, want = _operands(200, 264, 192)
    room = torch.zeros(200 * 264 + 4, dtype=torch.bfloat16, device=DEV)
    ops.gemm(x, w, room[4:].view(200, 264), bias=bias)
    assert (room[4:].view(200, 264).float() - (want + bias)).abs().max().item() <= 2 ** -8 * (1 + want.abs().max().item())
    room32 = torch.zeros(200 * 264 + 2, device=DEV)
    ops.gemm(x, w, room32[2:].view(200, 264), accumulate=True)
    assert (room32[2:].view(200, 264) - want).abs().max().item() <= 1e-4


@pytest.mark.parametrize("shifted", ["x", "w", "q_out", "k_pool", "v_pool", "table"])
@pytest.mark.parametrize("T,nq,nkv,hd,K", [(65, 2, 1, 64, 64), (512, 14, 2, 64, 896), (300, 28, 4, 128, 448)])
def test_rotating_with_operands_that_do_not_start_at_sixteen_bytes(T, nq, nkv, hd, K, shifted):
    """A caller that asks whether the product, the rotation and the cache write are one call asks by sizes alone; the call is taken
    wherever its operands start, with the result of aligned ones: to the bit where the same kernel runs, else within the roundings
    of the projections and the results to bfloat16."""
    from sprout_lm_amd import ops
    N, page, pages = (nq + 2 * nkv) * hd, 16, 40
    assert ops.fused_supported(ops.FUSED_ROPE, T, N, K, hd, hd, False, variant="halves")
    gen = torch.Generator(device=DEV).manual_seed(T)
    x, w, bias, _ = _operands(T, N, K)
    positions = torch.randint(0, 5000, (T,), device=DEV, generator=gen, dtype=torch.int32)
    slots = torch.randperm(page * pages, device=DEV, generator=gen)[:T].int()
    inv_freq = 1e4 ** (-torch.arange(hd // 2, device=DEV).float() / (hd // 2))
    table = torch.empty(T, hd // 2, 2, device=DEV)
    ops.rope_table(positions, inv_freq, table)

    def run(moved):
        place = lambda name, v: torch.empty(v.numel() + 4, dtype=v.dtype, device=DEV)[(8 // v.element_size() if name == moved else 0):][:v.numel()].view(v.shape).copy_(v)
        q_out, k, v = (torch.zeros(*shape, dtype=torch.bfloat16, device=DEV) for shape in ((T, nq * hd), (pages, nkv, page, hd), (pages, nkv, hd, page)))
        args = {name: place(name, v) for name, v in dict(x=x, w=w, q_out=q_out, k_pool=k, v_pool=v, table=table).items()}
        assert moved is None or args[moved].data_ptr() % 16 == 8
        ops.qkv_rope_cache(args["w"], bias, args["q_out"], positions, inv_freq, hd, slots, args["k_pool"], args["v_pool"], nq, nkv, hd,
                           x=args["x"], table=args["table"])
        return args["q_out"], args["k_pool"], args["v_pool"]

    for got, want in zip(run(shifted), run(None)):
        if shifted in ("v_pool", "table"):
            assert torch.equal(got, want)
        else:
            assert (got.float() - want.float()).abs().max().item() <= 2 ** -7 * (1 + want.float().abs().max().item())
