"""Gated products on blocks of an odd number of tile columns a wave: every such shape, with token and row edges, few steps along K, and the
activations, against float32 products of the same operands; and where the rule gives them a product."""
import pytest
import torch

from sprout_lm_amd import ops

DEV = "cuda"
# (tokens, gate and up rows, K) -> block; edges: one token over 256 and 288 tokens, rows that end within a wave's run and within a lane's
SIZES = [(193, 32800, 256, (256, 160)), (256, 33392, 256, (256, 160)), (511, 37888, 3584, (256, 160)), (289, 39312, 256, (320, 160)), (640, 37888, 3584, (320, 160)),
         (193, 49376, 640, (256, 224)), (767, 37888, 3584, (256, 224)), (257, 49376, 256, (288, 224)), (288, 50560, 448, (288, 224)),
         # shapes of an even number that sizes tested before now leave
         (193, 41088, 320, (256, 192)), (700, 21552, 640, (256, 256))]


def test_where_they_are_taken():
    try:
        ops.library()
    except Exception as e:      # no compiler here: nothing to ask
        pytest.skip(f"the kernel library cannot be built or loaded here: {e}")
    for T, N, K, shape in SIZES:
        assert (ops.quad_odd_plan(T, N, K) or ops.quad_plan(ops.PLAN_GATED, T, N, K))[:2] == shape, (T, N, K)
    assert ops.quad_odd_plan(640, 37888, 3584) == (320, 160, 2) and ops.quad_plan(ops.PLAN_GATED, 640, 37888, 3584)[1] % 64 == 0
    # 0.83, 0.91 and 0.81 of the time; 1.00, 1.00, 1.04 and 1.08 of it
    assert ops.quad_odd_plan(320, 37888, 3584) and ops.quad_odd_plan(640, 37888, 3584) and ops.quad_odd_plan(264, 55296, 5120)
    assert not any(ops.quad_odd_plan(*s) for s in ((264, 37888, 3584), (640, 9728, 896), (2048, 9728, 896), (2048, 37888, 3584)))


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K,shape", SIZES)
def test_gated(T, N, K, shape):
    g = torch.Generator(device=DEV).manual_seed(T + N)
    x, w = torch.randn(T, K, device=DEV, generator=g).bfloat16(), (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).bfloat16()
    I = N // 2
    full = x.float() @ w.float().T
    gates = torch.randn(T, 3, device=DEV, generator=g)
    for activation in ("silu", "gelu_tanh", "relu"):
        row = gates if activation == "relu" else None
        out = torch.full((T + 1, I), 7.0, dtype=torch.bfloat16, device=DEV)        # a row behind the last stays as it is
        ops.gate_up_silu(w, out[:T], x=x, activation=activation, row_gate=row, row_gate_column=1)
        a, u = full[:, :I], full[:, I:]
        act = {"silu": torch.nn.functional.silu, "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh"), "relu": torch.relu}[activation]
        want = act(a) * u * (1.0 if row is None else torch.sigmoid(gates[:, 1:2]))
        # gate and up rounded to bfloat16 (eight bits: 2^-8 of each at most; the activations' slopes are below 1.13) and the product once more
        bound = 2.0 ** -8 * (1.13 * a.abs() * u.abs() + act(a).abs() * u.abs() + want.abs()) * 1.05 + 1e-3
        assert ((out[:T].float() - want).abs() <= bound).all()
        assert (out[T] == 7).all()
