"""The few-rows product that starts from a bias and writes a feed-forward's activation itself:
against float64 products of the same bfloat16 operands, over row groups (16, 32, 64 and 128 rows a
block, one and two strips a wave), widths that leave a strip or a wave partly empty, and each
activation; the parts' two routes against each other."""
import math

import pytest
import torch

from edge_infer_amd.csrc import lib

pytestmark = pytest.mark.gpu
DEV = "cuda"

PLAIN = {
    "relu2": lambda z: torch.relu(z) ** 2,
    "relu": torch.relu,
    "silu": lambda z: z * torch.sigmoid(z),
    "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh"),
}
GATED = {
    "silu": lambda g, u: PLAIN["silu"](g) * u,
    "gelu_tanh": lambda g, u: PLAIN["gelu_tanh"](g) * u,
    "clamped_swish": lambda g, u: (g.clamp(max=2.0) * torch.sigmoid(1.5 * g.clamp(max=2.0))
                                   * (u.clamp(-2.0, 2.0) + 1.0)),
}


def check(got, want):
    """One rounding to bfloat16 (2^-8 of a value either way, doubled for a value next to a power of
    two) and, for what the float32 sums and the activation's own arithmetic add, 1e-3 absolute: the
    products here are of order 1 and the activations' slopes below 20."""
    assert not got.isnan().any()
    bound = want.abs() * 2.0 ** -7 + 1e-3
    worst = ((got.double() - want).abs() - bound).max().item()
    assert worst <= 0, f"{worst:.3e} above the bound"


def operands(m, n, k):
    torch.manual_seed(m * 1000 + n + k)
    x = torch.randn(m, k, device=DEV).to(torch.bfloat16)
    w = (torch.randn(n, k, device=DEV) / math.sqrt(k)).to(torch.bfloat16)
    bias = torch.randn(n, device=DEV)
    return x, w, bias


SHAPES = [(1, 16, 8), (1, 100, 520), (7, 130, 256), (16, 1024, 1000), (17, 77, 512), (33, 2048, 264),
          (64, 18, 776), (65, 100, 256), (100, 16400, 136), (129, 66, 512), (256, 250, 1032)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("kind", list(PLAIN))
def test_plain_activation(m, n, k, kind):
    x, w, bias = operands(m, n, k)
    z = x.double() @ w.double().t()
    for packed in (True, False):
        for b in (None, bias):
            guard = torch.full((m + 1, n), 7.0, device=DEV, dtype=torch.bfloat16)
            out = guard[:m]
            out.fill_(float("nan"))
            lib.gemm_bf16_skinny_act(x, lib.pack_weight(w) if packed else w, n, out, packed, kind, bias=b)
            check(out, PLAIN[kind](z if b is None else z + b.double()))
            assert (guard[m] == 7.0).all()


@pytest.mark.parametrize("m,i,k", [(1, 16, 8), (5, 48, 520), (16, 512, 1000), (33, 208, 256),
                                   (65, 48, 256), (100, 8208, 136), (129, 80, 512), (256, 16, 1032)])
@pytest.mark.parametrize("kind", list(GATED))
def test_gated_with_a_bias(m, i, k, kind):
    x, w, bias = operands(m, 2 * i, k)
    z = (x.double() @ w.double().t() + bias.double()).reshape(m, i // 16, 2, 16)
    want = GATED[kind](z[:, :, 0], z[:, :, 1]).reshape(m, i)
    for packed in (True, False):
        out = torch.full((m, i), float("nan"), device=DEV, dtype=torch.bfloat16)
        lib.gemm_bf16_skinny_gated(x, lib.pack_weight(w) if packed else w, 2 * i, out, packed, kind,
                                   limit=2.0, alpha=1.5, bias=bias)
        check(out, want)


def test_refusals():
    x, w, bias = operands(2, 64, 64)
    out = torch.empty(2, 64, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(lib.KernelError, match="unknown kind"):
        lib.gemm_bf16_skinny_act(x, w, 64, out, False, "tanh")
    with pytest.raises(lib.KernelError, match="do not agree"):
        lib.gemm_bf16_skinny_act(x, w, 64, out[:, :32], False, "relu")
    with pytest.raises(lib.KernelError, match="bias"):
        lib.gemm_bf16_skinny_act(x, w, 64, out, False, "relu", bias=bias[:32])
    with pytest.raises(lib.KernelError, match="bias"):
        lib.gemm_bf16_skinny_gated(x, w, 64, out[:, :32].contiguous(), False, bias=bias[:32])
