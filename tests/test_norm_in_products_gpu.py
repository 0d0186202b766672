"""Products that add to the stream and leave its norm to the product that reads it, against the same
sums in float64."""
import pytest
import torch

from edge_infer_amd.csrc import lib

pytestmark = pytest.mark.gpu
BF16, F64 = torch.bfloat16, torch.float64
# A float32 sum of k products in any order is off by at most k 2^-24 of the sum of their
# magnitudes, and by about sqrt(k) 2^-24 of it in practice; the bound of k is what is asserted.
UNIT = 2.0 ** -24


def made(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g) * scale


@pytest.mark.parametrize("m,n,k", [
    (1, 64, 64), (1, 1024, 2048), (3, 16, 1088), (8, 4096, 4096), (15, 64, 448), (16, 1024, 3072),
    (7, 2048, 512), (5, 80, 4168), (9, 1024, 12288), (2, 4096, 12352), (16, 16, 8), (1, 192, 3104)])
def test_add_product(m, n, k):
    x, w = made((m, k), 1).to(BF16), made((n, k), 2, k ** -0.5).to(BF16)
    residual, weight = made((m, n), 3), 1.0 + 0.1 * made((n,), 4)
    dev = residual.cuda()
    rows = torch.full((m, n), float("nan"), dtype=BF16, device="cuda")
    stats = torch.full((m, n // 16), float("nan"), device="cuda")
    lib.gemm_bf16_add(x.cuda(), lib.pack_weight(w.cuda()), dev, weight.cuda(), rows, stats)
    exact = residual.to(F64) + x.to(F64) @ w.to(F64).t()
    magnitude = residual.to(F64).abs() + x.to(F64).abs() @ w.to(F64).abs().t()
    bound = (k + 2) * UNIT * magnitude
    assert ((dev.cpu().to(F64) - exact).abs() <= bound).all()
    assert torch.equal(rows.cpu(), (dev.cpu() * weight).to(BF16))       # one product, rounded once
    squares = dev.cpu().to(F64).square().view(m, n // 16, 16).sum(dim=2)
    assert torch.allclose(stats.cpu().to(F64), squares, rtol=16 * 2 * UNIT, atol=0.0)


@pytest.mark.parametrize("m", [1, 3, 8])
@pytest.mark.parametrize("n,k", [(64, 64), (1024, 1088), (1024, 2048), (16, 8), (1024, 3072), (2048, 3136),
                                 (80, 4168), (2048, 8192)])
def test_add_product_by_half_strips(m, n, k):
    """Eight columns a block, and a product that finishes the norm from sums of eight columns."""
    x, w = made((m, k), 1).to(BF16), made((n, k), 2, k ** -0.5).to(BF16)
    residual, weight = made((m, n), 3), 1.0 + 0.1 * made((n,), 4)
    dev = residual.cuda()
    rows = torch.full((m, n), float("nan"), dtype=BF16, device="cuda")
    stats = torch.full((m, n // 8), float("nan"), device="cuda")
    assert lib.add_parts(m, n) == n // 8 and lib.add_parts(9, n) == n // 16 and lib.add_parts(m, 4096) == 256
    lib.gemm_bf16_add(x.cuda(), lib.pack_weight(w.cuda()), dev, weight.cuda(), rows, stats)
    exact = residual.to(F64) + x.to(F64) @ w.to(F64).t()
    magnitude = residual.to(F64).abs() + x.to(F64).abs() @ w.to(F64).abs().t()
    assert ((dev.cpu().to(F64) - exact).abs() <= (k + 2) * UNIT * magnitude).all()
    assert torch.equal(rows.cpu(), (dev.cpu() * weight).to(BF16))
    squares = dev.cpu().to(F64).square().view(m, n // 8, 8).sum(dim=2)
    assert torch.allclose(stats.cpu().to(F64), squares, rtol=16 * UNIT, atol=0.0)
    if n % 64:
        return
    reader = made((96, n), 7, n ** -0.5).to(BF16)
    out = torch.empty((lib.skinny_gemm_splits(m, 96, n), m, 96), device="cuda")
    lib.gemm_bf16_skinny_packed(rows, lib.pack_weight(reader.cuda()), 96, out, stats=(stats, 1e-6))
    factor = (dev.cpu().to(F64).square().mean(dim=1, keepdim=True) + 1e-6).rsqrt()
    want = (rows.cpu().to(F64) @ reader.to(F64).t()) * factor
    bound = (2 * n + 8) * UNIT * (rows.cpu().to(F64).abs() @ reader.to(F64).abs().t()) * factor
    assert ((out.cpu().to(F64).sum(dim=0) - want).abs() <= bound).all()


@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("n,k", [(64, 64), (96, 1024), (4096, 1024), (6144, 4096), (1600, 2048), (32, 448)])
def test_products_finish_the_norm(m, n, k):
    """Sliced sums and the gated product of rows that carry their sums of squares."""
    stream, w = made((m, k), 5, 3.0), made((n, k), 6, k ** -0.5).to(BF16)
    rows = stream.to(BF16).cuda()
    squares = stream.square().view(m, k // 16, 16).sum(dim=2).cuda()
    eps = 1e-6
    packed = lib.pack_weight(w.cuda())
    factor = (stream.to(F64).square().mean(dim=1, keepdim=True) + eps).rsqrt()
    exact = (rows.cpu().to(F64) @ w.to(F64).t()) * factor
    magnitude = (rows.cpu().to(F64).abs() @ w.to(F64).abs().t()) * factor
    out = torch.empty((lib.skinny_gemm_splits(m, n, k), m, n), device="cuda")
    lib.gemm_bf16_skinny_packed(rows, packed, n, out, stats=(squares, eps))
    # (the factor: a sum of k squares, a division and a hardware square root, 4 units together)
    bound = (2 * k + 8) * UNIT * magnitude
    assert ((out.cpu().to(F64).sum(dim=0) - exact).abs() <= bound).all()
    act = torch.empty((m, n // 2), dtype=BF16, device="cuda")
    lib.gemm_bf16_skinny_gated(rows, packed, n, act, True, stats=(squares, eps))
    strips = exact.view(m, n // 32, 2, 16)
    gate, up = strips[:, :, 0].reshape(m, -1), strips[:, :, 1].reshape(m, -1)
    want = gate / (1.0 + (-gate).exp()) * up
    slack = bound.view(m, n // 32, 2, 16)
    # silu's slope is at most 1.1, its value at most |gate|; the result rounds to 8 bits
    most = (1.1 * slack[:, :, 0].reshape(m, -1) * up.abs() + gate.abs() * slack[:, :, 1].reshape(m, -1)
            + (2.0 ** -8 + 2.0 ** -20) * want.abs() + 1e-30)
    assert ((act.cpu().to(F64) - want).abs() <= most).all()


def test_refused():
    x, w = torch.zeros((17, 64), dtype=BF16, device="cuda"), torch.zeros((64, 64), dtype=BF16, device="cuda")
    res, one = torch.zeros((17, 64), device="cuda"), torch.ones(64, device="cuda")
    with pytest.raises(lib.KernelError):
        lib.gemm_bf16_add(x, lib.pack_weight(w), res, one, torch.zeros_like(x), torch.zeros((17, 4), device="cuda"))
    with pytest.raises(lib.KernelError):
        lib.gemm_bf16_skinny_packed(x, lib.pack_weight(w), 64, torch.zeros((1, 17, 64), device="cuda"),
                                    stats=(torch.zeros((17, 4), device="cuda"), 1e-6))
