"""The experts of few rows against float64: both products' splits of K among waves, at the edges of
the rule that chooses them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.mark.parametrize("experts,top,width,inter", [
    (16, 4, 2048, 704), (16, 4, 1024, 768), (5, 2, 192, 64), (8, 2, 2048, 1408), (8, 3, 1024, 1472),
    (3, 1, 2048, 2816), (64, 6, 256, 320)])
@pytest.mark.parametrize("rows", [1, 2, 7, 16, 17, 32, 33, 64])
def test_experts_of_few_rows(experts, top, width, inter, rows):
    from edge_infer_amd.csrc import lib
    g = torch.Generator().manual_seed(rows + inter)
    made = lambda *shape: torch.randn(shape, generator=g)
    gate, up, down = (made(experts, a, b).mul(b ** -0.5).to(torch.bfloat16)
                      for a, b in ((inter, width), (inter, width), (width, inter)))
    x = made(rows, width).to(torch.bfloat16)
    chosen = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)])
    weight = torch.rand((rows, top), generator=g) + 0.1
    padding = rows > 2                                     # one row that belongs to no sequence
    seq = torch.arange(rows, dtype=torch.int32)
    if padding:
        seq[1] = -1
    act = torch.full((rows * top, inter), float("nan"), dtype=torch.bfloat16, device="cuda")
    out = torch.full((top, rows, width), float("nan"), device="cuda")
    lib.moe_experts_few(x.cuda(), *(lib.pack_experts(w.cuda()) for w in (gate, up, down)),
                        chosen.int().cuda(), weight.cuda(), seq.cuda(), act, out)
    act, out = act.cpu().view(rows, top, inter), out.cpu()
    for r in range(rows):
        if padding and r == 1:
            assert out[:, r].isnan().all()
            continue
        for k in range(top):
            e, xr = int(chosen[r, k]), x[r].to(F64)
            z, u = gate[e].to(F64) @ xr, up[e].to(F64) @ xr
            exact = z * torch.sigmoid(z) * u
            # bfloat16 holds a value to 2^-9 of it; the float32 sums are far below that
            assert ((act[r, k].to(F64) - exact).abs() <= exact.abs() * 2 ** -8 + 1e-5).all()
            # given the rounded activations a float32 sum of `inter` products remains: at most
            # inter 2^-24 of the sum of their magnitudes
            a = act[r, k].to(F64)
            want = weight[r, k].to(F64) * (down[e].to(F64) @ a)
            bound = weight[r, k].to(F64) * (down[e].to(F64).abs() @ a.abs()) * (inter + 8) * 2.0 ** -24
            assert ((out[k, r].to(F64) - want).abs() <= bound).all()
