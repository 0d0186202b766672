"""The float32 product's matrix-core kernels at the edges of their tiles and pieces of K."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 4), (17, 20), (64, 128), (100, 1028), (130, 2052), (4099, 68),
                                 (65600, 36), (10500, 1028), (10411, 2052), (49411, 4)])
def test_products_of_every_number_of_rows_within_the_bound_and_the_same_bits(N, K):
    """Rows 1 .. 64 take the kernel of few rows, more the tiles of 32 x 32, 32 x 64 and 64 x 64 or those
    of 128 x 128 (257 and 300 rows of the outputs above 10,000, 65 and 100 of 49,411 too).
    A sum of K float32 products in any order is within K u sum |a w| of the exact one (u = 2^-24,
    and one more u for a product's own rounding); a row has the same bits in every kernel."""
    from edge_infer_amd.csrc import lib
    g = torch.Generator().manual_seed(N + K)
    a = torch.randn(300, K, generator=g).to("cuda")
    w = torch.randn(N, K, generator=g).to("cuda")
    exact = a.double() @ w.double().T
    bound = (K + 1) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    first = None
    for rows in (300, 257, 129, 100, 65, 64, 33, 32, 17, 16, 5, 1):
        out = torch.full((rows, N), float("nan"), device="cuda")
        lib.gemm_f32(a[:rows].contiguous(), w, out)
        assert bool(((out.double() - exact[:rows]).abs() <= bound[:rows]).all()), rows
        if first is None:
            first = out
        assert torch.equal(out, first[:rows]), rows


@pytest.mark.parametrize("N,K", [(7, 2052), (1027, 3072), (2047, 2048), (2048, 2064), (2055, 1024), (4096, 520)])
def test_narrow_strips_of_few_rows(N, K):
    """Strips of 8 outputs a block (up to 2,048 outputs) and of 16 with more steps asked for at a
    time (up to 4,096), at their edges: the bound of the test above, and the same bits as 64 rows."""
    from edge_infer_amd.csrc import lib
    g = torch.Generator().manual_seed(N + K)
    a = torch.randn(64, K, generator=g).to("cuda")
    w = torch.randn(N, K, generator=g).to("cuda")
    exact = a.double() @ w.double().T
    bound = (K + 1) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    wide = torch.full((64, N), float("nan"), device="cuda")
    lib.gemm_f32(a, w, wide)
    for rows in (16, 9, 8, 5, 4, 3, 1):
        out = torch.full((rows + 1, N), 7.0, device="cuda")
        lib.gemm_f32(a[:rows].contiguous(), w, out[:rows])
        assert bool(((out[:rows].double() - exact[:rows]).abs() <= bound[:rows]).all()), rows
        assert torch.equal(out[:rows], wide[:rows]), rows
        assert bool((out[rows] == 7.0).all()), rows


@pytest.mark.parametrize("N,K", [(17, 20), (100, 1028), (4099, 68), (1000, 3072)])
def test_where_the_operands_lie_does_not_change_the_bits(N, K):
    """Rows that begin at any float give the bits of rows that begin at a multiple of four."""
    from edge_infer_amd.csrc import lib
    g = torch.Generator().manual_seed(N + K)
    a, w = torch.randn(130, K, generator=g).to("cuda"), torch.randn(N, K, generator=g).to("cuda")

    def moved(x, by):
        room = torch.empty(x.numel() + 4, device="cuda")
        view = room[by:by + x.numel()].view(x.shape)
        return view.copy_(x)
    for rows in (130, 65, 40, 17, 8, 1):
        want = torch.empty(rows, N, device="cuda")
        lib.gemm_f32(a[:rows], w, want)
        for by_a, by_w in ((1, 0), (0, 1), (2, 3)):
            out = torch.empty(rows, N, device="cuda")
            lib.gemm_f32(moved(a[:rows], by_a), moved(w, by_w), out)
            assert torch.equal(out, want), (rows, by_a, by_w)
