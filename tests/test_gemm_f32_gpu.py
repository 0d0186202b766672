"""The float32 product's matrix-core kernels at the edges of their tiles and pieces of K."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 4), (17, 20), (64, 128), (100, 1028), (130, 2052), (4099, 68),
                                 (65600, 36)])
def test_products_of_every_number_of_rows_within_the_bound_and_the_same_bits(N, K):
    """Rows 1 .. 64 take the kernel of few rows, more the tiles of 32 x 32, 32 x 64 and 64 x 64.
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
