"""The product of operands that fit no tile, whose K-tiles two groups of waves share: every number of K-tiles around the pairs."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("K", [16, 17, 127, 128, 129, 250, 257, 383, 385, 511, 513, 641, 1160, 2047])
@pytest.mark.parametrize("M,N", [(1, 1), (17, 65), (64, 63), (130, 129), (65, 1001)])
def test_ragged_product_is_the_integer_product(L, dev, M, N, K):
    g = torch.Generator().manual_seed(M * N + K)
    a = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8)
    want = (a.double() @ w.double().T).to(torch.int32)   # (exact: below 2^53)
    assert torch.equal(L.gemm_i32(a.to(dev), w.to(dev)).cpu(), want)
