"""Which batched products of an inner dimension that 16 does not divide are copied with it padded, on the CPU."""
import pytest
import torch

import torch_int._CUDA as C


@pytest.mark.parametrize("batch,M,N,K,out_bytes,padded", [
    (19, 1110, 1110, 17, 4, True), (8, 1857, 1857, 100, 4, True), (151, 499, 499, 17, 4, True), (131, 1631, 128, 10, 4, True),   # lines of 32-bit outputs
    (19, 1110, 1110, 17, 1, False), (28, 400, 400, 100, 4, False), (160, 517, 517, 130, 4, False), (200, 1500, 80, 100, 4, False),
    (64, 1664, 1664, 25, 1, True), (4, 2048, 2048, 4097, 1, True), (160, 517, 128, 517, 1, False), (3, 300, 300, 100, 4, False)])
def test_products_whose_operands_are_copied(batch, M, N, K, out_bytes, padded):
    a, b = torch.ones((batch, M, K), dtype=torch.int8), torch.ones((batch, N, K), dtype=torch.int8)
    pa, pb, k = C._pad_products(a, b, batch, M, N, K, out_bytes)
    if padded:
        assert k == (K + 63) // 64 * 64 and pa.shape == (batch, M, k) and pb.shape == (batch, N, k)
        assert int(pa[:, :, K:].abs().sum()) == 0 and int(pb[:, :, K:].abs().sum()) == 0
    else:
        assert k == K and pa is a and pb is b
