"""Batched products of more work units than one launch takes."""
import pytest
import torch

from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,m,k,n", [(2 ** 24 + 3, 2, 2, 2), (2 ** 22 + 1, 3, 5, 4), (2 ** 21 + 7, 65, 1, 4)])
def test_batches_of_millions(batch, m, k, n):
    """2 x 2 products past 2^24 tiles (at 256 threads a tile, past the 2^32 threads HIP takes in a grid), and two
    launches' worth with one and two tiles an item."""
    g = torch.Generator(device="cuda").manual_seed(m)
    A = torch.randn((batch, m, k), device="cuda", generator=g)
    B = torch.randn((batch, k, n), device="cuda", generator=g)
    C = torch.full((batch, m, n), float("nan"), device="cuda")
    call("pcd_gemm_f32_batched", A.data_ptr(), B.data_ptr(), C.data_ptr(), batch, m, k, n, None)
    torch.cuda.synchronize()
    ref, size = torch.zeros_like(C), torch.zeros_like(C)
    for j in range(k):
        term = A[:, :, j, None] * B[:, j, None, :]
        ref += term
        size += term.abs()
    # k roundings of either sum, and of the products of the reference
    assert bool(((C - ref).abs() <= (2 * k + 1) * 2.0 ** -24 * size).all())
