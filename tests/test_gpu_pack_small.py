"""Operands packed with a thread per element and by tiles: the last size of the one and the first of the other."""
import pytest
import torch

from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("batch,m", [(1, 8192), (1, 8193), (4, 2048), (4, 2049), (1, 3), (3, 1)])
@pytest.mark.parametrize("ta", [0, 1])
def test_products_of_packed_operands(dtype, batch, m, ta):
    """K = 61 is padded to 64: batch x m rows of A are 2^19 packed elements, or just more, or a few."""
    if batch > 1:
        ta = 0   # batched products take both operands as they are
    k, n = 61, 20
    g = torch.Generator(device="cuda").manual_seed(m)
    A = torch.randn((batch, k, m) if ta else (batch, m, k), device="cuda", generator=g).to(TORCH[dtype])
    B = torch.randn((batch, k, n), device="cuda", generator=g).to(TORCH[dtype])
    C = torch.full((batch, m, n), float("nan"), device="cuda")
    if batch == 1:
        call(f"pcd_gemm_{dtype}", A.data_ptr(), B.data_ptr(), C.data_ptr(), m, k, n, ta, 0, 0.0, None)
    else:
        call(f"pcd_gemm_{dtype}_batched", A.data_ptr(), B.data_ptr(), C.data_ptr(), batch, m, k, n, None)
    torch.cuda.synchronize()
    for i in range(batch):
        a = (A[i].T if ta else A[i]).double()
        # fp32 sums of k products: k roundings (2^-24) of at most the sum of magnitudes
        bound = k * 2.0 ** -24 * (a.abs() @ B[i].double().abs())
        assert bool(((C[i].double() - a @ B[i].double()).abs() <= bound).all())
