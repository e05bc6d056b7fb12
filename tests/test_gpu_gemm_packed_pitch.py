"""Products whose packed operands' rows are longer than the kernel's K sweep."""
import pytest
import torch

from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu

TYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
# 128 x 128 tiles and, for the 16-bit types, 256 x 256: K within a stage's and
# within a line's remainder, K whole stages but half a line (there the other
# operand can be read in place), edge tiles, several products
CASES = [(1, 2944, 2130, 2048, 0, 1), (1, 2049, 2144, 2047, 0, 0), (1, 2056, 2144, 2047, 1, 0),
         (1, 2048, 2144, 2049, 1, 1), (1, 4100, 97, 4090, 0, 1), (3, 1500, 161, 1501, 0, 0),
         (3, 1500, 160, 1501, 0, 0), (1, 2047, 16, 2049, 0, 0), (1, 2048, 1, 2048, 0, 0)]


@pytest.mark.parametrize("batch,m,k,n,ta,tb", CASES)
@pytest.mark.parametrize("dtype", list(TYPES))
def test_packed_operands_of_any_k(dtype, batch, m, k, n, ta, tb):
    """Within the bound of a sum of K fp32 terms of the product in 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(m + k)
    A = torch.randn((batch, k, m) if ta else (batch, m, k), device="cuda", generator=g).to(TYPES[dtype])
    B = torch.randn((batch, n, k) if tb else (batch, k, n), device="cuda", generator=g).to(TYPES[dtype])
    C = torch.full((batch, m, n), float("nan"), device="cuda")
    if batch == 1:
        call("pcd_gemm_" + dtype, A.data_ptr(), B.data_ptr(), C.data_ptr(), m, k, n, ta, tb, 0.0, None)
    else:
        call("pcd_gemm_" + dtype + "_batched", A.data_ptr(), B.data_ptr(), C.data_ptr(), batch, m, k, n, None)
    torch.cuda.synchronize()
    for i in range(batch):
        a, b = A[i].double(), B[i].double()
        a, b = (a.T.contiguous() if ta else a), (b.T.contiguous() if tb else b)
        # K products rounded to 2^-24 each at most (16-bit ones are exact), K sums to 2^-24 of the
        # magnitudes' own sum
        bound = 2.0 * k * 2.0 ** -24 * (a.abs() @ b.abs())
        assert bool(((C[i].double() - a @ b).abs() <= bound + 1e-30).all())
