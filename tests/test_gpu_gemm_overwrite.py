"""Products that overwrite one of their operands."""
import pytest
import torch

from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu


# batched products take both operands as they are
CASES = [(1, n, ta, tb) for n in (2048, 500, 64) for ta in (0, 1) for tb in (0, 1)] + \
    [(6, 512, 0, 0), (40, 128, 0, 0), (3, 100, 0, 0)]


@pytest.mark.parametrize("batch,n,ta,tb", CASES)
@pytest.mark.parametrize("over", ["a", "b"])
def test_the_result_in_place_of_an_operand(batch, n, ta, tb, over):
    """Square fp32 products into A's or B's own memory equal those into memory apart, bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(n)
    A, B = (torch.randn((batch, n, n), device="cuda", generator=g) for _ in range(2))

    def product(a, b, c):
        if batch == 1:
            call("pcd_gemm_f32", a.data_ptr(), b.data_ptr(), c.data_ptr(), n, n, n, ta, tb, 0.0, None)
        else:
            call("pcd_gemm_f32_batched", a.data_ptr(), b.data_ptr(), c.data_ptr(), batch, n, n, n, None)
        torch.cuda.synchronize()
        return c

    want = product(A, B, torch.empty_like(A))
    got = product(A, B, A if over == "a" else B)
    assert torch.equal(got, want)
