"""fp32 products on the 128 x 128 tile, which multiplies three bf16 pieces of each operand: error against 64-bit sums,
and the fp32 infinities and NaNs of operands the pieces cannot carry."""
import numpy as np
import pytest
import torch

from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu


def product(A, B):
    """C = A B^T through pcd_gemm_f32; 2048 x 2048 outputs fill every CU with a 128 x 128 tile."""
    (m, k), n = A.shape, B.shape[0]
    C = torch.empty((m, n), device="cuda")
    call("pcd_gemm_f32", A.data_ptr(), B.data_ptr(), C.data_ptr(), m, k, n, 0, 1, 0.0, None)
    torch.cuda.synchronize()
    return C


def operands(k, seed, m=2048, n=2048):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((m, k), generator=g, device="cuda"), torch.randn((n, k), generator=g, device="cuda"))


# K of one, two, three and more stages of 16, a padded K, ragged rows and columns, magnitudes far from one
@pytest.mark.parametrize("m,n,k,scale", [(2048, 2048, 16, 1.0), (2048, 2048, 32, 1.0), (2048, 2048, 64, 1.0),
                                         (2048, 2048, 208, 1.0), (1921, 2040, 333, 1.0), (2048, 2048, 2048, 1.0),
                                         (2048, 2048, 512, 1e-18), (2048, 2048, 512, 1e18)])
def test_split_products_against_64_bits(m, n, k, scale):
    A, B = operands(k, k, m, n)
    A *= scale
    ref = A.double() @ B.double().T
    err = (product(A, B).double() - ref).norm() / ref.norm()
    # One rounding (2^-24 / sqrt(3) of the value in the mean square) per 16 elements of K of a sum that grows to its
    # final size, one when the small products join it, twice that; and the terms left out
    # (2^-27 of normal operands' products in the root mean square, 2^-24 at most), twice that.
    bound = 2 * 2.0 ** -24 / np.sqrt(3.0) * np.sqrt(np.ceil(k / 16.0) + 1) + 2.0 ** -26
    assert float(err) <= bound, (float(err), bound)


@pytest.mark.parametrize("special", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_special_operands_as_fp32_multiplies_them(special):
    """Rows and columns with an infinity, a NaN or a value whose bf16 rounding overflows: the class and sign of every
    result, and the finite values, as fp32 arithmetic gives them."""
    A, B = operands(256, 5)
    A[3, 17] = special
    A[700, 255] = special
    B[1500, 0] = special
    B[9] = 0.0
    C, ref = product(A, B), A.double() @ B.double().T
    ref32 = ref.float()                    # sums beyond the fp32 range become infinite
    assert torch.equal(torch.isnan(C), torch.isnan(ref32))
    assert torch.equal(torch.isinf(C) & (C > 0), torch.isinf(ref32) & (ref32 > 0))
    assert torch.equal(torch.isinf(C) & (C < 0), torch.isinf(ref32) & (ref32 < 0))
    ok = torch.isfinite(ref32) & (ref.abs() < 1e6)
    assert float((C.double() - ref)[ok].abs().max()) < 1e-4   # K = 256 unit normals: 5e-6 at most


@pytest.mark.parametrize("k", [16, 64, 208, 1024])
def test_operands_that_lose_most(k):
    """The products left out are largest, and all of one sign, where both operands are 1 + 2^-8 - 2^-17 times a power of
    two: 2^-24 of each product.  Beside that, at most one rounding (2^-24) of a growing sum per 16 elements of K, one
    of the small products' sum and one when it joins."""
    v = 1 + 2.0 ** -8 - 2.0 ** -17
    g = torch.Generator(device="cuda").manual_seed(k)
    e = torch.randint(-6, 7, (2, 2048, k), generator=g, device="cuda", dtype=torch.float32)
    A, B = v * torch.exp2(e[0]), v * torch.exp2(e[1])
    ref = A.double() @ B.double().T
    err = float(((product(A, B).double() - ref) / ref).abs().max())
    assert err <= 2.0 ** -24 * (1 + k / 16 + 2), err
