"""Products whose operands are read where they lie without filling whole tiles: every layout against the packed route
(the same operands one element off their alignment), bit for bit, and against float64."""
import numpy as np
import pytest
import torch

from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def off(t):
    """`t`'s values one element past an aligned address: never read in place."""
    buf = torch.zeros(t.numel() + 1, dtype=t.dtype, device="cuda")
    buf[1:] = t.reshape(-1)
    return buf[1:]


# the 32 x 32 (fp32), 64 x 64, 128 x 128 and 256 x 256 (16-bit) tiles; one row over, one short of a tile, the fewest
# rows and columns of a unit, one K stage and several, and a K that is no whole number of stages
SHAPES = [("f32", 4, 64, 4), ("f32", 33, 192, 100), ("f32", 260, 64, 36), ("f32", 1100, 48, 1100),
          ("f32", 1028, 784, 1100), ("f32", 2052, 16, 2044), ("f32", 1924, 208, 2180), ("f32", 300, 100, 260),
          ("bf16", 8, 64, 8), ("bf16", 72, 192, 328), ("f16", 1000, 128, 1160), ("bf16", 2056, 96, 1912),
          ("f16", 4104, 128, 4088), ("bf16", 130, 320, 4040)]


@pytest.mark.parametrize("dtype,m,k,n", SHAPES)
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_in_place_layouts_match_the_packed_route(dtype, m, k, n, ta, tb):
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    A = torch.randn((k, m) if ta else (m, k), device="cuda", generator=g).to(TORCH[dtype])
    B = torch.randn((n, k) if tb else (k, n), device="cuda", generator=g).to(TORCH[dtype])
    out = []
    for a, b in ((A, B), (off(A), off(B)), (A, off(B)), (off(A), B)):
        C = torch.full((m + 1, n), 3.0, device="cuda")   # a row past the end, to stay as it is
        call(f"pcd_gemm_{dtype}", a.data_ptr(), b.data_ptr(), C.data_ptr(), m, k, n, ta, tb, 0.5, None)
        torch.cuda.synchronize()
        assert bool((C[m] == 3.0).all())
        out.append(C[:m])
    ref = (A.t() if ta else A).double() @ (B.t() if tb else B).double() + 1.5
    for C in out:
        assert torch.equal(C, out[0])
    # fp32 sums of k products of unit normals: k roundings of a sum up to sqrt(k) large, 6 sigma of the largest value
    assert float((out[0].double() - ref).abs().max()) <= 6 * 2.0 ** -24 * np.sqrt(k) * np.sqrt(k) + 1e-6


@pytest.mark.parametrize("dtype,batch,m,k,n", [("f32", 5, 33, 64, 36), ("f32", 96, 200, 64, 200), ("f32", 3, 7, 16, 4),
                                               ("f32", 40, 100, 100, 52), ("bf16", 70, 130, 64, 136),
                                               ("f16", 9, 515, 128, 264), ("bf16", 11, 24, 40, 9), ("f32", 7, 5, 3, 2)])
def test_batched_products_in_one_launch(dtype, batch, m, k, n):
    g = torch.Generator(device="cuda").manual_seed(batch)
    A = torch.randn((batch, m, k), device="cuda", generator=g).to(TORCH[dtype])
    B = torch.randn((batch, k, n), device="cuda", generator=g).to(TORCH[dtype])
    out = []
    for a, b in ((A, B), (off(A), off(B))):
        C = torch.full((batch, m, n), float("nan"), device="cuda")
        call(f"pcd_gemm_{dtype}_batched", a.data_ptr(), b.data_ptr(), C.data_ptr(), batch, m, k, n, None)
        torch.cuda.synchronize()
        out.append(C)
    assert torch.equal(out[0], out[1])
    ref = torch.stack([a.double() @ b.double() for a, b in zip(A, B)])
    assert float((out[0].double() - ref).abs().max()) <= 6 * 2.0 ** -24 * k + 1e-6
