"""Products and settlings on both sides of the rules that choose the 128 x 128 tile where it does not fill every CU, and
the K ranges it is split into, against float64 and against the 64 x 64 tile."""
import numpy as np
import pytest
import torch

from predicitivecoding_amd import GenerativeSnapshot, PcDeviceModel
from predicitivecoding_amd._native import call

pytestmark = pytest.mark.gpu
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}

# 144 fp32 tiles in four K ranges, in two, in one; ragged edges and K; eight ranges of 1024 and one less; 128 tiles; a
# K just below the line; 16-bit tiles at and below it
SHAPES = [("f32", 1536, 4096, 1536), ("f32", 1501, 2052, 1499), ("f32", 1536, 2047, 1536), ("f32", 644, 8192, 636),
          ("f32", 640, 8176, 640), ("f32", 512, 2048, 4096), ("f32", 1600, 639, 1600), ("bf16", 1600, 640, 1600),
          ("f16", 1501, 700, 1499), ("bf16", 1600, 624, 1600)]


@pytest.mark.parametrize("dtype,m,k,n", SHAPES)
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_products_near_the_tile_rules(dtype, m, k, n, ta, tb):
    g = torch.Generator(device="cuda").manual_seed(m + k)
    A = torch.randn((k, m) if ta else (m, k), device="cuda", generator=g).to(TORCH[dtype])
    B = torch.randn((n, k) if tb else (k, n), device="cuda", generator=g).to(TORCH[dtype])
    a, b = (A.double().T if ta else A.double()), (B.double().T if tb else B.double())
    prod = a @ b
    first = None
    for _ in range(3):   # the counters of the K ranges start from zero each time
        C = torch.full((m + 1, n), 3.0, device="cuda")
        call(f"pcd_gemm_{dtype}", A.data_ptr(), B.data_ptr(), C.data_ptr(), m, k, n, ta, tb, 0.5, None)
        torch.cuda.synchronize()
        assert bool((C[m] == 3.0).all())
        # at most a rounding of 2^-24 of the running sum per two elements of K, independent ones adding in the square,
        # and two more for beta C and the result
        err = ((C[:m].double() - (prod + 1.5)).norm() / prod.norm()).item()
        assert err <= 2.0 ** -24 * np.sqrt(k / 2 + 2), err
        first = C if first is None else first
        assert torch.equal(C, first)


@pytest.mark.parametrize("width,rows", [(640, 2100), (632, 2100), (2048, 500), (1024, 1000), (1024, 700), (2048, 650)])
def test_settlings_near_the_tile_rules(width, rows):
    sizes = [width] * 4
    rng = np.random.default_rng(width)
    W = [rng.standard_normal((width, width)).astype(np.float32) / np.float32(np.sqrt(width)) for _ in range(3)]
    b = [rng.standard_normal(width).astype(np.float32) * np.float32(0.1) for _ in range(3)]
    model = PcDeviceModel(GenerativeSnapshot(sizes, 1, 0.1, 0.0, False, W, b), "f32")
    x = torch.randn(rows, width, generator=torch.Generator().manual_seed(1)).cuda()
    out = []
    for tile in (0, 64):
        model.set_option("tile", tile)
        top, states = torch.zeros(rows, width, device="cuda"), torch.zeros(rows * sum(sizes), device="cuda")
        energy = torch.zeros(6, rows, device="cuda")
        call("pcd_pc_relax", model.handle, x.data_ptr(), rows, 6, top.data_ptr(), states.data_ptr(),
             energy.data_ptr(), None)
        torch.cuda.synchronize()
        out.append((top, states, energy))
    for a, c in zip(*out):   # fp32 sums of up to 2048 products in two orders, six steps of them
        assert ((a - c).norm() / c.norm()).item() <= 6 * 2.0 ** -24 * np.sqrt(2048)
    model.close()


@pytest.mark.parametrize("m,k,n", [(3072, 1024, 768), (2048, 960, 1408), (1792, 1024, 1408), (1536, 704, 2560),
                                   (1536, 640, 2560), (4608, 1280, 768)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_16_bit_products_near_the_rules_for_k_rows(dtype, m, k, n, ta, tb):
    """Operands in K rows small and large, K on both sides of 1024 and 704; every one packed as well (one element off
    its alignment), whichever tile that takes."""
    check_layouts(dtype, m, k, n, ta, tb)


@pytest.mark.parametrize("m,k,n,ta,tb", [(1500, 2560, 160, 0, 0), (1500, 2496, 160, 0, 0), (400, 2560, 1000, 1, 1),
                                         (404, 2560, 1000, 1, 1), (1460, 2560, 160, 0, 0), (1500, 2560, 160, 1, 0)])
def test_fp32_products_near_the_rule_that_packs_a_small_operand(m, k, n, ta, tb):
    """K on both sides of 2560, 6e8 multiply-adds and less, an operand two fifths of the other and a bit more."""
    check_layouts("f32", m, k, n, ta, tb)


def check_layouts(dtype, m, k, n, ta, tb):
    g = torch.Generator(device="cuda").manual_seed(m + n)
    A = torch.randn((k, m) if ta else (m, k), device="cuda", generator=g).to(TORCH[dtype])
    B = torch.randn((n, k) if tb else (k, n), device="cuda", generator=g).to(TORCH[dtype])
    a, b = (A.double().T if ta else A.double()), (B.double().T if tb else B.double())
    off = [torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:] for t in (A, B)]
    for x, y in ((A, B), off):
        C = torch.full((m, n), float("nan"), device="cuda")
        call(f"pcd_gemm_{dtype}", x.data_ptr(), y.data_ptr(), C.data_ptr(), m, k, n, ta, tb, 0.0, None)
        torch.cuda.synchronize()
        # a rounding of 2^-24 of the running sum per two elements of K, independent ones adding in the square
        assert ((C.double() - a @ b).norm() / (a @ b).norm()).item() <= 2.0 ** -24 * np.sqrt(k / 2 + 2)
