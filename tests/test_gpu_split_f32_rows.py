"""fp32 on the 128 x 128 tile (three bf16 pieces of each operand): what a row or column with values beyond the pieces
gets, and that it changes nothing for its neighbours in the tile."""
import numpy as np
import pytest
import torch

from predicitivecoding_amd import GenerativeSnapshot, PcDeviceModel
from predicitivecoding_amd._native import call
from tests.test_gpu_shared_rows import network, settle

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def product(A, B, ta=0, tb=1):
    """C = op(A) op(B) of the operands stored for (ta, tb); 2048 x 2048 outputs fill every CU with a 128 x 128 tile."""
    (m, k), n = A.shape, B.shape[0]
    C = torch.empty((m, n), device="cuda")
    a = A.T.contiguous() if ta else A
    b = B if tb else B.T.contiguous()
    call("pcd_gemm_f32", a.data_ptr(), b.data_ptr(), C.data_ptr(), m, k, n, ta, tb, 0.0, None)
    torch.cuda.synchronize()
    return C


def operands(k, seed, m=2048, n=2048):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((m, k), generator=g, device="cuda"), torch.randn((n, k), generator=g, device="cuda"))


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 1), (1, 0)])
@pytest.mark.parametrize("special", [INF, NAN, 3.4e38])
def test_neighbours_keep_their_bits(ta, tb, special):
    A, B = operands(208, 7)
    C0 = product(A, B, ta, tb)
    rows, cols = [0, 37, 64, 127, 1000], [5, 96, 1151, 2047]
    for i, r in enumerate(rows):
        A[r, (17 * i) % 208] = special
    for i, c in enumerate(cols):
        B[c, 207 - 50 * i] = special
    C = product(A, B, ta, tb)
    keep_r = torch.tensor([r for r in range(2048) if r not in rows], device="cuda")
    keep_c = torch.tensor([c for c in range(2048) if c not in cols], device="cuda")
    assert torch.equal(C[keep_r][:, keep_c], C0[keep_r][:, keep_c])
    ref32 = (A.double() @ B.double().T).float()
    for part in (lambda v: v[rows][:, keep_c], lambda v: v[keep_r][:, cols]):
        assert torch.equal(torch.isnan(part(C)), torch.isnan(part(ref32)))
        assert torch.equal(torch.isinf(part(C)), torch.isinf(part(ref32)))


def model128(sizes, act, **kw):
    model = PcDeviceModel(network(sizes, act, **kw), "f32")
    for k, v in (("tile", 128), ("split_k", 0)):
        model.set_option(k, v)
    return model


SIZES = [150, 260, 140, 60]


@pytest.mark.parametrize("shared", [0, 1])
@pytest.mark.parametrize("special", [INF, NAN, 3.4e38])
def test_settling_rows_do_not_interact(shared, special):
    """The other rows' bits, and the row's own infinities, NaNs and finite values as on the 64 x 64 tile, which
    multiplies in fp32."""
    x = torch.randn(300, SIZES[0], generator=torch.Generator().manual_seed(1)).cuda()
    y = x.clone()
    y[7, 3] = special
    if special != 3.4e38:
        y[200] = special
    keep = [r for r in range(300) if r not in (7, 200)]
    model = model128(SIZES, 2)
    model.set_option("shared_rows", shared)
    for steps in (1, 2, 5):
        (top, states, energy), (top1, states1, energy1) = settle(model, x, steps), settle(model, y, steps)
        np.testing.assert_array_equal(top[keep], top1[keep])
        np.testing.assert_array_equal(energy[:, keep], energy1[:, keep])
        model.set_option("tile", 64)
        other = settle(model, y, steps)
        model.set_option("tile", 128)
        for a, b in zip((top1, states1, energy1), other):
            np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
            np.testing.assert_array_equal(np.isinf(a), np.isinf(b))
            ok = np.isfinite(a)
            assert np.max(np.abs(a[ok] - b[ok]) / (1 + np.abs(b[ok]))) <= 1e-5   # fp32 sums of up to 260 products, 5 steps
    model.close()


def test_ragged_order_does_not_matter():
    """Requests beside one that overflows, in either packing."""
    steps = np.array([6, 1, 4, 2, 6, 3] * 50, np.int32)
    x = torch.randn(300, SIZES[0], generator=torch.Generator().manual_seed(2))
    x[3] = INF
    x[100, 5] = NAN
    model = model128(SIZES, 2)
    out = []
    for order in (0, 1):
        model.set_option("ragged_order", order)
        out.append(model.relax_ragged(x.numpy(), np.arange(301, dtype=np.int32), steps))
    for a, b in zip(*out):
        np.testing.assert_array_equal(np.asarray(a), np.asarray(b))
    model.close()


# magnitudes from where three bf16 pieces hold every fp32 bit to the smallest subnormals; in every layout, as the
# operand's fragments come out of LDS in two ways
@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 1), (1, 0)])
@pytest.mark.parametrize("scale", [1e-32, 1e-33, 1e-34, 1e-36, 1e-38, 1e-41])
def test_small_operands_keep_their_bits(ta, tb, scale):
    """An operand whose third bf16 piece would be below bf16's range takes the fp32 MFMAs, in rows and in columns: one
    rounding (2^-24 / sqrt(3) in the mean square) per two of K = 64 elements, twice that."""
    A, B = operands(64, 9)
    A[:700] *= scale
    A[700:] *= 1e25
    A[1500, 63] = scale
    B[1900:] *= scale
    C, ref = product(A, B, ta, tb), A.double() @ B.double().T
    bound = 2 * 2.0 ** -24 / np.sqrt(3.0) * np.sqrt(64 / 2 + 1)
    parts = [(slice(700, 2048), slice(1900, 2048)), (slice(700, 2048), slice(0, 1900)), (1500, slice(0, 2048))]
    if scale > 1e-37:   # the products themselves in the normal range
        parts.append((slice(0, 700), slice(0, 1900)))
    for r, c in parts:
        err = (C[r, c].double() - ref[r, c]).norm() / ref[r, c].norm()
        assert float(err) <= bound, (r, c, float(err), bound)


@pytest.mark.parametrize("which", ["row", "column"])
@pytest.mark.parametrize("k", [0, 15, 16, 33, 207])
def test_one_small_operand_is_found_wherever_it_lies(which, k):
    """A single product is one rounding from exact; its neighbours keep their bits.  K elements of the first, middle and
    last stages; rows and columns of each of the waves' blocks."""
    A, B = operands(208, 3)
    C0 = product(A, B)
    at = torch.tensor([1, 33, 65, 97, 128 + 50, 2047], device="cuda")
    v = torch.full((6,), 1.2345678e-36, device="cuda")
    X, Y = (A, B) if which == "row" else (B, A)
    X[at] = 0.0
    X[at, k] = v
    Y[300, k] = 3.1415926e30
    C = product(A, B)
    got = C[at, 300] if which == "row" else C[300, at]
    want = v.double() * Y[300, k].double()
    assert float(((got.double() - want) / want).abs().max()) <= 2.0 ** -24
    keep = torch.ones(2048, dtype=torch.bool, device="cuda")
    keep[at] = False
    other = torch.ones(2048, dtype=torch.bool, device="cuda")
    other[300] = False
    a, b = (keep, other) if which == "row" else (other, keep)
    assert torch.equal(C[a][:, b], C0[a][:, b])


def test_small_states_settle_as_on_the_64_tile():
    """A linear network without biases scales: inputs of 2^-121 give the settling of unit inputs, scaled, where the
    64 x 64 tile's fp32 MFMAs do."""
    net = GenerativeSnapshot(SIZES, 0, 0.1, 0.0, False, network(SIZES, 0).weights,
                             [np.zeros(n, np.float32) for n in SIZES[:-1]])
    x = torch.randn(300, SIZES[0], generator=torch.Generator().manual_seed(4)).cuda()
    model = PcDeviceModel(net, "f32")
    model.set_option("tile", 128)
    unit = settle(model, x, 5)[0].astype(np.float64)
    small = settle(model, x * 2.0 ** -121, 5)[0].astype(np.float64) * 2.0 ** 121
    model.close()
    # fp32 roundings of 5 steps, and of states near 2^-126 to multiples of 2^-149: 2^-23 of them
    assert np.linalg.norm(small - unit) / np.linalg.norm(unit) <= 2e-6
