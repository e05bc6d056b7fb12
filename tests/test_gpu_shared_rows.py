"""Layers the input has not reached, settled once for the whole batch (option shared_rows), against settling every
sample's own: the same sums in the same order, so the same bits where no tile-dependent order is in play (split-K and
the K stagger off)."""
import numpy as np
import pytest
import torch

from predicitivecoding_amd import GenerativeSnapshot, PcDeviceModel

pytestmark = pytest.mark.gpu


def network(sizes, act, ffg=False, lam=0.0, precisions=None, seed=0):
    rng = np.random.default_rng(seed)
    W = [rng.standard_normal((a, b)).astype(np.float32) * np.float32(1.0 / np.sqrt(b)) for a, b in zip(sizes, sizes[1:])]
    b = [rng.standard_normal(a).astype(np.float32) * np.float32(0.2) for a in sizes[:-1]]
    return GenerativeSnapshot(sizes, act, 0.1, lam, ffg, W, b, precisions)


def settle(model, x, steps, noalloc=False):
    """(top, states, energy) of one settling of device rows, as host arrays."""
    from predicitivecoding_amd._native import call
    B, s = x.shape[0], model.sizes
    top = torch.full((B, s[-1]), 7.0, device="cuda")
    states, energy = torch.full((B * sum(s),), 7.0, device="cuda"), torch.full((steps, B), 7.0, device="cuda")
    args = (model.handle, x.data_ptr(), B, steps, top.data_ptr(), states.data_ptr(), energy.data_ptr(), None)
    call("pcd_pc_relax_noalloc" if noalloc else "pcd_pc_relax", *args)
    torch.cuda.synchronize()
    return top.cpu().numpy(), states.cpu().numpy(), energy.cpu().numpy()


def both(model, x, steps, **kw):
    out = []
    for on in (1, 0):
        model.set_option("shared_rows", on)
        out.append(settle(model, x, steps, **kw))
    return out


SIZES = [130, 200, 65, 96, 33, 20]


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("tile,batch", [(64, 65), (64, 300), (128, 129), (128, 400), (256, 257)])
def test_shared_rows_give_every_samples_bits(dtype, tile, batch):
    """Every step count from one (no layer but the first reached) past the one at which the input reaches the top."""
    with_all = PcDeviceModel(network(SIZES, 1, lam=1e-3, precisions=[1.0, 0.5, 2.0, 1.0, 3.0, 1.0]), dtype)
    for k, v in (("tile", tile), ("split_k", 0), ("k_stagger", 0)):
        with_all.set_option(k, v)
    x = torch.randn(batch, SIZES[0], generator=torch.Generator().manual_seed(batch)).cuda()
    for steps in range(1, len(SIZES) + 2):
        for a, b in zip(*both(with_all, x, steps)):
            np.testing.assert_array_equal(a, b, err_msg=f"steps {steps}")
    with_all.close()


@pytest.mark.parametrize("act", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("ffg", [False, True])
@pytest.mark.parametrize("use_graph", [0, 1])
def test_activations_warm_start_and_graphs(act, ffg, use_graph):
    model = PcDeviceModel(network(SIZES, act, ffg=ffg, seed=act), "f32")
    for k, v in (("tile", 64), ("split_k", 0), ("use_graph", use_graph)):
        model.set_option(k, v)
    x = torch.randn(150, SIZES[0], generator=torch.Generator().manual_seed(3)).cuda()
    for steps in (2, 9):
        for noalloc in (False, True):
            for a, b in zip(*both(model, x, steps, noalloc=noalloc)):
                np.testing.assert_array_equal(a, b)
    model.close()


def test_rows_left_by_other_calls_do_not_matter():
    """A larger batch, then one whose states overflow, leave their rows in the workspace; two levels have nothing to
    share; and by default (split-K, stagger, automatic tile) the two ways agree to rounding."""
    model = PcDeviceModel(network(SIZES, 1), "f32")
    model.set_option("tile", 128)
    model.set_option("split_k", 0)
    g = torch.Generator().manual_seed(1)
    x = torch.randn(700, SIZES[0], generator=g).cuda()
    want = [v.copy() for v in settle(model, x[:200].contiguous(), 8)]
    settle(model, x, 8)
    settle(model, x * float("inf"), 3)
    for a, b in zip(settle(model, x[:200].contiguous(), 8), want):
        np.testing.assert_array_equal(a, b)
    model.close()
    two = PcDeviceModel(network([100, 70], 1), "f32")
    two.set_option("tile", 64)
    for a, b in zip(*both(two, x[:, :100].contiguous(), 3)):
        np.testing.assert_array_equal(a, b)
    two.close()
    for dtype, tol in (("f32", 1e-5), ("bf16", 2e-3)):
        wide = PcDeviceModel(network([1024] * 5, 4, seed=9), dtype)
        for a, b in zip(*both(wide, torch.randn(1100, 1024, generator=g).cuda(), 12)):
            assert np.max(np.abs(a - b) / (1 + np.abs(b))) <= tol
        wide.close()
