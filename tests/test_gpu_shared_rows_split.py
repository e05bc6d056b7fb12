"""Layers the input has not reached keep the K ranges that their problems have for the whole batch: with split-K on,
settling them once gives every sample's own bits, in the allocation-free variant near its scratch's end too."""
import numpy as np
import pytest
import torch

from predicitivecoding_amd import PcDeviceModel
from tests.test_gpu_shared_rows import both, network, settle

pytestmark = pytest.mark.gpu

# the full phases fill the GPU unsplit, their one-row problems do not; and one whose full phases split
NETS = [([768] * 5, "f32", 1732), ([2048] * 6, "bf16", 319), ([2048] * 6, "f16", 319),
        ([640, 300, 300, 300, 20], "f32", 200)]


@pytest.mark.parametrize("net", range(len(NETS)))
@pytest.mark.parametrize("ffg", [False, True])
def test_same_bits_with_split_k(net, ffg):
    sizes, dtype, batch = NETS[net]
    model = PcDeviceModel(network(sizes, 1, ffg=ffg, seed=net), dtype)
    model.set_option("k_stagger", 0)   # a row tile's stagger is not the one row's
    x = torch.randn(batch, sizes[0], generator=torch.Generator().manual_seed(net)).cuda()
    for steps in (1, 3, len(sizes) + 1):
        (top, states, energy), every = both(model, x, steps)
        for a, b in zip((top, states, energy), every):
            np.testing.assert_array_equal(a, b, err_msg=f"steps {steps}")
        model.set_option("shared_rows", 1)
        for a, b in zip(settle(model, x, steps, noalloc=True), every):
            np.testing.assert_array_equal(a, b, err_msg=f"allocation-free, steps {steps}")
    model.close()


@pytest.mark.parametrize("net", [0, 1, 2])
def test_warm_start_errors_are_zero(net):
    """A layer that the feed-forward sweep set and nothing below has moved stays where it is, to the bit: its errors
    are exactly zero.  After step t that holds from layer t + 2 on."""
    sizes, dtype, batch = NETS[net]
    model = PcDeviceModel(network(sizes, 1, ffg=True, seed=net), dtype)
    x = torch.randn(batch, sizes[0], generator=torch.Generator().manual_seed(net)).cuda()
    one, two = (settle(model, x, steps)[1] for steps in (1, 2))
    at = batch * sum(sizes[:4])   # the states lie layer by layer
    assert np.abs(one[at - batch * sizes[3]:at]).max() > 0
    np.testing.assert_array_equal(one[batch * sum(sizes[:3]):at], two[batch * sum(sizes[:3]):at])
    model.close()


@pytest.mark.parametrize("net", range(len(NETS)))
def test_default_options_agree_to_rounding(net):
    """With the K stagger the one row sums in row tile 0's order.  16 bits: where that turns a state copy's rounding
    (2^-8 of it in bf16, 2^-11 in f16) it enters the neighbours by eta = 0.1 through weight rows and columns of norm 1,
    once in each of 8 steps.  fp32: bit for bit, it has no stagger."""
    sizes, dtype, batch = NETS[net]
    model = PcDeviceModel(network(sizes, 1, seed=net), dtype)
    x = torch.randn(batch, sizes[0], generator=torch.Generator().manual_seed(net)).cuda()
    tol = {"f32": 0.0, "bf16": 8 * 0.1 * 2.0**-8, "f16": 8 * 0.1 * 2.0**-11}[dtype]
    for a, b in zip(*both(model, x, 8)):
        assert np.max(np.abs(a - b) / (1 + np.abs(b))) <= tol
    model.close()
