"""The native host path behind the differentiable functions: inputs as callers hand them over
(strided views, host arrays), gradients of a subset of the inputs, a graph used twice."""
import numpy as np
import pytest
import torch

import custom_helper_op_amd as chop
from custom_helper_op_amd.configs import reference_test_case
from gpu_util import dev, host

pytestmark = pytest.mark.gpu

KEYS = ("ref", "src", "base_plane", "offsets", "Rs", "Ts")


@pytest.mark.parametrize("wanted", [(0,), (1,), (2,), (0, 1, 2)])
def test_gradients_of_a_subset_and_of_strided_inputs(wanted):
    print("\n[case] wanted %s" % (wanted,), flush=True)
    t = reference_test_case(3, 1, 2, 6, 7, 8, 5, np.float32, seed=2)
    plain = [dev(t[k]) for k in KEYS]
    cost, mask = chop.cost_volume_raw(*plain)
    up = torch.randn_like(cost)
    want = chop.cost_volume_grad(*plain, up, mask)
    # the same values as strided views; offsets and cameras as host arrays
    ins = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in plain[:3]] + [t[k] for k in KEYS[3:]]
    for i in wanted:
        ins[i].requires_grad_(True)
    got_cost, got_mask = chop.cost_volume(*ins)
    assert torch.equal(got_cost, cost) and torch.equal(got_mask, mask) and not got_mask.requires_grad
    grads = torch.autograd.grad(got_cost, [ins[i] for i in wanted], up, retain_graph=True)
    again = torch.autograd.grad(got_cost, [ins[i] for i in wanted], up)
    for i, g, h in zip(wanted, grads, again):
        assert g.shape == plain[i].shape
        np.testing.assert_allclose(host(g), host(want[i]), rtol=1e-5, atol=1e-4)
        np.testing.assert_allclose(host(h), host(g), rtol=1e-5, atol=1e-4)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(got_cost, [ins[wanted[0]]], up)


def test_no_graph_without_a_gradient_and_saved_inputs_are_guarded():
    t = reference_test_case(1, 1, 2, 6, 7, 8, 5, np.float32, seed=3)
    ins = [dev(t[k]) for k in KEYS]
    assert not chop.cost_volume(*ins)[0].requires_grad
    ins[1].requires_grad_(True)
    with torch.no_grad():
        assert not chop.cost_volume(*ins)[0].requires_grad
    cost, _ = chop.cost_volume(*ins)
    ins[0].add_(1.0)  # the backward pass would read a changed reference image
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        cost.sum().backward()
