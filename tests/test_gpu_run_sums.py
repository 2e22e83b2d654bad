"""Gradients of group correlation that keep one set of tap sums per group of two, four and eight channels
while a cell lasts: runs that end in the window, outside it, at a chunk's and at the sweep's end, views
that take turns, idle lanes, without the depth gradient, against the oracle."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import random_cameras
from gpu_util import assert_backward_close, dev, host

pytestmark = pytest.mark.gpu

# near / far / rotation / shift of the sweep: one cell for many depths, one cell per depth, cells outside
# every window position
SWEEPS = {"dense": (3.0, 3.4, 6.0, 0.3), "apart": (1.7, 16.0, 8.0, 0.4), "magnified": (0.3, 1.2, 25.0, 0.2)}


def _tensors(seed, B, N, H, W, C, D, near, far, rot, shift, real=np.float32):
    rng = np.random.default_rng(seed)
    ref = rng.standard_normal((B, H, W, C)).astype(real)
    src = rng.standard_normal((B, N, H, W, C)).astype(real)
    depth = rng.uniform(0.0, 0.05, (B, H, W, 1)) + np.linspace(near, far, D)
    Rs, Ts = random_cameras(rng, B, N, H, W, rot, shift)
    return rng, (ref, src, depth.astype(real), Rs.astype(real), Ts.astype(real))


@pytest.mark.parametrize("sweep", sorted(SWEEPS))
@pytest.mark.parametrize("C,sub,real", [(4, 2, "f4"), (8, 2, "f4"), (8, 4, "f4"), (16, 2, "f4"), (16, 8, "f4"),
                                        (24, 2, "f4"), (28, 4, "f4"), (32, 2, "f4"), (32, 4, "f4"), (64, 2, "f4"),
                                        (64, 8, "f4"), (16, 2, "f8"), (24, 4, "f8"), (32, 2, "f8")])
def test_run_sums(oracle, C, sub, real, sweep):
    D = {4: 1, 8: 7, 16: 9, 24: 8, 28: 19, 32: 19, 64: 17}[C]
    rng, args = _tensors(C + sub, 2, 3, 19, 26, C, D, *SWEEPS[sweep], np.dtype(real).type)
    d_args, G = [dev(x) for x in args], C // sub
    for reduce in ("MEAN", "MIN"):
        print("\n[case] C%d sub%d %s %s %s" % (C, sub, real, sweep, reduce), flush=True)
        cost, mask = oracle.cost_volume_v2_fwd(*args, reduce, G)
        cg = rng.standard_normal(cost.shape).astype(real)
        want = oracle.cost_volume_v2_bwd(*args, cg, mask, reduce, G)
        got = chop.cost_volume_grad_v2(*d_args, dev(cg), dev(mask), reduce, G)
        assert real == "f8" or _lib.load().chop_last_kernel_family() == 2
        for g, w in zip(got, want):
            assert_backward_close(host(g), w)
        got = chop.cost_volume_grad_v2(*d_args, dev(cg), dev(mask), reduce, G, need_depth_grad=False)
        for g, w in zip(got[:2], want):
            assert_backward_close(host(g), w)


@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
def test_views_in_turn(oracle, reduce):
    # (as many tiles of eight channels as let one workgroup take all views of its tile)
    rng, args = _tensors(7, 1, 2, 512, 656, 8, 3, 3.0, 3.2, 3.0, 0.2)
    d_args = [dev(x) for x in args]
    cost, mask = oracle.cost_volume_v2_fwd(*args, reduce, 4)
    cg = rng.standard_normal(cost.shape).astype(np.float32)
    got = chop.cost_volume_grad_v2(*d_args, dev(cg), dev(mask), reduce, 4)
    assert _lib.load().chop_last_views_per_workgroup() == 2
    for g, w in zip(got, oracle.cost_volume_v2_bwd(*args, cg, mask, reduce, 4)):
        assert_backward_close(host(g), w)


def test_infinite_reference_of_the_last_channel(oracle):
    # 24 channels: the idle lanes read along with the last one and must leave the next texel alone
    rng, args = _tensors(3, 1, 2, 15, 18, 24, 8, 3.0, 7.0, 6.0, 0.3)
    cost, mask = oracle.cost_volume_v2_fwd(*args, "MEAN", 12)
    cg = rng.standard_normal(cost.shape).astype(np.float32)
    want = oracle.cost_volume_v2_bwd(*args, cg, mask, "MEAN", 12)
    hot = args[0].copy()
    hot[..., -1] = np.inf
    got = chop.cost_volume_grad_v2(dev(hot), *[dev(x) for x in args[1:]], dev(cg), dev(mask), "MEAN", 12)
    assert_backward_close(host(got[0]), want[0])
    assert_backward_close(host(got[1])[..., :-1], want[1][..., :-1])
