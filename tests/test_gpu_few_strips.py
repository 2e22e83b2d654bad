"""Launches of the lane-per-channel kernels with few strips of pixels, whose depth segments are shorter
than a chunk: one depth, two, whole chunks, and the most segments a gradient is cut into; and forward
launches of the tiled kernels whose segments are single chunks.  Against the oracle: forward to the
bit (the tiled mean: its 1e-5), gradients at the bars of the element type."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import reference_test_case
from gpu_util import assert_backward_close, assert_forward_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
@pytest.mark.parametrize("C,H,W,D", [(3, 4, 4, 1), (3, 12, 16, 9), (5, 3, 5, 94), (3, 18, 19, 186), (3, 40, 50, 11),
                                     (33, 9, 11, 23), (12, 30, 40, 17), (8, 11, 13, 7), (32, 8, 9, 41)])
def test_few_strips(oracle, C, H, W, D, reduce, dtype):
    print("\n[case] %d %dx%dx%d %s %s" % (C, H, W, D, reduce, np.dtype(dtype).name), flush=True)
    t = reference_test_case(3, 1, 3, H, W, C, D, dtype, seed=C + D)
    args = tuple(t[k] for k in ("ref", "src", "base_plane", "offsets", "Rs", "Ts"))
    ins = [dev(x) for x in args]
    want_cost, mask = oracle.cost_volume_fwd(*args, reduce)
    cost, got_mask = chop.cost_volume_raw(*ins, reduce)
    assert np.array_equal(host(got_mask), mask)
    if _lib.load().chop_last_kernel_family() == 3 or reduce == "MIN":
        assert np.array_equal(host(cost), want_cost)
    else:
        assert_forward_close(host(cost), want_cost)
    cg = np.random.default_rng(2).standard_normal(want_cost.shape).astype(dtype)
    got = chop.cost_volume_grad(*ins, dev(cg), dev(mask), reduce)
    want = oracle.cost_volume_bwd(*args, cg, mask, reduce)
    for g, w in zip(got, want):
        assert_backward_close(host(g), w, 1e-4 if dtype == np.float32 else 1e-10)
