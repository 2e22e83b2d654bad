"""Launches with few pixel tiles: the depth segments are rounded down to whole chunks (one more
segment than asked for, the last one ragged).  Sizes on both sides of that rule, against the oracle."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import random_cameras
from gpu_util import assert_backward_close, assert_forward_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,H,W,D", [(64, 6, 9, 135), (64, 7, 10, 36), (64, 5, 6, 16), (32, 9, 11, 45),
                                     (32, 9, 11, 17), (16, 13, 15, 54), (8, 12, 14, 17), (4, 9, 17, 23)])
def test_few_tiles(oracle, C, H, W, D):
    rng = np.random.default_rng(C + D)
    f32 = np.float32
    N = 3
    ref, src = rng.standard_normal((1, H, W, C)).astype(f32), rng.standard_normal((1, N, H, W, C)).astype(f32)
    base = rng.uniform(0.0, 0.05, (1, H, W, 1)).astype(f32)
    Rs, Ts = random_cameras(rng, 1, N, H, W, 5.0, 0.2)
    args = (ref, src, base, np.linspace(3.0, 9.0, D, dtype=f32)[None], Rs.astype(f32), Ts.astype(f32))
    d_args = [dev(x) for x in args]
    for reduce in ("MEAN", "MIN"):
        print("\n[case] C%d %dx%d D%d %s" % (C, H, W, D, reduce), flush=True)
        want, want_mask = oracle.cost_volume_fwd(*args, reduce)
        cost, mask = chop.cost_volume_raw(*d_args, reduce)
        assert _lib.load().chop_last_kernel_family() == 2
        assert np.array_equal(host(mask), want_mask)
        assert_forward_close(host(cost), want)
        cg = rng.standard_normal(want.shape).astype(f32)
        got = chop.cost_volume_grad(*d_args, dev(cg), mask, reduce)
        for g, w in zip(got, oracle.cost_volume_bwd(*args, cg, want_mask, reduce)):
            assert_backward_close(host(g), w)
