"""The 32-channel gradients with the eight-row window in its tall form (8 x 6 texels over tiles of 4 x 2
pixels): five and six views, sweeps of 32 depths and more on images that give 16384 workgroups, sizes
that no tile divides, sweeps whose samples lie far apart; and one a little too small for it, which runs the
wide form.  Against the oracle at the float32 bar."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import random_cameras
from gpu_util import assert_backward_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["v1", "aggregate_mean", "aggregate_min", "feature"])
@pytest.mark.parametrize("N,H,W,D,near,tall", [(5, 131, 99, 33, 0.6, True), (6, 75, 77, 64, 3.0, True),
                                               (5, 123, 77, 33, 0.6, False)])
def test_tall_window(oracle, op, N, H, W, D, near, tall):
    print("\n[case] %s N%d %dx%dx%d near %g" % (op, N, H, W, D, near), flush=True)
    f32, C = np.float32, 32
    rng = np.random.default_rng(N + D)
    ref, src = rng.standard_normal((1, H, W, C)).astype(f32), rng.standard_normal((1, N, H, W, C)).astype(f32)
    Rs, Ts = (x.astype(f32) for x in random_cameras(rng, 1, N, H, W, 8.0, 0.3))
    base = rng.uniform(0.0, 0.05, (1, H, W, 1)).astype(f32)
    args = (ref, src, base, np.linspace(near, 9.0, D, dtype=f32)[None], Rs, Ts)
    extra = ()
    if op == "v1":
        shape, fwd, bwd, want_bwd = (1, H, W, D, C), chop.cost_volume_raw, chop.cost_volume_grad, oracle.cost_volume_bwd
    elif op == "feature":
        args = args[1:]
        shape, fwd, bwd = (1, H, W, D, N, C), chop.feature_aggregate_raw, chop.feature_aggregate_grad
        want_bwd = oracle.feature_aggregate_bwd
    else:
        extra = ("MIN" if op.endswith("min") else "MEAN",)
        shape, fwd, bwd = (1, H, W, D), chop.cost_aggregate_raw, chop.cost_aggregate_grad
        want_bwd = oracle.cost_aggregate_bwd
    ins = [dev(x) for x in args]
    mask = fwd(*ins, *extra)[1]
    cg = rng.standard_normal(shape).astype(f32)
    got = bwd(*ins, dev(cg), mask, *extra)
    assert _lib.load().chop_last_backward_window() == 8
    # the number of workgroups as the tall form counts them: tiles of 4 x 2 pixels, views, segments
    units = -(-H // 4) * -(-W // 2) * N * _lib.load().chop_last_segments()
    assert (units >= 16384) == tall
    for g, w in zip(got, want_bwd(*args, cg, host(mask), *extra)):
        assert_backward_close(host(g), w)
