"""Forward launches whose last depth segment is a short one: all first segments of a band of tiles go before
all second ones (not the narrow pixels').  Every width of a pixel, sizes that no tile and no band divides, one tile more or less than
a multiple of eight, against the oracle: to the bit where the evaluation is the plain one (minima, samples,
best pairs, float64), the float32 mean at its 1e-5."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import random_cameras
from gpu_util import assert_forward_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _tiles(request):
    print("\n[case] %s" % request.node.nodeid, flush=True)
    _lib.load().chop_set_kernel_family(3)
    yield
    _lib.load().chop_set_kernel_family(0)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("C,H,W,D", [(8, 23, 41, 7), (16, 33, 29, 9), (24, 17, 37, 18), (32, 18, 36, 17), (32, 2, 29, 9),
                                     (32, 2, 33, 35), (64, 11, 13, 19)])
def test_uneven_segments(oracle, C, H, W, D, dtype):
    N, lib = 3, _lib.load()
    rng = np.random.default_rng(C + D)
    ref, src = rng.standard_normal((2, H, W, C)).astype(dtype), rng.standard_normal((2, N, H, W, C)).astype(dtype)
    base = rng.uniform(0.0, 0.05, (2, H, W, 1)).astype(dtype)
    offsets = np.tile(np.linspace(1.5, 9.0, D), (2, 1)).astype(dtype)
    Rs, Ts = (x.astype(dtype) for x in random_cameras(rng, 2, N, H, W, 6.0, 0.3))
    args = (ref, src, base, offsets, Rs, Ts)
    grid = (ref, src, base + offsets[:, None, None, :], Rs, Ts)
    in_turn = 0
    for name, a, extra in (("cost_volume", args, ("MEAN",)), ("cost_volume", args, ("MIN",)),
                           ("cost_volume_v2", grid, ("MIN", C // 4)), ("cost_aggregate", args, ("MEAN",)),
                           ("cost_aggregate", args, ("MIN",)), ("cost_volume_v3", args, ("MIN", C // 4)),
                           ("feature_aggregate", args[1:], ())):
        if name == "cost_volume_v3" and C == 24:
            continue
        want, want_mask = getattr(oracle, name + "_fwd")(*a, *extra)
        got, mask = getattr(chop, name + "_raw")(*[dev(x) for x in a], *extra)
        assert lib.chop_last_kernel_shape() == 2
        in_turn += lib.chop_last_segments() < 0
        assert np.array_equal(host(mask), want_mask), name
        if "MEAN" in extra and dtype == np.float32 and C != 24:
            assert_forward_close(host(got), want)
        else:
            assert np.array_equal(host(got), want), name
    assert in_turn == (0 if C == 8 else 6 if C == 24 else 7)
