"""The shared reciprocal of the tiled kernels' reprojection: coordinates, accepted views and winners stay those
of two correctly rounded divisions, whatever the scale of the homogeneous coordinates (a projection and its
multiple by a power of two are the same camera), at the ends of the exponent's range, behind the camera, with
and without the half-pixel convention, where quotients near zero count."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import random_cameras
from gpu_util import assert_backward_close, dev, host

pytestmark = pytest.mark.gpu


def _tensors(real, seed=1, N=3, H=21, W=29, C=16, D=14, near=0.4, far=5.0, rot=20.0):
    rng = np.random.default_rng(seed)
    ref = rng.standard_normal((1, H, W, C)).astype(real)
    src = rng.standard_normal((1, N, H, W, C)).astype(real)
    base = rng.uniform(0.0, 0.05, (1, H, W, 1)).astype(real)
    offsets = np.linspace(near, far, D)[None].astype(real)
    Rs, Ts = (x.astype(real) for x in random_cameras(rng, 1, N, H, W, rot, 0.4))
    return rng, [ref, src, base, offsets, Rs, Ts]


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("real,power", [(np.float32, p) for p in (0, 40, -40, 70, -70, 100, -100)] +
                         [(np.float64, p) for p in (0, 520, -520, 900, -900)])
def test_scaled_cameras(oracle, real, power, half):
    rng, args = _tensors(real)
    plain = [dev(x) for x in args]
    scale = np.ldexp(real(1.0), power)
    args[4], args[5] = args[4] * scale, args[5] * scale
    d_args = [dev(x) for x in args]
    print("\n[case] %s 2^%d half %s" % (real.__name__, power, half), flush=True)
    cost, mask = chop.cost_volume_raw(*d_args, "MIN", half)
    assert _lib.load().chop_last_kernel_family() in (2, 3)
    want, want_mask = oracle.cost_volume_fwd(*args, "MIN", half)
    assert np.array_equal(host(mask), want_mask) and np.array_equal(host(cost), want)
    unscaled, unscaled_mask = chop.cost_volume_raw(*plain, "MIN", half)
    assert np.array_equal(host(mask), host(unscaled_mask)) and np.array_equal(host(cost), host(unscaled))
    cg = rng.standard_normal(want.shape).astype(real)
    got = chop.cost_volume_grad(*d_args, dev(cg), mask, "MIN", half)
    if abs(power) > (60 if real is np.float32 else 500):
        got = got[:2]  # (z * z in the depth gradient's chain leaves the range)
    for g, w in zip(got, oracle.cost_volume_bwd(*args, cg, want_mask, "MIN", half)):
        assert_backward_close(host(g), w)


@pytest.mark.parametrize("real", [np.float32, np.float64])
@pytest.mark.parametrize("half", [True, False])
def test_exact_coordinates(oracle, real, half):
    # an integer shift with divisors that are no powers of two: every quotient is exact or lies on the edge of
    # what is accepted; and cameras that put zeros, infinities and NaN into the divisions
    rng, args = _tensors(real, seed=2, N=6, rot=0.0)
    R, T = np.zeros((1, 6, 3, 3), real), np.zeros((1, 6, 3), real)
    R[:] = np.eye(3)
    for n, (k, tx) in enumerate(((3.0, 2.0), (7.0, 0.0), (0.1, 5.0))):
        R[0, n] *= real(k)
        T[0, n, 0] = 0.0
        R[0, n, 0, 2] = real(tx) * real(k)
    R[0, 3, 2, 2] = 0.0                  # divided by zero
    R[0, 4, 2, 2] = np.inf
    R[0, 5, 0, 0] = np.nan
    args[4], args[5] = R, T
    d_args = [dev(x) for x in args]
    cost, mask = chop.cost_volume_raw(*d_args, "MIN", half)
    want, want_mask = oracle.cost_volume_fwd(*args, "MIN", half)
    assert np.array_equal(host(mask), want_mask) and np.array_equal(host(cost), want)
