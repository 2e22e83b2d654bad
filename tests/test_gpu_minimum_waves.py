"""Gradients of the per-channel minimum in launches too large for three waves per SIMD, which take the
kernels that keep the winners as lane masks, and in small ones, which do not: ragged depths on either side
of a chunk's halves, idle lanes, 16-bit storage, with and without the depth gradient, against the oracle."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import quantise, random_cameras
from gpu_util import TORCH_DTYPE, assert_backward_close, dev, host, rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,N,H,W,D,storage", [
    (8, 4, 196, 131, 3, "f32"), (8, 4, 60, 40, 3, "f32"), (16, 4, 130, 101, 5, "f32"), (16, 3, 131, 140, 9, "bf16"),
    (16, 4, 40, 40, 7, "f16"), (24, 4, 66, 101, 11, "f32"), (32, 4, 66, 101, 4, "f32"), (32, 4, 67, 101, 13, "f32"),
    (32, 5, 58, 97, 5, "f16"), (32, 4, 30, 40, 13, "f32")])
def test_minimum(oracle, C, N, H, W, D, storage):
    rng = np.random.default_rng(C + D)
    f32 = np.float32
    ref = quantise(rng.standard_normal((1, H, W, C)).astype(f32), storage)
    src = quantise(rng.standard_normal((1, N, H, W, C)).astype(f32), storage)
    base = rng.uniform(3.0, 3.1, (1, H, W, 1)).astype(f32)
    offsets = np.linspace(0.0, 2.0, D)[None].astype(f32)
    Rs, Ts = (x.astype(f32) for x in random_cameras(rng, 1, N, H, W, 6.0, 0.3))
    args, td = (ref, src, base, offsets, Rs, Ts), TORCH_DTYPE[storage]
    d_args = [dev(ref, td), dev(src, td)] + [dev(x) for x in args[2:]]
    print("\n[case] C%d N%d %dx%dx%d %s" % (C, N, H, W, D, storage), flush=True)
    cost, mask = oracle.cost_volume_fwd(*args, "MIN")
    cg = quantise(rng.standard_normal(cost.shape).astype(f32), storage)
    want = oracle.cost_volume_bwd(*args, cg, mask, "MIN")
    for need in (True, False):
        got = chop.cost_volume_grad(*d_args, dev(cg, td), dev(mask), "MIN", need_depth_grad=need)
        assert _lib.load().chop_last_kernel_family() == 2
        for g, w in list(zip(got, want))[:3 if need else 2]:
            if storage == "f32":
                assert_backward_close(host(g), w)
            else:  # one rounding to the storage type: 8 significant bits at the least, 1e-2 of the value
                np.testing.assert_allclose(host(g), w, rtol=1e-2, atol=1e-2 * rms(w))
