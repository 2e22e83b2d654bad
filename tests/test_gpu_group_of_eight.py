"""Group correlation with groups of eight channels on the tiled kernels: a group is two lanes of a
pixel.  Every width, both reduces, ragged images and view counts, the default fill of the
cost-map layer, 16-bit storage, against the oracle; the maximum bit for bit."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import quantise, random_cameras
from gpu_util import TORCH_DTYPE, assert_backward_close, assert_forward_close, dev, host, rms

pytestmark = pytest.mark.gpu


def _tensors(seed, B, N, H, W, C, D, storage="f32"):
    rng = np.random.default_rng(seed)
    f32 = np.float32
    ref = quantise(rng.standard_normal((B, H, W, C)).astype(f32), storage)
    src = quantise(rng.standard_normal((B, N, H, W, C)).astype(f32), storage)
    depth = rng.uniform(3.0, 3.3, (B, H, W, 1)) + np.linspace(0.0, 3.0, D)
    Rs, Ts = random_cameras(rng, B, N, H, W, 6.0, 0.3)
    return rng, (ref, src, depth.astype(f32), Rs.astype(f32), Ts.astype(f32))


@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
@pytest.mark.parametrize("C,N,H,W,D", [(8, 1, 13, 21, 5), (8, 3, 512, 652, 2), (16, 4, 15, 19, 9),
                                       (32, 6, 17, 23, 11), (32, 3, 9, 30, 8), (64, 2, 14, 15, 19)])
def test_group_of_eight(oracle, C, N, H, W, D, reduce):
    rng, args = _tensors(C + N, 1, N, H, W, C, D)
    G = C // 8
    print("\n[case] C%d N%d %dx%d D%d %s" % (C, N, H, W, D, reduce), flush=True)
    lib = _lib.load()
    d_args = [dev(x) for x in args]
    want, want_mask = oracle.cost_volume_v2_fwd(*args, reduce, G)
    cost, mask = chop.cost_volume_v2_raw(*d_args, reduce, G)
    assert lib.chop_last_kernel_family() == 2
    assert np.array_equal(host(mask), want_mask)
    if reduce == "MIN":
        assert np.array_equal(host(cost), want)
    else:
        assert_forward_close(host(cost), want, atol=1e-5)
    cg = rng.standard_normal(want.shape).astype(np.float32)
    got = chop.cost_volume_grad_v2(*d_args, dev(cg), mask, reduce, G)
    assert lib.chop_last_kernel_family() == 2
    for g, w in zip(got, oracle.cost_volume_v2_bwd(*args, cg, want_mask, reduce, G)):
        assert_backward_close(host(g), w)


@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
@pytest.mark.parametrize("storage", ["f16", "bf16"])
def test_group_of_eight_16bit(oracle, storage, reduce):
    rng, args = _tensors(5, 2, 3, 11, 25, 32, 9, storage)
    td = TORCH_DTYPE[storage]
    d_args = [dev(args[0], td), dev(args[1], td)] + [dev(x) for x in args[2:]]
    print("\n[case] %s %s" % (storage, reduce), flush=True)
    want, want_mask = oracle.cost_volume_v2_fwd(*args, reduce, 4)
    cost, mask = chop.cost_volume_v2_raw(*d_args, reduce, 4)
    assert _lib.load().chop_last_kernel_family() == 2
    assert np.array_equal(host(mask), want_mask)
    seen = want_mask > 0 if reduce == "MEAN" else want_mask >= 0
    seen = np.broadcast_to(seen if seen.ndim == want.ndim else seen[..., None], want.shape)
    # one rounding to the storage type: 8 significant bits at the least, 1e-2 of the value
    np.testing.assert_allclose(host(cost)[seen], want[seen], rtol=1e-2, atol=1e-2 * rms(want[seen]))
    cg = quantise(rng.standard_normal(want.shape).astype(np.float32), storage)
    got = chop.cost_volume_grad_v2(*d_args, dev(cg, td), mask, reduce, 4)
    for g, w in zip(got, oracle.cost_volume_v2_bwd(*args, cg, want_mask, reduce, 4)):
        np.testing.assert_allclose(host(g), w, rtol=1e-2, atol=1e-2 * rms(w))
