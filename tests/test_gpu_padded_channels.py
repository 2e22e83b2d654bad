"""Gradients of 20, 24 and 28 channels on the tiled kernels: eight lanes of four channels per pixel,
the last of them idle.  Every op and reduce, 16-bit storage, dense and spread sweeps, against the
oracle; and an infinite last channel (the one the idle lanes read along) leaves the others alone."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import quantise, random_cameras
from gpu_util import TORCH_DTYPE, assert_backward_close, dev, host, rms

pytestmark = pytest.mark.gpu


def _tensors(seed, B, N, H, W, C, D, near, far, storage="f32"):
    rng = np.random.default_rng(seed)
    f32 = np.float32
    ref = quantise(rng.standard_normal((B, H, W, C)).astype(f32), storage)
    src = quantise(rng.standard_normal((B, N, H, W, C)).astype(f32), storage)
    base = rng.uniform(0.0, 0.05, (B, H, W, 1)).astype(f32)
    offsets = np.tile(np.linspace(near, far, D), (B, 1)).astype(f32)
    Rs, Ts = random_cameras(rng, B, N, H, W, 6.0, 0.3)
    return rng, (ref, src, base, offsets, Rs.astype(f32), Ts.astype(f32))


@pytest.mark.parametrize("near,far", [(4.0, 6.0), (0.5, 9.0)])
@pytest.mark.parametrize("C", [20, 24, 28])
def test_padded_channels(oracle, C, near, far):
    rng, args = _tensors(C, 2, 3, 21, 27, C, 13, near, far)
    d_args = [dev(x) for x in args]
    lib = _lib.load()

    def check(grad, bwd, shape, *tail):
        cg = rng.standard_normal(shape).astype(np.float32)
        got = grad(dev(cg))
        assert lib.chop_last_kernel_family() == 2
        for g, w in zip(got, bwd(cg)):
            assert_backward_close(host(g), w)

    for reduce in ("MEAN", "MIN"):
        print("\n[case] C%d %g..%g %s" % (C, near, far, reduce), flush=True)
        cost, mask = oracle.cost_volume_fwd(*args, reduce)
        check(lambda cg: chop.cost_volume_grad(*d_args, cg, dev(mask), reduce),
              lambda cg: oracle.cost_volume_bwd(*args, cg, mask, reduce), cost.shape)
        cost, mask = oracle.cost_aggregate_fwd(*args, reduce)
        check(lambda cg: chop.cost_aggregate_grad(*d_args, cg, dev(mask), reduce),
              lambda cg: oracle.cost_aggregate_bwd(*args, cg, mask, reduce), cost.shape)
        a2 = (args[0], args[1], args[2] + args[3][:, None, None, :], args[4], args[5])
        d2 = [dev(x) for x in a2]
        for G in [g for g in (C, C // 2, C // 4, C // 8) if C % g == 0 and C // g in (1, 2, 4, 8)]:
            cost, mask = oracle.cost_volume_v2_fwd(*a2, reduce, G)
            check(lambda cg: chop.cost_volume_grad_v2(*d2, cg, dev(mask), reduce, G),
                  lambda cg: oracle.cost_volume_v2_bwd(*a2, cg, mask, reduce, G), cost.shape)
    mapped, mask = oracle.feature_aggregate_fwd(*args[1:])
    check(lambda cg: chop.feature_aggregate_grad(*d_args[1:], cg, dev(mask)),
          lambda cg: oracle.feature_aggregate_bwd(*args[1:], cg, mask), mapped.shape)


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("C", [20, 24, 28])
def test_padded_channels_16bit(oracle, C, storage):
    rng, args = _tensors(C, 1, 2, 19, 22, C, 9, 3.0, 7.0, storage)
    td = TORCH_DTYPE[storage]
    cost, mask = oracle.cost_volume_fwd(*args)
    cg = quantise(rng.standard_normal(cost.shape).astype(np.float32), storage)
    got = chop.cost_volume_grad(dev(args[0], td), dev(args[1], td), *[dev(x) for x in args[2:]],
                                dev(cg, td), dev(mask))
    assert _lib.load().chop_last_kernel_family() == 2
    # one rounding to the storage type: 8 significant bits at the least, 1e-2 of the value
    for g, w in zip(got, oracle.cost_volume_bwd(*args, cg, mask)):
        np.testing.assert_allclose(host(g), w, rtol=1e-2, atol=1e-2 * rms(w))


def test_infinite_last_channel_stays_there(oracle):
    rng, args = _tensors(3, 1, 2, 15, 18, 24, 8, 3.0, 7.0)
    cost, mask = oracle.cost_volume_fwd(*args)
    cg = rng.standard_normal(cost.shape).astype(np.float32)
    want = oracle.cost_volume_bwd(*args, cg, mask)
    hot = args[1].copy()
    hot[..., -1] = np.inf
    got = chop.cost_volume_grad(dev(args[0]), dev(hot), *[dev(x) for x in args[2:]], dev(cg), dev(mask))
    assert_backward_close(host(got[0])[..., :-1], want[0][..., :-1])
    assert_backward_close(host(got[1])[..., :-1], want[1][..., :-1])
