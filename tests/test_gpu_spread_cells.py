"""Gradients of sweeps whose consecutive hypotheses land many texels apart (few planes close to
the cameras): the cells of a chunk of depths do not fit the scatter window of the tiled kernels
together, so the window follows the runs depth by depth, and on strongly magnified views single
cells go to memory by themselves.  Every width of the tiled kernels, against the oracle."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import random_cameras
from gpu_util import assert_backward_close, dev, host

pytestmark = pytest.mark.gpu


def _tensors(seed, B, N, H, W, C, D, near, far, rot, shift, f32=np.float32):
    rng = np.random.default_rng(seed)
    ref = rng.standard_normal((B, H, W, C)).astype(f32)
    src = rng.standard_normal((B, N, H, W, C)).astype(f32)
    base = rng.uniform(0.0, 0.05, (B, H, W, 1)).astype(f32)
    offsets = np.tile(np.linspace(near, far, D), (B, 1)).astype(f32)
    Rs, Ts = random_cameras(rng, B, N, H, W, rot, shift)
    return rng, (ref, src, base, offsets, Rs.astype(f32), Ts.astype(f32))


# near / far / rotation / shift: far apart; so close that a tile's own cells outgrow the window;
# spread near hypotheses followed by dense far ones (both forms in one walk)
SWEEPS = {"apart": (1.7, 16.0, 8.0, 0.4), "magnified": (0.3, 1.2, 25.0, 0.2),
          "mixed": (0.4, 60.0, 12.0, 0.3)}


@pytest.mark.parametrize("sweep", sorted(SWEEPS))
@pytest.mark.parametrize("C", [4, 8, 16, 32, 64])
def test_spread_cells(oracle, C, sweep):
    near, far, rot, shift = SWEEPS[sweep]
    N, D = (6, 19) if sweep == "mixed" else (2, 11)
    rng, args = _tensors(C, 1, N, 37, 51, C, D, near, far, rot, shift)
    d_args = [dev(x) for x in args]
    lib = _lib.load()
    for reduce in ("MEAN", "MIN"):
        print("\n[case] C%d %s %s" % (C, sweep, reduce), flush=True)
        cost, mask = oracle.cost_volume_fwd(*args, reduce)
        cg = rng.standard_normal(cost.shape).astype(np.float32)
        want = oracle.cost_volume_bwd(*args, cg, mask, reduce)
        for window in (0, 6, 8):
            lib.chop_set_backward_window(window)
            try:
                got = chop.cost_volume_grad(*d_args, dev(cg), dev(mask), reduce)
            finally:
                lib.chop_set_backward_window(0)
            assert lib.chop_last_kernel_family() == 2
            for g, w in zip(got, want):
                assert_backward_close(host(g), w)
        cost, mask = oracle.cost_aggregate_fwd(*args, reduce)
        cg = rng.standard_normal(cost.shape).astype(np.float32)
        got = chop.cost_aggregate_grad(*d_args, dev(cg), dev(mask), reduce)
        for g, w in zip(got, oracle.cost_aggregate_bwd(*args, cg, mask, reduce)):
            assert_backward_close(host(g), w)
        a2 = (args[0], args[1], args[2] + args[3][:, None, None, :], args[4], args[5])
        cost, mask = oracle.cost_volume_v2_fwd(*a2, reduce, C // 4)
        cg = rng.standard_normal(cost.shape).astype(np.float32)
        got = chop.cost_volume_grad_v2(*[dev(x) for x in a2], dev(cg), dev(mask), reduce, C // 4)
        for g, w in zip(got, oracle.cost_volume_v2_bwd(*a2, cg, mask, reduce, C // 4)):
            assert_backward_close(host(g), w)
        if C >= 8:
            cost, mask = oracle.cost_volume_v3_fwd(*args, reduce, C // 4)
            cg = rng.standard_normal(cost.shape).astype(np.float32)
            got = chop.cost_volume_grad_v3(*d_args, dev(cg), dev(mask), reduce, C // 4)
            for g, w in zip(got, oracle.cost_volume_v3_bwd(*args, cg, mask, reduce, C // 4)):
                assert_backward_close(host(g), w)
    mapped, mask = oracle.feature_aggregate_fwd(*args[1:])
    cg = rng.standard_normal(mapped.shape).astype(np.float32)
    got = chop.feature_aggregate_grad(*d_args[1:], dev(cg), dev(mask))
    for g, w in zip(got, oracle.feature_aggregate_bwd(*args[1:], cg, mask)):
        assert_backward_close(host(g), w)


@pytest.fixture
def tiles():
    """The tiled kernels wherever they can serve the shape, also where a lane per channel is the faster one."""
    lib = _lib.load()
    lib.chop_set_kernel_family(3)
    yield lib
    lib.chop_set_kernel_family(0)


@pytest.mark.parametrize("sweep", sorted(SWEEPS))
@pytest.mark.parametrize("C", [4, 8, 16, 24, 32, 64])
def test_spread_cells_float64(oracle, tiles, C, sweep):
    """The same sweeps in float64, whose windows are smaller (six rows at 32 channels, four in
    CostAggregate) and whose lanes own two pairs of channels apart: runs that end outside the window,
    windows that move inside a chunk, cells on their way to memory.  Each sum has a few hundred terms: 1e-10
    of the gradient's rms, as for the tiles on ordinary sweeps."""
    near, far, rot, shift = SWEEPS[sweep]
    N, D = (6, 19) if sweep == "mixed" else (2, 11)
    rng, args = _tensors(C, 1, N, 31, 43, C, D, near, far, rot, shift, np.float64)
    a2 = (args[0], args[1], args[2] + args[3][:, None, None, :], args[4], args[5])
    calls = [("cost_volume", args, ("MEAN",)), ("cost_volume", args, ("MIN",)),
             ("cost_aggregate", args, ("MEAN",)), ("cost_aggregate", args, ("MIN",)),
             ("cost_volume_v2", a2, ("MEAN", C // 4)), ("cost_volume_v2", a2, ("MIN", C // 2)),
             ("feature_aggregate", args[1:], ())]
    if C in (8, 16, 32, 64):
        calls += [("cost_volume_v3", args, ("MEAN", C // 4)), ("cost_volume_v3", args, ("MIN", C // 8))]
    for name, a, extra in calls:
        print("\n[case] C%d %s %s %s" % (C, sweep, name, extra), flush=True)
        cost, mask = getattr(oracle, name + "_fwd")(*a, *extra)
        cg = rng.standard_normal(cost.shape)
        grad = getattr(chop, {"cost_volume_v2": "cost_volume_grad_v2", "cost_volume_v3": "cost_volume_grad_v3"}
                       .get(name, name + "_grad"))
        got = grad(*[dev(x) for x in a], dev(cg), dev(mask), *extra)
        assert tiles.chop_last_kernel_shape() == 2
        for g, w in zip(got, getattr(oracle, name + "_bwd")(*a, cg, mask, *extra)):
            assert_backward_close(host(g), w, 1e-10)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("sweep", sorted(SWEEPS))
@pytest.mark.parametrize("C,sub", [(8, 1), (16, 2), (32, 1), (32, 2), (64, 2)])
def test_spread_cells_narrow_pairs(oracle, tiles, C, sub, sweep, dtype):
    """CostVolumeV3 with groups of one and two channels."""
    near, far, rot, shift = SWEEPS[sweep]
    N, D = (4, 19) if sweep == "mixed" else (2, 11)
    rng, args = _tensors(C + sub, 1, N, 27, 39, C, D, near, far, rot, shift, dtype)
    for reduce in ("MEAN", "MIN"):
        print("\n[case] C%d sub %d %s %s" % (C, sub, sweep, reduce), flush=True)
        cost, mask = oracle.cost_volume_v3_fwd(*args, reduce, C // sub)
        cg = rng.standard_normal(cost.shape).astype(dtype)
        got = chop.cost_volume_grad_v3(*[dev(x) for x in args], dev(cg), dev(mask), reduce, C // sub)
        assert tiles.chop_last_kernel_shape() == 2
        for g, w in zip(got, oracle.cost_volume_v3_bwd(*args, cg, mask, reduce, C // sub)):
            assert_backward_close(host(g), w, 1e-4 if dtype == np.float32 else 1e-10)


def test_spread_cells_views_take_turns(oracle):
    """Narrow pixels on an image large enough that the views of a tile share a workgroup."""
    rng, args = _tensors(1, 1, 2, 512, 652, 8, 3, 1.0, 9.0, 10.0, 0.4)
    cost, mask = oracle.cost_volume_fwd(*args)
    cg = rng.standard_normal(cost.shape).astype(np.float32)
    got = chop.cost_volume_grad(*[dev(x) for x in args], dev(cg), dev(mask))
    assert _lib.load().chop_last_views_per_workgroup() == 2
    for g, w in zip(got, oracle.cost_volume_bwd(*args, cg, mask)):
        assert_backward_close(host(g), w)


@pytest.mark.parametrize("C", [4, 8, 16, 32, 64])
def test_runs_of_seldom_winners(oracle, C):
    """One winner per voxel or group among six views: a view wins now and then, so its runs stay
    open while the sweep moves on and few of them end at a depth.  Dense planes (the runs left
    behind alone do not fit the window), planes far apart, and both in one sweep."""
    for near, far, rot, shift, D in ((2.0, 12.0, 4.0, 0.2, 47), SWEEPS["apart"] + (13,), SWEEPS["mixed"] + (33,)):
        print("\n[case] C%d planes %g to %g" % (C, near, far), flush=True)
        rng, args = _tensors(C + D, 1, 6, 29, 43, C, D, near, far, rot, shift)
        a2 = (args[0], args[1], args[2] + args[3][:, None, None, :], args[4], args[5])
        for name, a, groups in (("cost_aggregate", args, ()), ("cost_volume_v2", a2, (C // 4,)),
                                ("cost_volume_v3", args, (C // 4,))):
            if name == "cost_volume_v3" and C < 8:
                continue
            cost, mask = getattr(oracle, name + "_fwd")(*a, "MIN", *groups)
            cg = rng.standard_normal(cost.shape).astype(np.float32)
            grad = {"cost_aggregate": chop.cost_aggregate_grad, "cost_volume_v2": chop.cost_volume_grad_v2,
                    "cost_volume_v3": chop.cost_volume_grad_v3}[name]
            got = grad(*[dev(x) for x in a], dev(cg), dev(mask), "MIN", *groups)
            assert _lib.load().chop_last_kernel_family() == 2
            for g, w in zip(got, getattr(oracle, name + "_bwd")(*a, cg, mask, "MIN", *groups)):
                assert_backward_close(host(g), w)
