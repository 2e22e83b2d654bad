"""Float64 on the tile-shaped kernels: pixels of 4 to 64 channels, some lanes idle (20, 24, 28), one to
seven views (seven: the forward pass keeps a lane per channel), depth ranges that end inside a chunk.

Family 3 asks for them wherever they can serve the shape, family 2 for a lane per channel, and the shape
reported says that they ran (which of the two an unforced call takes: test_kernel_choice.py).  Forward both are the
plain evaluation: equal to each other and to the oracle to the bit.  Gradients: the sums come in
another order, each of up to a few hundred terms, so 1e-10 of the gradient's rms (the oracle's own
bar in float64) holds with three digits to spare.
"""
import numpy as np
import pytest
import torch

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import reference_test_case
from gpu_util import assert_backward_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print("\n[case] %s" % request.node.nodeid, flush=True)
    yield
    _lib.load().chop_set_kernel_family(0)


def _both(run, tiles=True):
    """`run` with the tiles asked for and with a lane per channel.  `tiles`: whether the tiles can serve it."""
    out = []
    for family, shape in ((3, 2 if tiles else 3), (2, 3)):
        _lib.load().chop_set_kernel_family(family)
        out.append([host(x) for x in run()])
        assert _lib.load().chop_last_kernel_family() == 3
        assert _lib.load().chop_last_kernel_shape() == shape
    return out


@pytest.mark.parametrize("C", [4, 8, 16, 20, 24, 28, 32, 64])
@pytest.mark.parametrize("N,H,W,D", [(1, 13, 17, 5), (2, 7, 9, 35), (4, 12, 10, 16), (7, 6, 11, 9)])
@pytest.mark.parametrize("op,reduce,groups", [("v1", "MEAN", 1), ("v1", "MIN", 1), ("v2", "MEAN", 4),
                                              ("v2", "MIN", 2), ("v2", "MEAN", "four"), ("v2", "MIN", "two"),
                                              ("aggregate", "MEAN", 1), ("aggregate", "MIN", 1),
                                              ("feature", "MEAN", 1)])
def test_tiles_against_lanes(oracle, C, N, H, W, D, op, reduce, groups):
    # (groups of a width in words: as many as the channels make of them)
    groups = {"four": C // 4, "two": C // 2}.get(groups, groups)
    can = op != "v2" or C // groups in (1, 2, 4) or (C // groups == 8 and C > 4)
    t = reference_test_case(3, 2, N, H, W, C, D, np.float64, seed=C + N)
    t["Ts"] = (t["Ts"] + np.linspace(-0.5, 0.5, N)[None, :, None]).astype(np.float64)
    args = tuple(t[k] for k in ("ref", "src", "base_plane", "offsets", "Rs", "Ts"))
    extra = (reduce,)
    if op == "v1":
        fwd, bwd = chop.cost_volume_raw, chop.cost_volume_grad
        want_fwd, want_bwd = oracle.cost_volume_fwd, oracle.cost_volume_bwd
    elif op == "aggregate":
        fwd, bwd = chop.cost_aggregate_raw, chop.cost_aggregate_grad
        want_fwd, want_bwd = oracle.cost_aggregate_fwd, oracle.cost_aggregate_bwd
    elif op == "feature":
        args, extra = args[1:], ()
        fwd, bwd = chop.feature_aggregate_raw, chop.feature_aggregate_grad
        want_fwd, want_bwd = oracle.feature_aggregate_fwd, oracle.feature_aggregate_bwd
    else:
        grid = (t["base_plane"] + t["offsets"][:, None, None, :]).astype(np.float64)
        args, extra = (t["ref"], t["src"], grid, t["Rs"], t["Ts"]), (reduce, groups)
        fwd, bwd = chop.cost_volume_v2_raw, chop.cost_volume_grad_v2
        want_fwd, want_bwd = oracle.cost_volume_v2_fwd, oracle.cost_volume_v2_bwd
    ins = [dev(x) for x in args]
    want = want_fwd(*args, *extra)
    for got in _both(lambda: fwd(*ins, *extra), can and C > 4 and N <= 6):
        for g, w in zip(got, want):
            assert np.array_equal(g, w)
    cg = np.random.default_rng(5).standard_normal(want[0].shape)
    grads = want_bwd(*args, cg, want[1], *extra)
    for got in _both(lambda: bwd(*ins, dev(cg), dev(want[1]), *extra), can):
        for g, w in zip(got, grads):
            assert_backward_close(g, w, 1e-10)


@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
@pytest.mark.parametrize("C,H,W,D", [(64, 7, 9, 11), (64, 7, 9, 12), (32, 128, 128, 5), (32, 127, 129, 5),
                                     (32, 128, 128, 6), (16, 181, 182, 2), (16, 181, 182, 3),
                                     (64, 181, 182, 12)])
def test_gradients_of_few_depths(C, H, W, D, reduce):
    """Sizes on both sides of the line below which the gradients of group correlation keep a lane per
    channel: 3/4 depth per lane of a pixel, and up to 32 channels only where the launch fills the chip.
    The oracle would take minutes at these sizes; the two families agree as above."""
    t = reference_test_case(3, 1, 2, H, W, C, D, np.float64, seed=C + D)
    grid = (t["base_plane"] + t["offsets"][:, None, None, :]).astype(np.float64)
    ins = [dev(x) for x in (t["ref"], t["src"], grid, t["Rs"], t["Ts"])]
    groups = 4 if C < 64 else 8     # (groups of sixteen channels are not on the tiles)
    cost, mask = chop.cost_volume_v2_raw(*ins, reduce, groups)
    cg = dev(np.random.default_rng(7).standard_normal(tuple(cost.shape)))
    here, lanes = _both(lambda: chop.cost_volume_grad_v2(*ins, cg, mask, reduce, groups))
    for g, w in zip(here, lanes):
        assert_backward_close(g, w, 1e-10)


@pytest.mark.parametrize("op", ["v1", "v2"])
@pytest.mark.parametrize("C,N,H,W,D", [(8, 1, 9, 7, 11), (8, 1, 9, 7, 12), (32, 2, 9, 7, 11), (32, 1, 9, 7, 11),
                                       (32, 4, 9, 7, 12), (32, 5, 9, 7, 12), (64, 2, 9, 7, 12),
                                       (64, 3, 9, 7, 12), (64, 3, 91, 91, 12), (64, 5, 91, 91, 12),
                                       (64, 6, 91, 91, 12)])
def test_lines_of_small_launches(op, C, N, H, W, D):
    """Sizes around which launches of few depths, few tiles or many views keep a lane per channel: forward
    equal to the bit, gradients as above."""
    t = reference_test_case(3, 1, N, H, W, C, D, np.float64, seed=C + N)
    if op == "v1":
        ins = [dev(t[k]) for k in ("ref", "src", "base_plane", "offsets", "Rs", "Ts")]
        fwd, bwd, extra = chop.cost_volume_raw, chop.cost_volume_grad, ("MEAN",)
    else:
        grid = (t["base_plane"] + t["offsets"][:, None, None, :]).astype(np.float64)
        ins = [dev(x) for x in (t["ref"], t["src"], grid, t["Rs"], t["Ts"])]
        fwd, bwd, extra = chop.cost_volume_v2_raw, chop.cost_volume_grad_v2, ("MEAN", 4 if C < 64 else 8)
    here, lanes = _both(lambda: fwd(*ins, *extra))
    for g, w in zip(here, lanes):
        assert np.array_equal(g, w)
    cg = dev(np.random.default_rng(9).standard_normal(here[0].shape))
    mask = dev(here[1])
    here, lanes = _both(lambda: bwd(*ins, cg, mask, *extra))
    for g, w in zip(here, lanes):
        assert_backward_close(g, w, 1e-10)


def test_gradient_reports_its_launch():
    """After a tile-shaped gradient in double: one view per workgroup, the one window there is; after any
    other gradient nothing; a forward pass in between changes neither."""
    lib = _lib.load()
    t = reference_test_case(3, 1, 2, 9, 7, 32, 9, np.float64, seed=1)
    ins = [dev(t[k]) for k in ("ref", "src", "base_plane", "offsets", "Rs", "Ts")]
    cost, mask = chop.cost_volume_raw(*ins)
    for family, views in ((3, 1), (2, 0), (3, 1), (1, 0)):
        lib.chop_set_kernel_family(family)
        chop.cost_volume_grad(*ins, cost, mask)
        lib.chop_set_kernel_family(5 - family if family > 1 else 3)
        chop.cost_volume_raw(*ins)
        assert lib.chop_last_views_per_workgroup() == views
        assert lib.chop_last_backward_window() == 0


def _shifted_view(C, H, W, shift, seed):
    """One view that sees every pixel moved by `shift` texels right and down, at the single depth 1."""
    rng = np.random.default_rng(seed)
    ref, src = rng.standard_normal((1, H, W, C)), rng.standard_normal((1, 1, H, W, C))
    Rs, Ts = np.eye(3)[None, None].copy(), np.array([shift, shift, 0.0])[None, None].copy()
    return ref, src, np.zeros((1, H, W, 1)), np.ones((1, 1)), Rs, Ts


def _gradients(op, args, cg, reduce):
    name = {"v1": "cost_volume", "aggregate": "cost_aggregate"}[op]
    ins = [dev(x) for x in args]
    _, mask = getattr(chop, name + "_raw")(*ins, reduce)
    _lib.load().chop_set_kernel_family(3)
    got = getattr(chop, name + "_grad")(*ins, dev(cg), mask, reduce)
    assert _lib.load().chop_last_kernel_shape() == 2
    return [host(g) for g in got], host(mask), name


@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
@pytest.mark.parametrize("op", ["v1", "aggregate"])
@pytest.mark.parametrize("C", [8, 16, 24, 32, 64])
def test_small_weights_keep_their_accuracy(oracle, op, C, reduce):
    """Both fractions 2^-20 short of one: the first texel receives the weight 2^-40 and nothing else.  A
    weight that is the product of its factors is right to an ulp of itself, one left over by subtraction
    to an ulp of one, 2^-12 of itself.  The bar: eight roundings of a gradient's chain, where the
    difference of sample and reference may cancel to a hundredth: 8 x 100 x 2^-53 < 1e-12."""
    args = _shifted_view(C, 6, 7, 1.0 - 2.0 ** -20, C)
    cg = np.random.default_rng(1).standard_normal((1, 6, 7, 1) + ((C,) if op == "v1" else ()))
    got, mask, name = _gradients(op, args, cg, reduce)
    want = getattr(oracle, name + "_bwd")(*args, cg, mask, reduce)
    corner, at = got[1][0, 0, 0, 0], want[1][0, 0, 0, 0]
    near = np.abs(at) > 0.01 * np.abs(at).max()
    assert near.sum() > C // 2
    np.testing.assert_allclose(corner[near], at[near], rtol=1e-12)


@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
@pytest.mark.parametrize("op", ["v1", "aggregate"])
@pytest.mark.parametrize("C", [4, 8, 16, 24, 32, 64])
def test_difference_of_a_finished_sample(oracle, op, C, reduce):
    """Samples that are small against the reference: four parts of 0.225 x 2^-52 each, whose sum changes the
    reference of one by an ulp and none of which does alone.  Every operation up to the difference is then exact
    or rounds as the plain evaluation's, so the reference's gradient is the oracle's to the bit."""
    args = list(_shifted_view(C, 6, 7, 0.5, C))
    args[0], args[1] = np.ones_like(args[0]), np.full_like(args[1], 0.9 * 2.0 ** -52)
    cg = np.ones((1, 6, 7, 1) + ((C,) if op == "v1" else ()))
    got, mask, name = _gradients(op, args, cg, reduce)
    want = getattr(oracle, name + "_bwd")(*args, cg, mask, reduce)
    plain = 2.0 / (C if op == "aggregate" else 1)
    assert np.any((want[0] != 0) & (want[0] != plain))     # (the ulp is there to be lost)
    if C in (4, 8, 16, 32, 64) or op == "v1":              # (1 / C is exact)
        assert np.array_equal(got[0], want[0])
    else:
        np.testing.assert_allclose(got[0], want[0], rtol=3e-16)


@pytest.mark.parametrize("op,C,N,sub", [("v1", 16, 1, 1), ("v2", 16, 1, 1), ("v2", 32, 2, 1), ("v2", 64, 1, 1),
                                        ("feature", 16, 3, 1)])
@pytest.mark.parametrize("H,W", [(32, 41), (256, 257)])
def test_rows_of_half_lines(op, C, N, sub, H, W):
    """Rows that leave in two stores of half a line each, through the caches (small launches) and past them
    (65536 pixels and more): the bits of the lane-per-channel kernels."""
    t = reference_test_case(3, 1, N, H, W, C, 3, np.float64, seed=C + N)
    for reduce in ("MEAN",) if op == "feature" else ("MEAN", "MIN"):
        if op == "v2":
            grid = (t["base_plane"] + t["offsets"][:, None, None, :]).astype(np.float64)
            ins = [dev(x) for x in (t["ref"], t["src"], grid, t["Rs"], t["Ts"])]
            run = lambda: chop.cost_volume_v2_raw(*ins, reduce, C // sub)
        else:
            ins = [dev(t[k]) for k in ("ref", "src", "base_plane", "offsets", "Rs", "Ts")]
            run = (lambda: chop.cost_volume_raw(*ins, reduce)) if op == "v1" else (
                lambda: chop.feature_aggregate_raw(*ins[1:]))
        tiles, lanes = _both(run)
        for g, w in zip(tiles, lanes):
            assert np.array_equal(g, w)
