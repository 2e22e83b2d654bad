"""CostVolumeV3 on the tiled kernels for every group width they take (1, 2, 4, 8 channels), float32 and
float64: forward cost and pairs to the bit of the oracle, gradients at the type's bar; ties (constant
images, doubled groups) and features that hold infinities, NaN and zeros, where the search of one
channel per group goes by the reference's largest and smallest value."""
import numpy as np
import pytest

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import reference_test_case
from gpu_util import assert_backward_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _tiles():
    """Every call on the tiled kernels, also those for which another is the faster one."""
    _lib.load().chop_set_kernel_family(3)
    yield
    _lib.load().chop_set_kernel_family(0)


KEYS = ("ref", "src", "base_plane", "offsets", "Rs", "Ts")


def _case(C, N, H, W, D, dtype, values, seed):
    t = reference_test_case(3, 1, N, H, W, C, D, dtype, seed=seed)
    rng = np.random.default_rng(seed)
    t["ref"] = rng.standard_normal(t["ref"].shape).astype(dtype)
    t["src"] = rng.standard_normal(t["src"].shape).astype(dtype)
    if values == "ties":
        t["ref"][..., : C // 2] = np.round(t["ref"][..., : C // 2])
        t["ref"][..., C // 2:] = t["ref"][..., : C // 2]
        t["src"] = np.ones_like(t["src"]) * np.sign(t["src"][..., :1])
    if values == "specials":
        for x in (t["ref"], t["src"]):
            hit = rng.random(x.shape)
            x[hit < 0.02], x[(hit > 0.02) & (hit < 0.05)] = np.inf, 0.0
            x[(hit > 0.05) & (hit < 0.07)], x[(hit > 0.07) & (hit < 0.08)] = -np.inf, np.nan
        t["ref"][0, 0, 0] = np.nan
        t["ref"][0, 1, 1] = -np.abs(t["ref"][0, 1, 1])
    return tuple(t[k] for k in KEYS)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("C", [8, 16, 32, 64])
@pytest.mark.parametrize("sub", [1, 2, 4, 8])
@pytest.mark.parametrize("values", ["normal", "ties", "specials"])
def test_narrow_groups(oracle, C, sub, dtype, values):
    G = C // sub
    for N, H, W, D in ((1, 9, 7, 5), (3, 6, 11, 19), (6, 5, 7, 8)):
        print("\n[case] C%d sub%d %s %s N%d" % (C, sub, np.dtype(dtype).name, values, N), flush=True)
        args = _case(C, N, H, W, D, dtype, values, C + N)
        ins = [dev(x) for x in args]
        for reduce in ("MEAN", "MIN"):
            with np.errstate(all="ignore"):
                want, want_mask = oracle.cost_volume_v3_fwd(*args, reduce, G)
            cost, mask = chop.cost_volume_v3_raw(*ins, reduce, G)
            assert _lib.load().chop_last_kernel_family() == (2 if dtype == np.float32 else 3)
            assert _lib.load().chop_last_kernel_shape() == 2
            assert np.array_equal(host(mask), want_mask)
            assert np.array_equal(host(cost), want, equal_nan=True)
            if values == "specials":
                continue  # (a gradient of infinities is NaN wherever it lands)
            cg = np.random.default_rng(1).standard_normal(want.shape).astype(dtype)
            got = chop.cost_volume_grad_v3(*ins, dev(cg), dev(want_mask), reduce, G)
            assert _lib.load().chop_last_kernel_shape() == 2
            for g, w in zip(got, oracle.cost_volume_v3_bwd(*args, cg, want_mask, reduce, G)):
                assert_backward_close(host(g), w, 1e-4 if dtype == np.float32 else 1e-10)
