"""Forward passes of 20, 24 and 28 channels on eight lanes per pixel, the last lanes idle: the same bits
as the lane-per-channel kernels, in every element type, and in float32 as the oracle."""
import numpy as np
import pytest
import torch

import custom_helper_op_amd as chop
from custom_helper_op_amd import _lib
from custom_helper_op_amd.configs import reference_test_case
from gpu_util import dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print("\n[case] %s" % request.node.nodeid, flush=True)
    yield
    _lib.load().chop_set_kernel_family(0)


@pytest.mark.parametrize("C", [20, 24, 28])
@pytest.mark.parametrize("N,H,W,D", [(1, 9, 13, 7), (2, 5, 7, 19), (3, 6, 5, 8), (6, 7, 9, 9), (7, 5, 6, 9)])
@pytest.mark.parametrize("reduce", ["MEAN", "MIN"])
def test_idle_lanes(oracle, C, N, H, W, D, reduce):
    t = reference_test_case(3, 2, N, H, W, C, D, np.float32, seed=C + N)
    t["Ts"] = (t["Ts"] + np.linspace(-0.5, 0.5, N)[None, :, None]).astype(np.float32)
    args = tuple(t[k] for k in ("ref", "src", "base_plane", "offsets", "Rs", "Ts"))
    grid = (t["base_plane"] + t["offsets"][:, None, None, :]).astype(np.float32)
    v2 = (t["ref"], t["src"], grid, t["Rs"], t["Ts"])
    fill = dev(np.float32(0.375).reshape(()))
    calls = {"v1": lambda dt: chop.cost_volume_raw(*_to(args, dt), reduce),
             "aggregate": lambda dt: chop.cost_aggregate_raw(*_to(args, None), reduce),
             "filled": lambda dt: chop.cost_aggregate_filled(*_to(args, None), fill, reduce),
             "feature": lambda dt: chop.feature_aggregate_raw(*_to(args[1:], None))}
    for sub in (1, 2, 4) + ((8,) if C == 24 else ()):
        calls["v2/%d" % sub] = lambda dt, sub=sub: chop.cost_volume_v2_raw(*_to(v2, dt), reduce, C // sub)
    want = {"v1": oracle.cost_volume_fwd(*args, reduce), "aggregate": oracle.cost_aggregate_fwd(*args, reduce),
            "feature": oracle.feature_aggregate_fwd(*args[1:]),
            "v2/4": oracle.cost_volume_v2_fwd(*v2, reduce, C // 4)}
    for name, call in calls.items():
        for dt in (None, torch.float16, torch.bfloat16) if name[0] == "v" else (None,):
            got = []
            for family, shape in ((3, 2 if N <= 6 else 3), (2, 3)):
                _lib.load().chop_set_kernel_family(family)
                got.append([host(x) for x in call(dt)[:2]])
                assert _lib.load().chop_last_kernel_family() == 3
                assert _lib.load().chop_last_kernel_shape() == shape
            for a, b in zip(*got):
                assert np.array_equal(a, b), (name, dt)
            if dt is None and name in want:
                for a, b in zip(got[0], want[name]):
                    assert np.array_equal(a, b), name


def _to(args, dtype):
    # 16-bit storage: the images only, the rest stays float32
    out = [dev(x) for x in args]
    return [x.to(dtype) if i < 2 else x for i, x in enumerate(out)] if dtype else out
