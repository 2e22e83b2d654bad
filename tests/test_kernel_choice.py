"""Which kernels a call is given to.  The choice is made on the host, from sizes, types and pointer
alignment alone, before anything is launched: without a GPU the launch then fails, and
`chop_last_kernel_shape` says what it would have run (1 a thread per element, 2 tile-shaped, 3 a lane per
channel).  Never run where there is a GPU: the pointers are no pointers."""
import ctypes

import pytest
import torch

from custom_helper_op_amd import _lib

pytestmark = pytest.mark.skipif(torch.cuda.device_count() > 0, reason="made-up pointers: only without a GPU")
GENERAL, TILES, LANES = 1, 2, 3
REDUCE = {"MEAN": 0, "MIN": 1}


@pytest.fixture(autouse=True)
def _unforced():
    yield
    _lib.load().chop_set_kernel_family(0)


def ran(op, direction, C, N, H, W, D, reduce="MEAN", dtype="f64", groups=0, B=1, family=0, offset=0):
    """The kernels a call would have run.  `groups`: 0 is groups of four channels."""
    lib = _lib.load()
    lib.chop_set_kernel_family(family)
    p = [ctypes.c_void_p(4096 + offset)] * 12
    dims = (B, H, W, C, D, N, H, W)
    g = groups or max(C // 4, 1)
    name, fwd, bwd = {"v1": ("cost_volume", 8, 11), "v2": ("cost_volume_v2", 7, 10),
                      "v3": ("cost_volume_v3", 8, 11), "layer": ("cost_aggregate", 8, 11),
                      "feat": ("feature_aggregate", 7, 9)}[op]
    head = (None, 1) if op == "feat" else (None, REDUCE[reduce], 1)
    tail = (g,) if op in ("v2", "v3") else ()
    if dtype in ("f16", "bf16"):
        head = (None, {"f16": 1, "bf16": 2}[dtype]) + head[1:]
        extra = 1 if op == "v1" else 0            # the depth_grid argument
        status = (getattr(lib, "chop_%s_fwd_16" % name)(*head, *dims, *tail, *p[:fwd + extra])
                  if direction == "f" else
                  getattr(lib, "chop_%s_bwd_16" % name)(*head, *dims, *tail, *p[:bwd + extra],
                                                        ctypes.c_void_p(4096), 1 << 50))
    else:
        status = getattr(lib, "chop_%s_%swd_%s" % (name, direction, dtype))(
            *head, *dims, *tail, *p[:fwd if direction == "f" else bwd])
    assert status == 5, lib.chop_last_error_string()     # CHOP_ERR_LAUNCH: no device
    return lib.chop_last_kernel_shape()


@pytest.mark.parametrize("op", ["v1", "v2", "v3", "layer", "feat"])
@pytest.mark.parametrize("direction", ["f", "b"])
def test_forced_and_unaligned(op, direction):
    """Every type at a size that the tile-shaped kernels take unasked, the families forced, and pointers off
    the 16-byte grid, which they decline (CostVolumeV3 has no forward pass with a lane per channel)."""
    for dtype in ("f32", "f64") + (("f16", "bf16") if op in ("v1", "v2") else ()):
        call = lambda **kw: ran(op, direction, 16, 3, 128, 160, 64, dtype=dtype, **kw)
        lanes = GENERAL if op == "v3" and direction == "f" else LANES
        assert call() == TILES
        assert call(family=3) == TILES
        assert call(family=2) == lanes
        assert call(family=1) == GENERAL
        assert call(offset={"f32": 4, "f64": 8}.get(dtype, 2)) == lanes
        assert call(offset={"f32": 4, "f64": 8}.get(dtype, 2), family=3) == lanes


def test_families_keep_their_codes():
    """`chop_last_kernel_family` says 3 for tiles in double and for idle lanes forward; the shape does not."""
    lib = _lib.load()
    assert ran("v1", "f", 24, 3, 128, 160, 64, dtype="f32") == TILES and lib.chop_last_kernel_family() == 3
    assert ran("v1", "b", 24, 3, 128, 160, 64, dtype="f32") == TILES and lib.chop_last_kernel_family() == 2
    assert ran("v1", "b", 32, 3, 128, 160, 64) == TILES and lib.chop_last_kernel_family() == 3
    assert ran("v1", "b", 32, 3, 128, 160, 64, family=2) == LANES and lib.chop_last_kernel_family() == 3


def test_asked_for():
    """Family 3: the tiles wherever they can serve the shape, and only there."""
    for C, N, want in ((4, 2, LANES), (8, 2, TILES), (64, 6, TILES), (64, 7, LANES), (12, 2, LANES), (28, 2, TILES)):
        assert ran("v1", "f", C, N, 9, 7, 6, family=3) == want
    assert ran("v1", "b", 4, 1, 9, 7, 6, family=3) == TILES
    assert ran("v2", "b", 64, 4, 38, 40, 6, "MIN", family=3) == TILES
    assert ran("v2", "b", 64, 4, 38, 40, 6, "MIN") == LANES


def sides(direction, lanes, tiles):
    """Calls on either side of a line: `(op, C, N, H, W, D, keywords)`."""
    for want, calls in ((LANES, lanes), (TILES, tiles)):
        for op, C, N, H, W, D, *kw in calls:
            kw = kw[0] if kw else {}
            assert ran(op, direction, C, N, H, W, D, **kw) == want, (op, C, N, H, W, D, kw)


def test_forward_launches_of_few_waves_keep_a_lane_per_channel():
    """Double and idle lanes: below a wave per SIMD the chain of one wave is all there is, and a lane per
    channel has the shorter one."""
    f32, low = dict(dtype="f32"), dict(reduce="MIN")
    sides("f",
          [("v1", 32, 3, 38, 40, 6), ("v1", 32, 3, 38, 40, 24), ("v1", 32, 2, 38, 40, 12), ("v1", 32, 1, 20, 24, 12),
           ("v1", 16, 3, 50, 56, 6), ("v2", 16, 3, 38, 40, 6), ("v2", 64, 6, 38, 40, 17), ("v2", 32, 3, 13, 15, 3),
           ("v1", 24, 3, 38, 40, 24, f32), ("v1", 20, 3, 38, 40, 12, dict(dtype="bf16")), ("v2", 28, 2, 38, 40, 8, f32),
           ("layer", 32, 4, 38, 40, 12), ("layer", 64, 3, 20, 24, 8), ("feat", 32, 4, 38, 40, 12),
           ("v2", 8, 1, 200, 260, 48, low), ("v1", 8, 1, 200, 260, 86, low),
           ("v1", 32, 5, 120, 160, 24, low), ("v1", 64, 6, 90, 110, 24, low), ("v1", 64, 5, 19, 21, 1),
           ("v1", 28, 1, 160, 200, 96, low)],
          [("v1", 32, 3, 50, 56, 24), ("v1", 32, 6, 50, 56, 24), ("v1", 32, 2, 38, 40, 24), ("v1", 32, 1, 38, 40, 12),
           ("v1", 16, 3, 60, 80, 8), ("v2", 16, 3, 50, 56, 12), ("v2", 64, 6, 60, 80, 8), ("v2", 32, 1, 13, 15, 3),
           ("v1", 24, 3, 60, 80, 12, f32), ("v1", 8, 5, 38, 40, 6), ("v1", 32, 6, 128, 160, 64), ("v1", 64, 3, 200, 260, 6),
           ("layer", 32, 4, 50, 56, 12), ("layer", 64, 3, 20, 24, 3), ("layer", 16, 4, 20, 24, 8), ("layer", 32, 1, 20, 24, 8),
           ("feat", 32, 4, 50, 56, 12), ("v1", 32, 3, 13, 15, 3, dict(dtype="f32")),
           ("v2", 8, 1, 200, 260, 24, low), ("v2", 8, 1, 200, 260, 48), ("v1", 8, 1, 100, 130, 86, dict(B=2, reduce="MIN")),
           ("v1", 32, 5, 120, 160, 48, low), ("v1", 32, 5, 120, 160, 24), ("v1", 32, 5, 100, 130, 12, dict(B=2, reduce="MIN")),
           ("v1", 64, 4, 19, 21, 1), ("feat", 16, 6, 19, 20, 1), ("v2", 32, 6, 58, 61, 4), ("v1", 28, 1, 160, 200, 32, low)])


@pytest.mark.parametrize("op", ["v1", "layer", "feat"])
def test_gradients_of_one_and_two_views_in_small_launches(op):
    """Double: little to share in a tile's window, and a longer chain than the strips' atomic additions."""
    sides("b",
          [(op, 4, 1, 60, 80, 8), (op, 8, 1, 38, 40, 6), (op, 32, 1, 38, 40, 12), (op, 24, 1, 20, 24, 12),
           (op, 64, 1, 38, 40, 20), (op, 4, 2, 38, 40, 6), (op, 64, 2, 20, 24, 12)],
          [(op, 4, 1, 120, 160, 12), (op, 8, 1, 60, 80, 24), (op, 32, 1, 60, 80, 6), (op, 32, 1, 38, 40, 24),
           (op, 64, 1, 60, 80, 3), (op, 16, 1, 38, 40, 12), (op, 4, 2, 60, 80, 24), (op, 4, 2, 20, 24, 3),
           (op, 64, 2, 38, 40, 12), (op, 8, 1, 38, 40, 6, dict(dtype="f32")), (op, 64, 1, 38, 40, 2)])


def test_correlation_gradients_of_one_view():
    sides("b",
          [("v2", 8, 1, 38, 40, 6), ("v2", 64, 1, 38, 40, 12), ("v2", 8, 1, 38, 40, 6, dict(reduce="MIN"))],
          [("v2", 32, 1, 38, 40, 6), ("v2", 8, 1, 60, 80, 24), ("v2", 16, 1, 38, 40, 6)])


def test_gradients_of_one_view_and_one_value_per_voxel():
    sides("b", [("layer", 8, 1, 90, 110, 6)], [("layer", 8, 1, 90, 110, 12), ("v1", 8, 1, 90, 110, 6)])


def test_correlation_gradients_of_few_depths():
    """Double: a workgroup's window costs the same for two depths as for a chunk, and the minimum passes over
    every view's voxels."""
    low = dict(reduce="MIN")
    sides("b",
          [("v2", 64, 2, 200, 260, 3), ("v2", 64, 4, 60, 80, 2), ("v2", 32, 4, 200, 260, 2), ("v2", 16, 4, 200, 260, 3)],
          [("v2", 64, 2, 200, 260, 4), ("v2", 64, 1, 200, 260, 3), ("v2", 32, 4, 200, 260, 3), ("v2", 16, 4, 120, 160, 3),
           ("v2", 16, 4, 200, 260, 4), ("v2", 8, 4, 200, 260, 1), ("v2", 64, 3, 90, 100, 8)])
    sides("b",
          [(op, C, N, H, W, D, low) for op, C, N, H, W, D in
           [("v2", 64, 2, 38, 40, 6), ("v2", 64, 6, 200, 260, 32), ("v2", 32, 4, 60, 80, 8), ("v2", 24, 6, 200, 260, 6),
            ("v2", 32, 2, 200, 260, 4), ("v2", 16, 3, 200, 260, 3), ("v2", 8, 3, 120, 160, 8), ("v2", 8, 6, 200, 260, 8),
            ("v2", 8, 2, 60, 80, 12), ("v2", 8, 1, 120, 160, 8), ("v2", 4, 3, 200, 260, 12), ("v2", 4, 1, 60, 80, 8)]],
          [(op, C, N, H, W, D, low) for op, C, N, H, W, D in
           [("v2", 64, 1, 200, 260, 4), ("v2", 32, 4, 200, 260, 9), ("v2", 32, 3, 60, 80, 4), ("v2", 32, 3, 200, 260, 5),
            ("v2", 16, 3, 120, 160, 3), ("v2", 16, 3, 200, 260, 4), ("v2", 8, 6, 120, 160, 8), ("v2", 8, 2, 120, 160, 9),
            ("v2", 8, 1, 200, 260, 8), ("v2", 4, 3, 200, 260, 1), ("v2", 4, 6, 60, 80, 8), ("v2", 4, 1, 200, 260, 13)]])


def test_gradients_of_the_best_pair_by_winner():
    """CostVolumeV3's minimum: one pair of groups of one view receives the voxel's gradient, while the tiles walk
    every view with all of a pixel's lanes.  More than 16 groups: a thread per voxel, otherwise a lane per
    channel."""
    f32 = dict(dtype="f32")
    for want, calls in (
            (GENERAL, [(32, 1, 2, 200, 260, 12, f32), (32, 1, 2, 20, 24, 32, f32), (64, 1, 2, 383, 534, 27, f32),
                       (64, 2, 4, 200, 260, 8, f32), (32, 1, 2, 200, 260, 32), (64, 1, 4, 200, 260, 8),
                       (64, 1, 1, 60, 80, 96), (64, 2, 2, 60, 80, 32),
                       (32, 1, 4, 300, 400, 27, f32)]),
            (LANES, [(8, 1, 1, 60, 80, 12, f32), (32, 2, 2, 20, 24, 12, f32), (32, 2, 4, 200, 260, 4, f32),
                     (16, 2, 3, 383, 534, 4, f32), (32, 4, 4, 200, 260, 8), (64, 8, 4, 60, 80, 12),
                     (64, 4, 2, 200, 260, 4), (64, 4, 6, 200, 260, 4)]),
            (TILES, [(32, 1, 2, 200, 260, 32, f32), (32, 1, 1, 200, 260, 12, f32), (64, 1, 1, 200, 260, 32, f32),
                     (64, 2, 1, 200, 260, 4, f32), (64, 2, 2, 200, 260, 32, f32), (64, 4, 4, 200, 260, 4, f32),
                     (8, 1, 1, 60, 80, 32, f32), (8, 1, 2, 60, 80, 4, f32), (16, 2, 3, 200, 260, 12, f32),
                     (32, 1, 2, 120, 160, 96), (16, 1, 4, 200, 260, 4), (32, 4, 2, 200, 260, 4),
                     (64, 8, 1, 200, 260, 4), (64, 8, 6, 120, 160, 12), (64, 4, 2, 60, 80, 96)])):
        for C, sub, N, H, W, D, *kw in calls:
            kw = dict(reduce="MIN", groups=C // sub, **(kw[0] if kw else {}))
            assert ran("v3", "b", C, N, H, W, D, **kw) == want, (C, sub, N, H, W, D, kw)
            kw["reduce"] = "MEAN"
            if D > 8 or "dtype" in kw:
                assert ran("v3", "b", C, N, H, W, D, **kw) == TILES
            assert ran("v3", "f", C, N, H, W, D, **dict(kw, reduce="MIN")) == TILES


def test_gradients_of_few_depths():
    """Double: a window costs the same for one depth as for a chunk, and the minimum of CostAggregate passes over
    every view's voxels."""
    low = dict(reduce="MIN")
    sides("b",
          [("v1", 64, 2, 200, 260, 1), ("v1", 64, 4, 60, 80, 2, low), ("v1", 28, 6, 200, 260, 2), ("layer", 64, 4, 200, 260, 1),
           ("layer", 64, 6, 120, 160, 8, low), ("layer", 64, 3, 60, 80, 4, low), ("layer", 24, 4, 200, 260, 4, low),
           ("layer", 20, 2, 200, 260, 2), ("layer", 32, 4, 200, 260, 4, low), ("layer", 8, 3, 200, 260, 2, low),
           ("layer", 8, 1, 38, 40, 1), ("v3", 64, 2, 200, 260, 8, dict(groups=8)), ("v3", 64, 4, 200, 260, 2),
           ("v3", 32, 2, 200, 260, 2), ("v3", 16, 4, 200, 260, 1), ("v3", 16, 4, 200, 260, 1, low)],
          [("v1", 64, 2, 200, 260, 2), ("v1", 64, 4, 200, 260, 3, low), ("v1", 28, 6, 60, 80, 2), ("v1", 32, 4, 200, 260, 1),
           ("v1", 64, 1, 200, 260, 1), ("layer", 64, 4, 200, 260, 9, low), ("layer", 64, 2, 200, 260, 4, low),
           ("layer", 24, 4, 60, 80, 4, low), ("layer", 32, 3, 200, 260, 4, low), ("layer", 8, 4, 60, 80, 2, low),
           ("feat", 64, 4, 200, 260, 1), ("v3", 64, 2, 200, 260, 9, dict(groups=8)), ("v3", 64, 2, 60, 80, 4),
           ("v3", 32, 2, 200, 260, 3), ("v3", 64, 4, 200, 260, 2, dict(dtype="f32")),
           ("layer", 64, 4, 200, 260, 4, dict(reduce="MIN", dtype="f32"))])


def test_correlation_gradients_by_group_width():
    """Double, minimum: the strips' time goes up with the number of groups.  Four channels: long sweeps too."""
    call = lambda C, sub, N, H, W, D, **kw: ("v2", C, N, H, W, D, dict(dict(reduce="MIN"), groups=C // sub, **kw))
    sides("b",
          [call(32, 8, 4, 200, 260, 8), call(32, 1, 4, 200, 260, 2), call(32, 2, 6, 60, 80, 2), call(8, 8, 4, 200, 260, 16),
           call(8, 4, 2, 330, 400, 8), call(8, 1, 2, 120, 160, 8), call(4, 4, 2, 120, 160, 16),
           call(4, 1, 4, 120, 160, 96), call(4, 2, 4, 330, 400, 32), call(4, 4, 3, 200, 260, 8),
           call(4, 1, 1, 60, 80, 16), call(4, 4, 2, 120, 160, 96, reduce="MEAN"), call(64, 4, 4, 38, 45, 1, reduce="MEAN")],
          [call(32, 1, 4, 200, 260, 8), call(32, 2, 4, 120, 160, 6), call(32, 1, 6, 60, 80, 8), call(8, 1, 4, 200, 260, 8),
           call(8, 2, 2, 330, 400, 8), call(8, 8, 1, 200, 260, 16), call(8, 4, 6, 120, 160, 8), call(4, 1, 2, 120, 160, 16),
           call(4, 1, 4, 200, 260, 8), call(4, 1, 1, 330, 400, 8), call(4, 4, 4, 60, 80, 96), call(4, 1, 2, 60, 80, 8, reduce="MEAN"),
           call(4, 4, 2, 120, 160, 32, reduce="MEAN")])


def segments(*args, **kw):
    """Depth segments of the call; negative: all tiles' first segments before all second ones."""
    ran(*args, **kw)
    return _lib.load().chop_last_segments()


def test_strips_are_cut_where_it_pays():
    """A lane per channel: launches below two waves per SIMD (gradients: one; half a wave for next to no
    depths) are cut below a chunk, into segments as even as their number allows."""
    bf16 = dict(dtype="bf16", family=2)
    assert segments("v1", "b", 3, 5, 100, 128, 9, B=2, **bf16) == 1         # 1600 strips
    assert segments("v1", "b", 3, 5, 100, 128, 9, **bf16) == 3              # 800 strips, 3 x 3
    assert segments("v1", "f", 3, 5, 100, 128, 9, B=2, **bf16) == 2         # 5 + 4
    assert segments("v1", "b", 64, 3, 38, 40, 6, family=2) == 1             # 1520 strips
    assert segments("v2", "b", 32, 5, 38, 40, 5, family=2) == 1             # 760 strips, five depths
    assert segments("v2", "b", 32, 5, 38, 40, 6, family=2) == 2
    assert segments("layer", "f", 64, 5, 26, 34, 3, family=2) == 1
    assert segments("layer", "f", 64, 5, 26, 34, 9, family=2) > 1
    assert segments("v1", "f", 64, 5, 26, 34, 3, family=2) == 2
    assert segments("v1", "f", 3, 2, 12, 16, 9, family=2) == 9              # twelve strips: depth by depth
    assert segments("v1", "b", 3, 2, 12, 16, 9, family=2) == 5
    assert segments("v1", "b", 12, 5, 50, 55, 36, family=2) == 5            # 688 strips, two segments anyway
    assert segments("v2", "b", 12, 2, 59, 77, 22, groups=3, family=2) == 3  # 1136 strips
    assert segments("v1", "b", 12, 2, 72, 90, 22, dtype="f32") == 2         # 1620 strips
    assert segments("v1", "b", 12, 2, 72, 90, 22) == 1
    assert segments("v1", "b", 5, 3, 100, 100, 12, dtype="f32") == 2        # 1250 strips
    assert segments("v1", "b", 5, 3, 100, 100, 12) == 1
    assert segments("layer", "f", 3, 5, 16, 21, 5, family=2) == 5
    assert segments("layer", "f", 32, 5, 30, 40, 5, family=2) == 1          # 600 strips


def test_many_taps_stay_in_one_round():
    """Five and six views that hold their taps side by side run two waves per SIMD: more than 2048 waves
    would be a second round."""
    assert segments("layer", "f", 8, 6, 135, 181, 24, reduce="MIN", dtype="f32") == 2
    assert segments("layer", "f", 8, 4, 135, 181, 24, reduce="MIN", dtype="f32") == 3
    assert segments("layer", "f", 8, 6, 135, 181, 24, reduce="MEAN", dtype="f32") == 3     # (three waves)
    assert segments("feat", "f", 32, 6, 44, 62, 107, dtype="f32") == -5     # 4 x 24 + 11
    assert segments("feat", "f", 32, 4, 44, 62, 107, dtype="f32") == -7     # 6 x 16 + 11
    assert segments("feat", "f", 8, 6, 139, 157, 33, dtype="f64") == 3      # 2 x 16 + 1, rounded down
    assert segments("feat", "f", 32, 6, 8, 12, 33, dtype="f32") == -5       # twelve tiles: single chunks


def test_launches_of_narrow_pixels_are_not_cut_past_the_caches():
    """Pieces of lines: more waves side by side keep more lines open than the caches hold."""
    f32 = dict(dtype="f32")
    assert segments("feat", "f", 4, 4, 314, 375, 19, **f32) == 1
    assert segments("feat", "f", 4, 4, 314, 375, 3, **f32) == 2             # 23 MB
    assert segments("feat", "f", 4, 1, 160, 208, 57, **f32) == 2
    assert segments("feat", "f", 4, 1, 236, 263, 33, **f32) == 3            # a wave to every SIMD
    assert segments("v1", "f", 4, 3, 120, 160, 100, **f32) == 4
    assert segments("v1", "f", 4, 3, 120, 160, 57, **f32) == 7
    assert segments("feat", "f", 8, 4, 236, 263, 19, **f32) == 1
    assert segments("feat", "f", 8, 4, 160, 208, 19, **f32) == 2


def test_uneven_segments_go_one_after_the_other():
    """Side by side a short last segment leaves every other compute unit idle; segments about as long as each
    other stay side by side, and so do narrow pixels with one value per voxel."""
    layer = dict(reduce="MIN", dtype="f32")
    assert segments("layer", "f", 32, 4, 135, 181, 17, **layer) == -2       # 16 + 1
    assert segments("layer", "f", 32, 4, 135, 181, 24, **layer) == -2       # 16 + 8
    assert segments("layer", "f", 32, 4, 135, 181, 31, **layer) == 2        # 16 + 15
    assert segments("layer", "f", 32, 4, 135, 181, 32, **layer) == 4        # 4 x 8
    assert segments("v1", "f", 32, 6, 114, 117, 21, dtype="f32") == -2      # 16 + 5
    assert segments("layer", "f", 8, 1, 326, 430, 82, **layer) == 7         # 6 x 12 + 10, narrow
    assert segments("layer", "f", 8, 6, 147, 154, 14, B=2, dtype="f32") > 0
    assert segments("feat", "f", 16, 1, 60, 80, 17, dtype="f32") < 0
    assert segments("v1", "f", 32, 2, 128, 160, 192, dtype="f32") == 8      # 8 x 24
    assert segments("v1", "f", 32, 2, 8, 8, 3, dtype="f32") == 1
