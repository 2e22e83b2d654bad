"""Host-side mirror of the reference's Python operator interface for the cost volume.

Same names, argument order, defaults and outputs as
custom_helper_op/python/ops/custom_helper_ops.py:32-197 (``cost_volume``,
``cost_volume_v2``, ``cost_volume_v3``, ``cost_aggregate``, ``feature_aggregate`` and the
gradients registered for them), with torch tensors standing in
for TensorFlow tensors: torch supplies device memory and the current HIP stream, the
arithmetic is done by ``libchop_costvol.so``.  Argument checks, allocation, the launches and the
gradients registered with autograd are C++ (``csrc/torch_ops.cpp``); the functions here name
its arguments.  The checks are the ones ``CostVolumeOp::Compute`` performs
(custom_helper_op/cc/kernels/cost_volume_kernels.cc:91-106, :220-243;
cost_volume_kernels_v2.cc:93-110), raised as ``InvalidArgumentError``.

float32/float64 follow the registered ops; float16/bfloat16 feature tensors use the
library's 16-bit storage extension (depth inputs and camera matrices must then be
float32).
"""
import torch

from . import _lib

_REDUCE = {"MEAN": 0, "MIN": 1}


class InvalidArgumentError(ValueError):
    """What ``OP_REQUIRES(..., errors::InvalidArgument(...))`` becomes on this side."""


# the operators' numbers in csrc/torch_ops.cpp
_V1, _V2, _AGGREGATE, _V3, _FEATURE = range(5)

_native_module = None


def _native():
    """The extension module, loaded at the first call (there is no fallback without it)."""
    global _native_module
    if _native_module is None:
        _lib.load()
        from . import _chop_torch
        _connect(_chop_torch)
        _native_module = _chop_torch
    return _native_module


def _connect(module):
    module.python_side(InvalidArgumentError, _lib.ChopError, _recorded)


def _reduce_code(reduce_method):
    if reduce_method not in _REDUCE:
        # the reference aborts the process here (LOG(FATAL), cost_volume_kernels.cc:71)
        raise InvalidArgumentError(
            "Invalid reduce method %r. Supported types: MEAN, MIN" % (reduce_method,))
    return _REDUCE[reduce_method]


def _require(cond, msg):
    if not cond:
        raise InvalidArgumentError(msg)


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _stream(t):
    return torch.cuda.current_stream(t.device).cuda_stream


def _prep(t, dtype, device, name):
    t = torch.as_tensor(t)
    _require(t.dtype == dtype, "%s must have dtype %s, got %s" % (name, dtype, t.dtype))
    _require(t.device == device, "%s must live on %s" % (name, device))
    return t.contiguous()


def cost_volume_raw(ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method="MEAN",
                    half_centor=True, depth_grid=None):
    """Forward op without autograd: returns ``(cost [B,H,W,D,C], cost_mask int32)``.
    ``depth_grid`` ([B,H,W,D] float32, 16-bit feature storage only) replaces
    ``base_plane + offsets`` (which may then be ``None``) by per-voxel hypotheses."""
    grid = depth_grid is not None
    return _native().forward(_V1, ref_image, src_images, depth_grid if grid else base_plane,
                             None if grid else offsets, Rs, Ts, reduce_method, 1, half_centor, grid,
                             None, False)


def cost_volume_grad(ref_image, src_images, base_plane, offsets, rs, ts, cost_grad, cost_mask,
                     reduce_method="MEAN", half_centor=True, need_depth_grad=True,
                     depth_grid=None):
    """The ``CostVolumeGrad`` op: ``(ref_image_grad, src_images_grad, base_plane_grad)``.
    With ``need_depth_grad=False`` the third result is ``None`` and the kernels skip the
    depth-derivative work (the registered op always computes it).  With ``depth_grid``
    (16-bit feature storage only) the third result is the gradient of ``depth_grid``,
    ``[B,H,W,D]``, zero on the voxels the mask skips."""
    grid = depth_grid is not None
    return _native().backward(_V1, ref_image, src_images, depth_grid if grid else base_plane,
                              None if grid else offsets, rs, ts, reduce_method, 1, half_centor, grid,
                              cost_grad, cost_mask, need_depth_grad)


def cost_volume_v2_raw(ref_image, src_images, depth_grid, Rs, Ts, reduce_method="MEAN", groups=None,
                       half_centor=True, default_cost=None):
    """``default_cost`` (a device scalar): written instead of the cost wherever no view was
    accepted -- ``CostMapLayerV2``'s fill, done by the op's own store."""
    return _native().forward(_V2, ref_image, src_images, depth_grid, None, Rs, Ts, reduce_method,
                             groups, half_centor, True, default_cost, False)


def cost_volume_grad_v2(ref_image, src_images, depth_grid, rs, ts, cost_grad, cost_mask,
                        reduce_method="MEAN", groups=None, half_centor=True,
                        need_depth_grad=True):
    """The ``CostVolumeGradV2`` op: ``(ref_image_grad, src_images_grad, depth_grid_grad)``;
    ``need_depth_grad=False`` as in :func:`cost_volume_grad`."""
    return _native().backward(_V2, ref_image, src_images, depth_grid, None, rs, ts, reduce_method,
                              groups, half_centor, True, cost_grad, cost_mask, need_depth_grad)


def cost_aggregate_raw(ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method="MEAN",
                       half_centor=True, default_cost=None):
    """The ``CostAggregate`` op without autograd: ``(cost [B,H,W,D], cost_mask int32 [B,H,W,D])``
    (shapes: custom_helper_op/cc/ops/custom_helper_ops.cc:46-58; checks:
    cost_aggregate_kernels.cc:85-106).  float32 and float64 only, as registered.
    ``default_cost`` as in :func:`cost_volume_v2_raw` (``CostMapLayer``'s fill)."""
    return _native().forward(_AGGREGATE, ref_image, src_images, base_plane, offsets, Rs, Ts,
                             reduce_method, 1, half_centor, False, default_cost, False)


def cost_aggregate_grad(ref_image, src_images, base_plane, offsets, rs, ts, cost_grad, cost_mask,
                        reduce_method="MEAN", half_centor=True, need_depth_grad=True):
    """The ``CostAggregateGrad`` op: ``(ref_image_grad, src_images_grad, base_plane_grad)``
    (checks: cost_aggregate_kernels.cc:196-226); ``need_depth_grad=False`` as in
    :func:`cost_volume_grad`."""
    return _native().backward(_AGGREGATE, ref_image, src_images, base_plane, offsets, rs, ts,
                              reduce_method, 1, half_centor, False, cost_grad, cost_mask,
                              need_depth_grad)


def cost_volume_v3_raw(ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method="MEAN",
                       groups=None, half_centor=True):
    """The ``CostVolumeV3`` op without autograd: ``(cost [B,H,W,D,1], cost_mask int32
    [B,H,W,D,1] (MEAN) or [B,H,W,D,3] (MIN: view, reference group, source group))``
    (shapes: custom_helper_op/cc/ops/custom_helper_ops.cc:311-347; checks:
    cost_volume_kernels_v3.cc:94-115).  float32 and float64, as registered."""
    return _native().forward(_V3, ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method,
                             groups, half_centor, False, None, False)


def cost_volume_grad_v3(ref_image, src_images, base_plane, offsets, rs, ts, cost_grad, cost_mask,
                        reduce_method="MEAN", groups=None, half_centor=True):
    """The ``CostVolumeGradV3`` op: ``(ref_image_grad, src_images_grad, base_plane_grad)``
    (checks: cost_volume_kernels_v3.cc:231-255)."""
    return _native().backward(_V3, ref_image, src_images, base_plane, offsets, rs, ts, reduce_method,
                              groups, half_centor, False, cost_grad, cost_mask, True)


def feature_aggregate_raw(src_images, base_plane, offsets, Rs, Ts, half_centor=True):
    """The ``FeatureAggregate`` op without autograd: ``(mapped_feature [B,H,W,D,N,C],
    mapped_mask int32 [B,H,W,D,N,1])``; H and W are base_plane's (shapes:
    custom_helper_op/cc/ops/custom_helper_ops.cc:414-440)."""
    return _native().forward(_FEATURE, None, src_images, base_plane, offsets, Rs, Ts, "MEAN", 1,
                             half_centor, False, None, False)


def feature_aggregate_grad(src_images, base_plane, offsets, rs, ts, mapped_feature_grad,
                           mapped_mask, half_centor=True):
    """The ``FeatureAggregateGrad`` op: ``(src_images_grad, base_plane_grad)``
    (checks: feature_aggregate_kernels.cc:176-210)."""
    return _native().backward(_FEATURE, None, src_images, base_plane, offsets, rs, ts, "MEAN", 1,
                              half_centor, False, mapped_feature_grad, mapped_mask, True)[1:]


# The differentiable functions: the op's forward with its registered gradient behind it
# (custom_helper_ops.py:41-61, :74-94, :107-131, :141-161, :174-195).  The incoming gradient of
# the mask is ignored; offsets, Rs and Ts receive none.
def cost_volume(ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method="MEAN",
                half_centor=True, name=None):
    """``custom_helper_op.cost_volume``: returns ``(cost, cost_mask)``; differentiable with
    respect to ref_image, src_images and base_plane."""
    del name
    return _native().forward(_V1, ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method, 1,
                             half_centor, False, None, True)


def cost_volume_v2(ref_image, src_images, depth_grid, Rs, Ts, reduce_method="MEAN", groups=None,
                   half_centor=True, name=None):
    """``custom_helper_op.cost_volume_v2``: returns ``(cost [B,H,W,D,groups], cost_mask)``."""
    del name
    return _native().forward(_V2, ref_image, src_images, depth_grid, None, Rs, Ts, reduce_method,
                             groups, half_centor, True, None, True)


def cost_aggregate(ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method="MEAN",
                   half_centor=True, name=None):
    """``custom_helper_op.cost_aggregate`` (custom_helper_ops.py:133-138): returns
    ``(cost [B,H,W,D], cost_mask [B,H,W,D])``; differentiable with respect to ref_image,
    src_images and base_plane."""
    del name
    return _native().forward(_AGGREGATE, ref_image, src_images, base_plane, offsets, Rs, Ts,
                             reduce_method, 1, half_centor, False, None, True)


def cost_volume_v3(ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method="MEAN",
                   groups=None, half_centor=True, name=None):
    """``custom_helper_op.cost_volume_v3`` (custom_helper_ops.py:99-104): returns
    ``(cost [B,H,W,D,1], cost_mask)``; differentiable with respect to ref_image, src_images and
    base_plane."""
    del name
    return _native().forward(_V3, ref_image, src_images, base_plane, offsets, Rs, Ts, reduce_method,
                             groups, half_centor, False, None, True)


def feature_aggregate(src_images, base_plane, offsets, Rs, Ts, half_centor=True, name=None):
    """``custom_helper_op.feature_aggregate`` (custom_helper_ops.py:166-171): returns
    ``(mapped_feature [B,H,W,D,N,C], mapped_mask [B,H,W,D,N,1])``; differentiable with respect
    to src_images and base_plane."""
    del name
    return _native().forward(_FEATURE, None, src_images, base_plane, offsets, Rs, Ts, "MEAN", 1,
                             half_centor, False, None, True)


def cost_volume_v2_filled(ref_image, src_images, depth_grid, Rs, Ts, default_cost,
                          reduce_method="MEAN", groups=None, half_centor=True):
    """CostVolumeV2 followed by ``where(valid(cost_mask), cost, default_cost)``, fused into one
    kernel; differentiable in the images, the depth grid and the scalar.  The op's registered gradient skips exactly the
    filled voxels, so it takes the upstream gradient as it is; ``CostMapLayerV2.call``
    (custom_layers.py:77-83)."""
    return _native().forward(_V2, ref_image, src_images, depth_grid, None, Rs, Ts, reduce_method,
                             groups, half_centor, True, default_cost, True)


def cost_aggregate_filled(ref_image, src_images, base_plane, offsets, Rs, Ts, default_cost,
                          reduce_method="MEAN", half_centor=True):
    """CostAggregate followed by the same fill, fused into one kernel (``CostMapLayer.call``,
    custom_layers.py:51-57)."""
    return _native().forward(_AGGREGATE, ref_image, src_images, base_plane, offsets, Rs, Ts,
                             reduce_method, 1, half_centor, False, default_cost, True)


class _Operator(torch.autograd.Function):
    """An operator and its registered gradient as a function of Python's autograd, for the modes of
    torch that record or refuse such a function and cannot see a native node."""

    @staticmethod
    def forward(ctx, op, ref_image, src_images, depth, offsets, Rs, Ts, reduce_method, groups,
                half_centor, grid, default_cost):
        cost, mask = _native().forward(op, ref_image, src_images, depth, offsets, Rs, Ts,
                                       reduce_method, groups, half_centor, grid, default_cost, False)
        ctx.save_for_backward(ref_image, src_images, depth, offsets, Rs, Ts, default_cost, mask)
        ctx.attrs = (op, reduce_method, groups, half_centor, grid)
        ctx.mark_non_differentiable(mask)
        return cost, mask

    @staticmethod
    def backward(ctx, grad_out, _grad_mask):
        *inputs, default_cost, mask = ctx.saved_tensors
        op, *attrs = ctx.attrs
        grads = _native().backward(op, *inputs, *attrs, grad_out, mask, ctx.needs_input_grad[3])
        default_grad = (_native().default_gradient(attrs[0], grad_out, mask, default_cost)
                        if ctx.needs_input_grad[11] else None)
        return (None, *grads, *[None] * 7, default_grad)


def _recorded(op, ref_image, src_images, depth, offsets, Rs, Ts, reduce_method, groups, half_centor,
              grid, default_cost):
    """What a differentiable function does while a trace is recorded, under the transforms of
    ``torch.func`` and where an input carries a forward-mode tangent; depth inputs and cameras are
    taken from where the caller has them, as in ``csrc/torch_ops.cpp``."""
    device = (src_images if op == _FEATURE else ref_image).device

    def there(x):
        return x if x is None else (x if torch.is_tensor(x) else torch.as_tensor(x)).to(device)

    offsets, Rs, Ts = there(offsets), there(Rs), there(Ts)
    if op == _V2:
        depth = there(depth)
    return _Operator.apply(op, ref_image, src_images, depth, offsets, Rs, Ts, reduce_method, groups,
                           half_centor, grid, default_cost)


class _DefaultFill(torch.autograd.Function):
    """``tf.where(valid(cost_mask), cost, default_cost)`` with its gradient, as one kernel each
    way (custom_helper_op/python/layers/custom_layers.py:52-57, :78-83)."""

    @staticmethod
    def forward(ctx, cost, cost_mask, default_cost, reduce_method):
        lib = _lib.load()
        red = _reduce_code(reduce_method)
        dt, dev = cost.dtype, cost.device
        _require(dt in (torch.float32, torch.float64), "dtype must be float32 or float64")
        cost = _prep(cost, dt, dev, "cost")
        cost_mask = _prep(cost_mask, torch.int32, dev, "cost_mask")
        default_cost = _prep(default_cost, dt, dev, "default_cost")
        _require(default_cost.numel() == 1, "default_cost must be a scalar")
        n_mask = cost_mask.numel()
        _require(n_mask > 0 and cost.numel() % n_mask == 0 or cost.numel() == 0,
                 "cost_mask must cover cost with a whole number of elements per entry")
        inner = cost.numel() // n_mask if n_mask else 1
        out = torch.empty_like(cost)
        fn = lib.chop_cost_default_fill_f32 if dt == torch.float32 else lib.chop_cost_default_fill_f64
        _lib.check(fn(_stream(out), red, n_mask, inner, _ptr(cost), _ptr(cost_mask),
                      _ptr(default_cost), _ptr(out)))
        ctx.save_for_backward(cost_mask)
        ctx.attrs = (red, n_mask, inner, default_cost.shape)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        lib = _lib.load()
        (cost_mask,) = ctx.saved_tensors
        red, n_mask, inner, dshape = ctx.attrs
        grad_out = grad_out.contiguous()
        cost_grad = torch.empty_like(grad_out)
        default_grad = torch.empty(dshape, dtype=grad_out.dtype, device=grad_out.device)
        fn = (lib.chop_cost_default_fill_grad_f32 if grad_out.dtype == torch.float32
              else lib.chop_cost_default_fill_grad_f64)
        _lib.check(fn(_stream(cost_grad), red, n_mask, inner, _ptr(grad_out), _ptr(cost_mask),
                      _ptr(cost_grad), _ptr(default_grad)))
        return cost_grad, None, default_grad, None


def cost_default_fill(cost, cost_mask, default_cost, reduce_method="MEAN"):
    """``where(cost_mask > 0, cost, default_cost)`` for MEAN, ``cost_mask >= 0`` for MIN: what
    ``CostMapLayer`` / ``CostMapLayerV2`` apply to the op's outputs; differentiable with respect
    to ``cost`` and the scalar ``default_cost``.  ``cost_mask`` may have one entry per cost
    element or one per row of the last axis."""
    return _DefaultFill.apply(cost, cost_mask, default_cost, reduce_method)


def combine_projection(ref_cam, src_cam, scale):
    """The relative projection the ops take, computed on the device
    (custom_helper_op/python/ops/op_tests/cost_volume_op_test.py:115-134).
    ``ref_cam [B,2,4,4]`` (or ``[2,4,4]``), ``src_cam [B,N,2,4,4]`` (or ``[2,4,4]``), ``scale [3]``
    -> ``(Rs [B,N,3,3], Ts [B,N,3])``; the unbatched form returns ``(R [3,3], T [3,1])`` like the
    reference helper."""
    if ref_cam.dim() != 3:
        return _native().combine_projection(ref_cam, src_cam, scale)
    _require(tuple(ref_cam.shape) == (2, 4, 4) and tuple(src_cam.shape) == (2, 4, 4),
             "cameras must be [2,4,4]")
    Rs, Ts = _native().combine_projection(ref_cam[None], src_cam[None, None], scale)
    return Rs[0, 0], Ts[0, 0][:, None]


def sample_coords(base_plane, offsets, Rs, Ts, src_hw, half_centor=True, depth_grid=None):
    """Diagnostic: per-(voxel, view) sample coordinates ``[B,H,W,D,N]`` as the kernels
    compute them: ``(sw, sh, fh, fw, state)``."""
    lib = _lib.load()
    if depth_grid is not None:
        dt, dev = depth_grid.dtype, depth_grid.device
        depth_grid = depth_grid.contiguous()
        B, H, W, D = depth_grid.shape
    else:
        dt, dev = base_plane.dtype, base_plane.device
        base_plane, offsets = base_plane.contiguous(), offsets.contiguous()
        B, H, W = base_plane.shape[:3]
        D = offsets.shape[1]
    Rs, Ts = _prep(Rs, dt, dev, "Rs"), _prep(Ts, dt, dev, "Ts")
    N = Rs.shape[1]
    shape = (B, H, W, D, N)
    sw, sh = (torch.empty(shape, dtype=dt, device=dev) for _ in range(2))
    fh, fw, st = (torch.empty(shape, dtype=torch.int32, device=dev) for _ in range(3))
    fn = (lib.chop_cost_volume_sample_coords_f32 if dt == torch.float32
          else lib.chop_cost_volume_sample_coords_f64)
    rc = fn(_stream(sw), int(half_centor), B, H, W, D, N, src_hw[0], src_hw[1], _ptr(base_plane),
            _ptr(offsets), _ptr(depth_grid), _ptr(Rs), _ptr(Ts), _ptr(sw), _ptr(sh), _ptr(fh),
            _ptr(fw), _ptr(st))
    _lib.check(rc)
    return sw, sh, fh, fw, st
