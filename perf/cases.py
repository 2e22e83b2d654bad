"""The work that users of this library have it do, as cases that can be timed and compared.

A case is one call (inference) or one forward + backward (training) of one of the plane-sweep
operators on synthetic features and cameras.  Sizes are those of the five benchmark workloads in
``custom_helper_op_amd/configs.py``, of the unit tests, and ragged ones between them.  Everything
runs through the differentiable functions and layers of the package, the way a network's
``forward`` and ``loss.backward()`` reach them.

Keys of a case: ``op`` (``v1`` CostVolume, ``v2`` CostVolumeV2, ``v3`` CostVolumeV3, ``feat``
FeatureAggregate, ``layer`` CostMapLayer, ``layer2`` CostMapLayerV2), ``dtype``, ``reduce``,
``train``, the sizes ``B N H W C D`` and ``groups``, ``depth_grad`` (whether the depth input wants a
gradient), ``spacing`` / ``near`` / ``far`` (the depth hypotheses) and ``rot`` / ``shift`` (largest
rotation in degrees and translation between the reference and a source camera).
"""
import math

import numpy as np
import torch

import custom_helper_op_amd as chop
from custom_helper_op_amd.configs import intrinsics, random_cameras

DTYPES = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16, "bf16": torch.bfloat16}
ELEMENT = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2}
GRID_OPS = ("v2", "layer2")     # per-voxel depth hypotheses instead of plane + offsets


def _case(name, op, dtype, reduce, train, B, N, H, W, C, D, groups=1, depth_grad=True,
          spacing="inverse", near=1.0, far=10.0, rot=5.0, shift=0.2):
    case = dict(op=op, dtype=dtype, reduce=reduce, train=train, B=B, N=N, H=H, W=W, C=C, D=D,
                groups=groups, depth_grad=depth_grad, spacing=spacing, near=near, far=far, rot=rot,
                shift=shift)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a small variance volume at inference (benchmark workload 1): one launch, all latency
        _case("tiny_variance_infer_f32", "v1", "f32", "MEAN", False, 1, 2, 64, 80, 8, 32,
              spacing="linear", near=2.0, far=6.0, shift=0.1),
        # the size of the unit tests, in their element type: RGB patches, gradient checks,
        # photometric losses on small crops; host overhead of a whole training pass
        _case("small_patch_train_f64", "v1", "f64", "MEAN", True, 1, 2, 12, 16, 3, 9,
              spacing="linear", near=18.0, far=32.0),
        # the standard variance cost volume of a multi-view stereo network in training
        # (benchmark workload 2, the headline)
        _case("mvsnet_stage_train_f32", "v1", "f32", "MEAN", True, 1, 2, 128, 160, 32, 192),
        # the same operator in the second registered element type
        _case("mvsnet_stage_train_f64", "v1", "f64", "MEAN", True, 1, 2, 128, 160, 32, 192),
        # a cascade's fine stage: few hypotheses around a coarse depth map that is detached
        # (benchmark workload 3)
        _case("cascade_fine_train_f16", "v1", "f16", "MEAN", True, 1, 4, 256, 320, 16, 32,
              depth_grad=False, spacing="field", near=5.0, far=5.0),
        # group-wise correlation at high resolution, eight refined hypotheses per pixel
        # (benchmark workload 4)
        _case("group_correlation_train_bf16", "v2", "bf16", "MEAN", True, 2, 4, 512, 640, 8, 8,
              groups=4, spacing="field", near=5.0, far=5.0),
        # large batch, many wide-baseline views, hypotheses close to the cameras
        # (benchmark workload 5): the largest
        _case("large_batch_train_f32", "v1", "f32", "MEAN", True, 4, 6, 288, 384, 32, 128,
              spacing="linear", near=0.5, far=20.0, rot=15.0, shift=0.5),
        # the cost-map layer with its default reduce and trainable fill, from raw cameras, on an
        # image size that no tile divides
        _case("cost_map_layer_train_f32", "layer", "f32", "MIN", True, 1, 3, 135, 181, 32, 48),
        # the second layer at inference: per-pixel hypotheses, eight correlation groups of 16-bit
        # features, an odd image size
        _case("cost_map_layer_v2_infer_f16", "layer2", "f16", "MIN", False, 1, 4, 237, 315, 32, 24,
              groups=8, spacing="field", near=5.0, far=5.0),
        # the best-group-pair volume
        _case("best_pair_train_f32", "v3", "f32", "MEAN", True, 1, 2, 120, 152, 32, 64, groups=4),
        # warped features for a network that aggregates the views itself
        _case("feature_warp_train_f32", "feat", "f32", "MEAN", True, 2, 3, 97, 129, 16, 40),
        # a channel count that is no power of two, per-channel minimum over the views
        _case("odd_channels_min_train_f32", "v1", "f32", "MIN", True, 1, 5, 63, 85, 24, 37),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choices(("v1", "v2", "layer", "layer2", "v3", "feat"), (6, 4, 3, 2, 2, 3))[0]
    if op in ("v1", "v2", "layer2"):
        dtype = rng.choices(("f32", "f64", "f16", "bf16"), (6, 2, 2, 2))[0]
    else:
        dtype = rng.choices(("f32", "f64"), (4, 1))[0]
    C = rng.choice((3, 8, 8, 16, 16, 16, 24, 32, 32, 32, 64))
    # elements sampled in one direction: an order below the largest listed case, less where a
    # wide element or an odd channel count makes each of them dearer
    most = 4e8 if dtype == "f64" or C in (3, 24) else 2e9
    while True:
        B, N = rng.choice((1, 1, 1, 2, 4)), rng.randint(1, 6)
        H = _log_int(rng, 12, 512)
        W = int(H * rng.uniform(1.0, 1.5))
        D = _log_int(rng, 4, 192)
        if B * N * H * W * D * C <= most:
            break
    groups = 1
    if op in GRID_OPS or op == "v3":
        groups = rng.choice([g for g in range(1, C + 1) if C % g == 0 and C // g <= 8])
    reduce = "MEAN" if op == "feat" else rng.choice(("MEAN", "MIN"))
    spacing = rng.choice(("inverse", "linear", "field"))
    near = round(math.exp(rng.uniform(math.log(0.5), math.log(3.0))), 3)
    far = round(near * rng.uniform(3.0, 20.0), 3)
    if spacing == "field":
        near = far = round(rng.uniform(4.0, 8.0), 3)
    return _case(None, op, dtype, reduce, rng.random() < 0.75, B, N, H, W, C, D, groups,
                 rng.random() < 0.7, spacing, near, far, round(rng.uniform(2.0, 15.0), 2),
                 round(rng.uniform(0.1, 0.5), 3))


def _depths(case, real, gen):
    """(base_plane [B,H,W,1], offsets [B,D]): planes of a sweep, or a few hypotheses around a smooth
    coarse depth map."""
    B, H, W, D, dev = case["B"], case["H"], case["W"], case["D"], "cuda"
    k = torch.arange(D, dtype=torch.float64, device=dev)
    if case["spacing"] == "field":
        mean = case["near"]
        grid = torch.randn((B, 1, 8, 10), generator=gen, device=dev, dtype=torch.float64)
        grid = mean * (1.0 + 0.2 * grid.clamp(-3.0, 3.0))
        base = torch.nn.functional.interpolate(grid, (H, W), mode="bilinear", align_corners=True)
        base, planes = base.reshape(B, H, W, 1), (k - D // 2) * 0.02 * mean
    else:
        base = torch.zeros((B, H, W, 1), dtype=torch.float64, device=dev)
        t = k / max(D - 1, 1)
        if case["spacing"] == "inverse":
            planes = 1.0 / (1.0 / case["near"] + t * (1.0 / case["far"] - 1.0 / case["near"]))
        else:
            planes = case["near"] + t * (case["far"] - case["near"])
    return base.to(real), planes.to(real).expand(B, D).contiguous()


def _raw_cameras(rng, case):
    """Extrinsics and intrinsics [B,2,4,4] and [B,N,2,4,4] of cameras around the reference."""
    B, N = case["B"], case["N"]
    cams = np.zeros((B, N + 1, 2, 4, 4))
    cams[:, :, 0] = np.eye(4)
    cams[:, :, 1, :3, :3] = intrinsics(case["H"], case["W"])
    for b in range(B):
        for n in range(1, N + 1):
            x, y, z = np.radians(rng.uniform(-case["rot"], case["rot"], 3))
            turns = (np.array([[1, 0, 0], [0, np.cos(x), -np.sin(x)], [0, np.sin(x), np.cos(x)]]),
                     np.array([[np.cos(y), 0, np.sin(y)], [0, 1, 0], [-np.sin(y), 0, np.cos(y)]]),
                     np.array([[np.cos(z), -np.sin(z), 0], [np.sin(z), np.cos(z), 0], [0, 0, 1]]))
            cams[b, n, 0, :3, :3] = turns[2] @ turns[1] @ turns[0]
            cams[b, n, 0, :3, 3] = rng.uniform(-case["shift"], case["shift"], 3)
    return cams[:, 0], cams[:, 1:]


def prepare(case, seed):
    dev, dt = torch.device("cuda"), DTYPES[case["dtype"]]
    real = torch.float64 if case["dtype"] == "f64" else torch.float32
    B, N, H, W, C, D = (case[k] for k in "BNHWCD")
    gen = torch.Generator(device=dev).manual_seed(seed)
    rng = np.random.default_rng(seed)
    s = dict(case=case)

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=real).to(dt)

    s["ref"], s["src"] = normal(B, H, W, C), normal(B, N, H, W, C)
    base, offsets = _depths(case, real, gen)
    if case["op"] in GRID_OPS:
        if case["spacing"] == "field":
            k = torch.arange(D, dtype=real, device=dev) - D // 2
            s["depth"] = (base * (1.0 + 0.02 * k)).contiguous()
        else:
            s["depth"] = (base + offsets[:, None, None, :]).contiguous()
    else:
        s["depth"], s["offsets"] = base, offsets
    if case["op"] in ("layer", "layer2"):
        ref_cam, src_cam = _raw_cameras(rng, case)
        s["ref_cam"] = torch.from_numpy(ref_cam).to(dev, real)
        s["src_cam"] = torch.from_numpy(src_cam).to(dev, real)
        s["scale"] = torch.ones(3, dtype=real, device=dev)
        kind = dict(reduce_method=case["reduce"], default_type="DYNAMIC")
        layer = (chop.CostMapLayer(**kind) if case["op"] == "layer"
                 else chop.CostMapLayerV2(groups=case["groups"], **kind))
        s["layer"] = layer.to(dev)
        with torch.no_grad():
            s["layer"].default_cost.fill_(0.25)
    else:
        Rs, Ts = random_cameras(rng, B, N, H, W, case["rot"], case["shift"])
        s["Rs"], s["Ts"] = (torch.from_numpy(x).to(dev, real) for x in (Rs, Ts))
    if case["train"]:
        s["upstream"] = normal(*_output_shape(case))
        if case["op"] != "feat":
            s["ref"].requires_grad_(True)
        s["src"].requires_grad_(True)
        s["depth"].requires_grad_(bool(case["depth_grad"]))
    return s


def _output_shape(case):
    B, N, H, W, C, D = (case[k] for k in "BNHWCD")
    tail = {"v1": (C,), "v2": (case["groups"],), "layer": (), "layer2": (case["groups"],), "v3": (1,),
            "feat": (N, C)}[case["op"]]
    return (B, H, W, D) + tail


def _forward(s):
    case = s["case"]
    op, reduce = case["op"], case["reduce"]
    if op == "v1":
        return chop.cost_volume(s["ref"], s["src"], s["depth"], s["offsets"], s["Rs"], s["Ts"], reduce)
    if op == "v2":
        return chop.cost_volume_v2(s["ref"], s["src"], s["depth"], s["Rs"], s["Ts"], reduce,
                                   case["groups"])
    if op == "v3":
        return chop.cost_volume_v3(s["ref"], s["src"], s["depth"], s["offsets"], s["Rs"], s["Ts"],
                                   reduce, case["groups"])
    if op == "feat":
        return chop.feature_aggregate(s["src"], s["depth"], s["offsets"], s["Rs"], s["Ts"])
    # the layers start from the cameras of the sample, as a data loader delivers them
    Rs, Ts = chop.combine_projection(s["ref_cam"], s["src_cam"], s["scale"])
    if op == "layer":
        return s["layer"]((s["ref"], s["src"], s["depth"], s["offsets"], Rs, Ts))
    return s["layer"]((s["ref"], s["src"], s["depth"], Rs, Ts))


def run(s):
    if not s["case"]["train"]:
        with torch.no_grad():
            cost, mask = _forward(s)
        return {"cost": cost, "mask": mask}
    cost, mask = _forward(s)
    wanted = [s[k] for k in ("ref", "src", "depth") if s[k].requires_grad]
    if "layer" in s:
        wanted.append(s["layer"].default_cost)
    grads = torch.autograd.grad(cost, wanted, s["upstream"])
    return {"cost": cost.detach(), "mask": mask, "grads": list(grads)}


def work(case):
    B, N, H, W, C, D = (case[k] for k in "BNHWCD")
    op, e = case["op"], ELEMENT[case["dtype"]]
    real = 8 if case["dtype"] == "f64" else 4
    pixels, voxels = B * H * W, B * H * W * D
    out = voxels * {"v1": C, "v2": case["groups"], "layer": 1, "layer2": case["groups"], "v3": 1,
                    "feat": N * C}[op]
    if op == "feat":
        masks = voxels * N
    elif case["reduce"] == "MEAN" or op == "layer":
        masks = voxels
    else:
        masks = 3 * voxels if op == "v3" else out
    ref = 0 if op == "feat" else pixels * C
    src = B * N * H * W * C
    depth = voxels if op in GRID_OPS else pixels
    offsets = 0 if op in GRID_OPS else B * D
    moved = (ref + src + out) * e + (depth + offsets + 12 * B * N) * real + masks * 4
    # per (voxel, view): the reprojection; per channel of it the sample (7) and the reduce (1 to 3)
    samples = voxels * N
    pairs = 2 * C * case["groups"] if op == "v3" else 0   # every group with every group
    flops = samples * (30 + C * {"feat": 7, "v2": 9, "layer2": 9}.get(op, 10) + pairs)
    if case["train"]:
        moved += (out + ref + src) * e
        # sample again, its gradient (2 to 3), the four taps (8) and, where wanted, d/d(depth) (9)
        flops += samples * (30 + C * (18 + (9 if case["depth_grad"] else 0)) + pairs)
        if case["depth_grad"]:
            moved += depth * real
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # sums in another order: 32-bit 1e-5, 64-bit far below; 16-bit results are rounded once
    return {"f32": {"rel": 1e-5}, "f64": {"rel": 1e-12}, "f16": {"rel": 2e-3}, "bf16": {"rel": 1e-2}}[
        case["dtype"]]
