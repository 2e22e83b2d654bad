"""What the native host path keeps of torch's machinery: saved-tensor hooks and checkpointing, the
types of errors, tracing, forward-mode and functional derivatives -- for every differentiable
function, on the GPU and, with the C ABI taken from the oracle (host_path.py), on the CPU."""
import ctypes

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as forward_ad
import torch.utils.checkpoint

import custom_helper_op_amd as chop
import host_path
from custom_helper_op_amd import _lib, ops
from custom_helper_op_amd.configs import reference_test_case

FORMS = ("cost_volume", "cost_volume_v2", "cost_volume_v3", "cost_aggregate", "feature_aggregate",
         "cost_volume_v2_filled", "cost_aggregate_filled")


@pytest.fixture(scope="module")
def cpu_module(tmp_path_factory):
    return host_path.build_module(tmp_path_factory.mktemp("host_path"))


@pytest.fixture(params=["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def device(request, monkeypatch):
    if request.param == "cpu":
        module = request.getfixturevalue("cpu_module")[0]
        ops._connect(module)
        monkeypatch.setattr(ops, "_native_module", module)
    return request.param


def _inputs(form, device, grad=True, seed=2):
    """Positional tensors of a differentiable function, and the function on them."""
    t = reference_test_case(3, 1, 2, 6, 7, 8, 5, np.float32, seed=seed)
    t = {k: torch.from_numpy(v).to(device) for k, v in t.items()}
    t["depth_grid"] = t["base_plane"] + t["offsets"][:, None, None, :]
    t["default"] = torch.full((), 0.25, device=device)
    v2 = "_v2" in form
    keys = [] if form == "feature_aggregate" else ["ref"]
    keys += ["src"] + (["depth_grid"] if v2 else ["base_plane", "offsets"]) + ["Rs", "Ts"]
    wanted = {"ref", "src", "depth_grid", "base_plane", "default"} if grad else ()
    keys += ["default"] if form.endswith("filled") else []
    ins = [t[k].requires_grad_(k in wanted) for k in keys]
    kw = {"groups": 2} if v2 or form == "cost_volume_v3" else {}
    return ins, lambda *a, **more: getattr(chop, form)(*a, **kw, **more)


def _gradients(ins, cost, seed=5):
    up = torch.randn(cost.shape, generator=torch.Generator().manual_seed(seed)).to(cost)
    return torch.autograd.grad(cost, [x for x in ins if x.requires_grad], up)


def _close(got, want):
    # float32 sums of one order against another: the order of the GPU's atomics is free
    for g, w in zip(got, want):
        torch.testing.assert_close(g, w, rtol=1e-5, atol=1e-5 * float(w.abs().max()))


class Mine(Exception):
    pass


@pytest.mark.parametrize("form", FORMS)
def test_checkpoint_of_the_bare_operator(form, device):
    """Its recomputation ends with an exception out of the pack hook, inside the operator's call."""
    ins, fn = _inputs(form, device)
    want = _gradients(ins, fn(*ins)[0])
    cost, mask = torch.utils.checkpoint.checkpoint(fn, *ins, use_reentrant=False)
    _close(_gradients(ins, cost), want)


@pytest.mark.parametrize("form", FORMS)
def test_hooks_see_the_saved_tensors_and_may_raise(form, device):
    ins, fn = _inputs(form, device)
    want, packed = _gradients(ins, fn(*ins)[0]), []

    def pack(x):
        packed.append(x)
        return x.detach().cpu()

    def raises(x):
        raise Mine(form)

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda x: x.to(device)):
        cost, mask = fn(*ins)
    assert len(packed) == len(ins) + 1
    _close(_gradients(ins, cost), want)
    with torch.autograd.graph.saved_tensors_hooks(raises, lambda x: x), pytest.raises(Mine, match=form):
        fn(*ins)
    with torch.autograd.graph.saved_tensors_hooks(lambda x: x, raises):
        cost, mask = fn(*ins)
    with pytest.raises(Mine, match=form):
        _gradients(ins, cost)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("grad", [False, True])
def test_trace_holds_the_operator(form, grad, device):
    ins, fn = _inputs(form, device, grad)
    traced = torch.jit.trace(lambda *a: fn(*a), tuple(ins))
    other, _ = _inputs(form, device, grad, seed=3)
    cost, mask = traced(*other)
    want_cost, want_mask = fn(*other)
    assert torch.equal(cost, want_cost) and torch.equal(mask, want_mask)
    if grad:
        _close(_gradients(other, cost), _gradients(other, want_cost))


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_is_refused(form, grad, device):
    """There is no forward derivative: an input with a tangent must not give a result without one."""
    ins, fn = _inputs(form, device, grad)
    with forward_ad.dual_level():
        for i in range(len(ins)):
            dual = [forward_ad.make_dual(x, torch.ones_like(x)) if k == i else x for k, x in enumerate(ins)]
            with pytest.raises(NotImplementedError, match="forward mode"):
                fn(*dual)
        assert fn(*ins)[0].requires_grad == grad


@pytest.mark.parametrize("form", FORMS)
def test_functional_transforms_are_refused(form, device):
    ins, fn = _inputs(form, device, grad=False)
    first, rest = ins[0], ins[1:]
    for call in (lambda: torch.func.grad(lambda x: fn(x, *rest)[0].sum())(first),
                 lambda: torch.func.vmap(lambda x: fn(x, *rest)[0])(first[None]),
                 lambda: torch.func.vmap(lambda z: fn(*ins)[0] + z)(torch.zeros(3, device=device)),
                 lambda: torch.func.jvp(lambda x: fn(x, *rest)[0], (first,), (first,))):
        with pytest.raises(RuntimeError, match="functorch transforms"):
            call()


@pytest.mark.parametrize("form", FORMS)
def test_errors_of_the_backward_pass_keep_their_types(form, device):
    ins, fn = _inputs(form, device)
    ndim = max(x.dim() for x in ins)
    with torch.autograd.graph.saved_tensors_hooks(lambda x: x, lambda x: x[:, :1] if x.dim() == ndim else x):
        cost, mask = fn(*ins)
    with pytest.raises(chop.InvalidArgumentError, match="must compate"):
        _gradients(ins, cost)


@pytest.mark.parametrize("form", FORMS)
def test_status_of_the_library_reaches_the_caller(form, cpu_module, monkeypatch):
    module, so = cpu_module
    ops._connect(module)
    monkeypatch.setattr(ops, "_native_module", module)
    status = ctypes.c_int.in_dll(ctypes.CDLL(so), "chop_test_status")
    ins, fn = _inputs(form, "cpu")
    cost, mask = fn(*ins)
    try:
        status.value = 5
        for call in (lambda: fn(*ins), lambda: _gradients(ins, cost)):
            with pytest.raises(_lib.ChopError, match="as the test asked") as caught:
                call()
            assert caught.value.code == 5
    finally:
        status.value = 0


@pytest.mark.parametrize("form", FORMS)
def test_what_hooks_give_back_is_checked(form, device):
    """Tensors of another type than the upstream gradient's, or another mask, never reach a kernel."""
    ins, fn = _inputs(form, device)
    for change, match in ((lambda x: x.double() if x.is_floating_point() else x, "grad must have dtype torch.float64"),
                          (lambda x: x if x.is_floating_point() else x.long(), "mask must have dtype torch.int32"),
                          (lambda x: x[:0] if x.is_floating_point() and x.dim() else x, "must compate"),
                          (lambda x: x if x.dim() else x.new_empty(0), "default_cost must be a scalar")):
        if "default" in match and not form.endswith("filled"):
            continue
        with torch.autograd.graph.saved_tensors_hooks(lambda x: x, change):
            cost, mask = fn(*ins)
        with pytest.raises(chop.InvalidArgumentError, match=match):
            _gradients(ins, cost)


def test_order_of_the_checks(device):
    """Types before shapes, and among the types the order in which the operators take them."""
    ins, fn = _inputs("cost_volume", device, grad=False)
    cost, mask = fn(*ins)
    ref, src, plane, offsets, Rs, Ts = ins
    grid = plane + offsets[:, None, None, :]
    for match, call in (
            ("Rs must have", lambda: chop.cost_volume(ref, src, plane.double(), offsets, Rs.double(), Ts)),
            ("cost_grad must have", lambda: chop.cost_volume_grad(ref, src, plane.double(), offsets, Rs, Ts,
                                                                  cost.double(), mask)),
            ("cost_grad must have", lambda: chop.cost_volume_grad(ref[0], src, plane, offsets, Rs, Ts,
                                                                  cost.double(), mask)),
            ("cost_mask must have", lambda: chop.cost_volume_grad(ref[0], src, plane, offsets, Rs, Ts, cost,
                                                                  mask.long())),
            ("base_plane must have", lambda: chop.cost_aggregate(ref, src, plane.double(), offsets, Rs.double(), Ts)),
            ("depth_grid must have", lambda: chop.cost_volume_v2(ref, src, grid.double(), Rs.double(), Ts, groups=2)),
            ("cost_grad must have", lambda: chop.cost_volume_grad_v2(ref[0], src, grid, Rs, Ts, cost.double(), mask,
                                                                     groups=2)),
            ("ref image must", lambda: chop.cost_volume_grad(ref[0], src, plane, offsets, Rs, Ts, cost, mask[0]))):
        with pytest.raises(chop.InvalidArgumentError, match=match):
            call()


@pytest.mark.parametrize("form", FORMS)
def test_half_centor_is_a_number(form, device):
    ins, fn = _inputs(form, device, grad=False)
    for bad, error in ((None, TypeError), ("no", ValueError), ([], TypeError)):
        with pytest.raises(error):
            fn(*ins, half_centor=bad)
    for yes, no in ((1, 0), (np.True_, np.False_)):
        assert torch.equal(fn(*ins, half_centor=yes)[0], fn(*ins, half_centor=True)[0])
        assert torch.equal(fn(*ins, half_centor=no)[0], fn(*ins, half_centor=False)[0])


@pytest.mark.parametrize("form", FORMS)
def test_strided_inputs_subsets_and_a_second_pass(form, device):
    plain, fn = _inputs(form, device)
    wanted = [i for i, x in enumerate(plain) if x.requires_grad]
    want = dict(zip(wanted, _gradients(plain, fn(*plain)[0])))
    for subset in [[i] for i in wanted] + [wanted]:
        ins = [x.detach() if x.dim() < 3 else x.detach().transpose(1, 2).contiguous().transpose(1, 2) for x in plain]
        for i in subset:
            ins[i].requires_grad_(True)
        cost, mask = fn(*ins)
        assert cost.requires_grad and not mask.requires_grad
        up = torch.randn(cost.shape, generator=torch.Generator().manual_seed(5)).to(cost)
        for retain in (True, False):
            _close(torch.autograd.grad(cost, [ins[i] for i in subset], up, retain_graph=retain), [want[i] for i in subset])
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(cost, [ins[i] for i in subset], up)
    with torch.no_grad():
        assert not fn(*plain)[0].requires_grad
    cost, mask = fn(*plain)
    with torch.no_grad():
        plain[wanted[0]].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        _gradients(plain, cost)
