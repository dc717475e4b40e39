"""Operators without a forward-mode derivative refuse dual tensors instead of dropping the tangent."""
import pytest
import torch
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _calls():
    import medvision_amd.ops as ops
    vol, img = torch.randn(1, 2, 8, 9, 10, device=DEV), torch.randn(1, 2, 9, 10, device=DEV)
    plain3 = torch.tensor([[0, 1, 1, 1, 6, 6, 6.]], device=DEV)
    plain2 = torch.tensor([[0, 1, 1, 6, 6.]], device=DEV)
    turned3 = torch.tensor([[0, 4, 4, 4, 5, 5, 5, .1, .2, .3]], device=DEV)
    turned2 = torch.tensor([[0, 4, 4, 5, 5, .1]], device=DEV)
    dcn = ops.ModulatedDeformConv3d(2, 2, 3, padding=1).to(DEV)
    off, mask = torch.zeros(1, 81, 8, 9, 10, device=DEV), torch.ones(1, 27, 8, 9, 10, device=DEV)
    return {
        "RoIAlign 3-D": (lambda x, r: ops.RoIAlign((2, 2, 2), 1.0, 2)(x, r), vol, plain3),
        "RoIAlign 2-D": (lambda x, r: ops.RoIAlign((2, 2), 1.0, 2)(x, r), img, plain2),
        "RoIAlignRotated 3-D": (lambda x, r: ops.RoIAlignRotated((2, 2, 2), 1.0, 2)(x, r), vol, turned3),
        "RoIAlignRotated 2-D": (lambda x, r: ops.RoIAlignRotated((2, 2), 1.0, 2)(x, r), img, turned2),
        "ModulatedDeformConv3d": (lambda x, o: dcn(x, o, mask), vol, off),
    }


@pytest.mark.parametrize("name", ["RoIAlign 3-D", "RoIAlign 2-D", "RoIAlignRotated 3-D", "RoIAlignRotated 2-D",
                                  "ModulatedDeformConv3d"])
@pytest.mark.parametrize("grad", [True, False])
def test_dual_tensors_are_refused(name, grad):
    run, x, second = _calls()[name]
    with torch.set_grad_enabled(grad), forward_ad.dual_level():
        with pytest.raises(NotImplementedError):
            run(forward_ad.make_dual(x, torch.ones_like(x)), second)
        with pytest.raises(NotImplementedError):
            run(x, forward_ad.make_dual(second, torch.ones_like(second)))
    with pytest.raises((NotImplementedError, RuntimeError)):
        torch.func.jvp(lambda t: run(t, second), (x,), (torch.ones_like(x),))
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: run(t, second))(x.unsqueeze(0))
    assert torch.isfinite(run(x, second)).all()


def _layers():
    import medvision_amd.ops as ops
    from medvision_amd.ops import (deform_conv_2d, deform_conv_3d, modulated_deform_conv_2d, modulated_deform_conv_3d,
                                   roi_align_nd, roi_align_rotated_nd)
    g = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g).to(DEV)
    vol, img = r(2, 4, 7, 8, 9), r(2, 4, 8, 9)
    plain3, plain2 = torch.tensor([[1, 1, 1, 1, 6, 6, 5.]], device=DEV), torch.tensor([[0, 1, 1, 6, 6.]], device=DEV)
    turned3 = torch.tensor([[1, 4, 4, 4, 5, 5, 5, .1, .2, .3]], device=DEV)
    turned2 = torch.tensor([[0, 4, 4, 5, 5, .1]], device=DEV)
    w3, w2, b = r(6, 4, 3, 3, 3), r(6, 4, 3, 3), r(6)
    return [
        (roi_align_nd.RoIAlign3DFunction, [vol], (plain3, (2, 2, 2), 1.0, 2)),
        (roi_align_nd.RoIAlign2DFunction, [img], (plain2, (2, 2), 1.0, 0, 1)),
        (roi_align_rotated_nd.RoIAlignRotated3DFunction, [vol], (turned3, (2, 2, 2), 1.0, 2, True, 1)),
        (roi_align_rotated_nd.RoIAlignRotated2DFunction, [img], (turned2, (2, 2), 1.0, 2)),
        (deform_conv_3d.DeformConv3dFunction, [vol, r(2, 81, 7, 8, 9), w3, b], (1, 1, 1, 1, 1, 64)),
        (deform_conv_2d.DeformConv2dFunction, [img, r(2, 18, 8, 9), w2, b], (1, 1, 1, 1, 1, 64)),
        (modulated_deform_conv_3d.ModulatedDeformConv3dFunction, [vol, r(2, 81, 7, 8, 9), r(2, 27, 7, 8, 9), w3, b], (1, 1)),
        (modulated_deform_conv_2d.ModulatedDeformConv2dFunction, [img, r(2, 18, 8, 9), r(2, 9, 8, 9), w2, b], (1, 1)),
    ]


@pytest.mark.parametrize("index", range(8))
def test_functions_and_their_subclasses_agree(index):
    """``forward`` and ``backward`` of the classes, as a subclass of them is run, against the native node."""
    base, leaves, rest = _layers()[index]

    class Counted(base):
        calls = 0

        @staticmethod
        def backward(ctx, grad):
            Counted.calls += 1
            return base.backward(ctx, grad)

    results = []
    for function in (base, Counted):
        ins = [t.clone().requires_grad_() for t in leaves]
        out = function.apply(*ins, *rest)
        results.append([out, *torch.autograd.grad(out, ins, torch.ones_like(out))])
    assert Counted.calls == 1
    for got, want in zip(*results):
        torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4 * float(want.abs().max()))


@pytest.mark.parametrize("index", range(8))
def test_traced_layers_run_their_operator(index):
    """torch.jit.trace records the operators as nodes: a traced call computes with the inputs that it is given."""
    function, leaves, rest = _layers()[index]
    consts = [a for a in rest if not torch.is_tensor(a)]
    inputs = [*leaves, *[a for a in rest if torch.is_tensor(a)]]

    def run(*tensors):
        return function.apply(*tensors, *consts) + 1

    with torch.no_grad():
        traced = torch.jit.trace(run, tuple(inputs))
        other = (leaves[0] * 2 + 1, *inputs[1:])
        torch.testing.assert_close(traced(*other), run(*other))
        assert not torch.equal(traced(*other), traced(*inputs))


def test_function_transforms_are_refused():
    """torch.func's gradient has no rule for the operators either: an error, as before, not a wrong result."""
    for function, leaves, rest in _layers():
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: function.apply(t, *leaves[1:], *rest).sum())(leaves[0])


@pytest.mark.parametrize("groups,dg", [(0, 1), (1, 0), (-1, 1), (1, -2)])
def test_groups_that_cannot_be_divided_by_are_refused(groups, dg):
    from medvision_amd.ops.deform_conv_2d import deform_conv
    from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    x, off, mask = torch.zeros(1, 4, 6, 6, device=DEV), torch.zeros(1, 18, 6, 6, device=DEV), torch.zeros(1, 9, 6, 6, device=DEV)
    weight, bias = torch.zeros(4, 4, 3, 3, device=DEV), torch.zeros(4, device=DEV)
    with pytest.raises(RuntimeError):
        modulated_deform_conv(x, off, mask, weight, bias, 1, 1, 1, groups, dg)
    with pytest.raises(RuntimeError):
        deform_conv(x, off, weight, bias, 1, 1, 1, groups, dg, 64)
