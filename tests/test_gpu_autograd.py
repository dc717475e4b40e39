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
