"""Gradients of fp32 heads of rotated boxes with one sample per cell, on both sides of the line between the owners' kernel and the
one with atomics, against the fp64 oracle."""
import pytest
import torch

from parity import BWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rois", [56, 57, 120])   # 90112 voxels: from 57 rois on the owners' kernel
@pytest.mark.parametrize("ratio", [0, 1])
def test_sparse_rotated_heads(oracle, rois, ratio):
    from medvision_amd.ops.roi_align_rotated_nd import roi_align_rotated_3d
    g = wl.gen(rois + ratio)
    images, channels, size, cells = 1, 192, (32, 44, 64), (4, 4, 4)
    at = torch.rand(rois, 3, generator=g) * torch.tensor(size[::-1])
    boxes = torch.cat([torch.zeros(rois, 1), at, torch.rand(rois, 3, generator=g) * 12 + 1, torch.rand(rois, 3, generator=g) - 0.5], 1)
    x = torch.zeros(images, channels, *size, device="cuda:0", requires_grad=True)
    out = roi_align_rotated_3d(x, boxes.to("cuda:0"), cells, 1.0, ratio)
    gy = torch.randn(out.shape, generator=g)
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, ratio, True, 1, True)
    assert_close(torch.autograd.grad(out, x, gy.to("cuda:0"))[0], want.reshape(x.shape), BWD_TOL[torch.float32], "gradient")
