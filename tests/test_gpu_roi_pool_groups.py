"""Pooled heads of few rois: small boxes take several channel groups per workgroup, large ones one; both kinds in one call,
around the groups' sizes, against the fp64 oracle."""
import pytest
import torch

from parity import FWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("channels", [1, 3, 4, 5, 16, 17, 34, 256])
@pytest.mark.parametrize("cells,ratio,width", [
    ((7, 7, 7), 2, 40),       # rows of whole pieces: from a copy of the features
    ((4, 5, 3), 0, 37),
    ((4, 4, 4), 1, 40),       # sparse boxes among them
    ((7, 7, 7), 1, 39),
])
def test_small_and_large_boxes(oracle, dtype, channels, cells, ratio, width):
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    size = (18, 33, width)
    g = wl.gen(channels + width + ratio)
    rois = 40
    extent = torch.exp(torch.rand(rois, 3, generator=g) * 4.2 - 0.5)        # 0.6 .. 40 voxels
    at = torch.rand(rois, 3, generator=g) * (torch.tensor(size[::-1]) + 4.0) - 4.0
    boxes = torch.cat([torch.randint(0, 2, (rois, 1), generator=g).float(), at, at + extent], 1)
    feat = torch.randn(2, channels, *size, generator=g).to(dtype)
    want = oracle.roi_align_forward(feat, boxes, cells, 1.0, ratio, True, 1, False)
    boxes[5, 0], want[5] = 2.0, 0.0       # no such image (the oracle does not check): zeros
    out = roi_align_3d(feat.to(DEV), boxes.to(DEV), cells, 1.0, ratio, 1)
    assert_close(out, want, FWD_TOL[dtype], "forward")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("channels,cells,ratio,order", [
    (3, (7, 7, 7), 4, 1),     # more entries than a lane keeps in registers of a small head
    (5, (2, 3, 8), 0, 1),     # more than four slices of a plane, grids above four
    (2, (1, 8, 2), 0, 1),     # a plane of all slices
    (9, (8, 7, 5), 0, 0),     # nearest voxels
    (40, (3, 3, 3), 0, 1),
])
def test_planes_of_large_boxes(oracle, dtype, channels, cells, ratio, order):
    """Boxes of more voxels than the staged form takes: rows in one slab and in several, planes beside the volume."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    size = (21, 90, 71)
    g = wl.gen(channels + sum(cells))
    boxes = torch.tensor([[0, 2.3, 1.7, 3.1, 26.4, 27.9, 17.2], [1, 0.2, 0.4, 0.3, 70.6, 89.5, 20.1], [0, 40.1, 30.6, 2.2, 70.9, 52.3, 19.0],
                          [1, -9.3, 60.5, -12.7, 14.0, 88.2, 13.9], [0, 30.2, -20.0, 12.5, 33.1, 110.0, 40.0], [1, 10.0, 2.0, 1.0, 11.0, 88.0, 20.0],
                          [0, 1.0, 20.5, 2.5, 70.0, 24.5, 18.5]])
    feat = torch.randn(2, channels, *size, generator=g).to(dtype)
    want = oracle.roi_align_forward(feat, boxes, cells, 1.0, ratio, True, order, False)
    out = roi_align_3d(feat.to(DEV), boxes.to(DEV), cells, 1.0, ratio, order)
    assert_close(out, want, FWD_TOL[dtype], "forward")
    if order == 1 and cells[0] >= 3 and dtype != torch.float16:
        feat[:, :, 0] = float("inf")      # slices that the last planes do not touch; planes beside the volume stay zero
        out = roi_align_3d(feat.to(DEV), boxes.to(DEV), cells, 1.0, ratio, order)
        assert torch.equal(out[:2, :, -1].cpu(), roi_align_3d(torch.where(feat.isinf(), 0.0, feat).to(dtype).to(DEV), boxes.to(DEV), cells, 1.0, ratio, order)[:2, :, -1].cpu())
        assert bool((out[3, :, 0] == 0).all())
