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
