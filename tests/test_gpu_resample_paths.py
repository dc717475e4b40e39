"""Resampling outputs on both sides of the line between the persistent tiled kernel and the one that reads its
taps from the caches, with rows of every alignment, against the fp64 oracle."""
import math

import pytest
import torch

from parity import FWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("size,out", [
    ((20, 22, 17), (16, 18, 16)),       # taps from the caches: partial tiles on every axis, odd rows
    ((6, 9, 2), (16, 16, 17)),          # two columns: boxes one column wide at the last column
    ((3, 1, 33), (4, 40, 40)),          # an axis of one voxel
    ((70, 90, 131), (64, 100, 116)),    # tiled: rows of no whole groups, boxes that end with the row
    ((60, 71, 13), (60, 120, 110)),     # tiled: rows shorter than a box's groups
    ((75, 201, 101), (40, 110, 52)),    # reduced by about two per axis: boxes beyond the LDS tile
    ((31, 250), (64, 70)),              # images, both kernels
    ((500, 401), (900, 801)),
])
def test_rows_of_any_alignment(oracle, dtype, size, out):
    import medvision_amd.ops as ops
    nd = len(size)
    g = wl.gen(sum(size) + sum(out))
    feat = torch.randn(2, 1, *size, generator=g).to(dtype)
    xyz = torch.tensor(size[::-1], dtype=torch.float32)
    ang = (torch.rand(2, 3 if nd == 3 else 1, generator=g) * 2 - 1) * math.radians(25)
    ang[1] = 0.0                                            # one roi without rotation, partly outside
    centre = xyz / 2 + torch.tensor([[0.3], [2.6]])
    rois = torch.cat([torch.tensor([[1.0], [0.0]]), centre, xyz * torch.tensor([[0.9], [1.1]]), ang], 1)
    fn = ops.affine_3d if nd == 3 else ops.affine_2d
    got = fn(feat.to(DEV), rois.to(DEV), out, 1.0, 1, True, 1)
    assert_close(got, oracle.roi_align_forward(feat, rois, out, 1.0, 1, True, 1, True), FWD_TOL[dtype], f"{size} -> {out}")
    if dtype == torch.float32:
        # label maps at order 0: integers and floats pick the same voxels
        labels = torch.randint(0, 9, feat.shape, generator=g, dtype=torch.int32).to(DEV)
        picked = fn(labels, rois.to(DEV), out, 1.0, 1, True, 0)
        assert torch.equal(picked, fn(labels.float(), rois.to(DEV), out, 1.0, 1, True, 0).int())
