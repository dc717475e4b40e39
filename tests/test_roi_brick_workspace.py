"""Scratch memory of the backward pass of fp16 heads on volumes: lists of rois per brick do not outgrow the kernel with atomics."""
import pytest

from medvision_amd import _lib


@pytest.mark.parametrize("dims,rois,lists", [
    ((2, 256, 24, 96, 96), 4000, True),
    ((1, 16, 64, 128, 128), 4000, True),        # 2048 bricks
    ((1, 16, 256, 256, 256), 8000, True),       # 32768 bricks: 1.05 GB of lists, a copy of 1.07 GB
    ((1, 16, 256, 256, 256), 8300, False),
    ((8, 16, 64, 128, 128), 60000, False),      # 3.9 GB of lists
])
def test_lists_are_no_larger_than_the_copy(dims, rois, lists):
    lib, code = _lib.load(), _lib.MV_F16
    copy = lib.mv_roi_align_backward_workspace_bytes(code, *dims)
    asked = lib.mv_roi_align_backward_write_workspace_bytes(code, 3, 0, *dims, rois, 7, 7, 7, 2, 1)
    assert asked <= max(copy, 256 << 20)
    assert asked >= copy
    if not lists:
        assert asked == copy


@pytest.mark.parametrize("cells,rois,served", [
    ((7, 7, 7), 4000, True),
    ((7, 7, 8), 4000, True),      # 13 kilobytes of a ring of 18
    ((8, 8, 8), 4000, False),     # 17 of them: box by box
    ((7, 8, 8), 4000, False),
    ((8, 8, 8), 1079, True),      # fewer than five rois for four of the 864 bricks
    ((8, 8, 8), 1080, False),
    ((4, 4, 4), 4000, True),      # small gradients: two fit their ring, however small it is
    ((5, 5, 5), 4000, True),
    ((2, 2, 2), 4000, True),
])
def test_gradients_that_fill_their_ring(cells, rois, served):
    from test_gpu_roi_brick import bricks_apply
    assert bricks_apply((2, 256, 24, 96, 96), rois, cells) == served


@pytest.mark.parametrize("rois,served", [(28, True), (29, False)])
def test_gradients_that_fill_their_ring_on_small_maps(rois, served):
    """1152 pairs of a brick and 16 channels: two rois for five of the 72 bricks."""
    from test_gpu_roi_brick import bricks_apply
    assert bricks_apply((1, 256, 24, 32, 48), rois, (8, 8, 8)) == served
