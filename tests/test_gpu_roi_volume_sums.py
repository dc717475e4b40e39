"""Gradients of heads on volumes: sums kept channels-last in a workspace, at the edges of the rule and of the tiles,
against the fp64 oracle."""
import pytest
import torch

from parity import BWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("size,channels,rois,cells,ratio", [
    ((9, 11, 13), 8, 6, (4, 4, 4), 2),       # fewest channels
    ((9, 11, 13), 7, 6, (4, 4, 4), 2),       # one fewer: sums in the gradient
    ((16, 16, 16), 33, 8, (4, 4, 4), 0),     # one cell per eight voxels, a channel beyond the tile
    ((16, 16, 16), 33, 7, (4, 4, 4), 0),     # just below
    ((5, 21, 34), 70, 40, (7, 5, 3), 1),
])
def test_fp32_plain(oracle, size, channels, rois, cells, ratio):
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(sum(size) + rois + channels)
    at = torch.rand(rois, 3, generator=g) * torch.tensor(size[::-1]) * 1.2 - 2.0
    boxes = torch.cat([torch.zeros(rois, 1), at, at + torch.rand(rois, 3, generator=g) * 12], 1)
    feat = torch.randn(1, channels, *size, generator=g)
    x = feat.to(DEV).requires_grad_()
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, ratio, 1)
    gy = torch.randn(out.shape, generator=g)
    out.backward(gy.to(DEV))
    want = oracle.roi_align_backward(gy, boxes, feat.shape, 1.0, ratio, True, 1, False)
    assert_close(x.grad, want, BWD_TOL[torch.float32], "backward")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("size,channels,rois,cells,ratio,reach", [
    ((5, 9, 11), 16, 4, (5, 5, 5), 2, 3),         # boxes of too few slices to be shared
    ((7, 9, 11), 16, 20, (5, 5, 5), 2, 7),        # about six slices: one or two workgroups
    ((1, 30, 34), 16, 6, (7, 7, 7), 1, 12),       # one slice
    ((21, 13, 10), 17, 9, (7, 7, 7), 2, 18),      # a second block of one channel
    ((14, 12, 9), 50, 30, (4, 3, 4), 0, 14),      # four blocks of sixteen channels, the last of two
    ((12, 12, 14), 40, 300, (5, 5, 5), 2, 9),     # three blocks, the last of eight channels, two workgroups per box
    ((12, 12, 14), 24, 30, (5, 5, 5), 2, 12),     # without matrix cores blocks of eight channels
    ((9, 12, 14), 9, 7, (7, 5, 7), 2, 9),         # of four
    ((12, 12, 14), 40, 520, (4, 3, 4), 2, 11),    # fp16: two blocks per workgroup, whose wavefronts share the slices of all but flat boxes
    ((24, 30, 34), 40, 16, (6, 5, 7), 3, 40),     # boxes beyond the dense matrices
    ((5, 40, 38), 35, 9, (10, 10, 10), 3, 36),    # wide boxes of few slices: one or two channels per workgroup, one or two parts
    ((20, 30, 30), 19, 3, (7, 6, 7), 2, 28),      # fp16: boxes beyond the matrix cores beside small ones; channels and parts by the box
    ((13, 24, 20), 29, 30, (9, 10, 9), 1, 24),    # more than eight cells: blocks of eight channels or fewer
    ((70, 12, 12), 20, 160, (2, 3, 2), 1, 90),    # boxes wider than the lists: sums per sample
    ((16, 16, 18), 16, 400, (12, 9, 10), 1, 10),  # more than eight cells per axis, three workgroups per box
    ((12, 12, 14), 16, 1023, (4, 4, 4), 2, 9),    # two workgroups per box
    ((12, 12, 14), 16, 1024, (4, 4, 4), 2, 9),    # one
])
def test_plain_boxes_shared_by_workgroups(oracle, dtype, size, channels, rois, cells, ratio, reach):
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(sum(size) + rois + channels)
    at = torch.rand(rois, 3, generator=g) * torch.tensor(size[::-1]) * 1.2 - 2.0
    boxes = torch.cat([torch.randint(0, 2, (rois, 1), generator=g).float(), at, at + torch.rand(rois, 3, generator=g) * reach], 1)
    feat = torch.zeros(2, channels, *size, dtype=dtype)
    x = feat.to(DEV).requires_grad_()
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, ratio, 1)
    gy = torch.randn(out.shape, generator=g).to(dtype)
    out.backward(gy.to(DEV))
    want = oracle.roi_align_backward(gy, boxes, feat.shape, 1.0, ratio, True, 1, False)
    assert_close(x.grad, want, BWD_TOL[dtype], "backward")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("size,channels,rois,cells,ratio,order,reach", [
    ((9, 11, 13), 8, 6, (4, 4, 4), 2, 1, 12),      # tiles with remainders, one group of channels
    ((8, 8, 12), 72, 20, (7, 7, 7), 0, 1, 9),      # rows of whole pieces, a second group with few channels
    ((5, 6, 7), 16, 200, (7, 7, 7), 1, 1, 5),      # few tiles: shared by workgroups
    ((4, 40, 8), 64, 700, (2, 2, 2), 2, 1, 3),     # more rois than a list
    ((12, 10, 9), 24, 8, (3, 5, 2), 2, 0, 14),     # nearest taps
    ((40, 40, 40), 8, 3, (2, 2, 2), 1, 1, 60),     # cells wider than a tile
    ((33, 47), 40, 9, (7, 7), 0, 1, 40),           # images
    ((16, 24), 8, 300, (14, 14), 2, 1, 20),
])
def test_rotated_by_tiles(oracle, dtype, size, channels, rois, cells, ratio, order, reach):
    from medvision_amd.ops.roi_align_rotated_nd import roi_align_rotated_2d, roi_align_rotated_3d
    g = wl.gen(sum(size) + rois + channels)
    nd = len(size)
    at = torch.rand(rois, nd, generator=g) * torch.tensor(size[::-1]) * 1.1 - 1.0
    angle = (torch.rand(rois, 3 if nd == 3 else 1, generator=g) - 0.5) * 6
    image = torch.randint(0, 2, (rois, 1), generator=g).float()
    boxes = torch.cat([image, at, torch.rand(rois, nd, generator=g) * reach + 0.5, angle], 1)
    feat = torch.zeros(2, channels, *size, dtype=dtype)
    x = feat.to(DEV).requires_grad_()
    run = roi_align_rotated_3d if nd == 3 else roi_align_rotated_2d
    out = run(x, boxes.to(DEV), cells, 1.0, ratio, True, order)
    gy = torch.randn(out.shape, generator=g).to(dtype)
    out.backward(gy.to(DEV), retain_graph=True)
    want = oracle.roi_align_backward(gy, boxes, feat.shape, 1.0, ratio, True, order, True)
    assert_close(x.grad, want, BWD_TOL[dtype], "backward")
    # an infinite gradient reaches the voxels of its cell alone
    gy[0, 0].view(-1)[0] = float("inf")
    x.grad = None
    out.backward(gy.to(DEV))
    unit = torch.zeros(out.shape)
    unit[0, 0].view(-1)[0] = 1.0
    hit = oracle.roi_align_backward(unit, boxes, feat.shape, 1.0, ratio, True, order, True).reshape(feat.shape) > 1e-6
    got = x.grad.cpu().double()
    assert not torch.isfinite(got[hit]).any()
    want = want.reshape(feat.shape)
    assert_close(torch.where(hit, want, got), want, BWD_TOL[dtype], "finite part")


@pytest.mark.parametrize("size,cells,ratio,reach", [
    ((40, 40, 40), (2, 2, 2), 0, 80),      # adaptive grids: cells of 10^4 samples
    ((150, 160), (2, 2), 0, 260),
    ((12, 14, 10), (2, 3, 2), 20, 9),      # 8000 samples, most of them in a few voxels
    ((1, 30, 30), (2, 2, 2), 12, 20),      # an axis of one voxel takes the samples of two
])
def test_cells_of_many_samples(oracle, size, cells, ratio, reach):
    """Rotated fp32 heads whose cells hold thousands of samples: the weights are summed as precisely as those of a few (a relative
    error of 1e-6; sums of a few hundred fp32 terms, and cell weights in units of 2^-30 of the largest they can be)."""
    from medvision_amd.ops.roi_align_rotated_nd import roi_align_rotated_2d, roi_align_rotated_3d
    nd, rois = len(size), 12
    g = wl.gen(sum(size) + ratio)
    at = torch.rand(rois, nd, generator=g) * torch.tensor(size[::-1])
    angle = (torch.rand(rois, 3 if nd == 3 else 1, generator=g) - 0.5) * 6
    boxes = torch.cat([torch.zeros(rois, 1), at, torch.rand(rois, nd, generator=g) * reach / 2 + reach / 2, angle], 1)
    x = torch.zeros(1, 16, *size, device=DEV, requires_grad=True)
    out = (roi_align_rotated_3d if nd == 3 else roi_align_rotated_2d)(x, boxes.to(DEV), cells, 1.0, ratio, True, 1)
    gy = torch.randn(out.shape, generator=g)
    out.backward(gy.to(DEV))
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, ratio, True, 1, True)
    error = float((x.grad.cpu().double() - want).norm() / want.norm())
    assert error < 1e-6, error


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("rotated", [False, True])
@pytest.mark.parametrize("sized", [False, True])
def test_backward_keeps_to_its_workspace(oracle, dtype, rotated, sized):
    """The entry points that replace the gradient stay within the workspace they are told of (`sized`), or within the size of the
    query that all backward entry points share: the paths that want more, the owners' and the channels-last sums, are left."""
    from medvision_amd import _lib
    lib, code = _lib.load(), _lib.MV_F16 if dtype == torch.float16 else _lib.MV_F32
    g = wl.gen(3 + rotated)
    dims, rois, cells = (2, 64, 9, 11, 13), 60, 7
    at = torch.rand(rois, 3, generator=g) * torch.tensor(dims[:1:-1])
    image = torch.randint(0, 2, (rois, 1), generator=g).float()
    extent = torch.rand(rois, 3, generator=g) * 8 + 1
    boxes = torch.cat([image, at, extent, torch.rand(rois, 3, generator=g)], 1) if rotated else torch.cat([image, at, at + extent], 1)
    gy = torch.randn(rois, dims[1], cells, cells, cells, generator=g).to(dtype)
    want = oracle.roi_align_backward(gy, boxes, dims, 1.0, 2, True, 1, rotated)
    size = (code, 3, int(rotated), *dims, rois, cells, cells, cells, 2, 1)
    full, shared = lib.mv_roi_align_backward_write_workspace_bytes(*size), lib.mv_roi_align_backward_workspace_bytes(code, *dims)
    assert full > shared or (dtype == torch.float16 and not rotated)
    grad, d_gy, d_rois = torch.full(dims, 7.0, dtype=dtype, device=DEV), gy.to(DEV), boxes.to(DEV)
    for given in (shared, full) if sized else (shared,):
        room = torch.full((full + 4096,), 0x5a, dtype=torch.uint8, device=DEV)
        call = (lib.mv_roi_align_backward_replace if sized else lib.mv_roi_align_backward_write)
        _lib.check(call(_lib.ptr(d_gy), _lib.ptr(d_rois), _lib.ptr(grad), code, 3, int(rotated), *dims, rois, cells, cells, cells,
                        1.0, 2, 1, 1, _lib.ptr(room), *([given] if sized else []), _lib.stream_of(grad)))
        assert bool((room[given:] == 0x5a).all())
        assert_close(grad, want, BWD_TOL[dtype], f"{given} bytes")
    if dtype == torch.float16 and sized:
        with pytest.raises(RuntimeError, match="workspace"):
            _lib.check(call(_lib.ptr(d_gy), _lib.ptr(d_rois), _lib.ptr(grad), code, 3, int(rotated), *dims, rois, cells, cells, cells,
                            1.0, 2, 1, 1, _lib.ptr(room), shared - 4, _lib.stream_of(grad)))
