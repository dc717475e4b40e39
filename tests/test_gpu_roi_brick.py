"""Gradients of fp16 heads of plain boxes on volumes by the voxels' owners (roi_brick_backward.hip): remainders of bricks and
channels, rows of cells at any alignment, shared bricks, gradients that are not finite, against the fp64 oracle."""
import ctypes

import pytest
import torch

from parity import BWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = BWD_TOL[torch.float16]


def boxes_of(g, images, size, rois, reach):
    at = torch.rand(rois, 3, generator=g) * torch.tensor(size[::-1]) * 1.2 - 2.0
    image = torch.randint(0, images, (rois, 1), generator=g).float()
    return torch.cat([image, at, at + torch.rand(rois, 3, generator=g) * reach], 1)


@pytest.mark.parametrize("images,channels,size,rois,cells,ratio,order,reach", [
    (2, 128, (9, 17, 33), 60, (7, 7, 7), 2, 1, 12),     # a voxel beyond the bricks on every axis
    (1, 320, (16, 24, 32), 9, (8, 8, 8), 2, 1, 20),     # whole bricks, rows of eight cells, a gradient that fills its ring
    (4, 80, (40, 33, 8), 50, (5, 6, 7), 0, 1, 20),      # one brick along x
    (2, 129, (9, 17, 33), 40, (5, 3, 7), 1, 1, 9),      # odd channels: gradients that start between two words
    (2, 128, (9, 17, 33), 74, (4, 4, 4), 2, 1, 9),      # one workgroup per brick
    (2, 128, (9, 17, 33), 300, (4, 4, 4), 2, 1, 9),     # four share one
    (1, 128, (16, 16, 120), 700, (7, 1, 2), 3, 1, 9),   # the last of seven regions along x is half empty
    (2, 128, (9, 17, 33), 1100, (2, 2, 2), 1, 1, 6),    # more rois than are tried at a time
    (2, 144, (20, 30, 30), 20, (3, 5, 2), 2, 0, 14),    # nearest taps
    (1, 256, (30, 30, 30), 6, (7, 7, 7), 1, 1, 200),    # boxes larger than the map
    (3, 64, (41, 20, 40), 1, (1, 1, 1), 1, 1, 3),       # one cell
])
def test_bricks(oracle, images, channels, size, rois, cells, ratio, order, reach):
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(sum(size) + rois + channels)
    boxes = boxes_of(g, images, size, rois, reach)
    x = torch.zeros(images, channels, *size, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, ratio, order)
    gy = torch.randn(out.shape, generator=g).half()
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, ratio, True, order, False).reshape(x.shape)
    # gradients at a word's start and between two words
    for shift in (0, 1):
        room = torch.zeros(gy.numel() + 1, dtype=torch.float16, device=DEV)
        room[shift:shift + gy.numel()] = gy.flatten().to(DEV)
        assert_close(torch.autograd.grad(out, x, room[shift:shift + gy.numel()].view(gy.shape), retain_graph=True)[0], want, TOL, f"shift {shift}")
    # an infinite gradient reaches the voxels of its cell alone
    gy[0, 0].view(-1)[0] = float("inf")
    unit = torch.zeros(out.shape)
    unit[0, 0].view(-1)[0] = 1.0
    # (weights are rounded to 11 bits, 2^-25 at the least)
    hit = oracle.roi_align_backward(unit, boxes, x.shape, 1.0, ratio, True, order, False).reshape(x.shape) > 1e-6
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    assert not torch.isfinite(got[hit]).any()
    assert_close(torch.where(hit, want, got), want, TOL, "finite part")


def test_sums_beyond_fp16(oracle):
    """Cells far smaller than a voxel: sums over y and x of gradients near the type's largest, which no fp16 number holds."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(5)
    size = (9, 17, 33)
    at = torch.rand(6, 3, generator=g) * 6 + 1
    boxes = torch.cat([torch.zeros(6, 1), at, at + 0.1], 1)
    x = torch.zeros(2, 128, *size, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), (7, 7, 7), 1.0, 2, 1)
    gy = (torch.randn(out.shape, generator=g) * 3000).half()
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, 2, True, 1, False).reshape(x.shape)
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    fits = want.abs() < 60000
    assert bool((got[~fits].abs() > 59000).all())
    assert_close(torch.where(fits, got, want), want, TOL, "gradient")


def test_keeps_to_its_workspace(oracle):
    """With the room that the query asks for, and with the room that the older kernels need, which then run."""
    from medvision_amd import _lib
    lib, code = _lib.load(), _lib.MV_F16
    g = wl.gen(3)
    dims, rois, cells = (2, 128, 9, 17, 33), 300, 7
    boxes = boxes_of(g, 2, dims[2:], rois, 9)
    gy = torch.randn(rois, dims[1], cells, cells, cells, generator=g).half()
    want = oracle.roi_align_backward(gy, boxes, dims, 1.0, 2, True, 1, False)
    size = (code, 3, 0, *dims, rois, cells, cells, cells, 2, 1)
    full, shared = lib.mv_roi_align_backward_write_workspace_bytes(*size), lib.mv_roi_align_backward_workspace_bytes(code, *dims)
    assert full > shared
    grad, d_gy, d_rois = torch.full(dims, 7.0, dtype=torch.float16, device=DEV), gy.to(DEV), boxes.to(DEV)
    for given in (shared, full):
        room = torch.full((full + 4096,), 0x5a, dtype=torch.uint8, device=DEV)
        grad.fill_(7.0)
        _lib.check(lib.mv_roi_align_backward_replace(_lib.ptr(d_gy), _lib.ptr(d_rois), _lib.ptr(grad), code, 3, 0, *dims, rois, cells, cells, cells,
                                                     1.0, 2, 1, 1, _lib.ptr(room), given, _lib.stream_of(grad)))
        assert bool((room[given:] == 0x5a).all())
        assert_close(grad, want, TOL, f"{given} bytes")


@pytest.mark.parametrize("images,channels,size,rois", [
    (1, 128, (32, 40, 64), 1300),    # 1280 pairs of a brick and 16 channels: three workgroups each
    (1, 128, (32, 40, 64), 1279),    # one roi short of eight per brick: one
    (1, 256, (9, 16, 17), 110),      # the most that share one
])
def test_more_workgroups_share_bricks_of_many_rois(oracle, images, channels, size, rois):
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(rois)
    boxes = boxes_of(g, images, size, rois, 7)
    x = torch.zeros(images, channels, *size, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), (2, 3, 2), 1.0, 1, 1)
    gy = torch.randn(out.shape, generator=g).half()
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, 1, True, 1, False).reshape(x.shape)
    assert_close(torch.autograd.grad(out, x, gy.to(DEV))[0], want, TOL, "gradient")


@pytest.mark.parametrize("scale", [1e-5, 1e-6])
def test_small_gradients(oracle, scale):
    """Gradients in the subnormal range: the result's own rounding (half a step of 2^-24) is what may be left, with the same again
    for the sums' operands."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(8)
    boxes = boxes_of(g, 1, (24, 40, 40), 300, 12)
    x = torch.zeros(1, 128, 24, 40, 40, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), (7, 7, 7), 1.0, 2, 1)
    gy = (torch.randn(out.shape, generator=g) * scale).half()
    want = torch.as_tensor(oracle.roi_align_backward(gy, boxes, x.shape, 1.0, 2, True, 1, False)).double().reshape(x.shape)
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    own = (want.half().double() - want).norm()
    # (weights of 11 bits, twice: below 1e-3 of the result)
    assert (got - want).norm() <= 1.1 * own + 1e-3 * want.norm()


def test_gradients_beyond_their_scale(oracle):
    """Large gradients in some cells of a roi and ordinary ones in the rest."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(9)
    boxes = boxes_of(g, 2, (9, 17, 33), 60, 12)
    x = torch.zeros(2, 128, 9, 17, 33, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), (7, 7, 7), 1.0, 2, 1)
    gy = torch.randn(out.shape, generator=g).half()
    gy[::3, ::5] *= 4000
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, 2, True, 1, False).reshape(x.shape)
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    want = torch.as_tensor(want).double()
    fits = want.abs() < 60000
    assert_close(torch.where(fits, got, want), want, TOL, "gradient")
    ordinary = torch.ones(128, dtype=torch.bool)
    ordinary[::5] = False
    assert_close(got[:, ordinary], want[:, ordinary], TOL, "channels of ordinary gradients")


@pytest.mark.parametrize("cells", [(4, 4, 4), (7, 7, 7), (8, 8, 8)])
def test_small_gradients_beside_large_ones(oracle, cells):
    """Channels of gradients near the type's largest beside channels in the subnormal range, in the same bricks: what may be left of the
    small ones is the result's own rounding, with weights of 11 bits, twice (below 1e-3 of the result)."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(11)
    boxes = boxes_of(g, 1, (24, 40, 40), 300, 12)
    x = torch.zeros(1, 128, 24, 40, 40, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, 2, 1)
    gy = torch.randn(out.shape, generator=g) * 1e-5
    gy[:, ::5] *= 1e9
    gy = gy.half()
    assert bool(torch.isfinite(gy).all()) and float(gy.abs().max()) > 3e4
    want = torch.as_tensor(oracle.roi_align_backward(gy, boxes, x.shape, 1.0, 2, True, 1, False)).double().reshape(x.shape)
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    small = torch.ones(128, dtype=torch.bool)
    small[::5] = False
    own = (want[:, small].half().double() - want[:, small]).norm()
    assert (got[:, small] - want[:, small]).norm() <= 1.1 * own + 1e-3 * want[:, small].norm()


class _Problem(ctypes.Structure):   # RoiProblem (csrc/roi_geometry.hpp)
    _fields_ = ([(n, ctypes.c_int) for n in ("ndim", "rotated", "N", "C", "D", "H", "W", "R", "od", "oh", "ow")] + [("scale", ctypes.c_double)] +
                [(n, ctypes.c_int) for n in ("sampling_ratio", "aligned", "order")] + [(n, ctypes.c_uint) for n in ("per_roi", "chunks")])


def bricks_apply(dims, rois, cells, ratio=2):
    """Whether the bricks' kernels serve a head."""
    from medvision_amd import _lib
    fn = _lib.load()._ZN2mv19roi_brick_workspaceEiRKNS_10RoiProblemE
    fn.restype, fn.argtypes = ctypes.c_size_t, [ctypes.c_int, ctypes.POINTER(_Problem)]
    problem = _Problem(3, 0, *dims, rois, *cells, 1.0, ratio, 1, 1, dims[1] * cells[0] * cells[1] * cells[2], 1)
    return fn(_lib.MV_F16, ctypes.byref(problem)) > 0


@pytest.mark.parametrize("size,rois", [((9, 17, 33), 60), ((9, 17, 33), 480), ((40, 33, 8), 60), ((40, 33, 8), 480)])
@pytest.mark.parametrize("kind", ["plus", "minus", "both", "nan", "all inf", "all nan"])
def test_gradients_that_are_not_finite(oracle, size, rois, kind):
    """One workgroup per brick and several, one brick along x and several: infinities reach their voxels with their sign, both signs and NaN as
    NaN, every other voxel keeps its sum."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(rois + size[2])
    channels = 160
    assert bricks_apply((2, channels, *size), rois, (4, 5, 4))
    boxes = boxes_of(g, 2, size, rois, 9)
    x = torch.zeros(2, channels, *size, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), (4, 5, 4), 1.0, 2, 1)
    gy = torch.randn(out.shape, generator=g).half()
    draw = torch.rand(gy.shape, generator=g)
    if kind.startswith("all"):
        gy = torch.full_like(gy, float("inf")) * torch.sign(gy) if kind == "all inf" else torch.full_like(gy, float("nan"))
    else:
        few = draw < 2e-4
        value = {"plus": torch.full_like(draw, float("inf")), "minus": torch.full_like(draw, -float("inf")), "nan": torch.full_like(draw, float("nan")),
                 "both": torch.where(draw < 1e-4, float("inf"), -float("inf"))}[kind]
        gy = torch.where(few, value.half(), gy)
    reach = lambda of: torch.as_tensor(oracle.roi_align_backward(of.half(), boxes, x.shape, 1.0, 2, True, 1, False)).reshape(x.shape)
    plus, minus = reach((gy == float("inf")) | gy.isnan()), reach((gy == -float("inf")) | gy.isnan())
    finite = reach(torch.where(gy.isfinite(), gy, 0))
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    sure, none = 1e-6, 0.0   # (weights between: too small for 16 bits)
    assert bool(got[(plus > sure) & (minus > sure)].isnan().all())
    assert bool((got[(plus > sure) & (minus == none)] == float("inf")).all())
    assert bool((got[(plus == none) & (minus > sure)] == -float("inf")).all())
    apart = (plus == none) & (minus == none)
    assert_close(torch.where(apart, got, finite.double()), finite, TOL, "finite part")
    assert kind.startswith("all") or float(apart.float().mean()) > 0.2


@pytest.mark.parametrize("size,rois,cells,ratio,low,high", [
    ((24, 40, 40), 60, (7, 7, 7), 2, 15, 24),     # slices of more than 14 x 16
    ((24, 40, 40), 60, (4, 5, 4), 0, 15, 24),     # adaptive grids; rows that stand twice and rows that do not
    ((40, 66, 64), 12, (7, 7, 7), 2, 33, 60),     # beyond 32 voxels
    ((24, 40, 40), 60, (2, 3, 4), 0, 70, 90),     # more than 64 samples along an axis, most of them before the map
    ((24, 40, 40), 15, (8, 8, 8), 0, 15, 24),     # eight rows
    ((24, 40, 40), 700, (4, 4, 4), 1, 15, 24),    # shared bricks
])
def test_large_boxes_keep_their_bits(oracle, size, rois, cells, ratio, low, high):
    """What may be left of boxes that were worked out in fp32: the result's own rounding, with weights and sums of 22 bits beside it (three roundings
    of 2^-22 and sums of a few hundred terms in fp32: below 1e-5 of the result)."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(sum(size) + rois + sum(cells))
    dims = (1, 128, *size)
    assert bricks_apply(dims, rois, cells, ratio)
    extent = torch.rand(rois, 3, generator=g) * (high - low) + low
    room = torch.tensor(size[::-1]) - extent
    at = torch.where(room > 0, torch.rand(rois, 3, generator=g) * room, torch.rand(rois, 3, generator=g) * 6 + 3 - extent)
    boxes = torch.cat([torch.zeros(rois, 1), at, at + extent], 1)
    x = torch.zeros(dims, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, ratio, 1)
    gy = torch.randn(out.shape, generator=g).half()
    want = torch.as_tensor(oracle.roi_align_backward(gy, boxes, dims, 1.0, ratio, True, 1, False)).double().reshape(dims)
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    own = (want.half().double() - want).norm()
    assert (got - want).norm() <= 1.01 * own + 1e-5 * want.norm()


@pytest.mark.parametrize("rois,cells,low,high", [
    (100, (7, 7, 7), 15, 24),
    (100, (4, 5, 4), 15, 24),
    (60, (7, 7, 7), 20, 38),
])
def test_large_boxes_keep_the_bits_of_small_gradients(oracle, rois, cells, low, high):
    """Gradients of 1e-5: the results are subnormal numbers, and what is left of the sums' bits may not show beside their rounding (a tenth of it at
    the most, half a hundredth of the error; less than half of that allowed)."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(rois + sum(cells) + high)
    dims = (1, 128, 24, 40, 40)
    assert bricks_apply(dims, rois, cells)
    extent = (torch.rand(rois, 3, generator=g) * (high - low) + low).minimum(torch.tensor([40., 40., 24.]))
    at = torch.rand(rois, 3, generator=g) * (torch.tensor([40., 40., 24.]) - extent)
    boxes = torch.cat([torch.zeros(rois, 1), at, at + extent], 1)
    x = torch.zeros(dims, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, 2, 1)
    gy = (torch.randn(out.shape, generator=g) * 1e-5).half()
    want = torch.as_tensor(oracle.roi_align_backward(gy, boxes, dims, 1.0, 2, True, 1, False)).double().reshape(dims)
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    own = (want.half().double() - want).norm()
    assert (got - want).norm() <= 1.002 * own


def test_long_boxes_of_large_gradients(oracle):
    """Boxes of all bits whose sums over rows go beyond fp16 (several cells per voxel on two axes, several voxels per cell on the third)."""
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(41)
    dims, rois, cells = (1, 128, 40, 24, 40), 12, (7, 7, 7)
    assert bricks_apply(dims, rois, cells)
    extent = torch.rand(rois, 3, generator=g) * torch.tensor([1.5, 1.5, 5.0]) + torch.tensor([1.5, 1.5, 33.0])
    at = torch.rand(rois, 3, generator=g) * (torch.tensor([40., 24., 40.]) - extent)
    boxes = torch.cat([torch.zeros(rois, 1), at, at + extent], 1)
    x = torch.zeros(dims, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, 2, 1)
    gy = (torch.randn(out.shape, generator=g) * 8000).half()
    want = torch.as_tensor(oracle.roi_align_backward(gy, boxes, dims, 1.0, 2, True, 1, False)).double().reshape(dims)
    assert 16376 < want.abs().max() < 65000
    got = torch.autograd.grad(out, x, gy.to(DEV))[0].cpu().double()
    own = (want.half().double() - want).norm()
    assert (got - want).norm() <= 1.01 * own + 1e-5 * want.norm()


@pytest.mark.parametrize("images,channels,size,rois", [
    (2, 128, (9, 17, 33), 480),      # eight share a brick, the most
    (4, 80, (40, 33, 8), 130),       # one brick along x: four share it
    (4, 80, (40, 33, 8), 800),       # eight
])
def test_shared_bricks(oracle, images, channels, size, rois):
    from medvision_amd.ops.roi_align_nd import roi_align_3d
    g = wl.gen(rois + channels)
    dims, cells = (images, channels, *size), (3, 4, 5)
    assert bricks_apply(dims, rois, cells)
    boxes = boxes_of(g, images, size, rois, 9)
    x = torch.zeros(dims, dtype=torch.float16, device=DEV, requires_grad=True)
    out = roi_align_3d(x, boxes.to(DEV), cells, 1.0, 2, 1)
    gy = torch.randn(out.shape, generator=g).half()
    want = oracle.roi_align_backward(gy, boxes, x.shape, 1.0, 2, True, 1, False).reshape(x.shape)
    assert_close(torch.autograd.grad(out, x, gy.to(DEV))[0], want, TOL, "gradient")
