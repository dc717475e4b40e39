"""Heads on images with plain boxes: the matrix-core kernels at the edges of their tiles and lists, forward and
backward, against the fp64 oracle."""
import pytest
import torch

from parity import BWD_TOL, FWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("size,channels,rois,cells,ratio,order,reach", [
    ((33, 47), 37, 9, (7, 7), 0, 1, 40),      # tiles and channels with remainders, boxes over the border
    ((16, 16), 8, 1, (8, 8), 2, 1, 16),       # one tile, whole cells
    ((40, 21), 5, 6, (14, 14), 2, 1, 30),     # the 16-cell kernels
    ((50, 64), 3, 40, (16, 9), 1, 0, 30),     # nearest taps, cells of both sizes
    ((20, 3), 4, 5, (5, 3), 2, 1, 12),        # rows shorter than a load
    ((9, 9), 2, 3, (1, 5), 0, 1, 9),          # a single row of cells
    ((300, 180), 4, 4, (7, 7), 0, 1, 290),    # more rows and columns than the forward lists hold
    ((24, 24), 16, 1100, (7, 7), 2, 1, 12),   # more rois than one look-through, several workgroups per tile
    ((260, 260), 64, 300, (7, 7), 2, 1, 60),  # features beyond an L2: rois ordered first
    ((12, 12), 3, 4, (3, 1), 2, 1, 9),        # too few cells for the matrix cores
])
def test_plane_heads(oracle, dtype, size, channels, rois, cells, ratio, order, reach):
    from medvision_amd.ops.roi_align_nd import roi_align_2d
    g = wl.gen(sum(size) + rois + channels)
    batch = 2
    feat = torch.randn(batch, channels, *size, generator=g).to(dtype)
    at = torch.rand(rois, 2, generator=g) * torch.tensor(size[::-1]) * 1.2 - 4.0
    extent = torch.rand(rois, 2, generator=g) * reach
    image = torch.randint(0, batch, (rois, 1), generator=g).float()
    boxes = torch.cat([image, at, at + extent], 1)
    x = feat.to(DEV).requires_grad_()
    out = roi_align_2d(x, boxes.to(DEV), cells, 0.5, ratio, order)
    assert_close(out, oracle.roi_align_forward(feat, boxes, cells, 0.5, ratio, True, order, False), FWD_TOL[dtype], "forward")
    gy = torch.randn(out.shape, generator=g).to(dtype)
    out.backward(gy.to(DEV))
    want = oracle.roi_align_backward(gy, boxes, feat.shape, 0.5, ratio, True, order, False)
    assert_close(x.grad, want, BWD_TOL[dtype], "backward")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("size,channels,rois,cells,ratio,order,reach", [
    ((48, 53), 37, 30, (7, 7), 0, 1, 30),     # 8-cell kernels, a group of channels with a remainder
    ((40, 44), 9, 24, (14, 11), 2, 1, 24),    # 16-cell kernels
    ((40, 44), 9, 24, (5, 3), 1, 0, 24),      # nearest taps
    ((24, 24), 16, 1100, (7, 7), 2, 1, 12),   # several workgroups per tile
])
def test_plane_heads_non_finite(oracle, dtype, size, channels, rois, cells, ratio, order, reach):
    """Infinite and NaN pixels and gradients reach what a sample's weight ties them to and nothing else."""
    from medvision_amd.ops.roi_align_nd import roi_align_2d
    g = wl.gen(sum(size) + rois + channels)
    feat = torch.randn(2, channels, *size, generator=g).to(dtype)
    extent = torch.rand(rois, 2, generator=g) * reach + 1.0
    at = torch.rand(rois, 2, generator=g) * (torch.tensor(size[::-1]) * 2.0 - extent)   # inside the image: no void samples
    boxes = torch.cat([torch.randint(0, 2, (rois, 1), generator=g).float(), at, at + extent], 1)
    centre, half = torch.tensor([size[1] // 2 + 0.3, size[0] // 2 + 0.2]), torch.tensor([cells[1], cells[0]]) / 2.0
    boxes[0] = torch.cat([torch.zeros(1), 2 * (centre - half), 2 * (centre + half)])   # samples every pixel around the first one
    bad = feat.clone()
    bad[0, 0, size[0] // 2, size[1] // 2] = float("inf")
    bad[1, channels - 1, size[0] // 3, size[1] - 1] = float("nan")    # the last column: its group is moved back into the row
    x = bad.to(DEV).requires_grad_()
    out = roi_align_2d(x, boxes.to(DEV), cells, 0.5, ratio, order)

    def compare(got, want, finite, tol, name):
        got, finite = got.detach().cpu().double(), finite.reshape(got.shape)
        assert not finite.all() and torch.equal(torch.isfinite(got), finite), name
        assert_close(torch.where(finite, got, 0.0), torch.where(finite, want.reshape(got.shape), 0.0), tol, name)

    def pooled(x):
        return oracle.roi_align_forward(x, boxes, cells, 0.5, ratio, True, order, False)

    # (the oracle multiplies nearest neighbours that are not picked by 0: the cells reached come from marks instead)
    marks = (~torch.isfinite(bad)).to(dtype)
    compare(out, pooled(torch.where(marks > 0, 0.0, bad)), pooled(marks) == 0, FWD_TOL[dtype], "forward")
    gy = torch.randn(out.shape, generator=g).to(dtype)
    gy[0, 0].view(-1)[0] = float("inf")
    gy[rois - 1, channels - 1].view(-1)[-1] = float("nan")
    out.backward(gy.to(DEV))

    def spread(t):
        return oracle.roi_align_backward(t, boxes, feat.shape, 0.5, ratio, True, order, False)

    marks = (~torch.isfinite(gy)).to(dtype)
    compare(x.grad, spread(torch.where(marks > 0, 0.0, gy)), spread(marks) == 0, BWD_TOL[dtype], "backward")


@pytest.mark.parametrize("dtype,exponents,normal", [(torch.float16, (-24, -15), -14), (torch.bfloat16, (-133, -126), -126)])
@pytest.mark.parametrize("cells", [(7, 7), (14, 14)])
def test_plane_heads_denormal_values(oracle, dtype, exponents, normal, cells):
    """16-bit pixels and gradients go to the matrix cores as they are: values below the type's normal ones keep their bits.  Results are
    off by half a unit in the last place (the smallest denormal's below 2^normal), and by 2^-16 of the terms' sum for weights whose
    sample lies next to a decision of the sampler."""
    from medvision_amd.ops.roi_align_nd import roi_align_2d
    g = wl.gen(sum(cells))
    rois, channels, size = 60, 34, (60, 70)
    at = torch.rand(rois, 2, generator=g) * torch.tensor(size[::-1]) * 0.9
    boxes = torch.cat([torch.randint(0, 2, (rois, 1), generator=g).float(), at, at + torch.rand(rois, 2, generator=g) * 30 + 1], 1)

    def values(*shape):
        e = exponents[0] + (exponents[1] - exponents[0]) * torch.rand(*shape, generator=g, dtype=torch.float64)
        return (torch.exp2(e) * (torch.randint(0, 2, shape, generator=g) * 2 - 1)).to(dtype)

    feat = values(2, channels, *size)
    x = feat.to(DEV).requires_grad_()
    out = roi_align_2d(x, boxes.to(DEV), cells, 1.0, 2, 1)
    gy = values(*out.shape)
    out.backward(gy.to(DEV))
    half = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8

    def check(got, of, name):
        want, terms = of(False), of(True)
        error = (got.detach().cpu().double() - want.reshape(got.shape)).abs().reshape(-1)
        bound = half * want.abs().clamp(min=2.0 ** normal).reshape(-1) + 2.0 ** -16 * terms.reshape(-1)
        assert float(want.abs().max()) > 0 and float((error / bound).max()) <= 1.0, name

    check(out, lambda a: oracle.roi_align_forward(feat.abs() if a else feat, boxes, cells, 1.0, 2, True, 1, False), "forward")
    check(x.grad, lambda a: oracle.roi_align_backward(gy.abs() if a else gy, boxes, feat.shape, 1.0, 2, True, 1, False), "backward")
