"""The input's gradient of deformable layers at the edges of the LDS tiles that sum it, against the fp64 oracle: every brick and tile,
counts of output channels around the slices that a wavefront keeps, samples on the tiles' and the input's borders."""
import pytest
import torch

from parity import BWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _gradient(oracle, dtype, batch, cin, cout, size, stride, groups, dg, offsets, seed, dilation=1):
    if len(size) == 3:
        from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    else:
        from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(seed)
    x, off, mask, w, b = wl.dcn_inputs(g, batch, cin, cout, size, 3, dg, groups, dtype, stride, dilation, dilation)
    off = offsets(off, g).to(dtype)
    leaves = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(*leaves, stride, dilation, dilation, groups, dg)
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    want = oracle.dcn3d_backward(x, off, mask, w, gy, True, stride, dilation, dilation, groups, dg)
    assert_close(leaves[0].grad, want[0], BWD_TOL[dtype], "input")
    assert_close(leaves[4].grad, want[4], BWD_TOL[dtype], "bias")   # (from 1024 rows of grad_output on several per workgroup)


def _borders(off, g):
    """Whole and half voxels up to beyond the tiles, a few samples exactly one voxel outside, a few very far away."""
    whole = torch.randint(-9, 10, off.shape, generator=g).float()
    pick = torch.rand(off.shape, generator=g)
    return torch.where(pick < 0.5, whole, torch.where(pick < 0.98, whole + 0.5, torch.where(pick < 0.99, -1.0, 3e4)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,size,stride,groups,dg", [
    (32, 32, (5, 9, 17), 1, 1, 1),        # volumes: a brick and a remainder along every axis
    (64, 96, (4, 8, 9), 1, 1, 2),         # three slices of grad_output, two deformable groups
    (32, 160, (6, 9, 10), 2, 1, 1),       # strided, more slices than four
    (48, 16, (9, 5, 25), 1, 1, 1),        # channel counts that are padded
    (32, 160, (9, 5, 25), 1, 1, 1),       # wide: 16-bit ones in bricks of 4 x 4 x 8 and a remainder along every axis
    (16, 64, (9, 13, 17), 2, 1, 1),       # of 2 x 4 x 4, strided
    (32, 64, (33, 35), 1, 1, 1),          # images: a brick of 32 x 32 (few workgroups of 16-bit ones: of 8 x 8) and a remainder
    (512, 32, (40, 37), 1, 1, 1),         # of 32 x 32 with 32-bit sums too
    (512, 64, (33, 67), 2, 1, 1),         # of 8 x 16, strided (fp32: of 16 x 16)
    (64, 288, (17, 33), 1, 1, 1),         # more slices than eight
    (64, 64, (31, 67), 2, 2, 2),          # strided, groups
    (512, 32, (20, 20), 1, 1, 1),         # many channel blocks
])
def test_samples_on_borders(oracle, dtype, cin, cout, size, stride, groups, dg):
    _gradient(oracle, dtype, 2, cin, cout, size, stride, groups, dg, _borders, cin + cout + sum(size))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,size,dilation,groups,dg", [
    (32, 32, (33, 35), 10, 1, 1),         # a slice or two of grad_output, bricks of 16 x 16 and a remainder
    (64, 96, (20, 50), 12, 1, 2),         # three (fp32: six), two deformable groups
    (64, 288, (17, 40), 13, 1, 1),        # more slices than eight
    (512, 160, (37, 21), 12, 1, 1),       # many channel blocks
    (64, 64, (48, 30), 9, 2, 1),          # groups
])
def test_images_with_taps_far_apart(oracle, dtype, cin, cout, size, dilation, groups, dg):
    _gradient(oracle, dtype, 2, cin, cout, size, 1, groups, dg, _borders, cin + cout + sum(size), dilation)


@pytest.mark.parametrize("dtype,batch,cout,size", [
    (torch.float16, 64, 160, (5, 7)),     # 2048 workgroups, bricks of which most groups do not exist
    (torch.bfloat16, 16, 160, (17, 33)),
    (torch.float32, 64, 96, (5, 7)),
    (torch.float16, 63, 160, (5, 7)),     # one image fewer: one block of channels per workgroup
])
def test_two_channel_blocks_per_workgroup(oracle, dtype, batch, cout, size):
    """Wide 16-bit images of 2048 and more workgroups of sixteen channels sum 32 channels in two turns (fp32 ones have workgroups of eight
    channels and one turn)."""
    _gradient(oracle, dtype, batch, 512, cout, size, 1, 1, 1, lambda off, g: off, batch + sum(size))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kernel,stride,dilation", [
    ((3, 3, 3), (2, 1, 1), (1, 1, 1)),
    ((3, 3, 3), (1, 1, 1), (3, 1, 1)),
    ((7, 3, 3), (1, 1, 1), (1, 1, 1)),
])
def test_small_gradients_beside_large_ones_along_one_axis(oracle, dtype, kernel, stride, dilation):
    """Layers that are strided, dilated or deep along one axis alone sum the input's gradient in 64 bits too: where the output's
    gradient is 2^-14 of what it is in the same brick, the sums are as good as anywhere (rounding of the result: 2^-11 / 2^-8)."""
    from medvision_amd import _C
    cin, cout, size = 32, 64, (9, 8, 40)
    g = wl.gen(sum(kernel) + sum(stride) + sum(dilation))
    pad = tuple((k - 1) * d // 2 for k, d in zip(kernel, dilation))
    out = [(n + 2 * p - (d * (k - 1) + 1)) // s + 1 for n, p, d, k, s in zip(size, pad, dilation, kernel, stride)]
    taps = kernel[0] * kernel[1] * kernel[2]
    x = torch.randn(1, cin, *size, generator=g).to(dtype)
    w = (torch.randn(cout, cin, *kernel, generator=g) / (cin * taps) ** 0.5).to(dtype)
    off = (torch.rand(1, 3 * taps, *out, generator=g) - 0.5).to(dtype)
    mask = torch.rand(1, taps, *out, generator=g).to(dtype)
    gy = torch.randn(1, cout, *out, generator=g)
    split = 20      # in the middle of a brick of eight columns
    gy[..., :split] *= 2.0 ** -6
    gy[..., split:] *= 2.0 ** 8
    gy = gy.to(dtype)
    ins = [t.to(DEV) for t in (x, w, torch.zeros(cout, dtype=dtype), off, mask)]
    sums = [torch.zeros_like(t) for t in ins]
    _C.modulated_deform_conv_3d_backward(ins[0], ins[1], ins[2], None, ins[3], ins[4], None, sums[0], sums[1], sums[2], sums[3], sums[4],
                                         gy.to(DEV), *kernel, *stride, *pad, *dilation, 1, 1, True)
    want = oracle.dcn3d_backward(x, off, mask, w, gy, True, stride, pad, dilation, 1, 1)[0].reshape(x.shape)
    edge = split - 3      # columns that no position beyond the split reaches
    got, want = sums[0].cpu().double()[..., :edge], want[..., :edge]
    assert float(want.abs().max()) < 1.0       # nothing of the large ones
    error = float((got - want).norm() / want.norm())
    assert error < (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8), error


@pytest.mark.parametrize("cin,cout,size,stride", [(64, 64, (24, 24), 1), (32, 288, (31, 20), 1), (64, 32, (32, 30), 2)])
def test_fp32_images_of_one_brick_are_rounded_once(oracle, cin, cout, size, stride):
    """Every addition of a tile's sums to the fp32 gradient rounds, so that fp32 images have bricks as large as the tiles hold while
    no brick fills the chip.  Whole weights and gradients and offsets in eighths: the terms and their 64-bit sums are exact, and an
    image of one brick is off by one rounding, 2^-24 of each value."""
    from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(cin + cout)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, size, 3, 1, 1, torch.float32, stride, 1, 1)
    off = torch.randint(-24, 25, off.shape, generator=g) / 8.0
    w = torch.randint(-127, 128, w.shape, generator=g).float()
    leaves = [t.to(DEV).requires_grad_(True) for t in (x, off, torch.ones_like(mask), w, b)]
    y = modulated_deform_conv(*leaves, stride, 1, 1, 1, 1)
    gy = torch.randint(-2047, 2048, y.shape, generator=g).float()
    y.backward(gy.to(DEV))
    want = oracle.dcn3d_backward(x, off, torch.ones_like(mask), w, gy, True, stride, 1, 1, 1, 1)[0].reshape(x.shape)
    error = (leaves[0].grad.cpu().double() - want).abs()
    worst = float((error / want.abs().clamp(min=1e-9)).max())
    assert worst <= 2.0 ** -24, worst * 2.0 ** 24


@pytest.mark.parametrize("size", [(120, 127), (101, 151)])      # rows at whole pieces of 16 bytes, rows at any element
@pytest.mark.parametrize("batch,cout", [(8, 128), (2, 64)])     # 1024 rows, a wavefront each; slabs of rows
def test_fp32_bias_of_long_rows(batch, cout, size):
    """The bias gradient of fp32 layers is a sum in fp32, in chains of at most a 512th of a row.  A chain of n normal values rounds n times
    at 0.4 * 2^-24 of the sum so far (rms), sqrt(n / 2) * 0.4 * 2^-24 of its result: 1e-7 of the sum of all chains for n = 30; the tree and
    the atomics above add as much.  (Chains of a 64th of a row: 3e-7.)"""
    from medvision_amd import _C
    g = torch.Generator(DEV).manual_seed(sum(size))
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    ins = x, w, b, off, mask = rand(batch, 32, *size), rand(cout, 32, 1, 1), rand(cout), rand(batch, 2, *size), rand(batch, 1, *size)
    gy, sums = rand(batch, cout, *size), [torch.zeros_like(t) for t in ins]
    gx, gw, gb, goff, gmask = sums
    _C.modulated_deform_conv_2d_backward(x, w, b, None, off, mask, None, gx, gw, gb, goff, gmask, gy, 1, 1, 1, 1, 0, 0, 1, 1, 1, 1, True)
    want = gy.double().sum((0, 2, 3))
    error = float((gb.double() - want).norm() / want.norm())
    assert error < 2e-7, error
