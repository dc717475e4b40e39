"""Modulated deformable layers at the edges of the matrix-core kernels' tiles, ranges and chunks, forward and backward,
against the fp64 oracle."""
import pytest
import torch

from parity import BWD_TOL, FWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,size,stride,groups,dg", [
    (32, 32, (3, 3, 7), 1, 1, 1),         # fewer positions than a tile
    (32, 64, (5, 8, 16), 1, 1, 1),        # whole tiles
    (96, 160, (4, 9, 5), 2, 1, 1),        # three chunks, rows with a remainder, stride 2
    (64, 64, (6, 5, 7), 1, 2, 2),         # groups
    (48, 16, (5, 7, 9), 1, 1, 2),         # channel counts that are padded
    (64, 288, (23, 29), 1, 1, 1),         # images: a chunk of 64, two passes over the rows
    (128, 96, (37, 41), 2, 1, 2),         # images: two deformable groups of one chunk each
    (256, 64, (9, 140), 1, 1, 1),         # images: four chunks, long rows
])
def test_matrix_core_layers(oracle, dtype, cin, cout, size, stride, groups, dg):
    nd = len(size)
    if nd == 3:
        from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    else:
        from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(cin + cout + sum(size))
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, size, 3, dg, groups, dtype, stride, 1, 1)
    off = off * 1.5   # corners inside and beyond the tiles of the input's gradient
    leaves = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(*leaves, stride, 1, 1, groups, dg)
    assert_close(y, oracle.dcn3d_forward(x, off, mask, w, b, stride, 1, 1, groups, dg), FWD_TOL[dtype], "forward")
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    want = oracle.dcn3d_backward(x, off, mask, w, gy, True, stride, 1, 1, groups, dg)
    for t, v, name in zip(leaves, want, ("input", "offset", "mask", "weight", "bias")):
        assert_close(t.grad, v, BWD_TOL[dtype], name)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,size,stride,dilation", [
    (32, 256, (40, 72), 1, 1),        # images with more output channels than 128
    (32, 64, (44, 80), 2, 1),         # strided
    (32, 64, (48, 72), 1, 12),        # taps far apart
    (32, 64, (6, 20, 48), 2, 1),      # volumes, strided
    (32, 160, (5, 9, 48), 1, 1),
    (32, 160, (5, 9, 40), 1, 1),      # (the split is in the middle of a brick)
])
def test_small_gradients_beside_large_ones(oracle, dtype, cin, cout, size, stride, dilation):
    """The gradient of the input keeps fp32 sums in strided and wide layers: where the output's gradient is 2^-14 of what it
    is a few columns further on, in the same brick, the sums are as good as anywhere (rounding of the result: 2^-11 / 2^-8)."""
    if len(size) == 3:
        from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    else:
        from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(cin + cout + sum(size))
    x, off, mask, w, b = wl.dcn_inputs(g, 1, cin, cout, size, 3, 1, 1, dtype, stride, dilation, dilation, offset_std=0.0)
    off = (torch.rand(off.shape, generator=g) - 0.5).to(dtype)
    leaves = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(*leaves, stride, dilation, dilation, 1, 1)
    gy = torch.randn(y.shape, generator=g)
    split = y.shape[-1] // 2 + 1
    gy[..., :split] *= 2.0 ** -6
    gy[..., split:] *= 2.0 ** 8
    gy = gy.to(dtype)
    y.backward(gy.to(DEV))
    want = oracle.dcn3d_backward(x, off, mask, w, gy, True, stride, dilation, dilation, 1, 1)[0].reshape(x.shape)
    edge = split * stride - 2 - dilation       # columns that no position beyond the split reaches
    got, want = leaves[0].grad.cpu().double()[..., :edge], want[..., :edge]
    assert float(want.abs().max()) < 1.0       # nothing of the large ones
    error = float((got - want).norm() / want.norm())
    assert error < (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8), error


@pytest.mark.parametrize("cin,cout,size", [(32, 32, (5, 12, 21)), (64, 32, (24, 40))])
def test_offset_gradient_of_nearly_equal_corners(oracle, cin, cout, size):
    """Offset gradients are formed from differences of the corners, channel by channel: an input of 64 and 64 + one step of fp16
    loses nothing.  Weights and gradients are whole numbers, so that their sums with the differences are exact in fp32 and
    only the blend over the rows rounds (four operations, 2^-24 each); with one sum per corner, 1000 times as large, what cancels
    would show in the small results."""
    nd, delta, dtype = len(size), 1 / 16, torch.float16
    if nd == 3:
        from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    else:
        from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(cin + sum(size))
    taps = 3 ** nd
    x = (64 + delta * torch.randint(0, 2, (1, cin, *size), generator=g)).to(dtype)
    w = torch.randint(-128, 129, (cout, cin, *[3] * nd), generator=g).to(dtype)
    gy = torch.randint(-128, 129, (1, cout, *size), generator=g).to(dtype)
    off = ((torch.rand(1, nd * taps, *size, generator=g) - 0.5) * 1.5).to(dtype)
    mask, b = torch.ones(1, taps, *size, dtype=dtype), torch.zeros(cout, dtype=dtype)
    leaves = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(*leaves, 1, 1, 1, 1, 1)
    got = torch.autograd.grad(y, leaves[1], gy.to(DEV))[0]
    want = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, 1, 1)[1].reshape(off.shape)
    inside = (slice(None), slice(nd - 1, None, nd), *[slice(2, -2)] * nd)     # along w, away from the zeros outside
    got, want = got.cpu().double()[inside], want[inside]
    terms = torch.einsum("ock,oq->ckq", w.double().flatten(2), gy.double()[0].flatten(1)).abs().sum(0)   # sum over c of |gcol|
    largest = (terms.reshape(1, taps, *size) * delta)[(slice(None), slice(None), *inside[2:])]
    worst = float((((got - want).abs() - 2.0 ** -11 * want.abs()) / largest).max())
    assert worst <= 2.0 ** -22, worst


@pytest.mark.parametrize("dtype,batch,cin,cout,size,groups,dg", [
    (torch.float16, 1, 64, 144, (101, 103), 1, 1),      # 64 positions, rows of 256 with a remainder, a last tile of 35 positions
    (torch.bfloat16, 2, 128, 272, (73, 71), 1, 2),      # two passes over the rows, a unit of one line
    (torch.float16, 1, 80, 144, (103, 101), 1, 1),      # units of ten pieces: no whole lines
    (torch.float32, 1, 32, 144, (203, 202), 1, 1),
    (torch.float16, 1, 64, 32, (5, 7, 11), 1, 1),       # 16 positions
    (torch.float32, 2, 96, 160, (6, 9, 11), 1, 3),
    (torch.bfloat16, 2, 128, 96, (9, 33, 30), 2, 1),    # 32 positions, groups of 48 rows
])
def test_columns_of_whole_lines(oracle, dtype, batch, cin, cout, size, groups, dg):
    """Corners read by whole cache lines (units of 128 bytes and multiples) and by halves, tiles of 16, 32 and 64 positions."""
    if len(size) == 3:
        from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    else:
        from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(cin + cout + sum(size))
    x, off, mask, w, b = wl.dcn_inputs(g, batch, cin, cout, size, 3, dg, groups, dtype, 1, 1, 1)
    off = off * 1.5
    with torch.no_grad():
        y = modulated_deform_conv(*[t.to(DEV) for t in (x, off, mask, w, b)], 1, 1, 1, groups, dg)
    assert_close(y, oracle.dcn3d_forward(x, off, mask, w, b, 1, 1, 1, groups, dg), FWD_TOL[dtype], "forward")


@pytest.mark.parametrize("dtype,batch,cin,cout,size", [
    (torch.float16, 192, 32, 144, (4, 4)),      # few positions, many images: workgroups of fewer rows
    (torch.bfloat16, 96, 32, 272, (3, 4)),
    (torch.float16, 200, 16, 256, (3, 3)),
    (torch.float16, 200, 16, 256, (7, 7)),      # 64 positions, of which 49
    (torch.bfloat16, 300, 16, 144, (9, 9)),     # 32 positions: 64 would leave more than an eighth idle
])
def test_many_small_images(oracle, dtype, batch, cin, cout, size):
    from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(batch + cin + cout + sum(size))
    x, off, mask, w, b = wl.dcn_inputs(g, batch, cin, cout, size, 3, 1, 1, dtype, 1, 1, 1)
    with torch.no_grad():
        y = modulated_deform_conv(*[t.to(DEV) for t in (x, off, mask, w, b)], 1, 1, 1, 1, 1)
    assert_close(y, oracle.dcn3d_forward(x, off, mask, w, b, 1, 1, 1, 1, 1), FWD_TOL[dtype], "forward")
