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
