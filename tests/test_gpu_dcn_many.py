"""Deformable layers of very many workgroups: more than a grid of one dimension holds (2^32 threads)."""
import pytest
import torch

from parity import BWD_TOL, assert_close

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("taps", [1, 3])
def test_many_images_of_one_pixel(taps):
    """65535 images of one pixel and 1056 channels: 4.3 million workgroups of 1024 threads sum the gradient of the input, and with 3 x 3 taps
    19 million of 256 threads form the others.  The pixel takes max(0, 1 - |p|) of every sample along each axis, so that all gradients are
    products of matrices, here in fp32."""
    from medvision_amd import _C
    batch, cin, cout, dtype = 65535, 1056, 32, torch.float16
    g = torch.Generator(DEV).manual_seed(taps)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    x, w, gy = rand(batch, cin, 1, 1), rand(cout, cin, taps, taps) / 8, rand(batch, cout, 1, 1)
    off, mask = rand(batch, 2 * taps * taps, 1, 1) / 2, torch.rand(batch, taps * taps, 1, 1, generator=g, device=DEV).to(dtype)
    bias = torch.zeros(cout, dtype=dtype, device=DEV)
    gx, gw, gb, goff, gmask = (torch.zeros_like(t) for t in (x, w, bias, off, mask))
    _C.modulated_deform_conv_2d_backward(x, w, bias, None, off, mask, None, gx, gw, gb, goff, gmask, gy, taps, taps, 1, 1,
                                         taps // 2, taps // 2, 1, 1, 1, 1, True)
    want_x, x, gy = torch.zeros(batch, cin, device=DEV), x.flatten(1).float(), gy.flatten(1).float()
    for k in range(taps * taps):
        at = off[:, 2 * k:2 * k + 2, 0, 0].float() + torch.tensor([k // taps - taps // 2, k % taps - taps // 2], device=DEV)
        share = (1 - at.abs()).clamp(min=0).prod(1, keepdim=True)
        column = gy @ w[:, :, k // taps, k % taps].float()
        weighted = mask[:, k, 0].float() * share
        want_x += weighted * column
        assert_close(gw[:, :, k // taps, k % taps], gy.t() @ (weighted * x), BWD_TOL[dtype], "weight")
        assert_close(gmask[:, k, 0], share * (x * column).sum(1, keepdim=True), BWD_TOL[dtype], "mask")
    assert_close(gx.flatten(1), want_x, BWD_TOL[dtype], "input")
