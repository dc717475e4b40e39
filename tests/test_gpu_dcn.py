"""GPU parity of the 3-D deformable convolutions (DCNv1 / DCNv2) and the displacement-field warp
against the fp64 oracle, through the drop-in modules and the `_C` shim."""
import pytest
import torch
import torch.nn.functional as F

from parity import BWD_TOL, FWD_TOL, assert_close
import workloads as wl

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    import medvision_amd.ops as ops_
    from medvision_amd import _lib
    _lib.load()
    return ops_


def _to(dev, *ts):
    return [None if t is None else t.to(dev) for t in ts]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("modulated,groups,dg,stride,pad,dil", [
    (True, 1, 1, 1, 1, 1), (True, 2, 2, 2, 1, 1), (False, 1, 2, 1, 2, 2), (False, 2, 1, 1, 0, 1)])
def test_functions_vs_oracle(ops, oracle, dtype, modulated, groups, dg, stride, pad, dil):
    from medvision_amd.ops.deform_conv_3d import deform_conv
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(40 + groups + 2 * dg + stride)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, 4, 6, (6, 7, 8), 3, dg, groups, dtype, stride, pad, dil,
                                       modulated)
    xs, offs, ms, ws, bs = [None if t is None else t.to(DEV).requires_grad_(True)
                            for t in (x, off, mask, w, b)]
    if modulated:
        y = modulated_deform_conv(xs, offs, ms, ws, bs, stride, pad, dil, groups, dg)
    else:
        y = deform_conv(xs, offs, ws, bs, stride, pad, dil, groups, dg, 64)
    want = oracle.dcn3d_forward(x, off, mask, w, b, stride, pad, dil, groups, dg)
    assert y.dtype == dtype
    assert_close(y, want, FWD_TOL[dtype], "forward")
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, stride, pad, dil, groups, dg)
    tol = BWD_TOL[dtype]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ws.grad, gw, tol, "grad weight")
    assert_close(bs.grad, gb, tol, "grad bias")
    if modulated:
        assert_close(ms.grad, gm, tol, "grad mask")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_config4_reduced_vs_oracle(ops, oracle, dtype):
    """Benchmark configuration 4 channel / kernel geometry (Cin 32, Cout 64, 3^3, pad 1, dg 1,
    offsets N(0,2), sigmoid mask) on a 12x12x16 volume so the CPU oracle finishes in seconds."""
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(3)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, 32, 64, (12, 12, 16), 3, 1, 1, dtype)
    xs, offs, ms, ws, bs = _to(DEV, x, off, mask, w, b)
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, 1, 1)
    want = oracle.dcn3d_forward(x, off, mask, w, b, 1, 1, 1, 1, 1)
    assert_close(y, want, FWD_TOL[dtype], "config 4 forward")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("modulated,groups,dg,stride,pad,dil,cin,cout", [
    (True, 2, 2, 1, 1, 1, 64, 128), (False, 1, 2, 2, 1, 2, 32, 32), (True, 1, 1, 1, 0, 1, 16, 160)])
def test_matrix_core_path_vs_oracle(ops, oracle, dtype, modulated, groups, dg, stride, pad, dil, cin, cout):
    """Shapes that take the MFMA forward (channels per group % 16 == 0, outputs per group % 32 == 0)
    with groups, deformable groups, stride, dilation and a ragged last position tile."""
    from medvision_amd.ops.deform_conv_3d import deform_conv
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(60 + groups + dg)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, (7, 9, 11), 3, dg, groups, dtype, stride, pad, dil,
                                       modulated)
    xs, offs, ms, ws, bs = _to(DEV, x, off, mask, w, b)
    if modulated:
        y = modulated_deform_conv(xs, offs, ms, ws, bs, stride, pad, dil, groups, dg)
    else:
        y = deform_conv(xs, offs, ws, bs, stride, pad, dil, groups, dg, 64)
    want = oracle.dcn3d_forward(x, off, mask, w, b, stride, pad, dil, groups, dg)
    assert_close(y, want, FWD_TOL[dtype], "mfma forward")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("modulated,groups,dg,stride,pad,dil,cin,cout,size", [
    (True, 1, 1, 1, 1, 1, 32, 64, (12, 12, 16)),    # config-4 geometry, Q % 8 == 0
    (True, 2, 2, 1, 1, 1, 64, 128, (7, 9, 11)),     # groups, deformable groups, ragged tiles, Q odd
    (False, 1, 2, 2, 1, 2, 64, 32, (9, 10, 12)),    # DCNv1, stride 2, dilation 2, two chunks per group
    (True, 1, 1, 1, 0, 1, 32, 96, (6, 7, 9)),       # no padding, three 32-row output blocks
    (False, 1, 1, 1, 1, 1, 160, 192, (5, 6, 7))])   # more than 128 channels in and out
def test_matrix_core_backward_vs_oracle(ops, oracle, dtype, modulated, groups, dg, stride, pad, dil,
                                        cin, cout, size):
    """Shapes that take the MFMA backward (channels per group / per deformable group % 32 == 0,
    outputs per group % 32 == 0): all five gradients against the fp64 oracle."""
    from medvision_amd.ops.deform_conv_3d import deform_conv
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(80 + groups + dg + cout)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, size, 3, dg, groups, dtype, stride, pad, dil,
                                       modulated)
    xs, offs, ms, ws, bs = [None if t is None else t.to(DEV).requires_grad_(True)
                            for t in (x, off, mask, w, b)]
    if modulated:
        y = modulated_deform_conv(xs, offs, ms, ws, bs, stride, pad, dil, groups, dg)
    else:
        y = deform_conv(xs, offs, ws, bs, stride, pad, dil, groups, dg, 64)
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, stride, pad, dil, groups, dg)
    tol = BWD_TOL[dtype]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ws.grad, gw, tol, "grad weight")
    assert_close(bs.grad, gb, tol, "grad bias")
    if modulated:
        assert_close(ms.grad, gm, tol, "grad mask")


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("size,offset_std,gy_scale", [
    ((12, 16, 16), 0.0, 1.0),       # every corner inside its brick's LDS tile
    ((12, 16, 16), 0.7, 1.0),       # offsets within the tile's margin
    ((12, 16, 16), 8.0, 1.0),       # most corners leave the tile: global atomics of the data kernel
    ((3, 5, 7), 2.0, 1.0),          # volume smaller than a brick
    ((9, 17, 10), 2.0, 3.0e4),      # ragged bricks; large and small gradients: the fixed-point scale
    ((9, 17, 10), 2.0, 1.0e-4)])    # of the LDS sums follows max |grad_output|
def test_input_gradient_through_lds_tiles(ops, oracle, dtype, size, offset_std, gy_scale):
    """Unit-stride 3^3 layers sum the input gradient of corners near their position in 64-bit
    fixed-point LDS tiles (the rest goes through global atomics): all gradients against the oracle
    for offsets from zero to far beyond the tile and for gradients of very different magnitude."""
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    if dtype == torch.float16 and gy_scale > 1e3:
        gy_scale = 200.0    # keep fp16 gradients finite
    g = wl.gen(400 + int(offset_std * 10) + size[0])
    x, off, mask, w, b = wl.dcn_inputs(g, 2, 32, 64, size, 3, 1, 1, dtype, 1, 1, 1, True, offset_std)
    xs, offs, ms, ws, bs = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, 1, 1)
    gy = (torch.randn(y.shape, generator=g) * gy_scale).to(dtype)
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, 1, 1)
    tol = BWD_TOL[dtype]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ms.grad, gm, tol, "grad mask")
    assert_close(ws.grad, gw, tol, "grad weight")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nd,cout,groups", [(3, 160, 1), (3, 512, 2), (2, 288, 1)])
def test_gradients_of_wide_layers(ops, oracle, dtype, nd, cout, groups):
    """More than 128 output channels per group (FPN layers): beyond what the scatter kernel keeps of
    grad_output in registers, so every corner of the input gradient goes through the data kernel."""
    g = wl.gen(470 + cout)
    if nd == 3:
        from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
        size = (5, 9, 12)
    else:
        from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
        size = (37, 40)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, 32 * groups, cout, size, 3, 1, groups, dtype, 1, 1, 1, True, 1.5)
    xs, offs, ms, ws, bs = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, groups, 1)
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    # (4-D tensors give the 2-D layer)
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, groups, 1)
    tol = BWD_TOL[dtype]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ms.grad, gm, tol, "grad mask")
    assert_close(ws.grad, gw, tol, "grad weight")


def test_input_gradient_through_lds_tiles_5x5x5(ops, oracle):
    """125 taps: 32 000 terms per tile voxel, the fixed-point scale leaves room for them."""
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(440)
    x, off, mask, w, b = wl.dcn_inputs(g, 1, 32, 32, (6, 9, 10), 5, 1, 1, torch.float32, 1, 2, 1, True, 1.0)
    xs, offs, ms, ws, bs = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 2, 1, 1, 1)
    gy = torch.randn(y.shape, generator=g)
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 2, 1, 1, 1)
    tol = BWD_TOL[torch.float32]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ms.grad, gm, tol, "grad mask")
    assert_close(ws.grad, gw, tol, "grad weight")


@pytest.mark.parametrize("budget,channels,size", [
    (0, 32, (7, 9, 11)),          # a single chunk of channels: no partial sums
    (0, 96, (7, 9, 11)),          # a tap at a time
    (140000, 96, (7, 9, 11)),     # two taps at a time, one at the end
    (0, 192, (70, 61)),           # 4096 positions of a tap at a time, and the rest
])
def test_weight_gradient_without_column_buffer(ops, oracle, budget, channels, size):
    """Layers whose partial sums (the shares of several chunks of channels in the offset and mask gradients) exceed the limit
    run in pieces of fewer taps or positions."""
    import importlib
    from medvision_amd import _C
    layer = importlib.import_module(f"medvision_amd.ops.modulated_deform_conv_{len(size)}d")
    old = _C.set_dcn_column_budget(budget)
    try:
        _weight_gradient_without_column_buffer(oracle, layer.modulated_deform_conv, channels, size)
    finally:
        _C.set_dcn_column_budget(old)


def _weight_gradient_without_column_buffer(oracle, modulated_deform_conv, channels, size):
    g = wl.gen(450)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, channels, 64, size, 3, 1, 1, torch.float16, 1, 1, 1, True, 2.0)
    xs, offs, ms, ws, bs = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, 1, 1)
    gy = torch.randn(y.shape, generator=g).half()
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, 1, 1)
    tol = BWD_TOL[torch.float16]
    assert_close(ws.grad, gw, tol, "grad weight")
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")


def test_input_gradient_with_non_finite_values(ops, oracle):
    """An infinity in grad_output makes the bound of the fixed-point sums non-finite: every corner
    then goes through the fp32 atomics, and NaN / infinity reach exactly the voxels the oracle's do."""
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(431)
    x, off, mask, w, b = wl.dcn_inputs(g, 1, 32, 32, (6, 8, 8), 3, 1, 1, torch.float32, 1, 1, 1, True, 1.0)
    xs, offs, ms, ws, bs = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, 1, 1)
    gy = torch.randn(y.shape, generator=g)
    gy[0, 3, 2, 4, 5] = float("inf")
    y.backward(gy.to(DEV))
    gx = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, 1, 1)[0]
    got = xs.grad.cpu()
    assert torch.equal(torch.isfinite(got), torch.isfinite(gx))
    fin = torch.isfinite(gx)
    assert_close(got[fin], gx[fin], BWD_TOL[torch.float32], "finite part of grad input")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_config4_full_size_properties(ops, dtype):
    """Full config-4 shape [2,32,48^3] -> Cout 64: zero offsets and unit mask reduce DCN to a plain
    convolution (checked against torch's conv3d in fp64 on the stored values), and the op is linear
    in the mask."""
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(5)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, 32, 64, (48, 48, 48), 3, 1, 1, dtype)
    xs, offs, ms, ws, bs = _to(DEV, x, off, mask, w, b)
    y0 = modulated_deform_conv(xs, torch.zeros_like(offs), torch.ones_like(ms), ws, bs, 1, 1, 1, 1, 1)
    ref = F.conv3d(xs.double(), ws.double(), bs.double(), 1, 1)
    assert_close(y0, ref, FWD_TOL[dtype], "zero-offset == conv3d")
    y1 = modulated_deform_conv(xs, offs, ms, ws, None, 1, 1, 1, 1, 1)
    y2 = modulated_deform_conv(xs, offs, ms * 0.5, ws, None, 1, 1, 1, 1, 1)
    assert_close(y2.float() * 2, y1.float(), 2 * FWD_TOL[dtype], "mask linearity")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_config4_full_size_backward_properties(ops, dtype):
    """The backward pass at the full config-4 size [2,32,48^3] -> 64 channels, where the CPU oracle
    would take minutes.  (1) Zero offsets and a unit mask make the layer a plain convolution: the
    gradients of input, weight and bias must equal torch's conv3d autograd in fp32.  (2) At the
    configuration's own offsets (sigma = 2 voxels) and mask the output is linear in the input, in
    the weight and in the mask, so <gy, y - bias> = <gx, x> = <gw, w> = <gmask, mask>; the offset
    gradient is checked through a central difference along a random direction (the trilinear form
    is piecewise linear in the offsets)."""
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    g = wl.gen(6)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, 32, 64, (48, 48, 48), 3, 1, 1, dtype)
    gy = torch.randn(2, 64, 48, 48, 48, generator=g).to(dtype)
    tol = {torch.float32: 1e-4, torch.float16: 4e-3, torch.bfloat16: 1.6e-2}[dtype]

    # (1) plain convolution
    xs, ws, bs = [t.to(DEV).requires_grad_(True) for t in (x, w, b)]
    offs = torch.zeros_like(off, device=DEV)
    ms = torch.ones_like(mask, device=DEV)
    y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, 1, 1)
    y.backward(gy.to(DEV))
    xr, wr, br = [t.to(DEV).float().requires_grad_(True) for t in (x, w, b)]
    F.conv3d(xr, wr, br, 1, 1).backward(gy.to(DEV).float())
    assert_close(xs.grad, xr.grad, tol, "grad input == conv3d")
    assert_close(ws.grad, wr.grad, tol, "grad weight == conv3d")
    assert_close(bs.grad, br.grad, tol, "grad bias == conv3d")
    del xr, wr, br, y

    # (2) adjoint identities at the real offsets
    xs, offs, ms, ws = [t.to(DEV).requires_grad_(True) for t in (x, off, mask, w)]
    y = modulated_deform_conv(xs, offs, ms, ws, None, 1, 1, 1, 1, 1)
    gyd = gy.to(DEV)
    y.backward(gyd)
    dot = lambda a, c: float((a.double() * c.double()).sum())
    lhs = dot(gyd, y)
    scale = float(gyd.double().norm() * y.double().norm())
    for name, grad, val in (("input", xs.grad, xs), ("weight", ws.grad, ws), ("mask", ms.grad, ms)):
        assert abs(dot(grad, val) - lhs) <= tol * scale, (name, dot(grad, val), lhs, scale)
    assert torch.isfinite(offs.grad).all()
    if dtype == torch.float32:   # a directional derivative needs the resolution of fp32 outputs
        # direction along the gradient's signs: the derivative is a sum of positive terms
        d = torch.randn(off.shape, generator=g).abs().to(DEV) * offs.grad.sign()
        eps = 1e-3
        with torch.no_grad():
            yp = modulated_deform_conv(xs, offs + eps * d, ms, ws, None, 1, 1, 1, 1, 1)
            ym = modulated_deform_conv(xs, offs - eps * d, ms, ws, None, 1, 1, 1, 1, 1)
        fd = dot(gyd, yp - ym) / (2 * eps)
        an = dot(offs.grad, d)
        # samples that cross a voxel boundary within +-eps (under 1 % of them) see a kink
        assert an > 0 and abs(fd - an) <= 3e-2 * an, (fd, an)


def test_modules_state_dict_and_autocast_training(ops):
    """Mirrors the reference's smoke script (test/ops_test_dcn.py:41-65): Adam steps under autocast
    with a GradScaler on a 1x3x5^3 input; here the loss must also go down."""
    torch.manual_seed(0)
    x = torch.rand(1, 3, 5, 5, 5, device=DEV)
    target = torch.ones(1, 7, 5, 5, 5, device=DEV)
    for cls, keys in ((ops.ModulatedDeformConv3dPack, {"weight", "bias", "conv_offset_mask.weight", "conv_offset_mask.bias"}),
                      (ops.DeformConv3dPack, {"weight", "bias", "conv_offset.weight", "conv_offset.bias"})):
        dcn = cls(in_channels=3, out_channels=7, kernel_size=3, stride=1, padding=1).to(DEV)
        assert set(dcn.state_dict().keys()) == keys
        opt = torch.optim.Adam(dcn.parameters(), lr=0.01)
        scaler = torch.amp.GradScaler("cuda")
        losses = []
        for _ in range(20):
            with torch.autocast("cuda", dtype=torch.float16):
                out = dcn(x)
                loss = F.binary_cross_entropy_with_logits(out.float(), target)
            opt.zero_grad()
            scaler.scale(loss).backward()
            scaler.step(opt)
            scaler.update()
            losses.append(float(loss))
        assert out.shape == (1, 7, 5, 5, 5)
        assert losses[-1] < losses[0]
    # zero-initialised offset branch: the pack equals a plain convolution at initialisation
    dcn = ops.ModulatedDeformConv3dPack(3, 7, 3, stride=1, padding=1).to(DEV)
    want = 0.5 * F.conv3d(x, dcn.weight, None, 1, 1) + dcn.bias.view(1, -1, 1, 1, 1)  # sigmoid(0) = .5
    assert_close(dcn(x), want, 1e-5, "pack at init")


def test_dcn_errors(ops):
    from medvision_amd import _C
    x = torch.randn(2, 4, 5, 5, 5, device=DEV)
    w = torch.randn(6, 4, 3, 3, 3, device=DEV)
    off = torch.zeros(2, 81, 5, 5, 5, device=DEV)
    b = torch.zeros(6, device=DEV)
    args = (3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1)
    with pytest.raises(RuntimeError, match="contiguous"):
        _C.deform_conv_3d_forward(x.transpose(3, 4), w, b, off, *args, 64)
    with pytest.raises(RuntimeError, match="kernel channels wont match"):
        _C.deform_conv_3d_forward(x, w[:, :3].contiguous(), b, off, *args, 64)
    with pytest.raises(RuntimeError, match="kernel shape wont match"):
        _C.deform_conv_3d_forward(x, w, b, off, 3, 3, 2, *args[3:], 64)
    with pytest.raises(RuntimeError, match="must divide im2col_step"):
        _C.deform_conv_3d_forward(x.repeat(2, 1, 1, 1, 1)[:3].contiguous(), w, b,
                                  off.repeat(2, 1, 1, 1, 1)[:3].contiguous(), *args, 2)
    with pytest.raises(RuntimeError, match="Not implemented on the CPU"):
        _C.deform_conv_3d_forward(x.cpu(), w.cpu(), b.cpu(), off.cpu(), *args, 64)
    with pytest.raises(RuntimeError, match="offset has shape"):
        _C.deform_conv_3d_forward(x, w, b, off[:, :80].contiguous(), *args, 64)
    # a tensor left on the host must raise on the host, not fault on the GPU
    with pytest.raises(RuntimeError, match="weight is on cpu"):
        _C.deform_conv_3d_forward(x, w.cpu(), b, off, *args, 64)
    with pytest.raises(RuntimeError, match="bias is on cpu"):
        _C.deform_conv_3d_forward(x, w, b.cpu(), off, *args, 64)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("modulated,groups,dg,stride,pad,dil,cin,cout,size", [
    (True, 1, 1, 1, 1, 1, 4, 6, (9, 11)),           # general kernels
    (False, 2, 2, 2, 1, 2, 4, 6, (10, 13)),
    (True, 1, 1, 1, 1, 1, 64, 64, (20, 24)),        # matrix-core forward and backward (16-bit, fp32)
    (False, 2, 1, 1, 0, 1, 64, 64, (13, 17)),
    (True, 1, 2, 2, 2, 2, 32, 96, (17, 19)),
    (True, 1, 1, 1, 1, 1, 256, 256, (10, 12))])     # FPN-sized layer: two channel chunks, two output passes
def test_2d_layers_vs_oracle(ops, oracle, dtype, modulated, groups, dg, stride, pad, dil, cin, cout, size):
    """The 2-D layers (offset channels 2k = rows, 2k+1 = columns) forward and all gradients."""
    from medvision_amd.ops.deform_conv_2d import deform_conv
    from medvision_amd.ops.modulated_deform_conv_2d import modulated_deform_conv
    g = wl.gen(120 + groups + dg + cout)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, size, 3, dg, groups, dtype, stride, pad, dil,
                                       modulated)
    xs, offs, ms, ws, bs = [None if t is None else t.to(DEV).requires_grad_(True)
                            for t in (x, off, mask, w, b)]
    if modulated:
        y = modulated_deform_conv(xs, offs, ms, ws, bs, stride, pad, dil, groups, dg)
    else:
        y = deform_conv(xs, offs, ws, bs, stride, pad, dil, groups, dg, 64)
    want = oracle.dcn2d_forward(x, off, mask, w, b, stride, pad, dil, groups, dg)
    assert y.dtype == dtype and y.shape == want.shape
    assert_close(y, want, FWD_TOL[dtype], "2-D forward")
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn2d_backward(x, off, mask, w, gy, True, stride, pad, dil, groups, dg)
    tol = BWD_TOL[dtype]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ws.grad, gw, tol, "grad weight")
    assert_close(bs.grad, gb, tol, "grad bias")
    if modulated:
        assert_close(ms.grad, gm, tol, "grad mask")


def test_2d_packs(ops):
    """Pack modules: zero-initialised offset branch == plain convolution; state-dict keys."""
    torch.manual_seed(0)
    x = torch.randn(2, 8, 12, 14, device=DEV)
    m1 = ops.DeformConv2dPack(8, 16, 3, padding=1).to(DEV)
    assert set(m1.state_dict()) == {"weight", "bias", "conv_offset.weight", "conv_offset.bias"}
    assert_close(m1(x), F.conv2d(x, m1.weight, m1.bias, padding=1), 1e-5, "v1 pack")
    m2 = ops.ModulatedDeformConv2dPack(8, 16, 3, padding=1, stride=2).to(DEV)
    assert set(m2.state_dict()) == {"weight", "bias", "conv_offset_mask.weight", "conv_offset_mask.bias"}
    assert_close(m2(x), 0.5 * F.conv2d(x, m2.weight, None, stride=2, padding=1) + m2.bias.view(1, -1, 1, 1),
                 1e-5, "v2 pack")
    m2(x).sum().backward()
    assert m2.conv_offset_mask.weight.grad is not None and m2.weight.grad is not None
    with pytest.raises(RuntimeError, match="offset has shape"):
        ops.DeformConv2d(8, 16, 3, 1, 1).to(DEV)(x, torch.zeros(2, 18, 12, 13, device=DEV))


def test_warp_int32_labels(ops, oracle):
    """int32 label maps at order 0: the voxel the float path picks (the reference converts the labels
    to float, warps and converts back, aug_cuda/aug_spatial.py:664-668), void positions are 0."""
    g = wl.gen(18)
    for shape in [(2, 2, 10, 12, 14), (2, 3, 20, 24)]:
        nd = len(shape) - 2
        seg = torch.randint(-5, 2 ** 20, shape, generator=g, dtype=torch.int32)
        off = torch.randn(shape[0], nd, *shape[2:], generator=g) * 3
        warp = ops.apply_offset_3d if nd == 3 else ops.apply_offset_2d
        got = warp(seg.to(DEV), off.to(DEV), 0)
        assert got.dtype == torch.int32
        want = oracle.deform_warp(seg.double(), off, 0)
        assert torch.equal(got.cpu().double(), want.double())
        assert float((want == 0).double().mean()) > 0.01     # positions outside the image
    with pytest.raises(RuntimeError, match="order 0 only"):
        ops.apply_offset_3d(torch.zeros(1, 1, 4, 4, 4, dtype=torch.int32, device=DEV),
                            torch.zeros(1, 3, 4, 4, 4, device=DEV), 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("order", [0, 1, 3])
def test_warp_vs_oracle(ops, oracle, dtype, order):
    g = wl.gen(8)
    img = torch.randn(2, 3, 10, 12, 14, generator=g).to(dtype)
    off = (torch.randn(2, 3, 10, 12, 14, generator=g) * 3).to(dtype)
    got = ops.apply_offset_3d(img.to(DEV), off.to(DEV), order)
    assert_close(got, oracle.deform_warp(img, off, order), FWD_TOL[dtype], "warp 3d")
    img2 = torch.randn(2, 3, 20, 24, generator=g).to(dtype)
    off2 = (torch.randn(2, 2, 20, 24, generator=g) * 3).to(dtype)
    got = ops.apply_offset_2d(img2.to(DEV), off2.to(DEV), order)
    assert_close(got, oracle.deform_warp(img2, off2, order), FWD_TOL[dtype], "warp 2d")
    # the reference's calling convention (identity weight through `_C.deform_3d`) gives the same
    from medvision_amd import _C
    eye = torch.eye(3, device=DEV, dtype=dtype).reshape(3, 3, 1, 1, 1)
    same = _C.deform_3d(img.to(DEV), eye, torch.zeros(3, device=DEV, dtype=dtype), off.to(DEV),
                        1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, order)
    assert torch.equal(same, ops.apply_offset_3d(img.to(DEV), off.to(DEV), order))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("order", [0, 1, 3])
def test_general_deform_vs_oracle(ops, oracle, dtype, order):
    """`_C.deform_3d` / `_C.deform_2d` with a real kernel and weight: the DCNv1 forward with the
    clamped samplers (csrc/cuda_aug/deform_3d_cuda.cu:43-152)."""
    from medvision_amd import _C
    g = wl.gen(300 + order)
    cases = [  # Cin, Cout, size, kernel, stride, pad, dil, groups, dg
        (4, 6, (6, 7, 8), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1, 1),
        (4, 70, (5, 9, 8), (2, 3, 1), (1, 2, 1), (0, 2, 1), (2, 1, 1), 2, 2),
        (6, 3, (7, 6, 9), (1, 1, 1), (1, 1, 1), (0, 0, 0), (1, 1, 1), 1, 3),
        (4, 4, (12, 11), (3, 2), (2, 1), (1, 0), (1, 2), 2, 1),
        (3, 5, (9, 10), (1, 1), (1, 1), (0, 0), (1, 1), 1, 1),
    ]
    for Cin, Cout, size, k, stride, pad, dil, groups, dg in cases:
        nd = len(size)
        x = torch.randn(2, Cin, *size, generator=g).to(dtype)
        w = (torch.randn(Cout, Cin // groups, *k, generator=g) * 0.3).to(dtype)
        b = torch.randn(Cout, generator=g).to(dtype)
        out = [(s + 2 * p - (d * (kk - 1) + 1)) // st + 1 for s, p, d, kk, st in zip(size, pad, dil, k, stride)]
        K = 1
        for kk in k:
            K *= kk
        off = (torch.randn(2, dg * nd * K, *out, generator=g) * 2.5).to(dtype)
        fn = _C.deform_3d if nd == 3 else _C.deform_2d
        got = fn(x.to(DEV), w.to(DEV), b.to(DEV), off.to(DEV), *k, *stride, *pad, *dil, groups, dg, 64, order)
        want = oracle.deform_conv(x, off, w, b, stride, pad, dil, groups, dg, order)
        assert tuple(got.shape) == tuple(want.shape)
        assert_close(got, want, FWD_TOL[dtype], f"deform_{nd}d {size} k={k} order={order}")
        assert float((want == b.double().view(1, -1, *([1] * nd))).double().mean()) < 0.9
    if order == 1 and dtype in (torch.float32, torch.float16):
        # an identity weight (the warp) and then a real 1x1x1 weight of the same shape and type: a
        # verdict remembered by address or version would send the second one down the warp path
        x = torch.randn(1, 4, 6, 7, 8, generator=g).to(dtype)
        off = (torch.randn(1, 3, 6, 7, 8, generator=g) * 1.5).to(dtype)
        zero = torch.zeros(4, dtype=dtype)
        for rep in range(3):
            eye = torch.eye(4).view(4, 4, 1, 1, 1).to(dtype).to(DEV)
            got = _C.deform_3d(x.to(DEV), eye, zero.to(DEV), off.to(DEV), 1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, 1)
            assert_close(got, oracle.deform_conv(x, off, eye.cpu(), zero, (1, 1, 1), (0, 0, 0), (1, 1, 1), 1, 1, 1),
                         FWD_TOL[dtype], "identity weight")
            del eye
            w = torch.randn(4, 4, 1, 1, 1, generator=g).to(dtype)
            wd = w.to(DEV)
            got = _C.deform_3d(x.to(DEV), wd, zero.to(DEV), off.to(DEV), 1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, 1)
            assert_close(got, oracle.deform_conv(x, off, w, zero, (1, 1, 1), (0, 0, 0), (1, 1, 1), 1, 1, 1),
                         FWD_TOL[dtype], "random 1x1x1 weight after an identity one")
            ident = torch.eye(4).view(4, 4, 1, 1, 1).to(dtype).to(DEV)
            ident.data.mul_(2.0)     # (a write that leaves the tensor's version alone)
            got = _C.deform_3d(x.to(DEV), ident, zero.to(DEV), off.to(DEV), 1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, 1)
            assert_close(got, oracle.deform_conv(x, off, ident.cpu(), zero, (1, 1, 1), (0, 0, 0), (1, 1, 1), 1, 1, 1),
                         FWD_TOL[dtype], "identity weight edited through .data")
            del wd, ident
    x = torch.zeros(2, 4, 4, 4, 4, device=DEV)
    with pytest.raises(RuntimeError, match="kernel shape wont match"):
        _C.deform_3d(x, torch.zeros(4, 4, 3, 3, 3, device=DEV), torch.zeros(4, device=DEV),
                     torch.zeros(2, 3, 4, 4, 4, device=DEV), 1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, 1)
    with pytest.raises(RuntimeError, match="kernel channels wont match"):
        _C.deform_3d(x, torch.zeros(4, 3, 1, 1, 1, device=DEV), torch.zeros(4, device=DEV),
                     torch.zeros(2, 3, 4, 4, 4, device=DEV), 1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, 1)
    with pytest.raises(RuntimeError, match="order 2 is not supported"):
        _C.deform_3d(x, torch.zeros(4, 4, 1, 1, 1, device=DEV), torch.zeros(4, device=DEV),
                     torch.zeros(2, 3, 4, 4, 4, device=DEV), 1, 1, 1, 1, 1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 64, 2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("cin,cout,dg,modulated", [(24, 40, 2, True), (16, 16, 1, True), (48, 24, 1, False)])
def test_channel_counts_padded_for_the_matrix_cores(ops, oracle, dtype, cin, cout, dg, modulated):
    """Layers whose channel counts are no multiples of 32 run the matrix-core kernels on zero-padded
    copies made inside the library: all outputs and gradients as without."""
    from medvision_amd.ops.deform_conv_3d import deform_conv
    from medvision_amd.ops.modulated_deform_conv_3d import modulated_deform_conv
    from medvision_amd import _C, _lib
    g = wl.gen(500 + cin + cout)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, (5, 8, 9), 3, dg, 1, dtype, 1, 1, 1, modulated)
    import ctypes
    shape = _lib.DcnShape(2, cin, 5, 8, 9, cout, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, dg)
    code = _lib.DTYPES[dtype]
    assert _lib.load().mv_dcn3d_forward_workspace_bytes(ctypes.byref(shape), code) > 0    # padded copies + layouts
    assert _lib.load().mv_dcn3d_backward_workspace_bytes(ctypes.byref(shape), code) > 0
    xs, offs, ms, ws, bs = [None if t is None else t.to(DEV).requires_grad_(True) for t in (x, off, mask, w, b)]
    if modulated:
        y = modulated_deform_conv(xs, offs, ms, ws, bs, 1, 1, 1, 1, dg)
    else:
        y = deform_conv(xs, offs, ws, bs, 1, 1, 1, 1, dg, 64)
    assert_close(y, oracle.dcn3d_forward(x, off, mask, w, b, 1, 1, 1, 1, dg), FWD_TOL[dtype], "forward")
    gy = torch.randn(y.shape, generator=g).to(dtype)
    y.backward(gy.to(DEV))
    gx, goff, gm, gw, gb = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, 1, dg)
    tol = BWD_TOL[dtype]
    assert_close(xs.grad, gx, tol, "grad input")
    assert_close(offs.grad, goff, tol, "grad offset")
    assert_close(ws.grad, gw, tol, "grad weight")
    assert_close(bs.grad, gb, tol, "grad bias")
    if modulated:
        assert_close(ms.grad, gm, tol, "grad mask")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cin,cout,groups,dg,modulated", [
    (24, 40, 1, 1, True), (40, 24, 2, 1, True), (48, 48, 2, 2, False), (48, 80, 2, 4, True), (24, 64, 1, 3, False),
    (8, 8, 1, 1, True), (4, 8, 1, 1, False)])
def test_raw_abi_with_any_channel_count(oracle, dtype, cin, cout, groups, dg, modulated):
    """mv_dcn3d_forward / mv_dcn3d_backward called straight through ctypes (no shim in between) with
    channel counts that are no multiples of 32, several weight groups and deformable groups that
    nest either way, layers of a few channels: results against the oracle, and on the matrix-core kernels
    (timed against a bound the general kernels miss by an order of magnitude)."""
    import ctypes
    from medvision_amd import _lib
    lib = _lib.load()
    g = wl.gen(900 + cin + cout + groups + dg)
    size = (12, 16, 24)
    x, off, mask, w, b = wl.dcn_inputs(g, 2, cin, cout, size, 3, dg, groups, dtype, 1, 1, 1, modulated)
    # An offset far below the rounding of the coordinate it is added to (4 - 6e-8) puts the sample ON a
    # voxel in the kernels' fp32 positions and just below it in the oracle's fp64 ones: the derivative
    # with respect to the offset jumps there, and either side is right.  Keep the draws off that case.
    off[off.abs() < 1e-4] = 0
    shape = _lib.DcnShape(2, cin, *size, cout, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, groups, dg)
    code = _lib.DTYPES[dtype]
    xs, offs, ms, ws, bs = _to(DEV, x, off, mask, w, b)
    y = torch.full((2, cout, *size), float("nan"), dtype=dtype, device=DEV)
    general = dtype == torch.bfloat16 and cin * cout < 256   # (bf16 layers of a few channels: general kernels, no copies)
    nf = lib.mv_dcn3d_forward_workspace_bytes(ctypes.byref(shape), code)
    assert nf > 0 or general
    wsf = torch.empty(max(nf, 16), dtype=torch.uint8, device=DEV)
    stream = _lib.stream_of(xs)

    def forward():
        _lib.check(lib.mv_dcn3d_forward(_lib.ptr(xs), _lib.ptr(offs), _lib.ptr(ms), _lib.ptr(ws), _lib.ptr(bs), _lib.ptr(y),
                                        ctypes.byref(shape), code, _lib.ptr(wsf), stream))
    forward()
    assert_close(y, oracle.dcn3d_forward(x, off, mask, w, b, 1, 1, 1, groups, dg), FWD_TOL[dtype], "forward")
    gy = torch.randn(y.shape, generator=g).to(dtype)
    gys = gy.to(DEV)
    gi, goff, gw, gb = torch.zeros_like(xs), torch.zeros_like(offs), torch.zeros_like(ws), torch.zeros_like(bs)
    gm = torch.zeros_like(ms) if modulated else None
    nb = lib.mv_dcn3d_backward_workspace_bytes(ctypes.byref(shape), code)
    assert nb > 0
    wsb = torch.empty(nb, dtype=torch.uint8, device=DEV)

    def backward():
        _lib.check(lib.mv_dcn3d_backward(_lib.ptr(xs), _lib.ptr(offs), _lib.ptr(ms), _lib.ptr(ws), _lib.ptr(gys), _lib.ptr(gi),
                                         _lib.ptr(goff), _lib.ptr(gm), _lib.ptr(gw), _lib.ptr(gb), ctypes.byref(shape), code,
                                         _lib.ptr(wsb), stream))
    backward()
    want = oracle.dcn3d_backward(x, off, mask, w, gy, True, 1, 1, 1, groups, dg)
    tol = BWD_TOL[dtype]
    assert_close(gi, want[0], tol, "grad input")
    assert_close(goff, want[1], tol, "grad offset")
    assert_close(gw, want[3], tol, "grad weight")
    assert_close(gb, want[4], tol, "grad bias")
    if modulated:
        assert_close(gm, want[2], tol, "grad mask")
    # the gradients accumulate: a second call doubles input / weight / bias gradients
    backward()
    assert_close(gi, 2 * want[0], tol, "grad input accumulates")
    assert_close(gw, 2 * want[3], tol, "grad weight accumulates")
    # timing: against the next larger layer that needs no padding (the layer the library runs inside);
    # the general kernels are 10 - 50 times slower than that
    unit = min(cin // groups, cin // dg)
    cin_n, cout_n = cin // unit * (-(-unit // 32) * 32), groups * (-(-(cout // groups) // 32) * 32)
    xn, offn, mn, wn, bn = _to(DEV, *wl.dcn_inputs(g, 2, cin_n, cout_n, size, 3, dg, groups, dtype, 1, 1, 1, modulated))
    shape_n = _lib.DcnShape(2, cin_n, *size, cout_n, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, groups, dg)
    yn = torch.empty((2, cout_n, *size), dtype=dtype, device=DEV)
    wsn = torch.empty(max(lib.mv_dcn3d_forward_workspace_bytes(ctypes.byref(shape_n), code),
                          lib.mv_dcn3d_backward_workspace_bytes(ctypes.byref(shape_n), code)), dtype=torch.uint8, device=DEV)
    gin, goffn, gwn, gbn = torch.zeros_like(xn), torch.zeros_like(offn), torch.zeros_like(wn), torch.zeros_like(bn)
    gmn = torch.zeros_like(mn) if modulated else None

    def forward_native():
        _lib.check(lib.mv_dcn3d_forward(_lib.ptr(xn), _lib.ptr(offn), _lib.ptr(mn), _lib.ptr(wn), _lib.ptr(bn), _lib.ptr(yn),
                                        ctypes.byref(shape_n), code, _lib.ptr(wsn), stream))

    def backward_native():
        _lib.check(lib.mv_dcn3d_backward(_lib.ptr(xn), _lib.ptr(offn), _lib.ptr(mn), _lib.ptr(wn), _lib.ptr(yn), _lib.ptr(gin),
                                         _lib.ptr(goffn), _lib.ptr(gmn), _lib.ptr(gwn), _lib.ptr(gbn), ctypes.byref(shape_n),
                                         code, _lib.ptr(wsn), stream))

    def timed(fn):
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(10):
            fn()
        stop.record()
        torch.cuda.synchronize()
        return start.elapsed_time(stop) / 10

    if general:
        return   # (fp32 columns for their few weight gradients)
    for fn, native in ((forward, forward_native), (backward, backward_native)):
        ms_call, ms_native = timed(fn), timed(native)
        print(f"\n{fn.__name__} {dtype} cin={cin} cout={cout} groups={groups} dg={dg}: {ms_call:.3f} ms, "
              f"[{cin_n} -> {cout_n}] without padding {ms_native:.3f} ms")
        assert ms_call < 2.5 * ms_native + 0.15, f"{fn.__name__} takes {ms_call:.3f} ms: not on the matrix-core kernels"
