"""CPU-side checks of the boundary: the shared library loads, exports every symbol the header
declares, and the host shim rejects bad arguments without touching a GPU."""
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_symbols():
    text = open(os.path.join(ROOT, "include", "medvision_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return set(re.findall(r"\b(mv_[a-z0-9_]+)\s*\(", text))


def test_library_exports_every_declared_symbol():
    from medvision_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        from medvision_amd import build
        build.build()
    lib = _lib.load()
    declared = _header_symbols()
    assert declared, "no symbols parsed from the header"
    assert declared == set(_lib.SIGNATURES), declared ^ set(_lib.SIGNATURES)
    for name in declared:
        assert getattr(lib, name) is not None
    assert lib.mv_version() >= 1


def test_workspace_queries_and_dims_need_no_gpu():
    from medvision_amd import _lib
    import ctypes
    lib = _lib.load()
    assert lib.mv_roi_align_backward_workspace_bytes(_lib.MV_F32, 2, 3, 4, 5, 6) == 0
    assert lib.mv_roi_align_backward_workspace_bytes(_lib.MV_F16, 2, 3, 4, 5, 6) == 4 * 2 * 3 * 4 * 5 * 6
    s = _lib.DcnShape(2, 32, 48, 48, 48, 64, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1)
    d, h, w = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert lib.mv_dcn3d_output_dims(ctypes.byref(s), ctypes.byref(d), ctypes.byref(h), ctypes.byref(w)) == 0
    assert (d.value, h.value, w.value) == (48, 48, 48)
    s2 = _lib.DcnShape(2, 32, 9, 10, 11, 64, 3, 2, 3, 2, 1, 2, 0, 1, 2, 1, 2, 1, 1, 1)
    assert lib.mv_dcn3d_output_dims(ctypes.byref(s2), ctypes.byref(d), ctypes.byref(h), ctypes.byref(w)) == 0
    assert (d.value, h.value, w.value) == ((9 - 3) // 2 + 1, (10 + 2 - 3) // 1 + 1, (11 + 4 - 3) // 2 + 1)
    bad = _lib.DcnShape(2, 30, 8, 8, 8, 64, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 4, 1)
    assert lib.mv_dcn3d_output_dims(ctypes.byref(bad), ctypes.byref(d), ctypes.byref(h), ctypes.byref(w)) == 1
    assert b"must divide group" in lib.mv_last_error()


def test_rotated_image_heads_get_room_for_the_channels_last_copy():
    """The forward query is not told whether the rois are rotated: what plain heads on images want (an order of the rois) must not
    take the place of the copy that rotated ones read."""
    from medvision_amd import _lib
    lib = _lib.load()
    for code, size in ((_lib.MV_F32, 4), (_lib.MV_BF16, 2), (_lib.MV_F16, 2)):
        for rois in (100, 1000):
            need = lib.mv_roi_align_forward_workspace_bytes_for_input(code, 2, 2, 64, 1, 64, 100, rois, 1, 14, 14, 2)
            assert need >= 2 * 64 * 64 * 100 * size
    assert lib.mv_roi_align_forward_workspace_bytes_for_input(_lib.MV_F32, 2, 2, 256, 1, 200, 304, 1000, 1, 7, 7, 2) >= 2 * 256 * 200 * 304 * 4


def test_resampled_images_need_no_workspace():
    """Images of resampling size keep their state in LDS: no tensor is allocated per call."""
    from medvision_amd import _lib
    lib = _lib.load()
    for code in (_lib.MV_F32, _lib.MV_F16, _lib.MV_BF16, _lib.MV_I32):
        assert lib.mv_roi_align_forward_workspace_bytes(code, 2, 3, 8, 1, 512, 512, 1) == 0
        assert lib.mv_roi_align_forward_workspace_bytes_for_input(code, 2, 8, 16, 1, 512, 512, 8, 1, 512, 512, 1) == 0


def test_host_shim_rejects_cpu_tensors_and_bad_rois():
    import medvision_amd.ops as ops
    feat = torch.randn(1, 2, 4, 5, 6)
    with pytest.raises(RuntimeError, match="RoIAlign is not implemented on CPU"):
        ops.RoIAlign((2, 2, 2), 1.0, 2)(feat, torch.zeros(1, 7))
    with pytest.raises(RuntimeError, match="RoIAlignRotated is not implemented on CPU"):
        ops.RoIAlignRotated((2, 2, 2), 1.0, 2)(feat, torch.zeros(1, 10))
    with pytest.raises(AssertionError):
        ops.RoIAlignRotated((2, 2, 2), 1.0, 2)(feat, torch.zeros(1, 10), order=2)
    with pytest.raises(TypeError):
        from medvision_amd.ops.roi_align_nd import roi_align_3d
        roi_align_3d(feat, torch.zeros(1, 7), [2, 2, 2], 1.0, 2, 1)
    with pytest.raises(NotImplementedError):
        ops.ModulatedDeformConv3dPack(2, 3, 3, padding=1)(feat)
    with pytest.raises(AssertionError, match="order 2 is not supported"):
        ops.affine_3d(feat, torch.zeros(1, 10), (2, 2, 2), 1.0, 1, True, 2)
    with pytest.raises(RuntimeError, match="affine is not implemented on CPU"):
        ops.affine_3d(feat, torch.zeros(1, 10), (2, 2, 2), 1.0, 1, True, 3)
    m = ops.DeformConv3dPack(2, 4, 3, padding=1, bias=False)
    assert set(m.state_dict()) == {"weight", "bias", "conv_offset.weight", "conv_offset.bias"}
    assert not m.bias.requires_grad and m.conv_offset.lr_mult == 0.1
    with pytest.raises(ValueError):
        ops.DeformConv3d(3, 4, 3, 1, 1, groups=2)


def test_product_does_not_import_the_oracle():
    import subprocess, sys
    code = ("import sys; sys.path.insert(0, %r); import medvision_amd.ops, medvision_amd._C; "
            "assert not any(m == 'oracle' or m.startswith('oracle.') for m in sys.modules)" % ROOT)
    subprocess.check_call([sys.executable, "-c", code])
    for dirpath, _, files in os.walk(os.path.join(ROOT, "medvision_amd")):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".h")):
                assert "oracle" not in open(os.path.join(dirpath, f)).read().lower(), f


def test_foreign_device_tensors_are_refused():
    """Every tensor handed to a kernel must sit on the input's device; the check runs on the host."""
    from medvision_amd import _C
    here, there = torch.zeros(2), torch.zeros(2, device="meta")
    _C._same_device(here, weight=here, bias=None)
    with pytest.raises(RuntimeError, match="weight is on meta"):
        _C._same_device(here, weight=there)
    with pytest.raises(RuntimeError, match="grad_input is on meta"):
        _C._same_device(here, output=here, grad_input=there)


def test_host_shim_cost_per_call(monkeypatch):
    """Host time of one call through the Python shim with the library stubbed out (argument checks,
    roi cast, workspace query cache, pointer and stream marshalling): the part of a launch that the
    shim adds on top of the C entry point.  Printed for the record; the bound is loose because the
    machine running the CPU suite is shared."""
    import ctypes
    import time
    import torch
    from medvision_amd import _C, _lib

    class Stub:
        def __getattr__(self, name):
            return lambda *a: 0

    class NoGuard:
        def __init__(self, t): pass
        def __enter__(self): pass
        def __exit__(self, *e): return False

    monkeypatch.setattr(_lib, "load", lambda: Stub())
    monkeypatch.setattr(_lib, "stream_of", lambda t: ctypes.c_void_p(0))
    monkeypatch.setattr(_C, "_require_cuda", lambda t, what: None)
    monkeypatch.setattr(_C, "_on_device", NoGuard)
    monkeypatch.setattr(_C, "_ws_bytes_cache", {})
    vol = torch.zeros(1, 1, 16, 16, 16, dtype=torch.float16)
    roi = torch.tensor([[0, 8, 8, 8, 16, 16, 16, 0, 0, 0]], dtype=torch.float32)
    out = torch.empty(1, 1, 16, 16, 16, dtype=torch.float16)
    call = lambda: _C.roi_align_rotated_3d_forward(vol, roi, out, 16, 16, 16, 1.0, 1, True, 1)
    for _ in range(200):
        call()
    best = 1e9
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(2000):
            call()
        best = min(best, (time.perf_counter() - t) / 2000 * 1e6)
    print(f"roi_align_rotated_3d_forward shim: {best:.1f} us per call")
    assert best < 2000.0   # (a sanity bound only: ~8 us on an idle core)


def test_dcn_backward_workspace_keeps_to_its_limit():
    """The partial sums of layers with several chunks of channels stay within the limit that the caller sets."""
    import ctypes
    from medvision_amd import _C, _lib
    lib = _lib.load()

    def need(shape, code=_lib.MV_F16):
        fn = lib.mv_dcn3d_backward_workspace_bytes if isinstance(shape, _lib.DcnShape) else lib.mv_dcn2d_backward_workspace_bytes
        return fn(ctypes.byref(shape), code)

    volume = _lib.DcnShape(2, 256, 48, 48, 48, 256, 5, 5, 5, 1, 1, 1, 2, 2, 2, 1, 1, 1, 1, 1)     # 3.5 GB of partial sums
    image = _lib.Dcn2dShape(8, 256, 100, 152, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    old = _C.set_dcn_column_budget(0)
    try:
        least = [need(s) for s in (volume, image)]
        for budget in (100 << 20, 1 << 30, 2 ** 63):
            _C.set_dcn_column_budget(budget)
            for s, low in zip((volume, image), least):
                assert low <= need(s) <= low + budget
        assert need(volume) - least[0] > 3 << 30
        _C.set_dcn_column_budget(1 << 30)
        assert need(volume) - least[0] > 1 << 29     # ... and use it
    finally:
        _C.set_dcn_column_budget(old)


def test_operator_functions_can_be_subclassed():
    """The ``*Function`` classes are autograd functions with ``forward`` and ``backward``; one that overrides them is run through
    its own."""
    import importlib
    for module, names in (("roi_align_nd", ("RoIAlign2DFunction", "RoIAlign3DFunction")),
                          ("roi_align_rotated_nd", ("RoIAlignRotated2DFunction", "RoIAlignRotated3DFunction")),
                          ("deform_conv_2d", ("DeformConv2dFunction",)), ("deform_conv_3d", ("DeformConv3dFunction",)),
                          ("modulated_deform_conv_2d", ("ModulatedDeformConv2dFunction",)),
                          ("modulated_deform_conv_3d", ("ModulatedDeformConv3dFunction",))):
        for name in names:
            base = getattr(importlib.import_module("medvision_amd.ops." + module), name)
            assert issubclass(base, torch.autograd.Function)

            class Twice(base):
                @staticmethod
                def forward(ctx, x, *rest):
                    return 2 * x

                @staticmethod
                def backward(ctx, grad):
                    return 3 * grad

            class Node(base):
                native = staticmethod(lambda x, add=1: x + add)

            class Same(Node):
                pass

            x = torch.ones(2, requires_grad=True)
            y = Twice.apply(x)
            y.sum().backward()
            assert y.tolist() == [2, 2] and x.grad.tolist() == [3, 3]
            assert Same.apply(1) == 2 and Same.apply(1, add=2) == 3     # nothing overridden: the native node


def test_whole_numbers_may_be_floats():
    """sampling_ratio, order and im2col_step go through int(): the calls get as far as the check of the device."""
    import medvision_amd.ops as ops
    from medvision_amd.ops.deform_conv_3d import deform_conv
    vol, plain, turned = torch.randn(1, 4, 6, 6, 6), torch.zeros(1, 7), torch.zeros(1, 10)
    weight, bias, off = torch.zeros(4, 4, 3, 3, 3), torch.zeros(4), torch.zeros(1, 81, 6, 6, 6)
    for run in (lambda: ops.roi_align_nd.roi_align_3d(vol, plain, (2, 2, 2), 1.0, 2.0, 1.0),
                lambda: ops.roi_align_rotated_nd.roi_align_rotated_3d(vol, turned, (2, 2, 2), 1.0, 2.0, True, 1.0),
                lambda: ops.affine_3d(vol, turned, (2, 2, 2), 1.0, 1.0, True, 1.0),
                lambda: ops.apply_offset_3d(vol, torch.zeros(1, 3, 6, 6, 6), 1.0),
                lambda: deform_conv(vol, off, weight, bias, 1, 1, 1, 1, 1, 64.0)):
        with pytest.raises(RuntimeError, match="CPU"):
            run()
    with pytest.raises(AssertionError, match="order 1.5 is not supported"):
        ops.affine_3d(vol, turned, (2, 2, 2), 1.0, 1, True, 1.5)
