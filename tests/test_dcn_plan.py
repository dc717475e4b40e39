"""The plan of the deformable backward's LDS sums (``dcn_scatter_plan``, host code): bricks, tiles and the width of the sums,
asked of the built library without a GPU."""
import ctypes
import math

import pytest

from medvision_amd import _lib


class _Dims(ctypes.Structure):   # DcnDims (csrc/dcn_common.hpp)
    _fields_ = [(n, ctypes.c_int) for n in (
        "B", "Cin", "D", "H", "W", "Cout", "kd", "kh", "kw", "sd", "sh", "sw", "pd", "ph", "pw", "dd", "dh", "dw",
        "groups", "dg", "nd", "Do", "Ho", "Wo", "K", "cpg", "opg", "cpd")] + [("Q", ctypes.c_long), ("P", ctypes.c_long)]


class _Shape(ctypes.Structure):   # ScatterShape (csrc/dcn_scatter.hpp)
    _fields_ = [(n, ctypes.c_int) for n in (
        "bd", "bh", "bw", "td", "th", "tw", "nbd", "nbh", "nbw", "terms", "narrow", "turns")]


def _plan(code, batch, cin, cout, size, kernel=3, stride=1, dilation=1, padding=None):
    """The plan of a layer, None where no brick fits."""
    nd = len(size)
    each = lambda v: (1,) * (3 - nd) + ((v,) * nd if isinstance(v, int) else tuple(v))
    k, s, d, n = each(kernel), each(stride), each(dilation), (1,) * (3 - nd) + tuple(size)
    p = tuple((a - 1) * b // 2 for a, b in zip(k, d)) if padding is None else (0,) * (3 - nd) + (padding,) * nd
    out = [(n[a] + 2 * p[a] - (d[a] * (k[a] - 1) + 1)) // s[a] + 1 for a in range(3)]
    dims = _Dims(batch, cin, *n, cout, *k, *s, *p, *d, 1, 1, nd, *out, math.prod(k), cin, cout, cin, math.prod(out), math.prod(n))
    fn = _lib.load()._ZN2mv16dcn_scatter_planERKNS_7DcnDimsEiRNS_12ScatterShapeE
    fn.restype, fn.argtypes = ctypes.c_bool, [ctypes.POINTER(_Dims), ctypes.c_int, ctypes.POINTER(_Shape)]
    shape = _Shape()
    return shape if fn(ctypes.byref(dims), code, ctypes.byref(shape)) else None


@pytest.mark.parametrize("code", [_lib.MV_F16, _lib.MV_BF16])
@pytest.mark.parametrize("kernel,stride,dilation,narrow,brick", [
    (3, 1, 1, 1, (2, 3, 3)),
    ((1, 3, 3), (2, 1, 1), 1, 1, (2, 2, 2)),      # every other slice, each by itself
    (3, 1, (2, 1, 1), 1, (2, 2, 2)),               # 19 bits for a term, not the 18 of the larger brick
    (3, (2, 1, 1), 1, 0, None),                    # strided
    (3, 1, (3, 1, 1), 0, None),                    # taps far apart
    ((7, 3, 3), 1, 1, 0, None),
    (3, (1, 2, 1), 1, 0, None),
    (3, 1, (1, 1, 3), 0, None),
    (3, 2, 1, 0, None),
])
def test_width_of_the_sums_of_volumes(code, kernel, stride, dilation, narrow, brick):
    """32-bit sums are for dense layers: with strides or taps far apart along any axis the sums have 64 bits, whatever the tiles hold."""
    shape = _plan(code, 2, 32, 64, (48, 48, 48), kernel, stride, dilation)
    assert shape.narrow == narrow
    if brick:
        assert (shape.bd, shape.bh, shape.bw) == brick


@pytest.mark.parametrize("code", [_lib.MV_F32, _lib.MV_F16, _lib.MV_BF16])
@pytest.mark.parametrize("cout", [64, 256])
@pytest.mark.parametrize("kernel,stride,dilation", [
    (3, 1, 9), (3, 1, 10), (3, 1, 12), (3, 1, 13), (3, 1, (12, 2)), (3, 1, (1, 12)), ((3, 5), (1, 2), (12, 1)),
])
def test_images_with_taps_far_apart_keep_their_tiles(code, cout, kernel, stride, dilation):
    """A tile of 44 x 44 voxels holds the reach of 3 x 3 taps up to dilation 13: their corners are summed in LDS."""
    shape = _plan(code, 2, 128, cout, (112, 208), kernel, stride, dilation)
    assert shape is not None
    st, dl, kn = ((v, v) if isinstance(v, int) else v for v in (stride, dilation, kernel))
    spare = min(t - ((1 << b) - 1) * s - (k - 1) * d - 1
                for t, b, s, k, d in zip((shape.th, shape.tw), (shape.bh, shape.bw), st, kn, dl))
    assert spare >= (4 if max(dl) <= 12 else 2)


@pytest.mark.parametrize("cout", [64, 128])
@pytest.mark.parametrize("kernel,dilation", [(3, 5), (11, 1), ((3, 5), (5, 2))])
def test_dense_images_of_far_reach(cout, kernel, dilation):
    """Where 32 x 32 positions leave fewer than four voxels to spare, 16 x 16 in the same tile, not 8 x 8 in a smaller one."""
    for code in (_lib.MV_F16, _lib.MV_BF16):
        shape = _plan(code, 2, 128, cout, (112, 208), kernel, 1, dilation)
        assert (shape.narrow, shape.bh, shape.bw, shape.th, shape.tw) == (1, 4, 4, 44, 44)


class _Dim3(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in "xyz"]


def _grid(workgroups, threads):
    fn = _lib.load()._ZN2mv11linear_gridEli
    fn.restype, fn.argtypes = _Dim3, [ctypes.c_long, ctypes.c_int]
    return fn(workgroups, threads)


@pytest.mark.parametrize("threads", [256, 512, 1024])
@pytest.mark.parametrize("workgroups", [1, 255, (1 << 22) - 1, 1 << 22, (1 << 22) + 1, 4239360, (1 << 24) - 1, 1 << 24, 19462005, (1 << 31) - 1])
def test_grids_of_many_workgroups(workgroups, threads):
    """A dimension of a grid has fewer than 2^32 threads: one row as long as that holds, then rows that leave no whole row idle."""
    g = _grid(workgroups, threads)
    assert g.x * threads < 1 << 32 and g.y <= 65535 and g.z == 1
    assert g.x * g.y >= workgroups > g.x * (g.y - 1)
    assert g.y == 1 or workgroups * threads >= 1 << 32


def test_a_volume_of_more_workgroups_than_a_row():
    """fp32 [16, 32 -> 32, 128 x 180 x 182] at dilation 2 has 4 239 360 workgroups of 1024 threads: the plan takes it."""
    shape = _plan(_lib.MV_F32, 16, 32, 32, (128, 180, 182), 3, 1, 2)
    assert shape.nbd * shape.nbh * shape.nbw * 16 * (32 // 8) == 4239360
    assert _grid(4239360, 1024).y == 2


class _Columns(ctypes.Structure):   # ColumnsPlan (csrc/dcn_forward_columns.hip)
    _fields_ = [(n, ctypes.c_int) for n in ("positions", "waves", "blocks")] + [(n, ctypes.c_long) for n in ("tiles", "chunks")]


def _columns(code, batch, cin, cout, size, groups):
    nd = len(size)
    kernel, n = (1,) * (3 - nd) + (3,) * nd, (1,) * (3 - nd) + tuple(size)
    pad = tuple(k // 2 for k in kernel)
    dims = _Dims(batch, cin, *n, cout, *kernel, 1, 1, 1, *pad, 1, 1, 1, groups, 1, nd, *n, math.prod(kernel), cin // groups, cout // groups, cin,
                 math.prod(n), math.prod(n))
    fn = _lib.load()._ZN2mv16dcn_columns_planERKNS_7DcnDimsEiRNS_11ColumnsPlanE
    fn.restype, fn.argtypes = None, [ctypes.POINTER(_Dims), ctypes.c_int, ctypes.POINTER(_Columns)]
    plan = _Columns()
    fn(ctypes.byref(dims), code, ctypes.byref(plan))
    return plan


@pytest.mark.parametrize("code", [_lib.MV_F32, _lib.MV_F16, _lib.MV_BF16])
@pytest.mark.parametrize("groups", [1, 2, 3])
@pytest.mark.parametrize("rows", [16, 64, 80, 128, 144, 256, 272, 512, 528])
def test_columns_grid_covers_the_layer_once(code, groups, rows):
    """The workgroups that start are those that the kernel numbers: its tiles of positions and, per group, its chunks of output channels."""
    kernels = {(16, 4, 1), (16, 4, 2), (16, 4, 4), (32, 4, 1), (32, 4, 2), (32, 4, 4)}
    for size in [(1, 1), (3, 3), (4, 4), (17, 1), (5, 5), (7, 7), (8, 8), (9, 9), (14, 14), (33, 47), (100, 152), (2, 2, 4), (5, 7, 11), (48, 48, 48)]:
        q = math.prod(size)
        for batch in [*range(1, 20), *range(20, 700, 7), 1024, 4096]:
            plan = _columns(code, batch, 32 * groups, rows * groups, size, groups)
            what = f"{size} x {batch}"
            assert (plan.positions, plan.waves, plan.blocks) in kernels | ({(64, 8, 2)} if len(size) == 2 else set()), what
            assert plan.tiles == -(-q // plan.positions), what
            assert plan.chunks == groups * -(-rows // (16 * plan.waves * plan.blocks)), what
