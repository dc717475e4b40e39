"""RoI construction and box transforms of the augmentation layer (CPU: numpy only).

Expected values are worked out by hand from the definition "window (start, end), scaled about its
centre by 1/s, moved by -extent * shift / s, turned by the angle", not by re-running the code's
formula."""
import math
import random

import numpy as np
import pytest
import torch

from medvision_amd.aug_cuda import geometry
from medvision_amd.aug_cuda import spatial


def test_frame_and_window_rois():
    r = geometry.frame_rois((4, 6, 8), 2)
    assert r.dtype == np.float32 and r.shape == (2, 10)
    assert r.tolist() == [[0, 4, 3, 2, 8, 6, 4, 0, 0, 0], [1, 4, 3, 2, 8, 6, 4, 0, 0, 0]]
    # 3-D: scale 1.25 -> the sampled box shrinks to 8/1.25 = 6.4 etc.; shift +0.1 of the width
    # moves the box centre by -8 * 0.1 / 1.25 = -0.64; the angle goes to the last column
    r = geometry.window_rois(3, [0, 0, 0], [8, 6, 4], [1.25] * 3, [0.1, 0.0, -0.1], [0.3])
    want = [0, 4 - 0.64, 3, 2 + 0.32, 6.4, 4.8, 3.2, 0, 0, 0.3]
    assert np.allclose(r[0], want, atol=1e-6)
    # 2-D rows have one angle; per-sample tables
    r = geometry.window_rois(2, [[0, 0], [2, 2]], [[8, 6], [10, 8]], [[2, 2], [1, 1]],
                             [[0, 0.5], [0, 0]], [[0.3], [-0.1]])
    assert np.allclose(r, [[0, 4, 3 - 1.5, 4, 3, 0.3], [1, 6, 5, 8, 6, -0.1]], atol=1e-6)


def test_map_and_clip_boxes():
    frame = (40.0, 30.0, 20.0)
    box = np.array([[10., 9., 8., 20., 15., 12., 1., 0.9]])
    same = geometry.map_boxes(3, box, frame, [1, 1, 1], [0, 0, 0], [0.0])
    assert np.allclose(same, box)
    # shift by +0.25 of the width: content (and boxes) move +10 voxels along x
    moved = geometry.map_boxes(3, box, frame, [1, 1, 1], [0.25, 0, 0], [0.0])
    assert np.allclose(moved[0, [0, 3]], [20, 30]) and np.allclose(moved[0, [1, 2, 4, 5]], box[0, [1, 2, 4, 5]])
    # scale 2 about the image centre (20, 15, 10)
    big = geometry.map_boxes(3, box, frame, [2, 2, 2], [0, 0, 0], [0.0])
    assert np.allclose(big[0, :6], [0, 3, 6, 20, 15, 14])
    # quarter turn of a rectangle centred on the image centre swaps its x and y extents; z stays
    cen = np.array([[20 - 6., 15 - 2., 5., 20 + 6., 15 + 2., 9., 0., 0.]])
    turned = geometry.map_boxes(3, cen, frame, [1, 1, 1], [0, 0, 0], [math.pi / 2])
    assert np.allclose(turned[0, :6], [20 - 2, 15 - 6, 5, 20 + 2, 15 + 6, 9])
    # a crop window starting at (5, 4, 3) moves boxes by -start
    crop = geometry.map_boxes(3, box, (16., 16., 16.), [1, 1, 1], [0, 0, 0], [0.0], start_xyz=(5, 4, 3))
    assert np.allclose(crop[0, :6], [5, 5, 5, 15, 11, 9])
    # clip: into [0, size-1]; boxes that collapse are dropped; extra columns survive
    boxes = np.array([[-3., 2., 1., 50., 10., 5., 7., 0.5], [45., 2., 1., 60., 10., 5., 3., 0.1]])
    kept = geometry.clip_boxes(boxes, (20, 30, 40))
    assert kept.tolist() == [[0., 2., 1., 39., 10., 5., 7., 0.5]]
    assert geometry.clip_boxes(np.zeros((0, 8)), (20, 30, 40)).shape == (0, 8)


def test_parameter_draws_follow_numpy_random_in_the_documented_order():
    import torch
    result = {"img": torch.zeros(1, 8, 9, 10), "img_dim": 3}
    stage = spatial.CudaCropRandomWithAffine((4, 5, 6), scale=0.2, shift=0.1, rotate=30)
    np.random.seed(7)
    stage._forward_params(result)
    np.random.seed(7)
    start = [np.random.randint(0, 8 - 4 + 1), np.random.randint(0, 9 - 5 + 1), np.random.randint(0, 10 - 6 + 1)]
    scale = 1 + np.random.uniform(-0.2, 0.2)
    shifts = [np.random.uniform(-0.1, 0.1) for _ in range(3)]
    angle = math.pi * np.random.uniform(-30, 30) / 180
    p = result["CudaCropRandomWithAffine_params"]
    assert tuple(p["start"]) == tuple(start[::-1]) and tuple(p["end"]) == (start[2] + 6, start[1] + 5, start[0] + 4)
    assert p["_scales"] == [scale] * 3 and p["_shifts"] == shifts and p["_rotate"] == [angle]
    rois = stage._rois()
    assert rois.shape == (1, 10) and rois[0, 9] == np.float32(angle) and rois[0, 7] == 0 and rois[0, 8] == 0
    # batch stage: one row of parameters per sample
    bstage = spatial.BatchCudaRandomAffine(1.0, scale=0.1, shift=0.1, rotate=10)
    bresult = {"img": torch.zeros(3, 1, 8, 9), "img_dim": 2}
    bstage._forward_params(bresult)
    bp = bresult["BatchCudaRandomAffine_params"]
    assert bp["scales"].shape == (3, 2) and bp["shifts"].shape == (3, 2) and bp["rotate"].shape == (3, 1)
    assert bstage._rois().shape == (3, 6) and bstage._rois()[:, 0].tolist() == [0, 1, 2]


def test_elastic_control_grid_and_gate():
    import torch
    stage = spatial.CudaRandomElasticDeformation(p=1.0, num_control_points=7, max_displacement=0.5)
    result = {"img": torch.zeros(1, 24, 30, 36), "img_dim": 3}
    np.random.seed(3)
    stage._forward_params(result)
    grid = result["CudaRandomElasticDeformation_params"]
    assert grid.shape == (7, 7, 7, 3) and grid.dtype == np.float32
    inner = grid[2:-2, 2:-2, 2:-2]
    assert np.all(grid[:2] == 0) and np.all(grid[:, -2:] == 0) and np.all(grid[:, :, :2] == 0)
    assert np.any(inner != 0)
    # |displacement| <= max_displacement * cell / 2 with cell = size / (points - 1), per component z, y, x
    limit = 0.5 * np.array([24, 30, 36]) / 6 / 2
    assert np.all(np.abs(inner) <= limit + 1e-6) and np.abs(inner[..., 2]).max() > limit[0]
    # the probability gate uses random.random(): p * latitude = 0 never fires
    gate = spatial.CudaRandomShift(p=0.5, shift=0.1)
    gate.setLatitude(0.0)
    random.seed(0)
    out = gate({"img": torch.zeros(1, 4, 4), "img_dim": 2, "img_fields": ["img"]})
    assert out["history"] == ["CudaRandomShift"] and "CudaRandomShift_params" not in out
    with pytest.raises(AssertionError):
        spatial.CudaRandomShift(p=0.0, shift=0.1)({"img": torch.zeros(1, 4, 4), "img_dim": 2})


def test_uploads_keep_double():
    """Control grids and rois that a caller gives in float64 stay float64 (the field is then resampled in float64)."""
    from medvision_amd._lib import native
    values = np.random.default_rng(0).standard_normal((2, 3, 5))
    for array, dtype in ((values, torch.float64), (values.astype(np.float32), torch.float32), (values.T, torch.float64),
                         (np.arange(6), torch.float32)):
        out = native.upload(array, torch.device("cpu"))
        assert out.dtype == dtype and out.is_contiguous()
        assert torch.equal(out, torch.from_numpy(np.ascontiguousarray(array)).to(dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("grid,dtype", [(np.float64, torch.float64), (np.float32, torch.float32), (np.int64, torch.float32)])
def test_elastic_field_keeps_the_control_grids_type(grid, dtype):
    import medvision_amd.aug_cuda as aug
    params = (np.random.default_rng(1).standard_normal((9, 9, 9, 3)) * 3).astype(grid)   # 17 KB in float64: more than one upload
    for points in (5, 9):
        stage = aug.CudaRandomElasticDeformation(1.0, points, 0.8)
        stage._init_params({"img": torch.zeros(1, 20, 24, 28, device="cuda"), "img_dim": 3})
        stage.params = params[:points, :points, :points]
        field = stage.dense_field(torch.device("cuda"))
        assert field.dtype == dtype and field.shape == (3, 20, 24, 28)


def test_native_window_rois_are_the_arrays_rows():
    """The roi of one window, built natively, has the bits of geometry.window_rois."""
    from medvision_amd._lib import native
    rng = np.random.default_rng(8)
    for k in range(200):
        dim = 2 + k % 2
        start = [int(v) for v in rng.integers(0, 40, dim)] if k % 3 else [0.0] * dim
        end = [s + float(v) for s, v in zip(start, rng.uniform(0.1, 300, dim))]
        scales, shifts, rotate = list(rng.uniform(0.5, 1.7, dim)), [rng.uniform(-0.3, 0.3) for _ in range(dim)], rng.uniform(-4, 4)
        want = geometry.window_rois(dim, start, end, scales, shifts, [rotate], index=np.arange(1))
        got = native.window_roi(dim, start, end, scales, shifts, rotate, torch.device("cpu"))
        assert got.dtype == torch.float32 and np.array_equal(got.numpy(), want)
    with pytest.raises(RuntimeError):
        native.window_roi(3, [0.0] * 3, [1.0] * 3, [1.0] * 2, [0.0] * 3, 0.0, torch.device("cpu"))


def test_elastic_stage_restored_from_an_older_state():
    """A state that holds the dense field under its public name, and a stage that never ran."""
    import pickle
    import numpy as np
    from medvision_amd.aug_cuda import CudaRandomElasticDeformation
    stage = CudaRandomElasticDeformation(1.0, 6, 0.5)
    old = {k: v for k, v in stage.__dict__.items() if k not in ('_field', '_device_grid', '_field_device')}
    for field in (None, np.ones(3)):
        again = CudaRandomElasticDeformation.__new__(CudaRandomElasticDeformation)
        again.__setstate__({**old, 'tmp_params': field})
        assert again.tmp_params is field and again._field is field
        assert again._device_grid is None
    assert pickle.loads(pickle.dumps(stage)).tmp_params is None


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("values", [
    (1.25, 0.1, 0.3),                                                            # scalars, as window_rois takes them
    ([1.25] * 3, 0.1, [0.3]),
    (np.array([1.1, 1.2, 1.3]), np.array([0.1, -0.2, 0.05]), np.array([0.3])),
    (np.float32(1.25), [0.1, 0.0, np.float32(0.2)], 1),
    ([[1.1, 1.2, 1.3]], [[0.1, -0.2, 0.05]], [[0.3]]),                           # rows of a table
    ([1.1, 1.2, 1.3], np.array([[0.1, -0.2, 0.05]]), np.array(0.3)),
])
def test_affine_stage_takes_what_window_rois_takes(dim, values):
    """Scalars, rows and tables from a stage's parameters: the roi of geometry.window_rois."""
    from medvision_amd.aug_cuda import CudaRandomAffine

    def cut(v):
        if isinstance(v, list):
            return [cut(x) for x in v] if isinstance(v[0], list) else v[:dim]
        return v[..., :dim] if isinstance(v, np.ndarray) and v.ndim else v

    class Given(CudaRandomAffine):
        def _affine(self):
            return tuple(cut(v) for v in values)

    stage = Given(1.0, 0.2, 0.1, 30)
    stage._init_params({"img": torch.zeros(1, *(12, 14, 16)[:dim]), "img_dim": dim})
    got = stage._uploaded_rois(torch.device("cpu"))
    assert np.array_equal(got.cpu().numpy(), stage._rois())
