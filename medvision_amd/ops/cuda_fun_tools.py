"""Functional resampling engines used by the augmentation layer.

Interface of the reference's ``medvision/ops/cuda_fun_tools.py``: ``affine_2d`` / ``affine_3d``
(:6-92) resample with rotated rois (Resize, RandomAffine, Crop); ``apply_offset_2d`` /
``apply_offset_3d`` (:94-167) warp an image by a dense displacement field
(RandomElasticDeformation).  Orders: 0 nearest, 1 linear, 3 cubic (Catmull-Rom).
"""
from .._lib import native


def affine_2d(features, rois, out_size, spatial_scale, sampling_ratio=0, aligned=True, order=1):
    """features [B,C,H,W], rois [n,6] = (b, cx, cy, w, h, angle) -> [n,C,*out_size]."""
    return native.affine(2, features, rois, out_size, spatial_scale, sampling_ratio, aligned, order)


def affine_3d(features, rois, out_size, spatial_scale, sampling_ratio=0, aligned=True, order=1):
    """features [B,C,D,H,W], rois [n,10] = (b, cx, cy, cz, w, h, d, ax, ay, az) -> [n,C,*out_size]."""
    return native.affine(3, features, rois, out_size, spatial_scale, sampling_ratio, aligned, order)


def apply_offset_2d(img, offset, order=1):
    """img [B,C,H,W], offset [B,2,H,W] (channel 0 = rows, 1 = columns): out(q) = img(q + offset(q))."""
    assert img.shape[2:] == offset.shape[2:]
    assert offset.shape[1] == 2
    return native.deform_warp(img, offset, order)


def apply_offset_3d(img, offset, order=1):
    """img [B,C,D,H,W], offset [B,3,D,H,W] (channels depth, height, width)."""
    assert img.shape[2:] == offset.shape[2:]
    assert offset.shape[1] == 3
    return native.deform_warp(img, offset, order)
