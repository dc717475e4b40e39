"""Timed cases of the framework: resampling, augmentation, detection heads and deformable convolutions.

Every case goes through the public entry points (``medvision_amd.ops``, ``medvision_amd.aug_cuda``) the way a
training or inference script calls them.  ``listed()`` holds fixed cases, ``draw()`` gives further ones of the
same ranges, ``prepare()`` makes what the caller has in hand on the GPU, ``run()`` makes one pass, ``work()``
says what a pass cannot do without and ``tolerance()`` how far two correct implementations may be apart.

Kinds of cases
    affine   ``affine_{2,3}d`` with one rotated full-frame roi per sample (RandomAffine), a forward pass
    resize   ``affine_3d`` with unrotated full-frame rois (Resize of a CT scan)
    augment  the stages Resize, RandomAffine, RandomElasticDeformation and CropRandomWithAffine on one sample
             with a label map
    head     ``RoIAlign`` / ``RoIAlignRotated`` of a detection head, forward alone or forward and backward
    dcn      ``ModulatedDeformConv{2,3}d`` layers, forward alone or forward and all five gradients
"""
import math

import numpy as np
import torch

import medvision_amd.aug_cuda as aug
import medvision_amd.ops as ops

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
BYTES = {"f16": 2, "bf16": 2, "f32": 4}


def listed():
    return [
        # one training patch through RandomAffine: a call whose launch and host work count
        {"name": "affine3d_patch_f32", "kind": "affine", "ndim": 3, "dtype": "f32", "batch": 1, "channels": 1,
         "d": 32, "h": 48, "w": 48},
        # RandomAffine of a batch of volumes: the resampling benchmark of this repository
        {"name": "affine3d_batch_f16", "kind": "affine", "ndim": 3, "dtype": "f16", "batch": 4, "channels": 1,
         "d": 128, "h": 128, "w": 128},
        # RandomAffine of one scan as it comes from the scanner: odd axes, rows that are not aligned
        {"name": "affine3d_scan_f32", "kind": "affine", "ndim": 3, "dtype": "f32", "batch": 1, "channels": 1,
         "d": 155, "h": 241, "w": 233},
        # Resize of CT scans to the working resolution: the largest inputs
        {"name": "resize_ct_f16", "kind": "resize", "dtype": "f16", "batch": 2, "d": 256, "h": 512, "w": 512,
         "out_d": 160, "out_h": 256, "out_w": 256},
        # an augmentation pipeline on one sample: host work, uploads and several launches per stage
        {"name": "augment_chain_f16", "kind": "augment", "dtype": "f16", "d": 128, "h": 256, "w": 256,
         "factor": 0.75, "patch": 96, "points": 8},
        # inference of a small 3-D head at full precision
        {"name": "head3d_small_f32", "kind": "head", "ndim": 3, "rotated": False, "train": False, "dtype": "f32",
         "batch": 2, "channels": 16, "d": 32, "h": 64, "w": 64, "rois": 128, "low": 4.0, "high": 24.0, "scale": 1.0,
         "cells": 7, "ratio": 2},
        # training step of a large 3-D head on an FPN level
        {"name": "head3d_train_f16", "kind": "head", "ndim": 3, "rotated": False, "train": True, "dtype": "f16",
         "batch": 2, "channels": 256, "d": 24, "h": 96, "w": 96, "rois": 4000, "low": 2.0, "high": 48.0,
         "scale": 0.25, "cells": 7, "ratio": 2},
        # training step of an image head at full precision, with the adaptive sampling grid that is the default
        {"name": "head2d_train_f32", "kind": "head", "ndim": 2, "rotated": False, "train": True, "dtype": "f32",
         "batch": 2, "channels": 256, "d": 1, "h": 200, "w": 304, "rois": 1000, "low": 16.0, "high": 256.0,
         "scale": 0.25, "cells": 7, "ratio": 0},
        # training step of a head with rotated boxes
        {"name": "head3d_rotated_train_f16", "kind": "head", "ndim": 3, "rotated": True, "train": True,
         "dtype": "f16", "batch": 2, "channels": 64, "d": 48, "h": 96, "w": 96, "rois": 1000, "low": 6.0,
         "high": 24.0, "scale": 1.0, "cells": 7, "ratio": 2},
        # inference of a modulated deformable layer on volumes
        {"name": "dcn3d_forward_f16", "kind": "dcn", "ndim": 3, "train": False, "dtype": "f16", "batch": 2,
         "cin": 32, "cout": 64, "d": 48, "h": 48, "w": 48, "kernel": 3, "stride": 1, "groups": 1, "spread": 2.0},
        # its training step
        {"name": "dcn3d_train_bf16", "kind": "dcn", "ndim": 3, "train": True, "dtype": "bf16", "batch": 2,
         "cin": 32, "cout": 64, "d": 48, "h": 48, "w": 48, "kernel": 3, "stride": 1, "groups": 1, "spread": 2.0},
        # training step of a modulated deformable layer of an image backbone
        {"name": "dcn2d_train_f16", "kind": "dcn", "ndim": 2, "train": True, "dtype": "f16", "batch": 8,
         "cin": 256, "cout": 256, "d": 1, "h": 100, "w": 152, "kernel": 3, "stride": 1, "groups": 1, "spread": 2.0},
    ]


# ---- more cases of the same ranges -------------------------------------------------------------------
def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_affine(rng):
    c = {"kind": "affine", "ndim": rng.choice([3, 3, 2]), "dtype": rng.choice(["f16", "f16", "f32", "f32", "bf16"])}
    if c["ndim"] == 3:   # one to eight volumes of one to four channels, up to 20 M voxels
        c.update(batch=_log(rng, 1, 8), channels=rng.choice([1, 1, 1, 2, 4]), d=_log(rng, 24, 192),
                 h=_log(rng, 32, 320), w=_log(rng, 32, 320))
    else:
        c.update(batch=_log(rng, 1, 16), channels=rng.choice([1, 3]), d=1, h=_log(rng, 64, 1024), w=_log(rng, 64, 1024))
    return c


def _draw_resize(rng):
    c = {"kind": "resize", "dtype": rng.choice(["f16", "f32"]), "batch": rng.choice([1, 2]), "d": _log(rng, 40, 256),
         "h": _log(rng, 128, 512)}
    c["w"] = c["h"] if rng.random() < 0.5 else _log(rng, 128, 512)
    plane = rng.uniform(0.4, 1.0)
    c.update(out_d=max(16, int(c["d"] * rng.uniform(0.5, 1.5))), out_h=max(16, int(c["h"] * plane)),
             out_w=max(16, int(c["w"] * plane)))
    return c


def _draw_augment(rng):
    c = {"kind": "augment", "dtype": rng.choice(["f16", "f32"]), "d": _log(rng, 64, 160), "h": _log(rng, 96, 280),
         "w": _log(rng, 96, 280), "factor": round(rng.uniform(0.6, 1.0), 3), "points": rng.choice([6, 7, 8, 10])}
    c["patch"] = max(16, int(min(c["d"], c["h"], c["w"]) * c["factor"] * rng.uniform(0.5, 0.95)))
    return c


def _draw_head(rng):
    c = {"kind": "head", "ndim": rng.choice([3, 3, 2]), "rotated": rng.random() < 0.3, "train": rng.random() < 0.6,
         "dtype": rng.choice(["f16", "f16", "f32", "f32", "bf16"]), "batch": rng.choice([1, 2, 4]),
         "ratio": rng.choice([0, 1, 2, 2])}
    if c["ndim"] == 3:
        c.update(channels=rng.choice([16, 32, 64, 128, 256]), d=_log(rng, 8, 64), h=_log(rng, 24, 128),
                 w=_log(rng, 24, 128), rois=_log(rng, 16, 4000), cells=rng.choice([4, 5, 7, 7]))
        c["scale"] = rng.choice([1.0, 0.5, 0.25])
        c.update(low=round(1.0 / c["scale"], 3), high=round(rng.uniform(8, 24) / c["scale"], 3))
    else:
        c.update(channels=rng.choice([64, 128, 256]), d=1, h=_log(rng, 25, 256), w=_log(rng, 25, 336),
                 rois=_log(rng, 16, 2000), cells=rng.choice([7, 7, 14]))
        c["scale"] = rng.choice([0.25, 0.125])
        c.update(low=round(3.0 / c["scale"], 3), high=round(rng.uniform(16, 64) / c["scale"], 3))
    return c


def _draw_dcn(rng):
    c = {"kind": "dcn", "ndim": rng.choice([3, 3, 2]), "train": rng.random() < 0.6,
         "dtype": rng.choice(["f16", "bf16", "f32"]), "batch": rng.choice([1, 2, 4]), "kernel": 3,
         "stride": rng.choice([1, 1, 1, 2]), "spread": round(rng.uniform(0.3, 3.0), 2)}
    if c["ndim"] == 3:
        c.update(cin=rng.choice([16, 32, 48, 64, 128]), cout=rng.choice([16, 32, 64, 128]), d=_log(rng, 6, 64),
                 h=_log(rng, 12, 64), w=_log(rng, 12, 64))
    else:
        c.update(cin=rng.choice([32, 64, 128, 256]), cout=rng.choice([64, 128, 256]), d=1, h=_log(rng, 16, 160),
                 w=_log(rng, 16, 240))
    c["groups"] = rng.choice([1, 1, 1, 2])   # deformable groups
    return c


def draw(rng):
    while True:
        maker = rng.choice([_draw_affine, _draw_affine, _draw_resize, _draw_augment, _draw_head, _draw_head, _draw_head,
                            _draw_dcn, _draw_dcn, _draw_dcn])
        c = maker(rng)
        if _cost(c) <= _MOST[c["kind"]]:
            return c


def _out_dims(c):
    """Spatial output size of a deformable layer (padding keeps the size at stride 1)."""
    half = c["kernel"] // 2
    dims = (c["d"], c["h"], c["w"]) if c["ndim"] == 3 else (c["h"], c["w"])
    return [(s + 2 * half - c["kernel"]) // c["stride"] + 1 for s in dims]


def _samples_per_roi(c):
    """Samples of one roi and channel, for the mean extent of the rois."""
    if c["ratio"] > 0:
        return (c["cells"] * c["ratio"]) ** c["ndim"]
    mean = (c["high"] - c["low"]) / math.log(c["high"] / c["low"]) * c["scale"]
    return (c["cells"] * max(1.0, math.ceil(mean / c["cells"]))) ** c["ndim"]


def _cost(c):
    """Rough size of a case among those of its kind: values interpolated."""
    kind = c["kind"]
    if kind == "affine":
        return c["batch"] * c["channels"] * c["d"] * c["h"] * c["w"]
    if kind == "resize":
        return c["batch"] * (c["d"] * c["h"] * c["w"] + c["out_d"] * c["out_h"] * c["out_w"])
    if kind == "augment":
        return c["d"] * c["h"] * c["w"]
    if kind == "head":   # a training step adds the backward pass; rotated boxes and 32-bit sums are the heavier ones
        weight = (3 if c["train"] else 1) * (2 if c["rotated"] else 1) * (1 if c["dtype"] == "f16" else 4)
        return weight * c["rois"] * c["channels"] * _samples_per_roi(c) + c["batch"] * c["channels"] * c["d"] * c["h"] * c["w"]
    taps = c["kernel"] ** c["ndim"]
    return (4 if c["train"] else 1) * c["batch"] * math.prod(_out_dims(c)) * c["cin"] * taps * 2 ** c["ndim"]


_MOST = {"affine": 20e6, "resize": 160e6, "augment": 9e6, "head": 8.6e9, "dcn": 6.2e9}


# ---- inputs --------------------------------------------------------------------------------------------
def _randn(shape, g, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _ct(shape, g, dtype):
    """Hounsfield-like values: air, soft tissue and bone."""
    u = torch.rand(shape, generator=g, device="cuda")
    n = torch.randn(shape, generator=g, device="cuda")
    v = torch.where(u < 0.3, torch.full_like(u, -1000.0), torch.where(u < 0.9, 40.0 + 30.0 * n, 700.0 + 200.0 * n))
    return v.to(dtype)


def _affine_rois(c, rng):
    """(b, centre, size, angles): RandomAffine's draws of +-30 degrees, 0.8 - 1.2 and +-8 % of the size."""
    size = np.array([c["w"], c["h"], c["d"]][:c["ndim"]], np.float64)
    rows = []
    for b in range(c["batch"]):
        centre = size / 2 + rng.uniform(-0.08, 0.08, c["ndim"]) * size
        angles = np.radians(rng.uniform(-30, 30, 3 if c["ndim"] == 3 else 1))
        rows.append([b, *centre, *(size / rng.uniform(0.8, 1.2)), *angles])
    return torch.tensor(np.array(rows, np.float32)).cuda()


def _head_rois(c, rng):
    """Proposals in the input's coordinates with log-uniform extents, inside the image."""
    n, nd = c["rois"], c["ndim"]
    size = np.array([c["w"], c["h"], c["d"]][:nd], np.float64) / c["scale"]
    extent = np.minimum(np.exp(rng.uniform(math.log(c["low"]), math.log(c["high"]), (n, nd))), size)
    index = rng.integers(0, c["batch"], (n, 1))
    low = rng.uniform(0, 1, (n, nd)) * (size - extent)
    if not c["rotated"]:
        rows = np.hstack([index, low, low + extent])
    else:
        angles = np.radians(rng.uniform(-30, 30, (n, 3 if nd == 3 else 1)))
        rows = np.hstack([index, low + extent / 2, extent, angles])
    return torch.tensor(rows.astype(np.float32)).cuda()


def prepare(case, seed):
    c, kind = case, case["kind"]
    dtype = DTYPES[c["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    s = {"kind": kind, "case": c}
    if kind == "affine":
        spatial = (c["d"], c["h"], c["w"])[3 - c["ndim"]:]
        s.update(x=_randn((c["batch"], c["channels"], *spatial), g, dtype), rois=_affine_rois(c, rng), size=spatial,
                 engine=ops.affine_3d if c["ndim"] == 3 else ops.affine_2d)
    elif kind == "resize":
        frame = [c["w"] / 2, c["h"] / 2, c["d"] / 2, c["w"], c["h"], c["d"], 0, 0, 0]
        s.update(x=_ct((c["batch"], 1, c["d"], c["h"], c["w"]), g, dtype), size=(c["out_d"], c["out_h"], c["out_w"]),
                 rois=torch.tensor([[b, *frame] for b in range(c["batch"])], dtype=torch.float32).cuda(),
                 engine=ops.affine_3d)
    elif kind == "augment":
        shape = (1, c["d"], c["h"], c["w"])
        s.update(img=_ct(shape, g, dtype), seed=seed % 2 ** 32,
                 seg=torch.randint(0, 3, shape, generator=g, device="cuda", dtype=torch.int32),
                 stages=[aug.CudaResize(factor=(c["factor"],) * 3), aug.CudaRandomAffine(1.0, 0.2, 0.1, 30),
                         aug.CudaRandomElasticDeformation(1.0, c["points"], 0.8),
                         aug.CudaCropRandomWithAffine((c["patch"],) * 3, 0.2, 0.1, 15)])
    elif kind == "head":
        cells = (c["cells"],) * c["ndim"]
        spatial = (c["d"], c["h"], c["w"])[3 - c["ndim"]:]
        layer = ops.RoIAlignRotated if c["rotated"] else ops.RoIAlign
        s.update(x=_randn((c["batch"], c["channels"], *spatial), g, dtype).requires_grad_(c["train"]),
                 rois=_head_rois(c, rng), layer=layer(cells, c["scale"], c["ratio"]))
        if c["train"]:
            s["grad"] = _randn((c["rois"], c["channels"], *cells), g, dtype)
    elif kind == "dcn":
        nd, taps = c["ndim"], c["kernel"] ** c["ndim"]
        cls = ops.ModulatedDeformConv3d if nd == 3 else ops.ModulatedDeformConv2d
        layer = cls(c["cin"], c["cout"], c["kernel"], stride=c["stride"], padding=c["kernel"] // 2,
                    deformable_groups=c["groups"]).cuda().to(dtype)
        bound = 1.0 / math.sqrt(c["cin"] * taps)
        with torch.no_grad():
            layer.weight.copy_((torch.rand(layer.weight.shape, generator=g, device="cuda") * 2 - 1) * bound)
            layer.bias.copy_((torch.rand(layer.bias.shape, generator=g, device="cuda") * 2 - 1) * bound)
        spatial = (c["d"], c["h"], c["w"])[3 - nd:]
        out = _out_dims(c)
        s.update(layer=layer, x=_randn((c["batch"], c["cin"], *spatial), g, dtype),
                 offset=_randn((c["batch"], c["groups"] * nd * taps, *out), g).mul_(c["spread"]).to(dtype),
                 mask=torch.sigmoid(_randn((c["batch"], c["groups"] * taps, *out), g)).to(dtype))
        if c["train"]:
            s["inputs"] = [s[k].requires_grad_() for k in ("x", "offset", "mask")] + [layer.weight, layer.bias]
            s["grad"] = _randn((c["batch"], c["cout"], *out), g, dtype)
    return s


# ---- one pass --------------------------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind in ("affine", "resize"):
        return s["engine"](s["x"], s["rois"], s["size"], 1.0, 1, True, 1)
    if kind == "augment":
        np.random.seed(s["seed"])   # the stages draw from numpy's generator
        sample = {"img": s["img"], "gt_seg": s["seg"], "img_dim": 3, "img_spacing": (1.0, 1.0, 1.0),
                  "img_fields": ["img"], "seg_fields": ["gt_seg"], "det_fields": []}
        for stage in s["stages"]:
            sample = stage(sample)
        return {"img": sample["img"], "gt_seg": sample["gt_seg"]}
    if kind == "head":
        if not s["case"]["train"]:
            with torch.no_grad():
                return s["layer"](s["x"], s["rois"])
        out = s["layer"](s["x"], s["rois"])
        return {"out": out, "grads": torch.autograd.grad(out, s["x"], s["grad"])}
    if not s["case"]["train"]:
        with torch.no_grad():
            return s["layer"](s["x"], s["offset"], s["mask"])
    out = s["layer"](s["x"], s["offset"], s["mask"])
    return {"out": out, "grads": torch.autograd.grad(out, s["inputs"], s["grad"])}


# ---- what a pass cannot do without -------------------------------------------------------------------------
def work(case):
    """Bytes: every input of the call read once, every output written once (the stages of a pipeline are calls
    of their own).  Operations: 2 * 2^ndim - 2 per interpolated value, two per product of a convolution."""
    c, kind = case, case["kind"]
    e = BYTES[c["dtype"]]
    if kind == "affine":
        n = c["batch"] * c["channels"] * c["d"] * c["h"] * c["w"]
        return {"bytes": 2 * n * e, "flops": (2 * 2 ** c["ndim"] - 2) * n}
    if kind == "resize":
        n = c["batch"] * c["out_d"] * c["out_h"] * c["out_w"]
        return {"bytes": (c["batch"] * c["d"] * c["h"] * c["w"] + n) * e, "flops": 14 * n}
    if kind == "augment":
        full = c["d"] * c["h"] * c["w"]
        small = math.prod(int(v * c["factor"]) for v in (c["d"], c["h"], c["w"]))
        crop = c["patch"] ** 3
        # resize, affine, warp (and its field of three fp32 components, once), crop
        values = (full + small) + 2 * small + 2 * small + 2 * crop
        return {"bytes": values * (e + 4) + small * 12, "flops": 14 * (3 * small + crop)}
    if kind == "head":
        features = c["batch"] * c["channels"] * c["d"] * c["h"] * c["w"]
        outs = c["rois"] * c["channels"] * c["cells"] ** c["ndim"]
        passes = 2 if c["train"] else 1
        return {"bytes": passes * (features + outs) * e, "flops": passes * (2 * 2 ** c["ndim"] - 2) * outs}
    taps, q = c["kernel"] ** c["ndim"], c["batch"] * math.prod(_out_dims(c))
    x, y = c["batch"] * c["cin"] * c["d"] * c["h"] * c["w"], c["cout"] * q
    aux, weights = c["groups"] * (c["ndim"] + 1) * taps * q, c["cout"] * c["cin"] * taps
    product = 2 * q * c["cout"] * c["cin"] * taps
    if not c["train"]:
        return {"bytes": (x + aux + weights + y) * e, "flops": product}
    return {"bytes": (3 * (x + aux + weights) + 2 * y) * e, "flops": 3 * product}


def tolerance(case):
    """16-bit results carry their own rounding and that of 16-bit operands; 32-bit ones the order of the sums."""
    rel = {"f16": 2e-3, "bf16": 1.2e-2, "f32": 1e-5}[case["dtype"]]
    if case["kind"] == "augment":   # a sample on the tie between two labels may go to either
        return {"rel": rel, "differ": 1e-3}
    return {"rel": rel}
