"""The workloads this library's speed is measured on.

Each case is one call, or one frame's share of calls, through a public entry
point of ``bfhip`` (the ctypes mirror of ``include/bf_cuda_*.h``), in the way a
program that serves six-camera + LiDAR frames makes it: contexts, plans and
output buffers are created once, inputs arrive on the GPU, and nothing is
copied back or waited for inside a pass.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` builds what a program has in hand before the call,
``run`` makes one pass, ``work`` says what the pass cannot do without,
``tolerance`` how far another correct implementation of the same precision may
be off, and ``exact`` computes the outputs in 64 bits with plain torch.
"""

import math
import os
import sys
import tempfile

import numpy as np
import torch

# The package folder of the tree this runs in (its root is the working folder).
sys.path.insert(0, os.path.join(os.getcwd(), "bevfusion.c_amd"))

import bfhip  # noqa: E402
from bfhip import bfw, frame_scene, lss_scene  # noqa: E402

DEV = "cuda:0"
F64 = torch.float64
IMAGE_H, IMAGE_W = 256, 704
GRID = (41, 1440, 1440)          # sparse encoder grid (z, y, x) of the frame runtime
CAPACITY = 160000                # voxel and sparse capacity of the frame runtime
POINT_CAPACITY = 300000
DEPTH_BINS, CONTEXT = 118, 80    # depth head outputs


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # Stateless linears (bf_cuda_gemm_f32).  One layer of the decoder's FFN
        # over 200 proposals: the smallest call, launch latency and host time.
        dict(name="linear_200x128x256", kind="linear", m=200, k=128, n=256, bias=True, relu=True),
        # Stage-1 QKV of one camera (64x176 tokens): a short reduction.
        dict(name="linear_11264x96x288", kind="linear", m=11264, k=96, n=288, bias=True,
             relu=False),
        # Stage-3 fc1 over six cameras' 16x44 tokens: a square-ish GEMM.
        dict(name="linear_4224x384x1536", kind="linear", m=4224, k=384, n=1536, bias=True,
             relu=False),
        # Stateless convolutions (bf_cuda_conv2d_f32).  The FPN's 3x3 at level 0
        # over six cameras.
        dict(name="conv3x3_6x256x32x88", kind="conv", batch=6, ci=256, co=256, h=32, w=88, k=3,
             stride=1, pad=1, transpose=False, bias=False, relu=True),
        # The BEV neck's transposed 2x2 upsampling of a 90x90 map.
        dict(name="deconv2x2_1x256x90x90", kind="conv", batch=1, ci=256, co=256, h=90, w=90, k=2,
             stride=2, pad=0, transpose=True, bias=True, relu=True),
        # Image backbone.  A two-camera thumbnail with odd merge grids and
        # padded windows: many launches on little data.
        dict(name="swin_2x56x112", kind="swin", cams=2, h=56, w=112),
        # The frame's six 256x704 images.
        dict(name="swin_6x256x704", kind="swin", cams=6, h=256, w=704),
        # Camera neck: FPN + depth head on the frame's three levels, and the
        # downsample of the pooled 360x360 map that follows the pooling.
        dict(name="neck_6x32x88", kind="neck", cams=6, h=32, w=88, bev_h=360, bev_w=360),
        # Lift-splat pooling of a frame whose calibration or augmentation
        # changed: cell lists from the calibration, then the pool.
        dict(name="lss_6x118x32x88", kind="lss", cams=6, bins=118, h=32, w=88, channels=80,
             gx=360, gy=360, gz=1),
        # BEV stage (fuser, SECOND, deblocks, shared conv, heatmap head).
        dict(name="bev_180x180", kind="bev", h=180, w=180),
        # TransFusion decoder, 200 proposals.
        dict(name="transfusion_180x180", kind="transfusion", h=180, w=180, proposals=200),
        # LiDAR side of a frame: depth images, voxels with means, sparse
        # encoder, on ten accumulated sweeps.
        dict(name="lidar_100000", kind="lidar", points=100000, sweeps=10),
    ]


def _log(rng, low, high):
    """A whole number, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _pick(rng, values):
    return values[rng.randrange(len(values))]


def draw(rng):
    kind = _pick(rng, ("linear", "linear", "conv", "conv", "swin", "neck", "lss", "bev",
                       "transfusion", "lidar"))
    if kind == "linear":
        while True:
            m, k, n = _log(rng, 1, 101376), _log(rng, 8, 3072), _log(rng, 3, 3072)
            if m * k * n <= 4224 * 384 * 1536 and m * (k + n) <= 4224 * (384 + 1536):
                break
        if rng.random() < 0.5:   # layer widths are mostly multiples of eight
            k, n = max(8, k // 8 * 8), max(8, n // 8 * 8)
        return dict(kind=kind, m=m, k=k, n=n, bias=rng.random() < 0.7, relu=rng.random() < 0.5)
    if kind == "conv":
        while True:
            transpose = rng.random() < 0.25
            k = 2 if transpose else _pick(rng, (1, 3, 3, 5))
            stride = 2 if transpose else _pick(rng, (1, 1, 2, 4 if k == 5 else 1))
            batch, ci, co = rng.randint(1, 6), _log(rng, 1, 512), _log(rng, 8, 512)
            h, w = _log(rng, 5, 256), _log(rng, 5, 704)
            if rng.random() < 0.5:
                ci, co = max(8, ci // 8 * 8), co // 8 * 8
            pad = 0 if transpose else k // 2
            c = dict(kind=kind, batch=batch, ci=ci, co=co, h=h, w=w, k=k, stride=stride, pad=pad,
                     transpose=transpose, bias=rng.random() < 0.5, relu=rng.random() < 0.5)
            oh, ow = _conv_out(c)
            limit = 6 * 32 * 88
            if (work(c)["flops"] <= 2 * limit * 256 * 256 * 9 and batch * h * w * ci <= limit * 512
                    and batch * oh * ow * co <= limit * 512):
                return c
    if kind == "swin":
        return dict(kind=kind, cams=rng.randint(1, 6), h=4 * _log(rng, 8, 64),
                    w=4 * _log(rng, 12, 176))
    if kind == "neck":
        return dict(kind=kind, cams=rng.randint(1, 6), h=_log(rng, 2, 32), w=_log(rng, 3, 88),
                    bev_h=2 * _log(rng, 4, 180), bev_w=2 * _log(rng, 4, 180))
    if kind == "lss":
        channels = _pick(rng, (80, 80, 64, 32, _log(rng, 3, 80)))
        return dict(kind=kind, cams=rng.randint(1, 6), bins=_log(rng, 4, 118), h=_log(rng, 3, 32),
                    w=_log(rng, 5, 88), channels=channels, gx=_log(rng, 20, 360),
                    gy=_log(rng, 20, 360), gz=1)
    if kind == "bev":
        return dict(kind=kind, h=2 * _log(rng, 4, 90), w=2 * _log(rng, 4, 90))
    if kind == "transfusion":
        h, w = _log(rng, 8, 180), _log(rng, 8, 180)
        return dict(kind=kind, h=h, w=w, proposals=_log(rng, 20, 200))
    return dict(kind=kind, points=_log(rng, 2000, 100000), sweeps=_pick(rng, (1, 5, 10)))


# ------------------------------------------------------------ seeded material
def _gen(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed(bfw.stream_key(seed, name) & 0x7FFFFFFFFFFFFFFF)
    return g


def _randn(seed, name, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=_gen(seed, name), device=DEV) * std + mean


def _rand(seed, name, shape, low=0.0, high=1.0):
    return torch.rand(shape, generator=_gen(seed, name), device=DEV) * (high - low) + low


class _Weights(bfw._Init):
    """Fan-in initialised layers, so that every layer's output stays O(1), the
    large ones drawn on the GPU."""

    def __init__(self, seed, gain):
        super().__init__(seed, "fan_in", gain)

    def weight(self, name, shape, fan_in):
        return _randn(self.seed, name, shape, self.gain / math.sqrt(fan_in)).cpu().numpy()


_TENSORS = {"swin": (bfw.swin_tensors, 1.0), "neck": (bfw.neck_tensors, 1.0),
            "bev": (bfw.bev_stage_tensors, 1.4), "transfusion": (bfw.transfusion_tensors, 1.0),
            "lidar": (bfw.lidar_backbone_tensors, 1.2)}


def _tensors(kind, seed):
    make, gain = _TENSORS[kind]
    return make(_Weights(seed, gain))


def _with_model(kind, seed, create):
    """create(model) on a checkpoint of this seed's weights."""
    with tempfile.TemporaryDirectory(prefix="cases_") as d:
        path = os.path.join(d, "m.bfw")
        bfw.write_bfw(_tensors(kind, seed), path)
        with bfhip.Model(path) as m:
            return create(m)


def _conv_out(c):
    if c["transpose"]:
        return tuple((v - 1) * c["stride"] - 2 * c["pad"] + c["k"] for v in (c["h"], c["w"]))
    return tuple((v + 2 * c["pad"] - c["k"]) // c["stride"] + 1 for v in (c["h"], c["w"]))


def _swin_levels(cams, h, w):
    """The three NCHW levels of an h x w feature grid, as the neck takes them."""
    h1, w1 = (h + 1) // 2, (w + 1) // 2
    return [(cams, 192, h, w), (cams, 384, h1, w1), (cams, 768, (h1 + 1) // 2, (w1 + 1) // 2)]


def _inputs(case, seed):
    """The call's input tensors, on the GPU, by name."""
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        t = dict(x=_randn(seed, "x", (m, k)), w=_randn(seed, "w", (n, k), k ** -0.5))
        return dict(t, b=_randn(seed, "b", (n,), 0.1) if case["bias"] else None)
    if kind == "conv":
        ci, co, k = case["ci"], case["co"], case["k"]
        shape = (ci, co, k, k) if case["transpose"] else (co, ci, k, k)
        fan = ci if case["transpose"] else ci * k * k
        t = dict(x=_randn(seed, "x", (case["batch"], ci, case["h"], case["w"])),
                 w=_randn(seed, "w", shape, fan ** -0.5))
        return dict(t, b=_randn(seed, "b", (co,), 0.1) if case["bias"] else None)
    if kind == "swin":
        # pixels in [0, 1], normalised with the ImageNet mean and deviation
        img = _rand(seed, "images", (case["cams"], 3, case["h"], case["w"]))
        mean = torch.tensor(bfw.IMAGENET_MEAN, device=DEV).view(1, 3, 1, 1)
        std = torch.tensor(bfw.IMAGENET_STD, device=DEV).view(1, 3, 1, 1)
        return dict(images=((img - mean) / std).contiguous())
    if kind == "neck":
        cams, h, w = case["cams"], case["h"], case["w"]
        levels = [_randn(seed, f"s{i}", s) for i, s in enumerate(_swin_levels(cams, h, w))]
        # a LiDAR return of 1-60 m in one pixel of twenty, zero elsewhere
        hit = _rand(seed, "hit", (cams, 1, 8 * h, 8 * w)) < 0.05
        depth = torch.where(hit, _rand(seed, "depth", hit.shape, 1.0, 60.0), 0.0)
        bev = _randn(seed, "bev", (1, CONTEXT, case["bev_h"], case["bev_w"]))
        return dict(s0=levels[0], s1=levels[1], s2=levels[2], depth=depth.contiguous(), bev=bev)
    if kind == "lss":
        n, d, h, w, c = (case[k] for k in ("cams", "bins", "h", "w", "channels"))
        scene = lss_scene.rig(0, 1, 1, 1, 1)   # the surround rig's calibration
        rng = np.random.default_rng(seed)
        yaw = rng.uniform(-0.3, 0.3)
        scene["extra_rotation"] = lss_scene._rot_z(yaw).reshape(1, 3, 3)
        scene["extra_translation"] = rng.uniform(-0.5, 0.5, (1, 3)).astype(np.float32)
        t = {}
        for key in lss_scene.CALIBRATION_KEYS:
            a = scene[key] if key.startswith("extra") else scene[key][:, :n]
            t[key] = torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV)
        xs = np.linspace(0, IMAGE_W - 1, w, dtype=np.float32)
        ys = np.linspace(0, IMAGE_H - 1, h, dtype=np.float32)
        ds = (1.0 + np.arange(d) * np.float32(59.0 / d)).astype(np.float32)
        f = np.stack(np.broadcast_arrays(xs.reshape(1, 1, w), ys.reshape(1, h, 1),
                                         ds.reshape(d, 1, 1)), -1)
        t["frustum"] = torch.from_numpy(np.ascontiguousarray(f, np.float32)).to(DEV)
        t["logits"] = _randn(seed, "logits", (1, n, d, h, w), 2.0)
        t["context"] = _randn(seed, "context", (1, n, c, h, w))
        return t
    if kind == "bev":
        # two post-ReLU maps, a third of the cells without any input
        x = _randn(seed, "bev", (1, 336, case["h"], case["w"])).relu()
        return dict(x=(x * (_rand(seed, "cells", (1, 1, case["h"], case["w"])) > 0.33)).contiguous())
    if kind == "transfusion":
        h, w = case["h"], case["w"]
        # a quiet background and 3x3 peaks where objects stand
        heat = _randn(seed, "heat", (1, 10, h, w), 0.8, -4.5)
        objects = max(1, h * w // 270)
        flat = (_rand(seed, "at", (objects,)) * (10 * h * w)).long().clamp_(max=10 * h * w - 1)
        peak = torch.zeros(10 * h * w, device=DEV)
        peak[flat] = 4.0
        peak = torch.nn.functional.max_pool2d(peak.view(1, 10, h, w), 3, 1, 1)
        return dict(shared=_randn(seed, "shared", (1, 128, h, w)),
                    heatmap=(heat + peak * _rand(seed, "height", (1, 10, h, w), 0.8, 1.5)).contiguous())
    pts = bfw.synthetic_points(seed, case["points"], sweeps=case["sweeps"])
    cal = frame_scene.calibration(seed)
    t = {k: torch.from_numpy(cal[k]).to(DEV)
         for k in ("lidar_augmentation", "lidar_to_image", "image_augmentation")}
    return dict(t, points=torch.from_numpy(pts).to(DEV))


def _lss_desc(case):
    return bfhip.lss_desc(1, case["cams"], case["bins"], case["h"], case["w"], case["channels"],
                          *_lss_grid(case))


def _lss_grid(case):
    cells = (case["gx"], case["gy"], case["gz"])
    return ((-54.0, -54.0, -10.0), (108.0 / cells[0], 108.0 / cells[1], 20.0 / cells[2]), cells)


# ----------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind, s = case["kind"], dict(_inputs(case, seed), case=case)
    empty = lambda *shape: torch.zeros(shape, device=DEV)  # noqa: E731
    if kind == "linear":
        s["out"] = empty(case["m"], case["n"])
    elif kind == "conv":
        s["out"] = empty(case["batch"], case["co"], *_conv_out(case))
    elif kind == "swin":
        s["net"] = _with_model(kind, seed, lambda m: bfhip.Swin(m, case["cams"], case["h"], case["w"]))
        s["outs"] = [empty(*shape) for shape in s["net"].output_shapes()]
    elif kind == "neck":
        cams, h, w = case["cams"], case["h"], case["w"]
        s["net"] = _with_model(kind, seed, lambda m: bfhip.CameraNeck(
            m, cams, h, w, case["bev_h"], case["bev_w"]))
        s["outs"] = (empty(cams, DEPTH_BINS, h, w), empty(cams, CONTEXT, h, w),
                     empty(1, CONTEXT, case["bev_w"] // 2, case["bev_h"] // 2))
    elif kind == "lss":
        s["plan"] = bfhip.LssPlan(_lss_desc(case))
        s["out"] = empty(1, case["channels"] * case["gz"], case["gx"], case["gy"])
    elif kind == "bev":
        s["net"] = _with_model(kind, seed, lambda m: bfhip.BevStage(m, case["h"], case["w"]))
        s["outs"] = tuple(empty(1, c, case["h"], case["w"]) for c in (512, 128, 10))
    elif kind == "transfusion":
        s["net"] = _with_model(kind, seed, lambda m: bfhip.TransFusion(
            m, case["h"], case["w"], case["proposals"]))
        s["outs"] = s["net"].outputs(DEV)
    else:
        s["raster"] = bfhip.DepthRaster(POINT_CAPACITY, 6, IMAGE_H, IMAGE_W)
        s["vox"] = bfhip.Voxelizer(bfhip.voxel_config(CAPACITY), POINT_CAPACITY)
        s["net"] = _with_model(kind, seed, lambda m: bfhip.LidarBackbone(m, 1, *GRID, CAPACITY))
        s["depth"] = empty(6, IMAGE_H, IMAGE_W)
        s["coords"] = torch.zeros((CAPACITY, 4), dtype=torch.int32, device=DEV)
        s["means"] = empty(CAPACITY, 5)
        s["count"] = torch.zeros(1, dtype=torch.int32, device=DEV)
        s["bev"] = empty(*s["net"].out_shape)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return bfhip.gemm_f32(s["x"], s["w"], s["b"], case["relu"], out=s["out"])
    if kind == "conv":
        st, pad = case["stride"], case["pad"]
        return bfhip.conv2d_f32(s["x"], s["w"], s["b"], (st, st), (pad, pad), case["transpose"],
                                case["relu"], out=s["out"])
    if kind == "swin":
        return s["net"].forward(s["images"], s["outs"])
    if kind == "neck":
        logits, ctx, down = s["outs"]
        s["net"].neck_forward(s["s0"], s["s1"], s["s2"], s["depth"], logits, ctx)
        s["net"].downsample_forward(s["bev"], down)
        return dict(logits=logits, context=ctx, downsample=down)
    if kind == "lss":
        s["plan"].prepare_calibration(s["frustum"], *(s[k] for k in lss_scene.CALIBRATION_KEYS))
        return s["plan"].forward(s["logits"], s["context"], s["out"])
    if kind == "bev":
        spatial, shared, heatmap = s["net"].forward(s["x"], s["outs"])
        return dict(spatial=spatial, shared=shared, heatmap=heatmap)
    if kind == "transfusion":
        return s["net"].forward(s["shared"], s["heatmap"], s["outs"])
    s["raster"].forward(s["points"], s["lidar_augmentation"], s["lidar_to_image"],
                        s["image_augmentation"], out=s["depth"])
    s["vox"].forward(s["points"], s["coords"], s["means"], s["count"])
    s["net"].forward(s["coords"], s["means"], s["count"], out=s["bev"])
    return {k: s[k] for k in ("depth", "coords", "means", "count", "bev")}


# --------------------------------------------------------- work and tolerance
_SWIN = tuple(zip((96, 192, 384, 768), (2, 2, 6, 2)))


def work(case):
    """Inputs read once and outputs written once (32-bit tensors at the
    interface, weights a context holds at 16 bits), and the multiply-adds of
    the layers."""
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4 * (m * k + n * k + m * n), flops=2 * m * k * n)
    if kind == "conv":
        oh, ow = _conv_out(case)
        n, ci, co, k = case["batch"], case["ci"], case["co"], case["k"]
        at = n * (case["h"] * case["w"] if case["transpose"] else oh * ow)
        return dict(bytes=4 * (n * ci * case["h"] * case["w"] + ci * co * k * k + n * co * oh * ow),
                    flops=2 * at * ci * co * k * k)
    if kind == "swin":
        b, h, w = case["cams"], case["h"] // 4, case["w"] // 4
        flops, params = 2 * b * h * w * 48 * 96, 48 * 96
        size = b * 3 * 16 * h * w
        for s, (c, depth) in enumerate(_SWIN):
            t = b * h * w
            flops += depth * t * (2 * 12 * c * c + 4 * 49 * c)
            params += depth * 12 * c * c
            size += t * c if s else 0
            if s < 3:
                h, w = (h + 1) // 2, (w + 1) // 2
                flops += 2 * b * h * w * 8 * c * c
                params += 8 * c * c
        return dict(bytes=4 * size + 2 * params, flops=flops)
    if kind == "neck":
        n, h, w = case["cams"], case["h"], case["w"]
        (_, _, h1, w1), (_, _, h2, w2) = _swin_levels(n, h, w)[1:]
        # the laterals' upper halves act before the upsampling (both linear)
        flops = 2 * n * (h2 * w2 * 768 * 256 + h1 * w1 * (384 * 256 + 9 * 256 * 256 + 256 * 256)
                         + h * w * (192 * 256 + 9 * 256 * 256))
        flops += 2 * n * (64 * h * w * 8 + 4 * h * w * 25 * 8 * 32 + h * w * 25 * 32 * 64)
        flops += 2 * n * h * w * (9 * 320 * 256 + 9 * 256 * 256 + 256 * 198)
        cells = case["bev_h"] * case["bev_w"]
        flops += 2 * cells * 9 * CONTEXT * CONTEXT * 3 // 2
        size = n * (192 * h * w + 384 * h1 * w1 + 768 * h2 * w2 + 64 * h * w + 198 * h * w)
        params = 448 * 256 + 1152 * 256 + 9 * 256 * (256 * 2 + 320 + 256) + 198 * 256 + 25 * 2304 \
            + 27 * CONTEXT * CONTEXT
        return dict(bytes=4 * (size + CONTEXT * cells * 5 // 4) + 2 * params, flops=flops)
    if kind == "lss":
        pixels = case["cams"] * case["h"] * case["w"]
        samples, c = pixels * case["bins"], case["channels"]
        cells = case["gx"] * case["gy"] * case["gz"]
        return dict(bytes=4 * (samples + pixels * c + cells * c + 3 * samples // case["cams"]),
                    flops=2 * samples * c)
    if kind == "bev":
        cells = case["h"] * case["w"]
        per = 9 * (336 * 256 + 256 * 128 + 5 * 128 * 128) + 128 * 256
        low = 9 * (128 * 256 + 5 * 256 * 256) + 4 * 256 * 256
        head = 9 * (512 * 128 + 128 * 128 + 128 * 10)
        return dict(bytes=4 * cells * (336 + 512 + 128 + 10) + 2 * (per + low + head),
                    flops=2 * cells * (per + head) + 2 * (cells // 4) * low)
    if kind == "transfusion":
        keys, p = case["h"] * case["w"], case["proposals"]
        flops = 2 * keys * (2 * 128 + 3 * 128 * 128) + 4 * p * keys * 128 + 4 * p * p * 128
        flops += 2 * p * (10 * 128 * 128 + 2 * 128 * 256 + 6 * 128 * 64 + 20 * 64)
        return dict(bytes=4 * (keys * 138 + p * 34), flops=flops)
    coords = _voxels(bfw.synthetic_points(0, case["points"], sweeps=case["sweeps"]))[0]
    flops, params = _lidar_flops(coords)
    out = 6 * IMAGE_H * IMAGE_W + 256 * 180 * 180 + 9 * len(coords)
    return dict(bytes=4 * (5 * case["points"] + out) + 2 * params, flops=flops)


def tolerance(case):
    """About four times what the present path is off from 64 bits at its worst
    over the ranges: bf16 operands in the stateless operators, fp16 operands
    chained over the layers of the backbone, neck and BEV stage, 32-bit sums in
    the pooling and the sparse encoder (which splits its operands in two)."""
    return {"linear": dict(rel=1e-2), "conv": dict(rel=1e-2), "swin": dict(rel=5e-3),
            "neck": dict(rel=3e-3), "lss": dict(rel=3e-6, max=3e-4), "bev": dict(rel=6e-3),
            "transfusion": dict(rel=3e-3), "lidar": dict(rel=8e-6, max=1e-3)}[case["kind"]]


# ------------------------------------------------------- the results in 64 bits
def _conv64(x, w, b=None, stride=1, pad=0):
    """NCHW convolution in 64 bits, one matrix product per tap."""
    w = w.to(DEV, F64)
    k = w.shape[2:]
    oh, ow = ((x.shape[2 + i] + 2 * pad - k[i]) // stride + 1 for i in (0, 1))
    x = torch.nn.functional.pad(x.to(DEV, F64), (pad, pad, pad, pad))
    out = torch.zeros((x.shape[0], w.shape[0], oh, ow), dtype=F64, device=DEV)
    for n in range(x.shape[0]):
        for i in range(k[0]):
            for j in range(k[1]):
                tap = x[n, :, i:i + stride * (oh - 1) + 1:stride, j:j + stride * (ow - 1) + 1:stride]
                out[n] += (w[:, :, i, j] @ tap.reshape(tap.shape[0], -1)).view(-1, oh, ow)
    return out if b is None else out + b.to(DEV, F64).view(1, -1, 1, 1)


def _deconv64(x, w, b, stride, pad):
    """Transposed convolution in 64 bits (weights [in, out, k, k])."""
    x, w = x.to(F64), w.to(DEV, F64)
    n, _, h, wd = x.shape
    k = w.shape[2]
    full = torch.zeros((n, w.shape[1], (h - 1) * stride + k, (wd - 1) * stride + k), dtype=F64,
                       device=DEV)
    for i in range(k):
        for j in range(k):
            tap = (w[:, :, i, j].t().contiguous() @ x.reshape(n, x.shape[1], -1)).view(n, -1, h, wd)
            full[:, :, i:i + stride * (h - 1) + 1:stride, j:j + stride * (wd - 1) + 1:stride] += tap
    out = full[:, :, pad:full.shape[2] - pad, pad:full.shape[3] - pad]
    return out if b is None else out + b.to(DEV, F64).view(1, -1, 1, 1)


class _Params:
    """The checkpoint's tensors by name, in 64 bits on the GPU."""

    def __init__(self, kind, seed):
        self.t = dict(_tensors(kind, seed))

    def __getitem__(self, name):
        return torch.from_numpy(self.t[name]).to(DEV, F64)

    def bn(self, x, name, eps):
        v = [self[f"{name}.{k}"].view(1, -1, *[1] * (x.dim() - 2))
             for k in ("weight", "bias", "running_mean", "running_var")]
        return (x - v[2]) / torch.sqrt(v[3] + eps) * v[0] + v[1]

    def cbr(self, x, w, bn, stride=1, pad=0, bias=None, relu=True, eps=1e-5):
        y = _conv64(x, self[w], None if bias is None else self[bias], stride, pad)
        y = self.bn(y, bn, eps) if bn else y
        return y.relu() if relu else y

    def norm(self, x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], self[name + ".weight"],
                                              self[name + ".bias"], 1e-5)

    def linear(self, x, w, b):
        return x @ self[w].t() + self[b]


def _window_attention64(p, q, x, heads, shift):
    """Shifted-window attention of [B, H, W, C]: pad, roll, mask, softmax."""
    b, h, w, c = x.shape
    hp, wp = -(-h // 7) * 7, -(-w // 7) * 7
    x = torch.nn.functional.pad(x, (0, 0, 0, wp - w, 0, hp - h))
    label = torch.zeros((hp, wp), device=DEV)
    if shift:
        x = torch.roll(x, (-shift, -shift), (1, 2))
        row = (torch.arange(hp, device=DEV) >= hp - 7).long() + (torch.arange(hp, device=DEV) >= hp - shift).long()
        col = (torch.arange(wp, device=DEV) >= wp - 7).long() + (torch.arange(wp, device=DEV) >= wp - shift).long()
        label = row[:, None] * 3 + col[None]
    cut = lambda v, n: v.view(n, hp // 7, 7, wp // 7, 7, -1).transpose(2, 3).reshape(  # noqa: E731
        -1, 49, v.shape[-1] if v.dim() == 4 else 1)
    region = cut(label.view(1, hp, wp, 1), 1)[:, :, 0]
    mask = (region[:, :, None] != region[:, None, :]).to(F64) * -100.0
    win = cut(x, b)
    qkv = p.linear(win, q + "attn.w_msa.qkv.weight", q + "attn.w_msa.qkv.bias")
    qkv = qkv.view(-1, 49, 3, heads, c // heads).permute(2, 0, 3, 1, 4).contiguous()
    table = p[q + "attn.w_msa.relative_position_bias_table"]
    index = torch.from_numpy(bfw.relative_position_index(7)).to(DEV)
    bias = table[index.reshape(-1)].view(49, 49, heads).permute(2, 0, 1)
    score = (qkv[0] * (c // heads) ** -0.5) @ qkv[1].transpose(-1, -2).contiguous() + bias
    score = score + mask.repeat(b, 1, 1)[:, None]
    y = (score.softmax(-1) @ qkv[2]).transpose(1, 2).reshape(-1, 49, c)
    y = p.linear(y, q + "attn.w_msa.proj.weight", q + "attn.w_msa.proj.bias")
    y = y.view(b, hp // 7, wp // 7, 7, 7, c).transpose(2, 3).reshape(b, hp, wp, c)
    if shift:
        y = torch.roll(y, (shift, shift), (1, 2))
    return y[:, :h, :w]


def _swin64(p, images):
    pre = "image_backbone."
    x = _conv64(images, p[pre + "patch_embed.projection.weight"],
                p[pre + "patch_embed.projection.bias"], 4).permute(0, 2, 3, 1)
    x = p.norm(x, pre + "patch_embed.norm")
    outs = []
    for s, (c, depth) in enumerate(_SWIN):
        for k in range(depth):
            q = f"{pre}stages.{s}.blocks.{k}."
            x = x + _window_attention64(p, q, p.norm(x, q + "norm1"), c // 32, 3 if k % 2 else 0)
            y = p.linear(p.norm(x, q + "norm2"), q + "ffn.layers.0.0.weight", q + "ffn.layers.0.0.bias")
            x = x + p.linear(torch.nn.functional.gelu(y), q + "ffn.layers.1.weight",
                             q + "ffn.layers.1.bias")
        if s:
            outs.append(p.norm(x, f"{pre}norm{s}").permute(0, 3, 1, 2).contiguous())
        if s < 3:
            q = f"{pre}stages.{s}.downsample."
            b, h, w, _ = x.shape
            x = torch.nn.functional.pad(x, (0, 0, 0, w % 2, 0, h % 2))
            # unfold order: channel, then tap (ky, kx)
            x = torch.stack([x[:, i::2, j::2] for i in (0, 1) for j in (0, 1)], -1).flatten(3)
            x = p.norm(x, q + "norm") @ p[q + "reduction.weight"].t()
    return outs


def _neck64(p, t):
    up = lambda x, like: torch.nn.functional.interpolate(  # noqa: E731
        x, size=like.shape[2:], mode="bilinear", align_corners=False)
    s0, s1, s2 = (t[k].to(F64) for k in ("s0", "s1", "s2"))
    n = "neck."
    x = p.cbr(torch.cat([s1, up(s2, s1)], 1), n + "lateral_convs.1.conv.weight", n + "lateral_convs.1.bn")
    x = p.cbr(x, n + "fpn_convs.1.conv.weight", n + "fpn_convs.1.bn", pad=1)
    x = p.cbr(torch.cat([s0, up(x, s0)], 1), n + "lateral_convs.0.conv.weight", n + "lateral_convs.0.bn")
    x = p.cbr(x, n + "fpn_convs.0.conv.weight", n + "fpn_convs.0.bn", pad=1)
    v = "vtransform."
    d = t["depth"]
    for conv, stride, pad in ((0, 1, 0), (3, 4, 2), (6, 2, 2)):
        d = p.cbr(d, f"{v}dtransform.{conv}.weight", f"{v}dtransform.{conv + 1}", stride, pad,
                  f"{v}dtransform.{conv}.bias")
    x = torch.cat([d, x], 1)
    for conv in (0, 3):
        x = p.cbr(x, f"{v}depthnet.{conv}.weight", f"{v}depthnet.{conv + 1}", 1, 1,
                  f"{v}depthnet.{conv}.bias")
    x = p.cbr(x, v + "depthnet.6.weight", None, bias=v + "depthnet.6.bias", relu=False)
    y = t["bev"]
    for conv, stride in ((0, 1), (3, 2), (6, 1)):
        y = p.cbr(y, f"{v}downsample.{conv}.weight", f"{v}downsample.{conv + 1}", stride, 1)
    return dict(logits=x[:, :DEPTH_BINS], context=x[:, DEPTH_BINS:], downsample=y.transpose(2, 3))


def _inverse3(m):
    """Cofactor inverses of [n, 3, 3] in the stated precision's own order."""
    a, b, c, d, e, f, g, h, i = (m[:, r, s] for r in range(3) for s in range(3))
    adj = [e * i - f * h, c * h - b * i, b * f - c * e, f * g - d * i, a * i - c * g, c * d - a * f,
           d * h - e * g, b * g - a * h, a * e - b * d]
    one = np.float32(1.0) / (a * adj[0] + b * adj[3] + c * adj[6])
    return np.stack([v * one for v in adj], -1).reshape(-1, 3, 3)


def _apply3(m, v):
    """Row sums left to right of m [n, 3, 3] on three arrays [n, ...]."""
    col = lambda r, s: m[:, r, s].reshape(-1, *[1] * (v[0].ndim - 1))  # noqa: E731
    return [col(r, 0) * v[0] + col(r, 1) * v[1] + col(r, 2) * v[2] for r in range(3)]


def _lss_cells(case, t):
    """The cell of every sample, -1 outside: a decision, so taken with the
    32-bit operations the interface defines (transform, then truncation)."""
    g = {k: t[k].cpu().numpy() for k in lss_scene.CALIBRATION_KEYS}
    f = t["frustum"].cpu().numpy()[None]
    n = case["cams"]
    wide = lambda v: v.reshape(n, -1, 1, 1, 1)  # noqa: E731
    post = wide(g["post_translation"][0])
    with np.errstate(all="ignore"):
        u = _apply3(_inverse3(g["post_rotation"][0]), [f[..., k] - post[:, k] for k in range(3)])
        q = [u[0] * u[2], u[1] * u[2], u[2]]
        k_inv, rot = _inverse3(g["intrinsics"][0]), g["camera_rotation"][0]
        comb = np.zeros((n, 3, 3), np.float32)
        for k in range(3):
            comb = comb + rot[:, :, k, None] * k_inv[:, None, k, :]
        move = wide(g["camera_translation"][0])
        l = [a + move[:, k] for k, a in enumerate(_apply3(comb, q))]
        l = _apply3(np.repeat(g["extra_rotation"], n, 0), l)
        l = [a + g["extra_translation"][0, k] for k, a in enumerate(l)]
        minimum, step, cells = _lss_grid(case)
        ok, c = True, []
        for k in range(3):
            v = (l[k] - np.float32(minimum[k])) / np.float32(step[k])
            v = np.where(np.isfinite(v) & (np.abs(v) < 1e9), v, np.float32(-1e6)).astype(np.int64)
            ok = ok & (v >= 0) & (v < cells[k])
            c.append(v)
    rank = (c[2] * cells[0] + c[0]) * cells[1] + c[1]
    return torch.from_numpy(np.where(ok, rank, -1)).to(DEV)


def _lss64(case, t):
    cell = _lss_cells(case, t)
    prob = t["logits"][0].to(F64).softmax(1)
    ctx = t["context"][0].to(F64)
    out = torch.zeros((case["gx"] * case["gy"] * case["gz"], case["channels"]), dtype=F64, device=DEV)
    for n in range(case["cams"]):
        live = cell[n] >= 0
        row = (prob[n][..., None] * ctx[n].permute(1, 2, 0))[live]
        out.index_add_(0, cell[n][live], row)
    gz = case["gz"]
    out = out.view(gz, case["gx"], case["gy"], -1).permute(3, 0, 1, 2)
    return out.reshape(1, -1, case["gx"], case["gy"])


def _bev64(p, x):
    for name, bn in [("fuser.conv.0", "fuser.conv.1")] + [
            (f"backbone_2d.blocks.0.{3 * k + 1}", f"backbone_2d.blocks.0.{3 * k + 2}") for k in range(6)]:
        x = p.cbr(x, name + ".weight", bn, 1, 1, eps=1e-3)
    up0 = p.cbr(x, "backbone_2d.deblocks.0.0.weight", "backbone_2d.deblocks.0.1", eps=1e-3)
    for k in range(6):
        x = p.cbr(x, f"backbone_2d.blocks.1.{3 * k + 1}.weight", f"backbone_2d.blocks.1.{3 * k + 2}",
                  1 if k else 2, 1, eps=1e-3)
    up1 = p.bn(_deconv64(x, p["backbone_2d.deblocks.1.0.weight"], None, 2, 0),
               "backbone_2d.deblocks.1.1", 1e-3).relu()
    spatial = torch.cat([up0, up1], 1)
    d = "dense_head."
    shared = p.cbr(spatial, d + "shared_conv.weight", None, 1, 1, d + "shared_conv.bias", False)
    heat = p.cbr(shared, d + "heatmap_head.0.conv.weight", d + "heatmap_head.0.bn", 1, 1, eps=1e-3)
    heat = p.cbr(heat, d + "heatmap_head.1.weight", None, 1, 1, d + "heatmap_head.1.bias", False)
    return dict(spatial=spatial, shared=shared, heatmap=heat)


def _proposals(heatmap, count):
    """(scores, flat indices) of the proposals: 32-bit two-branch logistic with
    a correctly rounded exponential, 3x3 maxima (classes 8 and 9 exempt, no
    others on the border), highest score first, ties by index."""
    x = heatmap[0].to(F64)
    e = torch.exp(-x.abs()).float()
    score = torch.where(x >= 0, 1.0 / (1.0 + e), e / (1.0 + e))
    local = torch.full_like(score, math.inf)
    if min(score.shape[1:]) > 2:
        local[:, 1:-1, 1:-1] = torch.nn.functional.max_pool2d(score[None], 3, 1)[0]
    local[8:] = score[8:]
    score = torch.where(score == local, score, 0.0).reshape(-1)
    at = torch.sort(score, descending=True, stable=True).indices[:count]
    return score, at


def _transfusion64(p, t, case):
    h, w, count = case["h"], case["w"], case["proposals"]
    keys = h * w
    score, at = _proposals(t["heatmap"], count)
    label, index = at // keys, at % keys
    feat = t["shared"][0].to(F64).reshape(128, keys).t()
    d, head = "dense_head.decoder.", "dense_head.prediction_head."
    conv = lambda x, name: x @ p[name + ".weight"][:, :, 0].t() + p[name + ".bias"]  # noqa: E731
    query = feat[index] + p["dense_head.class_encoding.weight"][:, :, 0].t()[label] \
        + p["dense_head.class_encoding.bias"]

    def posembed(name, cells):
        q = f"{d}{name}.position_embedding_head."
        xy = torch.stack([cells % w, cells // w], 1).to(F64) + 0.5
        return conv(p.bn(conv(xy, q + "0"), q + "1", 1e-5).relu(), q + "3")

    def attend(name, q, kv):
        weight, bias = p[f"{d}{name}.in_proj_weight"], p[f"{d}{name}.in_proj_bias"]
        part = [(x @ weight[128 * i:128 * i + 128].t() + bias[128 * i:128 * i + 128]).view(-1, 8, 16)
                .transpose(0, 1).contiguous() for i, x in enumerate((q, kv, kv))]
        prob = (part[0] * 0.25 @ part[1].transpose(1, 2).contiguous()).softmax(-1)
        out = (prob @ part[2]).transpose(0, 1).reshape(-1, 128)
        return p.linear(out, f"{d}{name}.out_proj.weight", f"{d}{name}.out_proj.bias")

    pos = posembed("self_posembed", index)
    both = query + pos
    query = p.norm(query + attend("self_attn", both, both), d + "norm1")
    key = posembed("cross_posembed", torch.arange(keys, device=DEV)) + feat
    query = p.norm(query + attend("multihead_attn", query + pos, key), d + "norm2")
    ffn = p.linear(query, d + "linear1.weight", d + "linear1.bias").relu()
    query = p.norm(query + p.linear(ffn, d + "linear2.weight", d + "linear2.bias"), d + "norm3")
    out = {}
    for key, name in (("center", "center"), ("height", "height"), ("dimension_log", "dim"),
                      ("rotation", "rot"), ("velocity", "vel"), ("heatmap_logits", "heatmap")):
        z = p.bn(query @ p[f"{head}{name}.0.0.weight"][:, :, 0].t(), f"{head}{name}.0.1", 1e-5)
        out[key] = conv(z.relu(), f"{head}{name}.1").t().contiguous()[None]
    out["center"][0, 0] += index % w + 0.5
    out["center"][0, 1] += torch.div(index, w, rounding_mode="floor") + 0.5
    out["query_scores"] = score.view(10, keys)[:, index].to(F64)[None]
    return dict(out, labels=None, indices=None)


# LiDAR: voxels and sites are whole numbers, found with numpy.
def _voxels(points):
    """(coordinates [V, 3] as (z, y, x) in first-encounter order, 64-bit means
    of each voxel's first ten points)."""
    lo, size = np.float32([-54, -54, -5]), np.float32([0.075, 0.075, 0.2])
    with np.errstate(all="ignore"):
        ok = np.isfinite(points).all(1) & (points[:, :3] >= lo).all(1) \
            & (points[:, :3] < np.float32([54, 54, 3])).all(1)
        kept = points[ok]
        cell = np.floor((kept[:, :3] - lo) / size).astype(np.int64)
    inside = (cell >= 0).all(1) & (cell < [1440, 1440, 40]).all(1)
    kept, cell = kept[inside], cell[inside]
    key = (cell[:, 2] * 1440 + cell[:, 1]) * 1440 + cell[:, 0]
    _, first, inverse = np.unique(key, return_index=True, return_inverse=True)
    rank = np.empty(len(first), np.int64)
    rank[np.argsort(first, kind="stable")] = np.arange(len(first))
    voxel = rank[inverse]
    order = np.argsort(voxel, kind="stable")
    counts = np.bincount(voxel, minlength=len(first))
    place = np.arange(len(voxel)) - (np.cumsum(counts) - counts)[voxel[order]]
    use = order[place < 10]
    sums = np.zeros((len(first), 5))
    np.add.at(sums, voxel[use], kept[use].astype(np.float64))
    coords = np.empty((len(first), 3), np.int64)
    coords[voxel] = cell[:, ::-1]
    return coords, sums / np.minimum(counts, 10)[:, None]


def _find(sites, dims, z, y, x):
    """Row of each cell (z, y, x) in `sites` (sorted keys, rows), -1 if none."""
    keys, rows = sites
    ok = (z >= 0) & (z < dims[0]) & (y >= 0) & (y < dims[1]) & (x >= 0) & (x < dims[2])
    key = (z * dims[1] + y) * dims[2] + x
    at = np.searchsorted(keys, key).clip(max=len(keys) - 1)
    return np.where(ok & (keys[at] == key), rows[at], -1)


def _sites(coords, dims):
    key = (coords[:, 0] * dims[1] + coords[:, 1]) * dims[2] + coords[:, 2]
    order = np.argsort(key)
    return key[order], order


def _lidar_layers():
    """(input channels, output channels, kernel, stride, padding, submanifold,
    weight, BN, residual conv) of the encoder, in order."""
    b = "backbone_3d."
    one, ch = (1, 1, 1), (16, 32, 64, 128)
    yield 5, 16, (3, 3, 3), one, one, True, b + "conv_input.0.weight", b + "conv_input.1", 0
    for s in range(4):
        if s:
            pad = (0 if s == 3 else 1, 1, 1)
            yield ch[s - 1], ch[s], (3, 3, 3), (2, 2, 2), pad, False, \
                f"{b}conv{s + 1}.0.0.weight", f"{b}conv{s + 1}.0.1", 0
        for k in range(2):
            q = f"{b}conv{s + 1}.{k + (1 if s else 0)}."
            for c in (1, 2):
                yield ch[s], ch[s], (3, 3, 3), one, one, True, f"{q}conv{c}.weight", f"{q}bn{c}", c
    yield 128, 128, (3, 1, 1), (2, 1, 1), (0, 0, 0), False, b + "conv_out.0.weight", b + "conv_out.1", 0


def _lidar_walk(coords):
    """Per layer: (layer, taps' input rows per output site, output coordinates,
    grid)."""
    dims, table = GRID, None
    for layer in _lidar_layers():
        _, _, kernel, stride, pad, subm = layer[:6]
        taps = [(i, j, k) for i in range(kernel[0]) for j in range(kernel[1]) for k in range(kernel[2])]
        sites = _sites(coords, dims)
        out, odims = coords, dims
        if not subm:
            odims = tuple((dims[a] + 2 * pad[a] - kernel[a]) // stride[a] + 1 for a in range(3))
            keys = []
            for tap in taps:
                v = coords + np.array(pad) - np.array(tap)
                o = v // np.array(stride)
                ok = (v >= 0).all(1) & (v % np.array(stride) == 0).all(1) & (o < np.array(odims)).all(1)
                o = o[ok]
                keys.append((o[:, 0] * odims[1] + o[:, 1]) * odims[2] + o[:, 2])
            key = np.unique(np.concatenate(keys))
            out = np.stack([key // (odims[1] * odims[2]), key // odims[2] % odims[1], key % odims[2]], 1)
            table = None
        if table is None or not subm:
            table = [_find(sites, dims, *(out * np.array(stride) - np.array(pad) + np.array(tap)).T)
                     for tap in taps]
        yield layer, table, out, odims
        if not subm:
            table = None
        coords, dims = out, odims


def _lidar_flops(coords):
    flops, params = 0, 0
    for (ci, co, kernel, *_), table, _, _ in _lidar_walk(coords):
        flops += 2 * ci * co * sum(int((rows >= 0).sum()) for rows in table)
        params += ci * co * len(table)
    return flops, params


def _lidar64(p, points):
    coords, means = _voxels(points)
    x = torch.from_numpy(means).to(DEV)
    held = None
    for (ci, co, _, _, _, _, weight, bn, part), table, out, dims in _lidar_walk(coords):
        if part == 1:
            held = x
        w = p[weight].reshape(len(table), ci, co)
        y = torch.zeros((len(out), co), dtype=F64, device=DEV)
        for k, rows in enumerate(table):
            rows = torch.from_numpy(rows).to(DEV)
            live = (rows >= 0).nonzero()[:, 0]
            y[live] += x[rows[live]] @ w[k]
        y = p.bn(y, bn, 1e-3)
        x = (y + held if part == 2 else y).relu()
    bev = torch.zeros((1, 128, *dims), dtype=F64, device=DEV)
    at = torch.from_numpy(out).to(DEV)
    bev[0, :, at[:, 0], at[:, 1], at[:, 2]] = x.t()
    full = torch.zeros((CAPACITY, 5), dtype=F64, device=DEV)
    full[:len(means)] = torch.from_numpy(means).to(DEV)
    return dict(depth=None, coords=None, means=full, count=None, bev=bev)


def exact(case, seed):
    kind, t = case["kind"], _inputs(case, seed)
    if kind == "linear":
        y = t["x"].to(F64) @ t["w"].to(F64).t().contiguous()
        y = y if t["b"] is None else y + t["b"].to(F64)
        return y.relu() if case["relu"] else y
    if kind == "conv":
        if case["transpose"]:
            y = _deconv64(t["x"], t["w"], t["b"], case["stride"], case["pad"])
        else:
            y = _conv64(t["x"], t["w"], t["b"], case["stride"], case["pad"])
        return y.relu() if case["relu"] else y
    if kind == "lss":
        return _lss64(case, t)
    p = _Params(kind, seed)
    if kind == "swin":
        return _swin64(p, t["images"])
    if kind == "neck":
        return _neck64(p, t)
    if kind == "bev":
        return _bev64(p, t["x"])
    if kind == "transfusion":
        return _transfusion64(p, t, case)
    return _lidar64(p, t["points"].cpu().numpy())
