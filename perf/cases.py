"""The work that programs built on this framework have it do, as cases that can be timed.

Whole calls: a network forward on a small tile and on a full patch, and a mirrored sliding
window.  Single layers through the C ABI, at the sizes and channel counts of the U-Nets that
the benchmark runs (six stages, 32 to 320 features, 128^3 patches, eight mirror views) and at
ragged ones: the stride-1, strided and bf16 convolutions, the transposed convolution and the
residual InstanceNorm.  The two ends of a raw case: preprocessing of a CT and restoration of
class logits to the scanner's grid.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call,
``run`` is one pass, ``exact`` the same result in float64 by plain torch.
"""

from __future__ import annotations

import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "nnunet-mlx_amd"))

from nnunet_mlx import _native  # noqa: E402
from nnunet_mlx.data.preprocessing import PreprocessPlan, preprocess_raw_case  # noqa: E402
from nnunet_mlx.model.network import build_network  # noqa: E402
from nnunet_mlx.model.topology import PlainConvUNetSpec  # noqa: E402
from nnunet_mlx.plans import ResamplingContract  # noqa: E402
from nnunet_mlx.prediction.restore import restore_class_labels_device  # noqa: E402
from nnunet_mlx.prediction.sliding_window import predict_device_logits  # noqa: E402
from nnunet_mlx.storage.synthetic import random_weights  # noqa: E402

SLOPE = 0.01


# ---- the cases -------------------------------------------------------------------------

def listed() -> list[dict]:
    conv = {"kind": "conv", "kz": 3, "ky": 3, "kx": 3, "sz": 1, "sy": 1, "sx": 1, "c2": 0}
    return [
        # a preview or a test of an installation: one small tile, where launches and host
        # work count and the deep stages are a few voxels
        {"name": "forward_tile32", "kind": "forward", "features": "32,64,128,256,320,320",
         "cin": 1, "classes": 3, "batch": 1, "d": 32, "h": 32, "w": 32},
        # one patch without mirroring: the single-patch forward of the benchmark
        {"name": "forward_patch128", "kind": "forward", "features": "32,64,128,256,320,320",
         "cin": 1, "classes": 3, "batch": 1, "d": 128, "h": 128, "w": 128},
        # a small CT as the predictor handles every volume: padding, six overlapping tiles,
        # eight mirror views, one full and one partial batch of views
        {"name": "window_mirrored", "kind": "window", "features": "32,64,128,256,320,320",
         "cin": 1, "classes": 3, "patch": 128, "d": 101, "h": 200, "w": 168, "mirror": True},
        # the most expensive layer of a forward: the full-resolution decoder convolution over
        # the upsampled tensor and the skip, for the eight views of one tile
        {"name": "conv_decoder", **conv, "c1": 32, "c2": 32, "cout": 32, "batch": 8,
         "d": 128, "h": 128, "w": 128},
        # a middle stage, eight views
        {"name": "conv_middle", **conv, "c1": 128, "cout": 128, "batch": 8,
         "d": 32, "h": 32, "w": 32},
        # a layer of a network whose patch is no multiple of any tile
        {"name": "conv_ragged", **conv, "c1": 64, "cout": 64, "batch": 4,
         "d": 37, "h": 61, "w": 43},
        # the first strided convolution of the encoder, eight views
        {"name": "conv_stride", **conv, "c1": 32, "cout": 64, "batch": 8, "sz": 2, "sy": 2,
         "sx": 2, "d": 128, "h": 128, "w": 128},
        # a stage-1 convolution in bf16, as the residual network of the benchmark runs it
        {"name": "conv_bf16", **conv, "kind": "conv_bf16", "c1": 64, "cout": 64, "batch": 4,
         "d": 64, "h": 80, "w": 80},
        # the last transposed convolution of the decoder, eight views
        {"name": "upsample", "kind": "upsample", "cin": 64, "cout": 32, "batch": 8,
         "d": 64, "h": 64, "w": 64},
        # the end of a residual block: InstanceNorm, shortcut and LeakyReLU
        {"name": "norm_residual", "kind": "norm", "channels": 32, "batch": 2,
         "d": 128, "h": 160, "w": 160, "residual": True},
        # a CT as the scanner writes it, to the plan's spacing (separate coarse axis)
        {"name": "preprocess_ct", "kind": "preprocess", "d": 120, "h": 512, "w": 512,
         "coarse": 2.5},
        # its class logits back on the scanner's grid
        {"name": "restore_labels", "kind": "restore", "classes": 3, "d": 300, "h": 534, "w": 534,
         "td": 120, "th": 512, "tw": 512},
    ]


def _log(rng, low: float, high: float) -> float:
    return float(np.exp(rng.uniform(np.log(low), np.log(high))))


def _size(rng, low: int, high: int) -> int:
    return int(round(_log(rng, low, high)))


def draw(rng) -> dict:
    kind = rng.choice(["forward", "window", "conv", "conv", "conv", "conv_split", "conv_bf16",
                       "upsample", "norm", "preprocess", "restore"])
    if kind == "forward":
        stages = rng.choice([3, 4, 5, 6])
        step = 2 ** (stages - 1)
        d, h, w = (step * max(1, round(_log(rng, 24, 128) / step)) for _ in range(3))
        return {"kind": "forward", "features": ",".join(str(min(320, 32 * 2 ** s)) for s in range(stages)),
                "cin": rng.choice([1, 2, 4]), "classes": rng.choice([2, 3, 4]),
                "batch": rng.choice([1, 1, 2, 4]), "d": d, "h": h, "w": w}
    if kind == "window":
        patch = rng.choice([32, 64, 96])
        most = {32: 2.4, 64: 2.0, 96: 1.5}[patch]
        d, h, w = (_size(rng, 0.6 * patch, most * patch) for _ in range(3))
        return {"kind": "window", "features": "32,64,128,256", "cin": 1,
                "classes": rng.choice([2, 3]), "patch": patch, "d": d, "h": h, "w": w,
                "mirror": rng.random() < 0.7}
    if kind in ("conv", "conv_split", "conv_bf16"):
        # the U-Net's halving: wide channels on small grids
        cout = rng.choice([32, 64, 96, 128, 192, 256, 320])
        c1 = rng.choice([32, cout, cout])
        side = 4096 / cout
        d, h, w = (_size(rng, max(4, 0.08 * side), max(6, side)) for _ in range(3))
        case = {"kind": "conv" if kind == "conv_split" else kind, "kz": 3, "ky": 3, "kx": 3,
                "sz": 1, "sy": 1, "sx": 1, "c1": c1, "c2": rng.choice([0, 0, cout]) if c1 == cout else 0,
                "cout": cout, "batch": rng.choice([1, 2, 4, 8]), "d": d, "h": h, "w": w}
        if kind == "conv_split":
            # strided, or one slice thick in z
            if rng.random() < 0.6:
                case.update(sz=rng.choice([1, 2]), sy=2, sx=2, c1=rng.choice([32, max(32, cout // 2)]), c2=0)
            else:
                case.update(kz=1)
        return case
    if kind == "upsample":
        cout = rng.choice([32, 64, 128, 256])
        side = 2048 / cout
        d, h, w = (_size(rng, max(4, 0.2 * side), side) for _ in range(3))
        return {"kind": "upsample", "cin": min(320, 2 * cout), "cout": cout,
                "batch": rng.choice([1, 2, 4, 8]), "d": d, "h": h, "w": w}
    if kind == "norm":
        channels = rng.choice([32, 64, 128, 320])
        side = 5120 / channels
        d, h, w = (_size(rng, max(4, 0.1 * side), side) for _ in range(3))
        return {"kind": "norm", "channels": channels, "batch": rng.choice([1, 2, 4]),
                "d": d, "h": h, "w": w, "residual": rng.random() < 0.5}
    if kind == "preprocess":
        return {"kind": "preprocess", "d": _size(rng, 40, 120), "h": _size(rng, 200, 512),
                "w": _size(rng, 200, 512), "coarse": rng.choice([1.5, 2.5, 5.0])}
    d, h, w = _size(rng, 40, 300), _size(rng, 160, 534), _size(rng, 160, 534)
    return {"kind": "restore", "classes": rng.choice([2, 3, 5]), "d": d, "h": h, "w": w,
            "td": max(8, int(d * rng.uniform(0.4, 1.3))), "th": int(h * rng.uniform(0.8, 1.3)),
            "tw": int(w * rng.uniform(0.8, 1.3))}


# ---- what a program holds before the call ------------------------------------------------

def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _activation(shape, gen) -> torch.Tensor:
    """What a hidden layer reads: LeakyReLU of a normalised tensor."""
    x = torch.randn(shape, generator=gen, device="cuda")
    return torch.where(x > 0, x, SLOPE * x)


def _spec(case: dict) -> PlainConvUNetSpec:
    features = tuple(int(f) for f in case["features"].split(","))
    n = len(features)
    return PlainConvUNetSpec(
        input_channels=case["cin"], num_classes=case["classes"], features=features,
        kernel_sizes=((3, 3, 3),) * n, strides=((1, 1, 1),) + ((2, 2, 2),) * (n - 1),
        encoder_convs=(2,) * n, decoder_convs=(2,) * (n - 1))


def _volume(shape, gen) -> torch.Tensor:
    """A normalised CT: smooth regions of different mean, and noise."""
    c, d, h, w = shape
    coarse = torch.randn((1, c, max(2, d // 16), max(2, h // 16), max(2, w // 16)), generator=gen,
                         device="cuda")
    smooth = torch.nn.functional.interpolate(coarse, size=(d, h, w), mode="trilinear")[0]
    return (smooth + 0.5 * torch.randn(shape, generator=gen, device="cuda")).contiguous()


def _conv_operands(case: dict, seed: int):
    gen = _generator(seed)
    grid = (case["batch"], case["d"], case["h"], case["w"])
    k = (case["kz"], case["ky"], case["kx"])
    x1 = _activation((*grid, case["c1"]), gen)
    # the second input of a decoder convolution is the skip; the first the upsampled tensor
    x2 = _activation((*grid, case["c2"]), gen) if case["c2"] else None
    cin = case["c1"] + case["c2"]
    w = torch.randn((case["cout"], *k, cin), generator=gen, device="cuda")
    w *= (2.0 / (1 + SLOPE ** 2) / (cin * k[0] * k[1] * k[2])) ** 0.5
    bias = 0.1 * torch.randn(case["cout"], generator=gen, device="cuda")
    return x1, x2, w, bias


def _upsample_operands(case: dict, seed: int):
    gen = _generator(seed)
    x = _activation((case["batch"], case["d"], case["h"], case["w"], case["cin"]), gen)
    w = torch.randn((case["cout"], 2, 2, 2, case["cin"]), generator=gen, device="cuda")
    w *= (2.0 / (1 + SLOPE ** 2) / (case["cout"] * 8)) ** 0.5
    bias = 0.1 * torch.randn(case["cout"], generator=gen, device="cuda")
    return x, w, bias


def _norm_operands(case: dict, seed: int):
    gen = _generator(seed)
    c = case["channels"]
    shape = (case["batch"], case["d"] * case["h"] * case["w"], c)
    # a convolution's output: every channel with a mean and a spread of its own
    x = torch.randn(shape, generator=gen, device="cuda")
    x = x * (0.5 + torch.rand(c, generator=gen, device="cuda")) + torch.randn(c, generator=gen, device="cuda")
    gamma = 1 + 0.1 * torch.randn(c, generator=gen, device="cuda")
    beta = 0.1 * torch.randn(c, generator=gen, device="cuda")
    residual = _activation(shape, gen) if case["residual"] else None
    return x.contiguous(), gamma, beta, residual


def _raw_ct(case: dict, seed: int) -> torch.Tensor:
    """int16 CT: air outside an elliptic body section, soft tissue inside."""
    gen = _generator(seed)
    d, h, w = case["d"], case["h"], case["w"]
    yy = (torch.arange(h, device="cuda") - h / 2) / (0.39 * h)
    xx = (torch.arange(w, device="cuda") - w / 2) / (0.45 * w)
    body = (yy[:, None] ** 2 + xx[None] ** 2) <= 1
    tissue = 40 + 60 * torch.randn((1, d, h, w), generator=gen, device="cuda")
    return torch.where(body, tissue, torch.full_like(tissue, -1000.0)).to(torch.int16).contiguous()


def _plan() -> PreprocessPlan:
    return PreprocessPlan.from_plans({
        "transpose_forward": [0, 1, 2], "transpose_backward": [0, 1, 2],
        "foreground_intensity_properties_per_channel": {
            "0": {"mean": 99.4, "std": 137.2, "percentile_00_5": -958.0, "percentile_99_5": 327.0}},
        "configurations": {"3d_fullres": {
            "spacing": [1.0, 0.7676, 0.7676], "normalization_schemes": ["CTNormalization"],
            "use_mask_for_norm": [False], "patch_size": [128, 128, 128],
            "resampling_fn_data": "resample_data_or_seg_to_shape",
            "resampling_fn_data_kwargs": {"is_seg": False, "order": 3, "order_z": 0,
                                          "force_separate_z": None}}},
    }, "3d_fullres")


_SPACING = 0.8       # in-plane, of the raw CT
_FINE = 0.7676       # in-plane, of the plan


def _winograd(case: dict) -> bool:
    """Stride-1 3x3x3 layers take the Winograd entry, as the network does."""
    return ((case["kz"], case["ky"], case["kx"], case["sz"], case["sy"], case["sx"])
            == (3, 3, 3, 1, 1, 1))


def prepare(case: dict, seed: int):
    kind = case["kind"]
    lib = _native.load()
    stream = _native.stream_handle()
    if kind in ("forward", "window"):
        spec = _spec(case)
        net = build_network(spec)
        net.load_weights(random_weights(spec, seed=seed, random_affine=True))
        gen = _generator(seed)
        if kind == "forward":
            x = _volume((case["batch"] * case["cin"], case["d"], case["h"], case["w"]), gen)
            x = x.reshape(case["batch"], case["cin"], case["d"], case["h"], case["w"])
            x = x.permute(0, 2, 3, 4, 1).contiguous()
        else:
            x = _volume((case["cin"], case["d"], case["h"], case["w"]), gen)
        return {"case": case, "net": net, "x": x}
    if kind in ("conv", "conv_bf16"):
        x1, x2, w, bias = _conv_operands(case, seed)
        k = _native.ints((case["kz"], case["ky"], case["kx"]))
        c1, c2, cout = case["c1"], case["c2"], case["cout"]
        top = float(w.abs().max())
        if kind == "conv" and _winograd(case):
            scale = lib.nnx_winograd_weight_scale(top)
            packed = torch.empty(lib.nnx_conv3d_winograd_packed_bytes(cout, c1, c2),
                                 dtype=torch.uint8, device="cuda")
            _native.check(lib.nnx_conv3d_winograd_pack_weight(
                _native.ptr(w), cout, c1, c2, scale, _native.ptr(packed), stream))
        else:
            scale = lib.nnx_split_weight_scale(top)
            packed = torch.empty(lib.nnx_conv3d_split_packed_bytes(cout, k, c1, c2),
                                 dtype=torch.uint8, device="cuda")
            pack = lib.nnx_conv3d_bf16_pack_weight if kind == "conv_bf16" else lib.nnx_conv3d_split_pack_weight
            _native.check(pack(_native.ptr(w), cout, k, c1, c2, scale, _native.ptr(packed), stream))
        out = [(case[a] + 2 * (case["k" + b] // 2) - case["k" + b]) // case["s" + b] + 1
               for a, b in (("d", "z"), ("h", "y"), ("w", "x"))]
        y = torch.empty((case["batch"], *out, cout), device="cuda")
        return {"case": case, "x1": x1, "x2": x2, "packed": packed, "scale": scale, "bias": bias,
                "y": y, "k": k, "s": _native.ints((case["sz"], case["sy"], case["sx"])),
                "size": _native.ints((case["d"], case["h"], case["w"]))}
    if kind == "upsample":
        x, w, bias = _upsample_operands(case, seed)
        k = _native.ints((2, 2, 2))
        scale = lib.nnx_split_weight_scale(float(w.abs().max()))
        packed = torch.empty(lib.nnx_tconv3d_split_packed_bytes(case["cout"], k, case["cin"]),
                             dtype=torch.uint8, device="cuda")
        _native.check(lib.nnx_tconv3d_split_pack_weight(
            _native.ptr(w), case["cout"], k, case["cin"], scale, _native.ptr(packed), stream))
        y = torch.empty((case["batch"], 2 * case["d"], 2 * case["h"], 2 * case["w"], case["cout"]),
                        device="cuda")
        return {"case": case, "x": x, "packed": packed, "scale": scale, "bias": bias, "y": y,
                "k": k, "size": _native.ints((case["d"], case["h"], case["w"]))}
    if kind == "norm":
        x, gamma, beta, residual = _norm_operands(case, seed)
        nbytes = lib.nnx_instnorm_workspace_bytes(case["batch"], x.shape[1], case["channels"])
        return {"case": case, "x": x, "gamma": gamma, "beta": beta, "residual": residual,
                "y": torch.empty_like(x),
                "work": torch.empty(nbytes, dtype=torch.uint8, device="cuda")}
    if kind == "preprocess":
        return {"case": case, "raw": _raw_ct(case, seed), "plan": _plan(),
                "properties": {"spacing": (case["coarse"], _SPACING, _SPACING)}}
    gen = _generator(seed)
    logits = _volume((case["classes"], case["d"], case["h"], case["w"]), gen)
    contract = ResamplingContract(function_name="resample_data_or_seg_to_shape", order=1,
                                  order_z=0, force_separate_z=None)
    return {"case": case, "logits": (4 * logits).permute(1, 2, 3, 0).contiguous().half(),
            "target": (case["td"], case["th"], case["tw"]), "contract": contract,
            "current": (1.0, _FINE, _FINE),
            "new": (case["d"] / case["td"], _FINE * case["h"] / case["th"],
                    _FINE * case["w"] / case["tw"])}


# ---- one pass ------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return state["net"](state["x"])
    if kind == "window":
        return predict_device_logits(
            state["net"], state["x"], patch_size=(case["patch"],) * 3,
            num_classes=case["classes"], mirroring_axes=(0, 1, 2) if case["mirror"] else ())
    if kind == "preprocess":
        return preprocess_raw_case(state["raw"], state["properties"], state["plan"]).data
    if kind == "restore":
        return restore_class_labels_device(state["logits"], state["target"], state["current"],
                                           state["new"], state["contract"]).view(torch.int16)
    lib = _native.load()
    ptr = _native.ptr
    stream = _native.stream_handle()
    if kind in ("conv", "conv_bf16"):
        if kind == "conv" and _winograd(case):
            status = lib.nnx_conv3d_winograd(
                ptr(state["x1"]), case["c1"], ptr(state["x2"]), case["c2"], ptr(state["packed"]),
                state["scale"], ptr(state["bias"]), ptr(state["y"]), case["batch"], state["size"],
                case["cout"], stream)
        else:
            entry = lib.nnx_conv3d_bf16 if kind == "conv_bf16" else lib.nnx_conv3d_split
            status = entry(
                ptr(state["x1"]), case["c1"], ptr(state["x2"]), case["c2"], ptr(state["packed"]),
                state["scale"], ptr(state["bias"]), ptr(state["y"]), case["batch"], state["size"],
                case["cout"], state["k"], state["s"], stream)
    elif kind == "upsample":
        status = lib.nnx_tconv3d_split(
            ptr(state["x"]), case["cin"], ptr(state["packed"]), state["scale"], ptr(state["bias"]),
            ptr(state["y"]), case["batch"], state["size"], case["cout"], state["k"], stream)
    else:
        x = state["x"]
        status = lib.nnx_instnorm_lrelu(
            ptr(x), ptr(state["y"]), case["batch"], x.shape[1], case["channels"], None,
            ptr(state["gamma"]), ptr(state["beta"]), 1e-5, 1, SLOPE, ptr(state["residual"]),
            ptr(state["work"]), state["work"].numel(), stream)
    _native.check(status, kind)
    return state["y"]


# ---- what a pass cannot do without -----------------------------------------------------------

def _forward_work(features, cin: int, classes: int, voxels: float) -> tuple[float, float]:
    """(multiply-add FLOPs of the convolutions, weight bytes) of one forward of `voxels`."""
    flops = weights = 0.0
    n = len(features)
    for s, f in enumerate(features):
        vox = voxels / 8 ** s
        for ci in (cin if s == 0 else features[s - 1], f):
            flops += 54.0 * ci * f * vox
            weights += 27.0 * ci * f
    for s in range(n - 2, -1, -1):
        vox, f = voxels / 8 ** s, features[s]
        flops += 2.0 * features[s + 1] * f * vox + 54.0 * 2 * f * f * vox + 54.0 * f * f * vox
        weights += 8.0 * features[s + 1] * f + 81.0 * f * f
    return flops + 2.0 * features[0] * classes * voxels, 4.0 * weights


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "preprocess":
        vox = case["d"] * case["h"] * case["w"]
        new = (case["coarse"] * case["d"]) * (_SPACING / _FINE) ** 2 * case["h"] * case["w"]
        return {"bytes": 2.0 * vox + 4.0 * new, "flops": 0.0}
    if kind == "restore":
        return {"bytes": 2.0 * case["classes"] * case["d"] * case["h"] * case["w"]
                + 2.0 * case["td"] * case["th"] * case["tw"], "flops": 0.0}
    vox = float(case["d"] * case["h"] * case["w"])
    if kind in ("forward", "window"):
        features = [int(f) for f in case["features"].split(",")]
        if kind == "forward":
            views = case["batch"] * vox
        else:
            tiles = 1
            for a in "dhw":
                extent = max(case[a], case["patch"])
                tiles *= -(-2 * (extent - case["patch"]) // case["patch"]) + 1
            views = tiles * (8 if case["mirror"] else 1) * float(case["patch"]) ** 3
            # one pass over the volume and its logits, whatever the overlap
        flops, weights = _forward_work(features, case["cin"], case["classes"], views)
        moved = vox * (case["batch"] if kind == "forward" else 1)
        return {"bytes": weights + 4.0 * moved * (case["cin"] + case["classes"]), "flops": flops}
    if kind == "norm":
        tensors = 3 if case["residual"] else 2
        return {"bytes": 4.0 * tensors * case["batch"] * vox * case["channels"], "flops": 0.0}
    if kind == "upsample":
        return {"bytes": 4.0 * (case["batch"] * vox * (case["cin"] + 8 * case["cout"])
                                + 8 * case["cin"] * case["cout"]),
                "flops": 16.0 * case["cin"] * case["cout"] * case["batch"] * vox}
    cin, taps = case["c1"] + case["c2"], case["kz"] * case["ky"] * case["kx"]
    out = case["batch"]
    for a, b in (("d", "z"), ("h", "y"), ("w", "x")):
        out *= (case[a] - 1) // case["s" + b] + 1
    return {"bytes": 4.0 * (case["batch"] * vox * cin + out * case["cout"] + taps * cin * case["cout"]),
            "flops": 2.0 * taps * cin * case["cout"] * out}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "restore":
        return "exact"
    if kind in ("forward", "window"):
        # logits behind up to 22 convolutions: 3e-6 to 5e-6 from float64
        return {"rel": 2e-5, "max": 1e-3}
    if kind == "conv_bf16":
        # operands rounded to bf16: 2.4e-3 from float64
        return {"rel": 1e-2, "max": 1e-1}
    if kind in ("conv", "upsample"):
        # split products: 2e-7 to 5e-7 from float64
        return {"rel": 2e-6, "max": 5e-5}
    # float32 arithmetic of a few operations, or float64 rounded once
    return {"rel": 1e-6, "max": 2e-5}


# ---- the same in float64 ------------------------------------------------------------------------

def _conv64(x, w, bias, k, s):
    """(N, D, H, W, C) float64 convolution, one matrix product a tap."""
    p = [v // 2 for v in k]
    x = torch.nn.functional.pad(x, (0, 0, p[2], p[2], p[1], p[1], p[0], p[0]))
    out = [(x.shape[1 + i] - k[i]) // s[i] + 1 for i in range(3)]
    y = torch.zeros((x.shape[0], *out, w.shape[0]), dtype=torch.float64, device=x.device)
    for a in range(k[0]):
        for b in range(k[1]):
            for c in range(k[2]):
                tap = x[:, a:a + s[0] * (out[0] - 1) + 1:s[0], b:b + s[1] * (out[1] - 1) + 1:s[1],
                        c:c + s[2] * (out[2] - 1) + 1:s[2]]
                flat = tap.reshape(-1, x.shape[-1]) @ w[:, a, b, c].t().contiguous()
                y += flat.reshape(y.shape)
    return y if bias is None else y + bias


def _tconv64(x, w, bias):
    n, d, h, v, _ = x.shape
    cout = w.shape[0]
    y = x.reshape(-1, x.shape[-1]) @ w.reshape(cout * 8, -1).t().contiguous()
    y = y.reshape(n, d, h, v, cout, 2, 2, 2).permute(0, 1, 5, 2, 6, 3, 7, 4)
    return y.reshape(n, 2 * d, 2 * h, 2 * v, cout) + bias


def _norm64(x, gamma, beta, residual=None):
    dims = tuple(range(1, x.dim() - 1))
    mean = x.mean(dims, keepdim=True)
    var = ((x - mean) ** 2).mean(dims, keepdim=True)
    y = (x - mean) / torch.sqrt(var + 1e-5) * gamma + beta
    if residual is not None:
        y = y + residual
    return torch.where(y > 0, y, SLOPE * y)


def _forward64(case: dict, seed: int, x):
    spec = _spec(case)
    w = {k: torch.from_numpy(v).cuda().double()
         for k, v in random_weights(spec, seed=seed, random_affine=True).items()}
    n = len(spec.features)

    def block(name, v, stride):
        y = _conv64(v, w[name + ".conv.weight"], w[name + ".conv.bias"], (3, 3, 3), (stride,) * 3)
        return _norm64(y, w[name + ".norm.weight"], w[name + ".norm.bias"])

    skips = []
    for s in range(n):
        for j in range(2):
            x = block(f"enc{s}.block{j}", x, 2 if s and not j else 1)
        skips.append(x)
    for d in range(n - 1):
        x = _tconv64(x, w[f"up{d}.weight"], w[f"up{d}.bias"])
        x = block(f"dec{d}.block0", torch.cat((x, skips[n - 2 - d]), -1), 1)
        x = block(f"dec{d}.block1", x, 1)
    head = w[f"seg{n - 2}.weight"].reshape(case["classes"], -1).t().contiguous()
    flat = x.reshape(-1, x.shape[-1]) @ head + w[f"seg{n - 2}.bias"]
    return flat.reshape(*x.shape[:-1], case["classes"])


def _spline_matrix(n: int, m: int) -> torch.Tensor:
    """Cubic spline interpolation of n samples at m pixel-centred points (edge samples
    repeated 12 times before the coefficients are solved), as a matrix."""
    pad = 12
    size = n + 2 * pad
    basis = np.zeros((size, size))
    for i in range(size):
        basis[i, i] += 4 / 6
        for j in (i - 1, i + 1):
            basis[i, -j if j < 0 else (2 * size - 2 - j if j >= size else j)] += 1 / 6
    edge = np.zeros((size, n))
    edge[np.arange(size), np.clip(np.arange(size) - pad, 0, n - 1)] = 1
    coefficients = np.linalg.solve(basis, edge)
    at = (np.arange(m) + 0.5) * n / m - 0.5 + pad
    first = np.floor(at).astype(int)
    t = at - first
    taps = ((1 - t) ** 3 / 6, (3 * t ** 3 - 6 * t ** 2 + 4) / 6,
            (-3 * t ** 3 + 3 * t ** 2 + 3 * t + 1) / 6, t ** 3 / 6)
    matrix = sum(tap[:, None] * coefficients[first + o - 1] for o, tap in enumerate(taps))
    return torch.from_numpy(matrix).cuda()


def _preprocess64(case: dict, seed: int):
    x = _raw_ct(case, seed)[0].double()
    x = (x.clamp(-958.0, 327.0) - 99.4) / 137.2
    old = tuple(x.shape)
    new = [int(round(o * s / t)) for o, s, t in
           zip(old, (case["coarse"], _SPACING, _SPACING), (1.0, _FINE, _FINE))]
    separate = case["coarse"] / _SPACING > 3
    planes = (1, 2) if separate else (0, 1, 2)
    low = x.amin(planes, keepdim=True)
    high = x.amax(planes, keepdim=True)
    for axis in planes:
        matrix = _spline_matrix(old[axis], new[axis])
        moved = x.movedim(axis, -1).contiguous()
        x = (moved.reshape(-1, old[axis]) @ matrix.t().contiguous()).reshape(*moved.shape[:-1], -1)
        x = x.movedim(-1, axis)
    x = torch.minimum(torch.maximum(x, low), high)
    if separate and new[0] != old[0]:
        at = np.clip(np.floor((np.arange(new[0]) + 0.5) * old[0] / new[0]), 0, old[0] - 1)
        x = x[torch.from_numpy(at.astype(np.int64)).cuda()]
    return x[None]


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "forward":
        gen = _generator(seed)
        x = _volume((case["batch"] * case["cin"], case["d"], case["h"], case["w"]), gen)
        x = x.reshape(case["batch"], case["cin"], case["d"], case["h"], case["w"])
        return _forward64(case, seed, x.permute(0, 2, 3, 4, 1).double().contiguous())
    if kind in ("conv", "conv_bf16"):
        x1, x2, w, bias = _conv_operands(case, seed)
        x = x1 if x2 is None else torch.cat((x1, x2), -1)
        return _conv64(x.double(), w.double(), bias.double(),
                       (case["kz"], case["ky"], case["kx"]), (case["sz"], case["sy"], case["sx"]))
    if kind == "upsample":
        x, w, bias = _upsample_operands(case, seed)
        return _tconv64(x.double(), w.double(), bias.double())
    if kind == "norm":
        x, gamma, beta, residual = _norm_operands(case, seed)
        return _norm64(x.double(), gamma.double(), beta.double(),
                       None if residual is None else residual.double())
    if kind == "preprocess":
        return _preprocess64(case, seed)
    return None  # labels are whole numbers; a mirrored window takes minutes in float64
