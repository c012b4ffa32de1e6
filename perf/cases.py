"""The framework's work as a user has it done: the per-frame path of the sparse refiner and the operators it is made of.

A frame of PromptMoGe goes through: nearest-fill of the LiDAR prompt, K refine steps (each a prompt fit, the residual
features, voxelisation, the sparse network and the log-depth update), the final metric fit with the metric depth, and
the prompt gauge. A caller who keeps the reference's own model code instead plugs in the refiner module alone, or the
`flex_gemm` operators (maps, convolutions, pooling). Every case calls the public Python entry points of
`promptmoge_amd`, with inputs on the GPU, and returns all that the call computes.

`listed()` names twelve cases over that range, `draw(rng)` gives more of the same kinds with other sizes and options,
`prepare` makes a case's inputs and handles, `run` is one call, `work` the bytes and operations it cannot do without,
`tolerance` what two correct implementations may differ by, and `exact` the same result in 64 bits in plain torch.
"""
from __future__ import annotations

import contextlib
import functools
import math

import numpy as np
import torch
import torch.nn.functional as F

DEVICE = "cuda"
RESOLUTION = 256.0  # voxel keys per unit of log depth (the reference's depth_resolution)
TRIM, MIN_POINTS = 0.2, 32
CLIP1, CLIP2, CLIP_LINEAR = 4.0, 2.5, 4.0  # activation clips of the int8 refiners (about the 99.9th percentile)
TAPS_SURFACE = 5.5  # active taps per voxel of a 480x640 depth map with 5 mm noise
TAPS_GENERIC = 10.0  # and of a smooth surface set
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


# ---------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # The metric fit as the model's own code calls it (fit_scale_shift, default 4 rounds), on a phone's 192x256
        # LiDAR map: the smallest call, all latency.
        {"name": "fit_lidar", "kind": "fit", "B": 1, "h": 192, "w": 256, "iters": 4},
        # nearest_fill of a prompt at the high-resolution size: scattered holes and a window-sized patch without returns.
        {"name": "fill_hires", "kind": "fill", "B": 1, "h": 756, "w": 1008, "holes": 0.2, "patch": 64},
        # The prompt gauge that `infer` applies after the loop: depth at model size, prompt at LiDAR size.
        {"name": "gauge", "kind": "gauge", "B": 1, "H": 480, "W": 640, "h": 192, "w": 256, "degree": 2},
        # One refine step with final fit and depth of the small on-device model (B: 240x320, 4 int8 layers, C = 32).
        {"name": "step_small", "kind": "step", "precision": "int8", "B": 1, "H": 240, "W": 320, "dh": 240, "dw": 320,
         "C": 32, "blocks": 2, "K": 1, "iters": 10, "soft": False, "gate": False, "anchor": 0.0, "stream": "own"},
        # The headline step (A: 480x640, 6 int8 layers, C = 48), with final fit and depth.
        {"name": "step_int8", "kind": "step", "precision": "int8", "B": 1, "H": 480, "W": 640, "dh": 480, "dw": 640,
         "C": 48, "blocks": 3, "K": 1, "iters": 10, "soft": False, "gate": False, "anchor": 0.0, "stream": "own"},
        # A whole high-resolution frame (H: 756x1008, 6 int8 layers, C = 64, 3 steps and the final fit): the largest.
        {"name": "frame_hires", "kind": "step", "precision": "int8", "B": 1, "H": 756, "W": 1008, "dh": 756, "dw": 1008,
         "C": 64, "blocks": 3, "K": 3, "iters": 10, "soft": False, "gate": False, "anchor": 0.0, "stream": "own"},
        # A step of the half-precision teacher (T: 480x640, 6 fp16 layers, C = 64).
        {"name": "step_fp16", "kind": "step", "precision": "fp16", "B": 1, "H": 480, "W": 640, "dh": 480, "dw": 640,
         "C": 64, "blocks": 3, "K": 1, "iters": 10, "soft": False, "gate": False, "anchor": 0.0, "stream": "own"},
        # A refine step around the deployed five-level int8 U-Net, at the headline size.
        {"name": "unet_step", "kind": "unet_step", "precision": "int8", "channels": "32 64 128 256 256", "B": 1,
         "H": 480, "W": 640, "enc": 1024, "iters": 10, "stream": "own"},
        # The teacher's U-Net as a module plugged into the model's own code, which runs on the default stream.
        {"name": "unet_fp16", "kind": "unet", "precision": "fp16", "channels": "32 64 128 256 512", "B": 1,
         "H": 480, "W": 640, "enc": 1024, "stream": "default"},
        # flex_gemm's SubmanifoldConv3d on a surface set of the size of the U-Net's second level, its map kept.
        {"name": "conv_bf16", "kind": "conv", "dtype": "bf16", "n": 183_582, "C": 64, "bias": True},
        # flex_gemm's level step in fp32, as the model's own code makes it: level-0 map and convolution, the pooling
        # to level 1, its map and convolution, and the nearest upsampling back.
        {"name": "level_fp32", "kind": "level", "dtype": "fp32", "H": 240, "W": 320, "C": 32},
        # The int8 convolution of a large surface set (1M voxels, C = 128) with the map's row order kept beside it.
        {"name": "conv_int8", "kind": "conv_i8", "n": 1_000_000, "C": 128, "ordered": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "fill", "gauge", "step", "step", "unet_step", "unet", "conv", "level", "conv_i8"])
    if kind == "fit":
        return {"kind": kind, "B": rng.choice([1, 1, 2]), "h": _log_int(rng, 48, 756), "w": _log_int(rng, 64, 1008),
                "iters": rng.choice([4, 10])}
    if kind == "fill":
        return {"kind": kind, "B": rng.choice([1, 1, 2]), "h": _log_int(rng, 96, 756), "w": _log_int(rng, 128, 1008),
                "holes": round(rng.uniform(0.05, 0.5), 3), "patch": _log_int(rng, 8, 64)}
    if kind == "gauge":
        H, W = _log_int(rng, 240, 756), _log_int(rng, 320, 1008)
        f = rng.choice([1.0, 0.5, 0.4])
        return {"kind": kind, "B": rng.choice([1, 1, 2]), "H": H, "W": W, "h": max(24, int(H * f)),
                "w": max(32, int(W * f)), "degree": rng.choice([1, 2, 2])}
    if kind == "step":
        precision = rng.choice(["int8", "int8", "fp16"])
        H, W = (_log_int(rng, 96, 756), _log_int(rng, 128, 1008)) if precision == "int8" else (
            _log_int(rng, 96, 480), _log_int(rng, 128, 640))
        f = rng.choice([1.0, 1.0, 0.5])
        return {"kind": kind, "precision": precision, "B": 1 if H * W > 100_000 else rng.choice([1, 2]), "H": H, "W": W,
                "dh": max(1, int(H * f)), "dw": max(1, int(W * f)), "C": rng.choice([16, 32, 48, 64]),
                "blocks": rng.choice([2, 3]), "K": rng.choice([1, 2]), "iters": rng.choice([4, 10]),
                "soft": rng.random() < 0.3, "gate": rng.random() < 0.3,
                "anchor": rng.choice([0.0, 0.0, 0.3]), "stream": rng.choice(["own", "own", "default"])}
    if kind in ("unet_step", "unet"):
        precision, channels = rng.choice([("int8", "32 64 128 256 256"), ("int8", "16 32 64 128"),
                                          ("int8", "48 96 192"), ("fp16", "32 64 128 256 512"),
                                          ("fp16", "32 64 128 256")])
        case = {"kind": kind, "precision": precision, "channels": channels, "B": 1, "H": 16 * _log_int(rng, 6, 30),
                "W": 16 * _log_int(rng, 8, 40), "enc": rng.choice([256, 1024])}
        if kind == "unet_step":
            case["iters"] = rng.choice([4, 10])
        case["stream"] = rng.choice(["own", "default"])
        return case
    if kind == "conv":
        dtype = rng.choice(["fp16", "bf16", "fp32"])
        C = rng.choice([32, 48, 64, 96, 128, 256]) if dtype != "fp32" else rng.choice([16, 32, 48, 64])
        return {"kind": kind, "dtype": dtype, "n": _log_int(rng, 2_000, 400_000 if C <= 64 else 100_000), "C": C,
                "bias": rng.random() < 0.8}
    if kind == "level":
        return {"kind": kind, "dtype": rng.choice(["fp32", "fp16"]), "H": _log_int(rng, 96, 480),
                "W": _log_int(rng, 128, 640), "C": rng.choice([16, 32, 64])}
    return {"kind": "conv_i8", "n": _log_int(rng, 10_000, 900_000), "C": rng.choice([64, 128]),
            "ordered": rng.random() < 0.5}


# ------------------------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed) * 7919 + 17)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEVICE)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEVICE)


def _room(g, B, H, W):
    """Depth maps [B, H, W] (fp64, 0.5-6 m) of rooms made of eight planes, seen by a pinhole camera."""
    y = ((torch.arange(H, device=DEVICE, dtype=torch.float64) - H / 2) / (0.8125 * W)).view(1, H, 1)
    x = ((torch.arange(W, device=DEVICE, dtype=torch.float64) - W / 2) / (0.8125 * W)).view(1, 1, W)
    D = torch.full((B, H, W), 6.0, dtype=torch.float64, device=DEVICE)
    for _ in range(8):
        n = _normal(g, B, 3).double()
        n[:, 2] = -n[:, 2].abs() - 0.6
        p = torch.stack([_uniform(g, B) - 0.5, _uniform(g, B) - 0.5, torch.ones(B, device=DEVICE)], 1).double()
        p = p * (0.8 + 5.2 * _uniform(g, B, 1).double())
        c = (n * p).sum(1).view(B, 1, 1)
        nd = n[:, 0].view(B, 1, 1) * x + n[:, 1].view(B, 1, 1) * y + n[:, 2].view(B, 1, 1)
        t = torch.where(nd < -1e-6, c / nd, torch.full_like(D, 6.0))
        D = torch.minimum(D, torch.where(t > 0, t, torch.full_like(D, 6.0)))
    return D.clamp(0.5, 6.0), x.expand(B, H, W), y.expand(B, H, W)


def _scene(seed, B, H, W, dh, dw):
    """Point map (x/z, y/z, logz) [B, H, W, 3] of a network that is a few percent off in a smooth way and 5 mm noisy,
    in an affine frame (depth ~ 1.3 exp(logz) + 0.05); the LiDAR prompt [B, dh, dw] with 5 mm noise and 3 % outliers;
    its confidence in {0, 1, 2} with shares 0.1, 0.2, 0.7."""
    g = _gen(seed)
    D, x, y = _room(g, B, H, W)
    smooth = F.interpolate(_normal(g, B, 1, 6, 8), size=(H, W), mode="bicubic", align_corners=True)[:, 0].double()
    net = D * (1.0 + 0.015 * smooth) + 0.005 * _normal(g, B, H, W).double()
    logz = torch.log(((net - 0.05) / 1.3).clamp_min(0.05))
    points = torch.stack([x, y, logz], -1).float().contiguous()
    iy = (torch.arange(dh, device=DEVICE) * H) // dh
    ix = (torch.arange(dw, device=DEVICE) * W) // dw
    lidar = D[:, iy][:, :, ix] + 0.005 * _normal(g, B, dh, dw).double()
    out = _uniform(g, B, dh, dw) < 0.03
    lidar = torch.where(out, lidar * (0.5 + _uniform(g, B, dh, dw).double()), lidar).float().contiguous()
    u = _uniform(g, B, dh, dw)
    conf = (u >= 0.1).float() + (u >= 0.3).float()
    return points, lidar, conf.contiguous()


def _surface(seed, n):
    """`n` unique voxels (0, x, y, z) in increasing order: sheets over the (x, y) plane, smooth height fields with one
    voxel per column and sheet, so that a voxel has about nine or ten of its 27 neighbours."""
    g = _gen(seed)
    side = max(24, int(math.sqrt(n / 3.0)))
    grid = torch.arange(side, device=DEVICE)
    X, Y = torch.meshgrid(grid, grid, indexing="ij")
    got, total, k = [], 0, 0
    while total < n:
        h = F.interpolate(_normal(g, 1, 1, 6, 6), size=(side, side), mode="bicubic", align_corners=True)[0, 0]
        z = (64 * k + 32 + (0.06 * side * h).clamp(-28, 28)).round().long()
        got.append((X * side + Y) * 4096 + z)
        total += side * side
        k += 1
    key = torch.cat([q.reshape(-1) for q in got]).unique()[:n]
    coords = torch.stack([torch.zeros_like(key), key // 4096 // side, key // 4096 % side, key % 4096], 1)
    return coords.int().contiguous(), (1, side, side, 64 * k)


@functools.lru_cache(maxsize=4)
def _refiner_weights(C, blocks, precision):
    """A single-level refiner whose updates are about a percent of the depth, as a trained one's are."""
    from promptmoge_amd import spec

    w = spec.make_weights(C, blocks, seed=3, precision=precision)
    w.out_w, w.out_b = w.out_w * np.float32(0.02), w.out_b * np.float32(0.02)
    for b in w.blocks:
        b.clip1, b.clip2 = CLIP1, CLIP2
    return w


@functools.lru_cache(maxsize=2)
def _unet_weights(channels, enc):
    from promptmoge_amd import unet_weights

    w = unet_weights.make_unet_weights([int(c) for c in channels.split()], enc, seed=1)
    w.out_w, w.out_b = w.out_w * np.float32(0.02), w.out_b * np.float32(0.02)
    for layer in w.quantised_layers().values():
        if hasattr(layer, "clip1"):
            layer.clip1, layer.clip2 = CLIP1, CLIP2
        else:
            layer.clip = CLIP_LINEAR
    return w


def _encoder(case, seed):
    """Encoder feature and bias map of a U-Net's token grid."""
    channels = [int(c) for c in case["channels"].split()]
    ds = 2 ** (len(channels) - 1)
    g = _gen(seed + 1_000_003)
    h, w = case["H"] // ds, case["W"] // ds
    return _normal(g, case["B"], case["enc"], h, w), 0.1 * _normal(g, case["B"], channels[-1], h, w)


# ----------------------------------------------------------------------------------------------------- prepare and run
def _inputs(case, seed):
    """A case's input tensors, by name."""
    k = case["kind"]
    if k == "fit":
        points, lidar, conf = _scene(seed, case["B"], case["h"], case["w"], case["h"], case["w"])
        return {"z": torch.exp(points[..., 2]).contiguous(), "target": lidar, "mask": conf >= 2}
    if k == "fill":
        _, lidar, conf = _scene(seed, case["B"], case["h"], case["w"], case["h"], case["w"])
        g = _gen(seed + 11)
        hole = _uniform(g, *lidar.shape) < case["holes"]
        for b in range(case["B"]):
            for _ in range(4):
                i, j = (int(v) for v in (_uniform(g, 2) * torch.tensor([case["h"], case["w"]], device=DEVICE)).long())
                hole[b, i:i + case["patch"], j:j + case["patch"]] = True
        return {"depth": torch.where(hole, torch.zeros_like(lidar), lidar), "conf": conf}
    if k == "gauge":
        points, lidar, conf = _scene(seed, case["B"], case["H"], case["W"], case["h"], case["w"])
        return {"depth": (1.3 * torch.exp(points[..., 2]) + 0.05).contiguous(), "lidar": lidar, "conf": conf}
    if k == "step":
        points, lidar, conf = _scene(seed, case["B"], case["H"], case["W"], case["dh"], case["dw"])
        return {"points": points, "lidar": lidar, "conf": conf}
    if k in ("unet", "unet_step"):
        points, lidar, conf = _scene(seed, case["B"], case["H"], case["W"], case["H"], case["W"])
        enc, bias = _encoder(case, seed)
        if k == "unet_step":
            return {"points": points, "lidar": lidar, "conf": conf, "enc": enc, "bias": bias}
        g = _gen(seed + 5)
        n = case["B"] * case["H"] * case["W"]
        prompt = torch.stack([0.02 * _normal(g, n), _uniform(g, n)], 1).contiguous()
        return {"feats": points.reshape(n, 3), "prompt": prompt, "enc": enc, "bias": bias}
    if k == "level":
        points, _, _ = _scene(1, 1, case["H"], case["W"], case["H"], case["W"])  # one scene: its voxel counts
        zq = torch.round(points[0, ..., 2] * RESOLUTION).int()
        z = zq - zq.min()
        i, j = torch.meshgrid(torch.arange(case["H"], device=DEVICE), torch.arange(case["W"], device=DEVICE),
                              indexing="ij")
        coords = torch.stack([torch.zeros_like(z), i.int(), j.int(), z], -1).reshape(-1, 4).contiguous()
        feats = 0.5 * _normal(_gen(seed + 7), coords.shape[0], case["C"])
        return {"coords": coords, "shape": (1, case["H"], case["W"], int(z.max()) + 1),
                "feats": feats.to(DTYPES[case["dtype"]])}
    coords, shape = _surface(seed, case["n"])
    g = _gen(seed + 3)
    if k == "conv":
        return {"coords": coords, "shape": shape,
                "feats": (0.5 * _normal(g, coords.shape[0], case["C"])).to(DTYPES[case["dtype"]])}
    x = torch.randint(-127, 128, (coords.shape[0], case["C"]), generator=g, device=DEVICE, dtype=torch.int8)
    return {"coords": coords, "shape": shape, "x": x}


def _conv_weights(C, index):
    """A layer's parameters, on the CPU in fp32: the same in every state, as a model's are."""
    g = torch.Generator().manual_seed(100 + index)
    return 0.05 * torch.randn(C, 3, 3, 3, C, generator=g), 0.05 * torch.randn(C, generator=g)


def _conv_module(case, index):
    from promptmoge_amd.flex_gemm import nn as fnn

    m = fnn.SubmanifoldConv3d(case["C"], case["C"], 3, bias=case.get("bias", True))
    w, b = _conv_weights(case["C"], index)
    with torch.no_grad():
        m.weight.copy_(w)
        if m.bias is not None:
            m.bias.copy_(b)
    return m.to(DEVICE, DTYPES[case["dtype"]]).requires_grad_(False)


@functools.lru_cache(maxsize=1)
def _own_stream():
    """The one stream of a program that keeps its own (a captured step replays only off the default stream)."""
    return torch.cuda.Stream()


def prepare(case, seed):
    k = case["kind"]
    s = dict(_inputs(case, seed), case=case, stream=_own_stream() if case.get("stream") == "own" else None)
    if k == "step":
        from promptmoge_amd.refiner import RefinerStep

        def make(final):
            return RefinerStep(_refiner_weights(case["C"], case["blocks"], case["precision"]), case["B"], case["H"],
                               case["W"], case["dh"], case["dw"], precision=case["precision"],
                               fit_iters=case["iters"], soft_gate=case["soft"], output_gate=case["gate"],
                               anchor=case["anchor"], final_fit=final, post_depth=final)

        s["last"] = make(True)
        s["mid"] = make(False) if case["K"] > 1 else None
        s["out"] = [torch.empty_like(s["points"]) for _ in range(min(case["K"], 2))]
    elif k == "unet_step":
        from promptmoge_amd.unet import UNetStep

        s["step"] = UNetStep(_unet_weights(case["channels"], case["enc"]), case["B"], case["H"], case["W"],
                             precision=case["precision"], fit_iters=case["iters"], final_fit=True, post_depth=True)
        s["out"] = torch.empty_like(s["points"])
    elif k == "unet":
        from promptmoge_amd.unet import UNetRefiner

        s["module"] = UNetRefiner(_unet_weights(case["channels"], case["enc"]), precision=case["precision"])
    elif k == "conv":
        from promptmoge_amd.flex_gemm import ops as fops

        s["module"] = _conv_module(case, 0)
        s["cache"] = fops.build_submanifold_cache(s["coords"], s["shape"], (3, 3, 3))
    elif k == "level":
        from promptmoge_amd.flex_gemm import nn as fnn

        s["conv0"], s["conv1"] = _conv_module(case, 0), _conv_module(case, 1)
        s["pool"], s["up"] = fnn.SparsePool3d(2, 2), fnn.SparseUpsample3d(2)
    elif k == "conv_i8":
        from promptmoge_amd import ops, spec

        C = case["C"]
        w, b = _conv_weights(C, 2)
        q, scale = spec.quantize_weight(w.numpy())
        s["w"] = torch.from_numpy(q).to(DEVICE)
        s["w_scale"], s["bias"] = torch.from_numpy(scale).to(DEVICE), b.to(DEVICE)
        if case["ordered"]:
            _, _, rows, mask = ops.nmap_hash(s["coords"], s["shape"], rows=True, row_mask=True)
            s["order"], s["order_mask"], s["map"] = ops.row_order(mask, rows, window=0 if C == 128 else 1 << 18)
        else:
            s["map"], s["tile_mask"], _ = ops.nmap_hash(s["coords"], s["shape"])
    torch.cuda.synchronize()  # the inputs were made on the default stream
    return s


def run(s):
    case = s["case"]
    with torch.cuda.stream(s["stream"]) if s["stream"] is not None else contextlib.nullcontext():
        return _RUN[case["kind"]](s, case)


def _run_fit(s, case):
    from promptmoge_amd import ops

    return ops.fit_scale_shift(s["z"], s["target"], s["mask"], case["iters"])


def _run_fill(s, case):
    from promptmoge_amd import prompt

    return prompt.nearest_fill(s["depth"], s["conf"])


def _run_gauge(s, case):
    from promptmoge_amd import prompt

    return prompt.prompt_gauge_poly(s["depth"], s["lidar"], s["conf"], case["degree"])


def _run_step(s, case):
    src, fits = s["points"], []
    for k in range(case["K"]):
        dst = s["out"][k % 2]
        step = s["last"] if k == case["K"] - 1 else s["mid"]
        prompt, final = step(src, s["lidar"], s["conf"], out=dst)
        src = dst
    return {"points": src, "prompt": prompt, "final": final, "depth": step.depth}


def _run_unet_step(s, case):
    prompt, final = s["step"](s["points"], s["lidar"], s["conf"], s["enc"], s["bias"], out=s["out"])
    return {"points": s["out"], "prompt": prompt, "final": final, "depth": s["step"].depth}


def _run_unet(s, case):
    shape = torch.Size([case["B"], case["H"], case["W"], 1024, 3])
    return s["module"](s["feats"], None, shape, s["enc"], prompt_feats=s["prompt"], encoder_bias_map=s["bias"])


def _run_conv(s, case):
    shape = torch.Size([*s["shape"], case["C"]])
    return s["module"](s["feats"], s["coords"], shape, neighbor_cache=s["cache"])[0]


def _run_level(s, case):
    shape = torch.Size([*s["shape"], case["C"]])
    x0, cache0 = s["conv0"](s["feats"], s["coords"], shape)
    pooled, coords1, shape1, pool_cache = s["pool"](x0, s["coords"], shape)
    x1, cache1 = s["conv1"](pooled, coords1, shape1)
    up = s["up"](x1, coords1, shape1, output_coords=s["coords"], output_shape=shape, neighbor_cache=pool_cache.T)[0]
    return {"x0": x0, "pooled": pooled, "coords1": coords1, "x1": x1, "up": up}


def _run_conv_i8(s, case):
    from promptmoge_amd import ops

    kw = {"a_scale": CLIP1 / 127, "w_scale": s["w_scale"], "bias": s["bias"], "out_mult": 127 / 20.0}
    if case["ordered"]:
        return ops.spconv_i8_ordered(s["x"], s["map"], s["order"], s["order_mask"], s["w"], ops.EPI_Q, **kw)
    return ops.spconv_i8(s["x"], s["map"], s["tile_mask"], s["w"], ops.EPI_Q, **kw)


_RUN = {"fit": _run_fit, "fill": _run_fill, "gauge": _run_gauge, "step": _run_step, "unet_step": _run_unet_step,
        "unet": _run_unet, "conv": _run_conv, "level": _run_level, "conv_i8": _run_conv_i8}


# ------------------------------------------------------------------------------------------------- work and tolerance
def _fits_work(pixels, times):
    return {"bytes": 12.0 * pixels * times, "flops": 0.0}


def work(case):
    k = case["kind"]
    if k == "fit":
        n = case["B"] * case["h"] * case["w"]
        return {"bytes": 9.0 * n, "flops": 20.0 * n * (case["iters"] + 1)}
    if k == "fill":
        return {"bytes": 16.0 * case["B"] * case["h"] * case["w"], "flops": 0.0}
    if k == "gauge":
        return {"bytes": case["B"] * (8.0 * case["H"] * case["W"] + 8.0 * case["h"] * case["w"]),
                "flops": 3.0 * 60 * case["B"] * case["h"] * case["w"]}
    if k == "step":  # the point map, LiDAR and confidence in and the point map and depth out, per step; the weights
        m, C, layers = case["B"] * case["H"] * case["W"], case["C"], 2 * case["blocks"]
        lp = case["B"] * case["dh"] * case["dw"]
        elt = 1 if case["precision"] == "int8" else 2
        return {"bytes": case["K"] * (24.0 * m + 8.0 * lp + layers * 27 * C * C * elt) + 4.0 * m,
                "flops": case["K"] * layers * 2.0 * C * C * TAPS_SURFACE * m}
    if k in ("unet", "unet_step"):
        ch = [int(c) for c in case["channels"].split()]
        m, elt = case["B"] * case["H"] * case["W"], 1 if case["precision"] == "int8" else 2
        share = [1.0, 0.6, 0.16, 0.036, 0.0084]  # voxels per level, measured on 480x640 maps
        taps = [TAPS_SURFACE, 8.0, 9.0, 9.0, 9.0]
        convs = [4] * (len(ch) - 1) + [4]
        flops = sum(n * 2.0 * c * c * t * s * m for n, c, t, s in zip(convs, ch, taps, share))
        weights = sum(n * 27.0 * c * c * elt for n, c in zip(convs, ch))
        ds = 4 ** (len(ch) - 1)
        enc = 4.0 * (case["enc"] + ch[-1]) * m / ds
        io = (24.0 + 4.0 + 16.0 if k == "unet_step" else 12.0 + 8.0 + 4.0) * m
        return {"bytes": io + enc + weights, "flops": flops}
    elt = {"fp32": 4, "fp16": 2, "bf16": 2}.get(case.get("dtype"), 1)
    C = case["C"]
    if k == "level":
        m = case["H"] * case["W"]
        rows = m + 0.6 * m
        return {"bytes": rows * (2.0 * C * elt + 16) + 0.6 * m * C * elt + m * C * elt + 2 * 27.0 * C * C * elt,
                "flops": 2.0 * C * C * (TAPS_SURFACE * m + 8.0 * 0.6 * m)}
    return {"bytes": case["n"] * (2.0 * C * elt + 4 * TAPS_GENERIC) + 27.0 * C * C * elt,
            "flops": 2.0 * C * C * TAPS_GENERIC * case["n"]}


def tolerance(case):
    k = case["kind"]
    if k == "fill":
        return "exact"  # copies of input values
    if k in ("fit", "gauge"):
        return {"rel": 1e-6}  # fp64 sums, fp32 results: 4e-8 off the result in 64 bits
    if k == "step":
        # A fit that differs in its last bit moves some int8 codes (or fp16 roundings): 4e-6 off the result in 64
        # bits. Later steps voxelise the moved points: a key that rounds the other way changes its neighbourhood, and
        # three steps are 7e-3 off.
        return {"rel": 1e-4, "max": 0.1} if case["K"] == 1 else {"rel": 2e-2, "max": 0.5}
    if k == "unet_step":
        return {"rel": 4e-3, "max": 0.2} if case["precision"] == "int8" else {"rel": 1e-2, "max": 0.5}  # 8e-4 seen
    if k == "unet":
        return {"rel": 2e-2, "max": 0.5}  # 1e-3 to 1e-2 seen: the coarse levels' LayerNorms amplify a rounding
    if k == "conv_i8":
        return {"differ": 1e-5}  # exact sums; the requantisation's ties
    return {"fp32": {"rel": 2e-6, "max": 1e-5}, "fp16": {"rel": 1e-3, "max": 1e-2},
            "bf16": {"rel": 7e-3, "max": 5e-2}}[case["dtype"]]


# --------------------------------------------------------------------------------------------- the same work in 64 bits
def _taps(coords, shape):
    """Index lists (rows, sources) of the 27 taps of a voxel set's submanifold map."""
    c = coords.long()
    ext = [int(v) for v in shape[:4]]
    key = ((c[:, 0] * ext[1] + c[:, 1]) * ext[2] + c[:, 2]) * ext[3] + c[:, 3]
    sk, order = key.sort()
    for di in (-1, 0, 1):
        for dj in (-1, 0, 1):
            for dz in (-1, 0, 1):
                q = c[:, 1:] + torch.tensor([di, dj, dz], device=c.device)
                ok = (q >= 0).all(1)
                for d in range(3):
                    ok &= q[:, d] < ext[d + 1]
                qk = ((c[:, 0] * ext[1] + q[:, 0]) * ext[2] + q[:, 1]) * ext[3] + q[:, 2]
                pos = torch.searchsorted(sk, qk).clamp_max(sk.numel() - 1)
                rows = (ok & (sk[pos] == qk)).nonzero()[:, 0]
                yield rows, order[pos[rows]]


def _conv64(x, taps, w):
    """Submanifold convolution of fp64 rows with a weight (Co, 27, Ci)."""
    out = torch.zeros(x.shape[0], w.shape[0], dtype=torch.float64, device=x.device)
    for v, (rows, src) in enumerate(taps):
        out.index_add_(0, rows, x[src] @ w[:, v].T)
    return out


def _t64(a):
    return torch.as_tensor(np.asarray(a, np.float32)).double().to(DEVICE)


class _Layers64:
    """The refiners' layers in fp64: the int8 contract's codes and scales, or plain products of fp16 weights."""

    def __init__(self, int8):
        self.int8 = int8

    def weight(self, w):
        """(matrix as (Co, ...) fp64, per-channel scale or 1)."""
        w = _t64(w)
        if not self.int8:
            return w.half().double(), 1.0
        s = (w.abs().flatten(1).amax(1) / 127).clamp_min(1e-12)
        return torch.round(w / s.view(-1, *[1] * (w.ndim - 1))).clamp(-127, 127), s

    def codes(self, x, clip):
        """The layer's input as it multiplies the weight, and the factor to undo it."""
        if not self.int8:
            return x, 1.0
        return torch.round(x * (127.0 / clip)).clamp(-127, 127), clip / 127.0

    def conv(self, x, clip, taps, w, b):
        q, a = self.codes(x, clip)
        w, s = self.weight(w)
        return _conv64(q, taps, w.reshape(w.shape[0], 27, -1)) * (a * s) + _t64(b)

    def linear(self, x, lin):
        q, a = self.codes(x, lin.clip)
        w, s = self.weight(lin.w)
        return (q @ w.T) * (a * s) + _t64(lin.b)

    def block(self, x, taps, b):
        h = F.silu(F.layer_norm(x, (x.shape[1],), _t64(b.gamma), _t64(b.beta), 1e-6))
        h = F.silu(self.conv(h, b.clip1, taps, b.w1, b.b1))
        return x + self.conv(h, b.clip2, taps, b.w2, b.b2)

    def input(self, feats, w, prompt):
        x = feats @ _t64(w.in_w).T + _t64(w.in_b)
        return x if prompt is None else x + prompt @ _t64(w.pr_w).T + _t64(w.pr_b)

    def output(self, x, w):
        return x @ _t64(w.out_w).reshape(-1) + _t64(w.out_b).reshape(-1)[0]


def _voxels(logz):
    B, H, W = logz.shape
    zq = torch.round(logz * RESOLUTION).long()
    z = zq - zq.amin((1, 2), keepdim=True)
    b, i, j = torch.meshgrid(*[torch.arange(n, device=DEVICE) for n in (B, H, W)], indexing="ij")
    return torch.stack([b, i, j, z], -1).reshape(-1, 4), [B, H, W, int(z.max()) + 1]


def _coarser(coords, shape):
    """The voxels of the next level (both spatial dims and depth halved) and each voxel's parent."""
    out = [shape[0]] + [-(-s // 2) for s in shape[1:]]
    c = coords.clone()
    c[:, 1:] //= 2
    key = ((c[:, 0] * out[1] + c[:, 1]) * out[2] + c[:, 2]) * out[3] + c[:, 3]
    u, parent = key.unique(return_inverse=True)
    c = torch.stack([u // (out[1] * out[2] * out[3]), u // (out[2] * out[3]) % out[1], u // out[3] % out[2],
                     u % out[3]], 1)
    return c, out, parent


def _mean_pool(x, parent, n):
    s = torch.zeros(n, x.shape[1], dtype=x.dtype, device=x.device).index_add_(0, parent, x)
    return s / torch.bincount(parent, minlength=n).double().view(-1, 1)


def _single64(points, prompt, w, int8):
    B, H, W, _ = points.shape
    L = _Layers64(int8)
    coords, shape = _voxels(points[..., 2])
    taps = list(_taps(coords, shape))
    x = L.input(points.reshape(-1, 3), w, None if prompt is None else prompt)
    for b in w.blocks:
        x = L.block(x, taps, b)
    return L.output(x, w).view(B, H, W)


def _unet64(feats, logz, prompt, enc, bias, w, int8):
    L = _Layers64(int8)
    coords, shape = _voxels(logz)
    x, skips, levels = L.input(feats, w, prompt), [], []
    depth = len(w.channels)
    for k in range(depth):
        taps = list(_taps(coords, shape))
        for b in w.down[k]:
            x = L.block(x, taps, b)
        if k < depth - 1:
            fine = coords
            coords, shape, parent = _coarser(coords, shape)
            levels.append((taps, parent, fine))
            skips.append(x)
            x = L.linear(_mean_pool(x, parent, coords.shape[0]), w.pool[k])
    at = lambda m: m.double()[coords[:, 0], :, coords[:, 1], coords[:, 2]]  # noqa: E731
    e = L.linear(at(enc), w.enc) + at(bias)
    x = L.linear(F.silu(L.linear(torch.cat([x, e], 1), w.fuse0)), w.fuse2)
    for b in w.bott:
        x = L.block(x, taps, b)
    for i in range(depth - 1):
        taps, parent, _ = levels[depth - 2 - i]
        x = L.linear(x, w.up[i])[parent] + skips[depth - 2 - i]
        for b in w.dec[i]:
            x = L.block(x, taps, b)
    return L.output(x, w)


def _fit64(z, target, mask, iters):
    """Trimmed least squares of target ~ s z + t, per batch item; fp64 [B, 2]."""
    got = []
    for b in range(z.shape[0]):
        zz, tt = z[b][mask[b]].double().reshape(-1), target[b][mask[b]].double().reshape(-1)
        n, s, t = zz.numel(), 1.0, 0.0
        if n >= MIN_POINTS:
            k = min(max(int(np.float32(1.0 - TRIM) * np.float32(n)), MIN_POINTS), n)
            keep = torch.ones_like(zz, dtype=torch.bool)
            for it in range(iters + 1):
                a, c = zz[keep], tt[keep]
                ma, mc = a.mean(), c.mean()
                var = ((a - ma) ** 2).sum()
                s = float(((a - ma) * (c - mc)).sum() / var)
                t = float(mc - s * ma)
                if it < iters:
                    r = (s * zz + t - tt).abs() / tt.clamp_min(1e-3)
                    keep = r <= r.kthvalue(k).values
        got.append([s, t])
    return torch.tensor(got, dtype=torch.float64, device=DEVICE)


def _nearest(n, m):
    return (torch.arange(n, device=DEVICE).float() * (torch.tensor(m, device=DEVICE).float() / n)).floor().long()


def _resized(case, lidar, conf, H, W):
    d = lidar[:, _nearest(H, lidar.shape[1]).clamp_max(lidar.shape[1] - 1)]
    c = conf[:, _nearest(H, lidar.shape[1]).clamp_max(lidar.shape[1] - 1)]
    ix = _nearest(W, lidar.shape[2]).clamp_max(lidar.shape[2] - 1)
    return d[:, :, ix].double(), (c[:, :, ix].double() / 2).clamp(0, 1)


def _affine64(logz, d, c, st, soft=False):
    daff = (d - st[:, 1].view(-1, 1, 1)) / st[:, 0].view(-1, 1, 1).clamp_min(1e-6)
    ok = (d > 0) & (daff > 1e-4)
    log_d = torch.where(ok, torch.log(daff.clamp_min(1e-4)), logz)
    return log_d, ((0.15 + 0.85 * c) if soft else c) * ok


def _step64(case, points, lidar, conf, network, soft=False, gate=False, anchor=0.0, final=True):
    """A refine step in fp64: `network(points, prompt features)` gives the update of the log depth."""
    B, H, W, _ = points.shape
    logz = points[..., 2]
    d, c = _resized(case, lidar, conf, H, W)
    valid = (d > 0) & (c >= 0.999)
    st = _fit64(torch.exp(logz), d, valid, case["iters"])
    log_d, g = _affine64(logz, d, c, st, soft)
    new = logz + network(points, torch.stack([(log_d - logz) * g, g], -1).reshape(-1, 2))
    if gate:
        u = torch.where(d > 0, 1 - c * (1 - ((d - 3) / 2).clamp(0, 1)), torch.ones_like(d))
        new = logz + (0.1 + 0.9 * u) * (new - logz)
    if anchor > 0:
        log_d, g = _affine64(new, d, c, _fit64(torch.exp(new), d, valid, case["iters"]))
        new = new + anchor * g * (log_d - new)
    out = {"points": torch.cat([points[..., :2], new[..., None]], -1), "prompt": st}
    if final:
        z = F.adaptive_avg_pool2d(torch.exp(new)[:, None], lidar.shape[1:])[:, 0]
        fit = _fit64(z, lidar.double(), (conf >= 2) & (lidar > 0) & (z > 0), case["iters"])
        depth = fit[:, 0].view(-1, 1, 1) * torch.exp(new) + fit[:, 1].view(-1, 1, 1)
        out["final"], out["depth"] = fit, torch.where(depth > 0, depth, torch.full_like(depth, float("inf")))
    return out


def _gauge64(depth, lidar, conf, degree, iters=3):
    B, H, W = depth.shape
    h, w = lidar.shape[1:]

    def basis(n, m):
        v, u = torch.meshgrid(torch.linspace(-1, 1, n, dtype=torch.float64, device=DEVICE),
                              torch.linspace(-1, 1, m, dtype=torch.float64, device=DEVICE), indexing="ij")
        terms = [torch.ones_like(u), u, v] + ([u * u, u * v, v * v] if degree >= 2 else [])
        return torch.stack(terms, -1)

    out = torch.ones(B, H, W, dtype=torch.float64, device=DEVICE)
    z = F.adaptive_avg_pool2d(depth.double()[:, None], (h, w))[:, 0]
    for b in range(B):
        m = (conf[b] >= 2) & (lidar[b] > 0) & (z[b] > 0)
        if int(m.sum()) < 200:
            continue
        y, A = torch.log(lidar[b][m].double()) - torch.log(z[b][m]), basis(h, w)[m]
        wt = torch.ones_like(y)
        for it in range(iters):
            Aw = A * wt[:, None]
            coef = torch.linalg.solve(Aw.T @ Aw, Aw.T @ (y * wt))
            r = (y - A @ coef).abs()
            wt = (2 * (1.4826 * r.median() + 1e-4) / r.clamp_min(1e-6)).clamp_max(1.0)
        out[b] = torch.exp(basis(H, W) @ coef)
    return out


def _fill64(depth, conf):
    """Every missing pixel takes its nearest valid pixel's depth (ties: smaller column, then smaller row)."""
    out, c_out = depth.double().clone(), conf.double().clone()
    B, h, w = depth.shape
    rows = torch.arange(h, device=DEVICE)
    cols = torch.arange(w, device=DEVICE)
    for b in range(B):
        valid = depth[b] > 0
        if not bool(valid.any()):
            continue
        up = torch.where(valid, rows.view(-1, 1), -10 ** 6).cummax(0).values
        down = torch.where(valid, rows.view(-1, 1), 10 ** 6).flip(0).cummin(0).values.flip(0)
        near = torch.where(rows.view(-1, 1) - up <= down - rows.view(-1, 1), up, down)  # the nearest row per column
        for i in range(h):
            d2 = (near[i] - i).long() ** 2 + (cols.view(-1, 1) - cols) ** 2
            best = (d2 * w + cols).amin(1) % w
            out[b, i] = depth[b][near[i][best], best].double()
        c_out[b] = torch.where(valid, c_out[b], torch.ones_like(c_out[b]))
    return out, c_out


def exact(case, seed):
    s = _inputs(case, seed)
    k = case["kind"]
    if k == "fit":
        st = _fit64(s["z"], s["target"], s["mask"], case["iters"])
        return st[:, 0], st[:, 1]
    if k == "fill":
        return _fill64(s["depth"], s["conf"])
    if k == "gauge":
        return _gauge64(s["depth"], s["lidar"], s["conf"], case["degree"])
    if k == "step":
        w = _refiner_weights(case["C"], case["blocks"], case["precision"])
        points = s["points"].double()
        for i in range(case["K"]):
            r = _step64(case, points, s["lidar"], s["conf"],
                        lambda p, f: _single64(p, f, w, case["precision"] == "int8"), case["soft"], case["gate"],
                        case["anchor"], final=i == case["K"] - 1)
            points = r["points"]
        return r
    if k in ("unet", "unet_step"):
        w, int8 = _unet_weights(case["channels"], case["enc"]), case["precision"] == "int8"
        if k == "unet":
            logz = s["feats"][:, 2].double().view(case["B"], case["H"], case["W"])
            return _unet64(s["feats"].double(), logz, s["prompt"].double(), s["enc"].double(), s["bias"].double(), w,
                           int8).view(-1, 1)
        net = lambda p, f: _unet64(p.reshape(-1, 3), p[..., 2], f, s["enc"].double(),  # noqa: E731
                                   s["bias"].double(), w, int8).view(p.shape[:3])
        return _step64(case, s["points"].double(), s["lidar"], s["conf"], net)
    if k == "conv_i8":
        return None  # whole numbers
    dt = DTYPES[case["dtype"]]

    def conv(x, coords, shape, index):
        w, b = (t.to(dt).double().to(DEVICE) for t in _conv_weights(case["C"], index))
        y = _conv64(x, _taps(coords, shape), w.reshape(case["C"], 27, case["C"]))
        return y + b if case.get("bias", True) else y

    x = s["feats"].double()
    if k == "conv":
        return conv(x, s["coords"], s["shape"], 0)
    x0 = conv(x, s["coords"], s["shape"], 0)
    coords1, shape1, parent = _coarser(s["coords"].long(), list(s["shape"]))
    pooled = _mean_pool(x0, parent, coords1.shape[0])
    x1 = conv(pooled, coords1, shape1, 1)
    return {"x0": x0, "pooled": pooled, "coords1": None, "x1": x1, "up": x1[parent]}
