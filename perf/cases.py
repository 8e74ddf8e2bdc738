"""Performance cases of the library: what its users run, over the sizes they run it at.

Whole networks go through the device-pointer entry points with HIP graphs on, as a serving program
calls them; the layers go through the kernel entry points on device buffers; photos are decoded
RGBA8 host arrays, as an image loader hands them over. Every kind has a plain float64 restatement
(`exact`). Tolerances are about four times what the library was measured to differ from it or, where
one call's roundings feed the next, what a reordered sum changes.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "splatting-rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import splathip  # noqa: E402
from splathip import specs, synth  # noqa: E402

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
DEV = "cuda"
_held = {}   # the contexts a program keeps: one per loaded network, one for the kernels


# --- the cases ----------------------------------------------------------------------------------

def listed():
    return [
        # One photo in fp32, the precision the reference's DA3 binary defaults to: the smallest
        # whole call, ~200 short launches.
        {"name": "da3_one_view_f32", "kind": "da3", "V": 1, "H": 504, "W": 504, "dtype": "f32"},
        # The six-photo reconstruction of a capture in bf16 (27x36 patches a view).
        {"name": "da3_six_views_bf16", "kind": "da3", "V": 6, "H": 378, "W": 504, "dtype": "bf16"},
        # MapAnything on six photos, the benchmark's default workload.
        {"name": "ma_six_views_bf16", "kind": "ma", "V": 6, "H": 392, "W": 518, "dtype": "bf16"},
        # A DA3-Small cross-view block of six photos in fp32: one sequence of all tokens.
        {"name": "block_da3_global_f32", "kind": "block", "S": 1, "L": 5838, "dim": 384, "dtype": "f32"},
        # A MapAnything encoder block of six photos: per-view attention, 1024 wide.
        {"name": "block_encoder_bf16", "kind": "block", "S": 6, "L": 1037, "dim": 1024, "dtype": "bf16"},
        # An information-sharing block over 24 photos' tokens and the scale token: the long sequence.
        {"name": "block_global_24_views_bf16", "kind": "block", "S": 1, "L": 24889, "dim": 768, "dtype": "bf16"},
        # Three thumbnails (11x17 patches): ragged rows, a few tiles a launch, latency counts.
        {"name": "block_small_ragged_f16", "kind": "block", "S": 3, "L": 188, "dim": 384, "dtype": "f16"},
        # A residual convolution unit of MapAnything's DPT head at a quarter of the resolution.
        {"name": "unit_256_bf16", "kind": "unit", "V": 6, "H": 112, "W": 148, "C": 256, "dtype": "bf16"},
        # The same unit of the DA3-Small head, fp32.
        {"name": "unit_64_f32", "kind": "unit", "V": 6, "H": 108, "W": 144, "C": 64, "dtype": "f32"},
        # MapAnything's output stage in f16 (the reference binary's default precision): 3x3 to 128
        # channels, resize to the image, 3x3 with ReLU.
        {"name": "tail_f16", "kind": "tail", "V": 6, "R": 28, "Cc": 37, "dtype": "f16"},
        # Six decoded 3-megapixel photos to MapAnything's model input.
        {"name": "photos_six_3mp", "kind": "photos", "n": 6, "H": 1512, "W": 2016},
        # Cameras, unprojection and multi-view cleaning of six views.
        {"name": "geometry_six_views", "kind": "geometry", "V": 6, "H": 378, "W": 504},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "unit", "unit", "tail", "da3", "ma", "photos", "geometry"])
    if kind == "block":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        dim = rng.choice([384, 768, 1024])
        V, patches = _log_int(rng, 1, 24 if dtype != "f32" else 8), rng.randint(12, 37) * rng.randint(9, 37)
        if rng.random() < 0.5:
            return {"kind": kind, "S": V, "L": 1 + patches, "dim": dim, "dtype": dtype}
        return {"kind": kind, "S": 1, "L": min(V * (1 + patches) + rng.randint(0, 1), 24889), "dim": dim, "dtype": dtype}
    if kind == "unit":
        C = rng.choice([64, 128, 256])
        s = rng.choice([1, 2, 4])
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        return {"kind": kind, "V": _log_int(rng, 1, 8), "H": s * rng.randint(12, 37), "W": s * rng.randint(12, 37),
                "C": C, "dtype": dtype}
    if kind == "tail":
        return {"kind": kind, "V": _log_int(rng, 1, 8), "R": rng.randint(12, 37), "Cc": rng.randint(12, 37),
                "dtype": rng.choice(["bf16", "f16"])}
    if kind == "da3":
        long, short = 504, 14 * rng.randint(18, 36)
        H, W = (long, short) if rng.random() < 0.5 else (short, long)
        return {"kind": kind, "V": rng.randint(1, 6), "H": H, "W": W, "dtype": rng.choice(["f32", "bf16", "f16"])}
    if kind == "ma":
        W, H = rng.choice([(392, 518), (518, 392), (518, 336), (336, 518), (518, 294), (294, 518)])
        return {"kind": kind, "V": rng.randint(1, 6), "H": H, "W": W, "dtype": "bf16"}
    if kind == "photos":
        W = _log_int(rng, 640, 4032)
        return {"kind": kind, "n": rng.randint(1, 4), "H": int(W * rng.choice([0.5625, 0.667, 0.75, 1.333])) | 1, "W": W}
    return {"kind": kind, "V": rng.randint(2, 12), "H": 14 * rng.randint(18, 36), "W": 14 * rng.randint(24, 37)}


# --- what a program has in hand -----------------------------------------------------------------

def _context(key, load=None):
    if key not in _held:
        ctx = splathip.Context(0)
        if load is not None:
            load(ctx)
        _held[key] = ctx
    return _held[key]


def _weights(kind):
    """The network's checkpoint: one trained model serves every input. LayerScale 1, so that every
    block weighs in the outputs."""
    shapes = synth.da3_shapes(specs.DA3_VARIANTS["small"]) if kind == "da3" else synth.ma_shapes(specs.MA_SPECS["baseline_l"])
    return synth.generate(shapes, seed=7, layer_scale=1.0)


def _network(kind, dtype):
    def load(ctx):
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "w.safetensors")
            synth.save(path, _weights(kind))
            if kind == "da3":
                # The middle view is the reference: the automatic choice is a comparison of nearly
                # equal scores, which a rounding of the class tokens could decide either way.
                ctx.load_da3(path, "small", dtype, specs.REF_MIDDLE)
            else:
                ctx.load_mapanything(path, specs.MA_SPECS["baseline_l"], dtype)
        ctx.set_graphs(True)
    return _context((kind, dtype), load)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, device=DEV, generator=g) * scale


def _views(c, seed):
    """Photos of one scene, normalised: smooth colour fields shared by the views, with detail."""
    g = _gen(seed)
    V, H, W = c["V"], c["H"], c["W"]
    y = torch.linspace(0, 1, H, device=DEV)[:, None]
    x = torch.linspace(0, 1, W, device=DEV)[None, :]
    img = torch.full((V, 3, H, W), 0.5, device=DEV)
    for v in range(V):
        for ch in range(3):
            for _ in range(4):
                f = torch.rand(3, device=DEV, generator=g)
                img[v, ch] += 0.12 * torch.sin(6.28 * ((0.5 + 2.5 * f[0]) * x + (0.5 + 2.5 * f[1]) * y + f[2]))
    img += 0.05 * (torch.rand(V, 3, H, W, device=DEV, generator=g) - 0.5) * 3.46
    mean = torch.tensor(specs.IMAGENET_MEAN, device=DEV).view(1, 3, 1, 1)
    std = torch.tensor(specs.IMAGENET_STD, device=DEV).view(1, 3, 1, 1)
    return ((img.clamp(0, 1) - mean) / std).contiguous()


def _block_inputs(c, seed):
    """A pre-norm block with its LayerNorms folded into qkv and fc1, as the library's loader lays
    it out, and the residual rows."""
    g = _gen(seed)
    d, T, td = c["dim"], c["S"] * c["L"], TORCH[c["dtype"]]
    s = {"x": _randn(g, T, d) + _randn(g, d, scale=0.5)}
    for name, n, k in (("qkv", 3 * d, d), ("proj", d, d), ("fc1", 4 * d, d), ("fc2", d, 4 * d)):
        s["w_" + name] = _randn(g, n, k, scale=k ** -0.5).to(td)
        s["b_" + name] = _randn(g, n, scale=0.1)
        if name in ("qkv", "fc1"):
            s["c1_" + name] = s["w_" + name].double().sum(1).float()
    s["ls1"] = 0.1 + 0.4 * torch.rand(d, device=DEV, generator=g)
    s["ls2"] = 0.1 + 0.4 * torch.rand(d, device=DEV, generator=g)
    return s


def _conv_weights(g, cout, cin, td):
    """[cout, 9 * cin] rows, k = (ky * 3 + kx) * cin + ci (9 * cin is a multiple of 64 here)."""
    return _randn(g, cout, 9 * cin, scale=(9 * cin) ** -0.5).to(td), _randn(g, cout, scale=0.1)


def _unit_inputs(c, seed):
    g = _gen(seed)
    td, C = TORCH[c["dtype"]], c["C"]
    s = {"x": _randn(g, c["V"], c["H"], c["W"], C).to(td)}
    s["w1"], s["b1"] = _conv_weights(g, C, C, td)
    s["w2"], s["b2"] = _conv_weights(g, C, C, td)
    return s


def _tail_inputs(c, seed):
    g = _gen(seed)
    td = TORCH[c["dtype"]]
    s = {"x": _randn(g, c["V"], 8 * c["R"], 8 * c["Cc"], 256).to(td)}
    s["w1"], s["b1"] = _conv_weights(g, 128, 256, td)
    s["w2"], s["b2"] = _conv_weights(g, 128, 128, td)
    return s


def _photo_arrays(c, seed):
    g = _gen(seed)
    out = []
    for _ in range(c["n"]):
        y = torch.arange(c["H"], device=DEV)[:, None, None]
        x = torch.arange(c["W"], device=DEV)[None, :, None]
        f = torch.rand(4, device=DEV, generator=g)
        k = torch.tensor([17.0, 23.0, 31.0], device=DEV)
        rgb = 127 + 90 * torch.sin(x / (k + 9 * f[0]) + y / (29 + 40 * f[1]) + 6 * f[2]) + 12 * torch.randn(
            c["H"], c["W"], 3, device=DEV, generator=g)
        alpha = torch.full((c["H"], c["W"], 1), 255.0, device=DEV)
        out.append(torch.cat([rgb, alpha], 2).clamp(0, 255).to(torch.uint8).cpu().numpy())
    return out


def _geometry_inputs(c, seed):
    """Cameras close together looking at one surface whose depth maps disagree by a few percent."""
    g = _gen(seed)
    V, H, W = c["V"], c["H"], c["W"]
    y = torch.linspace(0, 1, H, device=DEV)[:, None]
    x = torch.linspace(0, 1, W, device=DEV)[None, :]
    f = torch.rand(3, device=DEV, generator=g)
    surface = 2.0 + 0.4 * torch.sin(5 * x + 6 * f[0]) + 0.3 * torch.cos(4 * y + 6 * f[1])
    depth = surface * (1 + 0.03 * _randn(g, V, H, W))
    pose = torch.zeros(V, 9, device=DEV)
    pose[:, :3] = _randn(g, V, 3, scale=0.05)
    pose[:, 3:6] = _randn(g, V, 3, scale=0.02)
    pose[:, 6] = 1.0
    pose[:, 7:] = 0.9 + 0.1 * torch.rand(V, 2, device=DEV, generator=g)
    return {"depth": depth.contiguous(), "pose": pose, "conf": 1 + torch.exp(_randn(g, V, H, W)),
            "fg": (torch.rand(V, H, W, device=DEV, generator=g) < 0.9).to(torch.uint8)}


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, device=DEV, dtype=dtype)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("da3", "ma"):
        V, H, W = c["V"], c["H"], c["W"]
        s = {"c": c, "ctx": _network(kind, c["dtype"]), "images": _views(c, seed)}
        if kind == "da3":
            s["out"] = {"depth": _empty(V, H, W), "depth_conf": _empty(V, H, W),
                        "ray_logits": _empty(V, 7, 8 * (H // 14), 8 * (W // 14)), "pose_encoding": _empty(V, 9),
                        "camera_tokens": _empty(V, 768)}
            s["ref"] = _empty(1, dtype=torch.int32)
        else:
            s["out"] = {"raw": _empty(V, 6, H, W), "quaternion": _empty(V, 4), "translation": _empty(V, 3),
                        "scale": _empty(1), "points": _empty(V, H, W, 3), "conf": _empty(V, H, W),
                        "mask": _empty(V, H, W, dtype=torch.uint8)}
        s["ptrs"] = {k: t.data_ptr() for k, t in s["out"].items()}
    elif kind == "block":
        d, T, td = c["dim"], c["S"] * c["L"], TORCH[c["dtype"]]
        s = {"c": c, "ctx": _context("kernels"), **_block_inputs(c, seed)}
        s["out"] = {"qkv": _empty(T, 3 * d, dtype=td), "att": _empty(T, d, dtype=td), "x1": _empty(T, d),
                    "hid": _empty(T, 4 * d, dtype=td), "x2": _empty(T, d)}
        s["st0"], s["st1"], s["st2"] = (_empty(T, d // 64, 2) for _ in range(3))
        if c["dtype"] != "f32":
            s["h0"], s["h1"], s["h2"] = (_empty(T, d, dtype=td) for _ in range(3))
    elif kind == "unit":
        s = {"c": c, "ctx": _context("kernels"), **_unit_inputs(c, seed)}
        s["out"] = {"mid": torch.empty_like(s["x"]), "y": torch.empty_like(s["x"])}
    elif kind == "tail":
        td = TORCH[c["dtype"]]
        s = {"c": c, "ctx": _context("kernels"), **_tail_inputs(c, seed)}
        H, W = 14 * c["R"], 14 * c["Cc"]
        s["out"] = {"a": _empty(c["V"], 8 * c["R"], 8 * c["Cc"], 128, dtype=td), "up": _empty(c["V"], H, W, 128, dtype=td),
                    "y": _empty(c["V"], H, W, 128, dtype=td)}
    elif kind == "photos":
        W, H = splathip.ma_input_size([(c["W"], c["H"])] * c["n"])
        s = {"c": c, "ctx": _context("kernels"), "photos": _photo_arrays(c, seed)}
        s["out"] = {"images": _empty(c["n"], 3, H, W), "foreground": _empty(c["n"], H, W, dtype=torch.uint8)}
    else:
        V, H, W = c["V"], c["H"], c["W"]
        s = {"c": c, "ctx": _context("kernels"), **_geometry_inputs(c, seed)}
        s["out"] = {"cameras": _empty(V, 16, dtype=torch.float64), "points": _empty(V, H, W, 3), "conf": _empty(V, H, W)}
    torch.cuda.synchronize()
    return s


# --- one pass -------------------------------------------------------------------------------------

def run(s):
    c, ctx, out = s["c"], s["ctx"], s["out"]
    kind = c["kind"]
    if kind == "da3":
        ctx.da3_forward_raw_device(s["images"].data_ptr(), c["V"], c["H"], c["W"], s["ptrs"], s["ref"].data_ptr())
        return {**out, "reference_view": s["ref"]}
    if kind == "ma":
        ctx.ma_forward_device(s["images"].data_ptr(), c["V"], c["H"], c["W"], s["ptrs"])
        return out
    if kind == "photos":
        ctx.ma_model_inputs_device(s["photos"], out["images"].data_ptr(), out["foreground"].data_ptr())
        return out
    if kind == "geometry":
        ctx.kernel_reconstruct(c["V"], c["H"], c["W"], depth=s["depth"].data_ptr(), pose_encoding=s["pose"].data_ptr(),
                               conf=s["conf"].data_ptr(), foreground=s["fg"].data_ptr(),
                               cameras=out["cameras"].data_ptr(), points=out["points"].data_ptr(),
                               conf_out=out["conf"].data_ptr())
        return out
    dt = splathip.DTYPES[c["dtype"]]
    if kind == "unit":
        V, H, W, C = c["V"], c["H"], c["W"], c["C"]
        ctx.kernel_conv2d(dt, s["x"].data_ptr(), V, H, W, C, s["w1"].data_ptr(), C, 9 * C, 3, 1, s["b1"].data_ptr(), 1, 0,
                          0, out["mid"].data_ptr())
        ctx.kernel_conv2d(dt, out["mid"].data_ptr(), V, H, W, C, s["w2"].data_ptr(), C, 9 * C, 3, 1, s["b2"].data_ptr(), 1,
                          0, s["x"].data_ptr(), out["y"].data_ptr())
        return out
    if kind == "tail":
        V, h, w, H, W = c["V"], 8 * c["R"], 8 * c["Cc"], 14 * c["R"], 14 * c["Cc"]
        ctx.kernel_conv2d(dt, s["x"].data_ptr(), V, h, w, 256, s["w1"].data_ptr(), 128, 9 * 256, 3, 1, s["b1"].data_ptr(),
                          0, 0, 0, out["a"].data_ptr())
        ctx.kernel_resize_bilinear(dt, out["a"].data_ptr(), V, h, w, 128, out["up"].data_ptr(), H, W)
        ctx.kernel_conv2d(dt, out["up"].data_ptr(), V, H, W, 128, s["w2"].data_ptr(), 128, 9 * 128, 3, 1,
                          s["b2"].data_ptr(), 0, 1, 0, out["y"].data_ptr())
        return out
    S, L, d = c["S"], c["L"], c["dim"]
    T, f32 = S * L, c["dtype"] == "f32"
    p = lambda k: s[k].data_ptr()  # noqa: E731
    o = lambda k: out[k].data_ptr()  # noqa: E731
    ctx.kernel_ln_stats(p("x"), T, d, 64, p("st0"), dt, 0 if f32 else p("h0"))
    ctx.kernel_gemm_ln(dt, p("x") if f32 else p("h0"), T, d, p("w_qkv"), 3 * d, d, p("b_qkv"), 0, o("qkv"), f32,
                       ln_in=p("st0"), c1=p("c1_qkv"))
    ctx.kernel_attention(dt, o("qkv"), o("att"), S, L, d // 64)
    ctx.kernel_gemm_ln(dt, o("att"), T, d, p("w_proj"), d, d, p("b_proj"), 0, o("x1"), True, gamma=p("ls1"), res=p("x"),
                       ln_out=p("st1"), copy=0 if f32 else p("h1"))
    ctx.kernel_gemm_ln(dt, o("x1") if f32 else p("h1"), T, d, p("w_fc1"), 4 * d, d, p("b_fc1"), 2, o("hid"), f32,
                       ln_in=p("st1"), c1=p("c1_fc1"))
    ctx.kernel_gemm_ln(dt, o("hid"), T, 4 * d, p("w_fc2"), d, 4 * d, p("b_fc2"), 0, o("x2"), True, gamma=p("ls2"),
                       res=o("x1"), ln_out=p("st2"), copy=0 if f32 else p("h2"))
    return out if f32 else {**out, "x2_copy": s["h2"]}


# --- bytes and operations ---------------------------------------------------------------------------

def _vit_flops(T, S, L, d, hidden):
    return 2.0 * T * (4 * d * d + 2 * d * hidden) + 4.0 * S * L * L * d


def _fusion_flops(F, V, sizes):
    """Residual units and 1x1s of a fusion chain, `sizes` coarse to fine (pixels a view)."""
    return sum(2.0 * V * px * (9 * F * F * (2 if i == 0 else 4) + F * F) for i, px in enumerate(sizes))


def _adapter_flops(V, P, quarter, hin, dims, F):
    """1x1 projections, resizes (x4, x2, 1, /2) and the 3x3 to F features of the four levels."""
    c0, c1, c2, c3 = dims
    fl = sum(2.0 * V * P * h * c for h, c in zip(hin, dims))
    fl += 2.0 * V * P * (16 * c0 * c0 + 4 * c1 * c1) + 2.0 * V * quarter * 9 * c3 * c3
    return fl + 2.0 * V * 9 * F * (16 * P * c0 + 4 * P * c1 + P * c2 + quarter * c3)


def work(case):
    c, kind = case, case["kind"]
    es = 4 if c.get("dtype") == "f32" else 2
    if kind in ("da3", "ma"):
        V, H, W = c["V"], c["H"], c["W"]
        R, Cc = H // 14, W // 14
        P, n, q, hw = R * Cc, R * Cc + 1, ((R + 1) // 2) * ((Cc + 1) // 2), H * W
        if kind == "da3":
            fl = 2.0 * V * P * 588 * 384 + 8 * _vit_flops(V * n, V, n, 384, 1536) + 4 * _vit_flops(V * n, 1, V * n, 384, 1536)
            fl += _adapter_flops(V, P, q, [768] * 4, (48, 96, 192, 384), 64) + 2 * _fusion_flops(64, V, (q, P, 4 * P, 16 * P))
            fl += 2.0 * V * 64 * P * 9 * (64 * 32 * 6 + 32 * 32) + 2.0 * V * hw * (9 * 32 * 32 + 64) + 2.0 * V * 64 * P * 7 * 32
            return {"bytes": V * hw * (12 + 8) + 28.0 * 64 * P * V + 26.8e6 * es, "flops": fl}
        fl = 2.0 * V * P * 588 * 1024 + 24 * _vit_flops(V * n, V, n, 1024, 4096) + 2.0 * V * n * 1024 * 768
        T = V * n + 1
        fl += 12 * _vit_flops(T, 1, T, 768, 3072) + 12 * _vit_flops(V * n, V, n, 768, 3072)
        fl += _adapter_flops(V, P, q, (1024, 768, 768, 768), (96, 192, 384, 768), 256)
        fl += _fusion_flops(256, V, (q, P, 4 * P, 16 * P)) + 2.0 * V * 64 * P * 9 * 256 * 128 + 2.0 * V * hw * (9 * 128 * 128 + 6 * 128)
        fl += 2.0 * V * P * 784 * (768 + 6 * 784)
        return {"bytes": V * hw * (12 + 24 + 12 + 4 + 1.0) + 500e6 * es, "flops": fl}
    if kind == "block":
        d, T = c["dim"], c["S"] * c["L"]
        # In: the rows and the weights; out: every result that `run` returns (and the second copy).
        by = T * d * 4.0 + 12.0 * d * d * es + T * d * (3 + 1 + 4) * es + T * d * 8.0 + (0 if es == 4 else T * d * 2.0)
        return {"bytes": by, "flops": _vit_flops(T, c["S"], c["L"], d, 4 * d)}
    if kind == "unit":
        px, C = c["V"] * c["H"] * c["W"], c["C"]
        return {"bytes": 3.0 * px * C * es + 18.0 * C * C * es, "flops": 36.0 * px * C * C}
    if kind == "tail":
        lo, hi = 64 * c["V"] * c["R"] * c["Cc"], 196 * c["V"] * c["R"] * c["Cc"]
        return {"bytes": (lo * (256 + 128) + 2.0 * hi * 128) * es, "flops": 18.0 * (lo * 256 * 128 + hi * 128 * 128)}
    if kind == "photos":
        W, H = splathip.ma_input_size([(c["W"], c["H"])] * c["n"])
        taps = 6 * max(1.0, c["W"] / W)
        return {"bytes": c["n"] * (4.0 * c["H"] * c["W"] + 13.0 * H * W),
                "flops": c["n"] * 8.0 * taps * (H * c["W"] + H * W)}
    px = c["V"] * c["H"] * c["W"]
    return {"bytes": px * (4 + 4 + 1 + 12 + 4.0), "flops": px * (30.0 + 40.0 * (c["V"] - 1))}


def tolerance(case):
    """Measured against `exact`, worst output: networks f32 8.8e-7, bf16 6.9e-3, f16 1.4e-3; layers
    f32 6.3e-7, bf16 2.4e-3, f16 3.6e-4; geometry (f64, points stored as f32) 2.5e-8."""
    kind, dtype = case["kind"], case.get("dtype")
    if kind == "photos":
        return "exact"   # bytes: the crate's own f32 order, then a table of 256 normalised values
    if kind == "geometry":
        return {"rel": 1e-7, "max": 1e-6}
    if kind in ("da3", "ma"):
        return {"f32": {"rel": 4e-6, "max": 4e-4}, "bf16": {"rel": 2.5e-2, "max": 0.5, "differ": 5e-3},
                "f16": {"rel": 6e-3, "max": 0.1, "differ": 2e-3}}[dtype]
    return {"f32": {"rel": 3e-6, "max": 1e-4}, "bf16": {"rel": 1e-2, "max": 0.1}, "f16": {"rel": 1.5e-3, "max": 0.02}}[dtype]


# --- the same in 64 bits --------------------------------------------------------------------------

def _d(t):
    return t.to(DEV, torch.float64)


def _ln(x, w=None, b=None, eps=1e-6):
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w + b


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))


def _attend(q, k, v, heads, S):
    """q, k, v [S * L, heads * 64], softmax(q k^T / 8) v per sequence and head, 4096 queries at a time."""
    out, L = torch.empty_like(q), q.shape[0] // S
    for s in range(S):
        for h in range(heads):
            r, cols = slice(s * L, (s + 1) * L), slice(64 * h, 64 * h + 64)
            kt, vh, qh = k[r, cols].t().contiguous(), v[r, cols].contiguous(), q[r, cols].contiguous()
            for a in range(0, L, 4096):
                e = min(L, a + 4096)
                out[s * L + a:s * L + e, cols] = torch.softmax(qh[a:e] @ kt / 8, 1) @ vh
    return out


def _conv3(x, w, b=None, stride=1):
    """3x3, padding 1; x [V, H, W, Cin], w [Cout, 3, 3, Cin]."""
    V, H, W, C = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    out = torch.zeros(V * Ho * Wo, w.shape[0], dtype=x.dtype, device=x.device)
    for ky in range(3):
        for kx in range(3):
            tap = xp[:, ky:ky + stride * (Ho - 1) + 1:stride, kx:kx + stride * (Wo - 1) + 1:stride]
            out += tap.reshape(-1, C) @ w[:, ky, kx].t()
    out = out if b is None else out + b
    return out.reshape(V, Ho, Wo, -1)


def _resize(x, H, W):
    """Bilinear, aligned corners; x [V, h, w, C]."""
    def axis(n, m):
        at = torch.arange(m, dtype=torch.float64, device=DEV) * ((n - 1) / (m - 1) if m > 1 else 0.0)
        lo = at.floor().long().clamp(max=n - 1)
        return lo, (lo + 1).clamp(max=n - 1), at - lo
    y0, y1, fy = axis(x.shape[1], H)
    x0, x1, fx = axis(x.shape[2], W)
    rows = x[:, y0] * (1 - fy)[None, :, None, None] + x[:, y1] * fy[None, :, None, None]
    return rows[:, :, x0] * (1 - fx)[None, None, :, None] + rows[:, :, x1] * fx[None, None, :, None]


def _exact_block(c, seed):
    s = {k: _d(v) for k, v in _block_inputs(c, seed).items()}
    d = c["dim"]

    def folded(x, name):
        m = x.mean(1, keepdim=True)
        rstd = 1 / torch.sqrt(((x - m) ** 2).mean(1, keepdim=True) + 1e-6)
        return rstd * (x @ s["w_" + name].t() - m * s["c1_" + name]) + s["b_" + name]
    qkv = folded(s["x"], "qkv")
    att = _attend(qkv[:, :d], qkv[:, d:2 * d], qkv[:, 2 * d:], d // 64, c["S"])
    x1 = s["x"] + s["ls1"] * (att @ s["w_proj"].t() + s["b_proj"])
    hid = _gelu(folded(x1, "fc1"))
    x2 = x1 + s["ls2"] * (hid @ s["w_fc2"].t() + s["b_fc2"])
    out = {"qkv": qkv, "att": att, "x1": x1, "hid": hid, "x2": x2}
    return out if c["dtype"] == "f32" else {**out, "x2_copy": x2}


class _Net:
    """Weights of a checkpoint in float64 on the GPU, by name."""

    def __init__(self, kind, prefix=""):
        self.w, self.prefix = _weights(kind), prefix

    def __call__(self, name):
        return _d(torch.from_numpy(self.w[self.prefix + name]))

    def has(self, name):
        return self.prefix + name in self.w

    def lin(self, x, name):
        w = self(name + ".weight")
        y = x @ w.reshape(w.shape[0], -1).t()
        return y + self(name + ".bias") if self.has(name + ".bias") else y

    def ln(self, x, name, eps):
        return _ln(x, self(name + ".weight"), self(name + ".bias"), eps)

    def conv3(self, x, name, stride=1):
        w = self(name + ".weight").permute(0, 2, 3, 1).contiguous()
        return _conv3(x, w, self(name + ".bias") if self.has(name + ".bias") else None, stride)

    def conv_t(self, x, name, s):
        w = self(name + ".weight")                      # [Cin, Cout, s, s]
        V, H, W, C = x.shape
        y = (x.reshape(-1, C) @ w.reshape(C, -1)).reshape(V, H, W, w.shape[1], s, s)
        return y.permute(0, 1, 4, 2, 5, 3).reshape(V, H * s, W * s, w.shape[1]) + self(name + ".bias")

    def block(self, x, name, heads, S, shape=None):
        """Pre-norm block on rows [T, d]; shape(q): the qk-norm and rotation of q or k rows."""
        d = x.shape[1]
        qkv = self.lin(self.ln(x, name + ".norm1", 1e-6), name + ".attn.qkv")
        q, k, v = qkv[:, :d], qkv[:, d:2 * d], qkv[:, 2 * d:]
        if shape is not None:
            q, k = shape(q, name + ".attn.q_norm"), shape(k, name + ".attn.k_norm")
        x = x + self.lin(_attend(q, k, v, heads, S), name + ".attn.proj") * self(name + ".ls1.gamma")
        h = _gelu(self.lin(self.ln(x, name + ".norm2", 1e-6), name + ".mlp.fc1"))
        return x + self.lin(h, name + ".mlp.fc2") * self(name + ".ls2.gamma")

    def unit(self, x, name):
        return self.conv3(self.conv3(x.clamp(min=0), name + ".conv1").clamp(min=0), name + ".conv2") + x

    def fuse(self, x, skip, name, H, W):
        if skip is not None:
            x = x + self.unit(skip, name + ".resConfUnit1")
        return self.lin(_resize(self.unit(x, name + ".resConfUnit2"), H, W), name + ".out_conv")

    def tokens(self, images, base):
        """[V, 1 + P, d]: class token and 14x14 patches with the resized positional embedding."""
        V, _, H, W = images.shape
        R, Cc = H // 14, W // 14
        x = images.reshape(V, 3, R, 14, Cc, 14).permute(0, 2, 4, 1, 3, 5).reshape(V, R * Cc, 588)
        x = self.lin(x, base + ".patch_embed.proj")
        pos = self(base + ".pos_embed")[0]
        grid = pos[1:].reshape(37, 37, -1)
        if (R, Cc) != (37, 37):
            grid = torch.einsum("rac,ka->rkc", torch.einsum("abc,ra->rbc", grid, _bicubic(R)), _bicubic(Cc))
        x = torch.cat([self(base + ".cls_token").expand(V, 1, -1), x], 1)
        return x + torch.cat([pos[:1], grid.reshape(R * Cc, -1)])


def _bicubic(n, src=37, a=-0.75):
    m = torch.zeros(n, src, dtype=torch.float64)
    for o in range(n):
        at = (o + 0.5) * src / (n + 0.1) - 0.5
        lo = math.floor(at)
        for k in range(lo - 1, lo + 3):
            t = abs(at - k)
            w = ((a + 2) * t - (a + 3)) * t * t + 1 if t <= 1 else ((a * t - 5 * a) * t + 8 * a) * t - 4 * a
            m[o, min(max(k, 0), src - 1)] += w
    return m.to(DEV)


def _uv(C, R, Cc, aspect):
    """[R, Cc, C] position code added to DA3's head maps."""
    diag, q = math.hypot(aspect, 1), C // 4
    fr = 100.0 ** (torch.arange(q, dtype=torch.float64, device=DEV) / q)

    def code(n, span):
        edge = span / diag * (n - 1) / n
        a = torch.linspace(-edge, edge, n, dtype=torch.float64, device=DEV)[:, None] / fr
        return 0.1 * torch.cat([a.sin(), a.cos()], 1)
    u, v = code(Cc, aspect), code(R, 1.0)
    return torch.cat([u[None].expand(R, Cc, -1), v[:, None].expand(R, Cc, -1)], 2)


def _pyramid(net, hooks, name, resize, rn, uv=None):
    out = []
    for k, x in enumerate(hooks):
        x = net.lin(x, name % k)
        x = x if uv is None else x + uv(x.shape[3], x.shape[1], x.shape[2])
        if k < 2:
            x = net.conv_t(x, resize[k], 4 if k == 0 else 2)
        elif k == 3:
            x = net.conv3(x, resize[3], 2)
        out.append(net.conv3(x, rn(k)))
    return out


def _exact_da3(c, seed):
    net = _Net("da3", "model.")
    images = _views(c, seed).double()
    V, H, W = c["V"], c["H"], c["W"]
    R, Cc, d, base = H // 14, W // 14, 384, "backbone.pretrained"
    P, n = R * Cc, R * Cc + 1
    x = net.tokens(images, base).reshape(V * n, d)
    p = torch.arange(P, device=DEV)
    within = torch.cat([torch.zeros(1, 2, device=DEV).long(), torch.stack([p // Cc + 1, p % Cc + 1], 1)]).repeat(V, 1).double()
    across = (within > 0).double()
    freq = 100.0 ** (-torch.arange(16, dtype=torch.float64, device=DEV) / 16)

    def rotate(pos):
        ang = (pos[:, :, None] * freq)[:, None]                       # [T, 1, 2, 16]

        def shape(t, norm):
            t = net.ln(t.reshape(V * n, 6, 64), norm, 1e-5).reshape(V * n, 6, 2, 2, 16)
            a, b = t[..., 0, :], t[..., 1, :]
            return torch.stack([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], 3).reshape(V * n, d)
        return shape
    ref = V // 2 if V >= 3 else 0
    near, hooks, tokens = x, [], None
    for i in range(12):
        if i == 4:
            cam = net(base + ".camera_token")[0]
            x = x.reshape(V, n, d).clone()
            x[:, 0] = cam[1]
            x[ref, 0] = cam[0]
            x = x.reshape(V * n, d)
        name = "%s.blocks.%d" % (base, i)
        if i >= 4 and i % 2 == 1:
            x = net.block(x, name, 6, 1, rotate(across))
        else:
            x = near = net.block(x, name, 6, V, rotate(within) if i >= 4 else None)
        if i in (5, 7, 9, 11):
            both = torch.cat([near, net.ln(x, base + ".norm", 1e-5)], 1)
            hooks.append(net.ln(both, "head.norm", 1e-5).reshape(V, n, 2 * d)[:, 1:].reshape(V, R, Cc, 2 * d))
            tokens = torch.cat([near, x], 1).reshape(V, n, 2 * d)[:, 0]
    uv = lambda C, r, cc: _uv(C, r, cc, W / H)  # noqa: E731
    s = "head.scratch."
    pyr = _pyramid(net, hooks, "head.projects.%d", ["head.resize_layers.%d" % k for k in range(4)],
                   lambda k: s + "layer%d_rn" % (k + 1), uv)

    def chain(suffix):
        y = None
        for k in (3, 2, 1, 0):
            h, w = (pyr[k - 1].shape[1:3] if k else (8 * R, 8 * Cc))
            y = net.fuse(pyr[3] if k == 3 else y, None if k == 3 else pyr[k], s + "refinenet%d%s" % (k + 1, suffix), h, w)
        return y
    y = _resize(net.conv3(chain(""), s + "output_conv1"), H, W) + uv(32, H, W)
    logits = net.lin(net.conv3(y, s + "output_conv2.0").clamp(min=0), s + "output_conv2.2")
    y = chain("_aux")
    for i in range(5):
        y = net.conv3(y, s + "output_conv1_aux.3.%d" % i)
    y = _ln(net.conv3(y + uv(32, 8 * R, 8 * Cc), s + "output_conv2_aux.3.0"), eps=1e-5).clamp(min=0)
    rays = net.lin(y, s + "output_conv2_aux.3.5").permute(0, 3, 1, 2)
    h = tokens
    for k in (0, 2):
        h = net.lin(h, "cam_dec.backbone.%d" % k).clamp(min=0)
    pose = torch.cat([net.lin(h, "cam_dec.fc_t"), net.lin(h, "cam_dec.fc_qvec"), net.lin(h, "cam_dec.fc_fov.0").clamp(min=0)], 1)
    return {"depth": logits[..., 0].exp(), "depth_conf": 1 + logits[..., 1].exp(), "ray_logits": rays,
            "pose_encoding": pose, "camera_tokens": tokens, "reference_view": None}


def _exact_ma(c, seed):
    net = _Net("ma")
    images = _views(c, seed).double()
    V, H, W = c["V"], c["H"], c["W"]
    R, Cc, d, q = H // 14, W // 14, 768, "info_sharing."
    P, n = R * Cc, R * Cc + 1
    x = net.tokens(images, "encoder.model").reshape(V * n, 1024)
    for i in range(24):
        x = net.block(x, "encoder.model.blocks.%d" % i, 16, V)
    x = x.reshape(V, n, 1024)
    fused = net.ln(x[:, 1:], "fusion_norm_layer", 1e-6)
    seq = net.lin(torch.cat([fused, x[:, :1]], 1), q + "proj_embed")
    seq[0] += net(q + "view_pos_table")[0]
    x = torch.cat([seq.reshape(V * n, d), net("scale_token")[None]])
    hooks = [fused.reshape(V, R, Cc, 1024)]
    for i in range(24):
        name = q + "self_attention_blocks.%d" % i
        x = net.block(x, name, 12, 1) if i % 2 == 0 else torch.cat([net.block(x[:-1], name, 12, V), x[-1:]])
        if i in (11, 17, 23):
            y = net.ln(x, q + "norm", 1e-6)
            hooks.append(y[:-1].reshape(V, n, d)[:, :P].reshape(V, R, Cc, d))
    t = net.lin(y[-1:], "scale_head.proj")
    for k in range(2):
        t = net.lin(t, "scale_head.mlp.%d.0" % k).clamp(min=0)
    scale = net.lin(t, "scale_head.output_proj").exp().clamp(min=1e-8).reshape(1)
    h = "dense_head.0."
    pyr = _pyramid(net, hooks, h + "input_process.%d.0.0", [h + "input_process.%d.0.1" % k for k in range(4)],
                   lambda k: h + "input_process.%d.1" % k)
    y = None
    for k in (3, 2, 1, 0):
        a = pyr[3] if k == 3 else y[:, :pyr[k].shape[1], :pyr[k].shape[2]]
        y = net.fuse(a, None if k == 3 else pyr[k], h + "scratch.refinenet%d" % (k + 1), 2 * a.shape[1], 2 * a.shape[2])
    y = _resize(net.conv3(y, "dense_head.1.conv1"), H, W)
    raw = net.lin(net.conv3(y, "dense_head.1.conv2.0").clamp(min=0), "dense_head.1.conv2.2")
    r = net.lin(hooks[3], "pose_head.proj")
    for blk in range(2):
        z = r
        for k in (1, 2, 3):
            z = net.lin(z, "pose_head.res_conv.%d.res_conv%d" % (blk, k)).clamp(min=0)
        r = r + z
    r = r.reshape(V, P, -1).mean(1)
    for k in (0, 2):
        r = net.lin(r, "pose_head.more_mlps.%d" % k).clamp(min=0)
    quat = net.lin(r, "pose_head.fc_rot")
    ray = raw[..., :3] / raw[..., :3].norm(dim=-1, keepdim=True).clamp(min=1e-8)
    return {"raw": raw.permute(0, 3, 1, 2), "quaternion": quat / quat.norm(dim=1, keepdim=True).clamp(min=1e-8),
            "translation": net.lin(r, "pose_head.fc_t") * scale, "scale": scale,
            "points": ray * raw[..., 3:4].exp() * scale, "conf": 1 + raw[..., 4].exp(), "mask": None}


def _lanczos(n_in, n_out):
    """Rows of normalised Lanczos3 weights [n_out, n_in] (shrinking)."""
    ratio = n_in / n_out
    at = (torch.arange(n_out, dtype=torch.float64) + 0.5) * ratio
    i = torch.arange(n_in, dtype=torch.float64)
    t = (i[None] + 0.5 - at[:, None]) / ratio
    w = torch.where(t.abs() < 3, torch.sinc(t) * torch.sinc(t / 3), torch.zeros_like(t))
    return (w / w.sum(1, keepdim=True)).to(DEV)


def _exact_photos(c, seed):
    tw, th = splathip.ma_input_size([(c["W"], c["H"])] * c["n"])
    scale = max(tw / c["W"], th / c["H"]) + 1e-8
    if scale >= 1:
        return None
    rw, rh = int(c["W"] * scale), int(c["H"] * scale)
    left, top = (rw - tw) // 2, (rh - th) // 2
    wy, wx = _lanczos(c["H"], rh)[top:top + th], _lanczos(c["W"], rw)[left:left + tw]
    mean = torch.tensor(specs.IMAGENET_MEAN, device=DEV).double()
    std = torch.tensor(specs.IMAGENET_STD, device=DEV).double()
    out = []
    for p in _photo_arrays(c, seed):
        planes = [wy @ _d(torch.from_numpy(p[..., k].copy())) @ wx.t() for k in range(3)]
        rgb = (torch.stack(planes).clamp(0, 255) + 0.5).floor()
        out.append((rgb / 255 - mean[:, None, None]) / std[:, None, None])
    return {"images": torch.stack(out), "foreground": None}


def _exact_geometry(c, seed):
    s = {k: _d(v) for k, v in _geometry_inputs(c, seed).items()}
    V, H, W = c["V"], c["H"], c["W"]
    px = torch.arange(W, dtype=torch.float64, device=DEV)[None].expand(H, W)
    py = torch.arange(H, dtype=torch.float64, device=DEV)[:, None].expand(H, W)
    cams = []
    for e in s["pose"]:
        x, y, z, w = (e[3:7] / e[3:7].norm()).tolist()
        rot = torch.tensor([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                            [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                            [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]], dtype=torch.float64, device=DEV)
        cams.append((rot, e[:3], W / 2 / math.tan(float(e[8]) / 2), H / 2 / math.tan(float(e[7]) / 2)))
    r0, t0 = cams[0][:2]
    cams = [(r0.t() @ r, r0.t() @ (t - t0), fx, fy) for r, t, fx, fy in cams]
    points = torch.empty(V, H, W, 3, dtype=torch.float64, device=DEV)
    for v, (r, t, fx, fy) in enumerate(cams):
        d = s["depth"][v]
        points[v] = torch.stack([(px - W / 2) / fx * d, (py - H / 2) / fy * d, d], 2) @ r.t() + t
    seen = points.float().double()
    conf = s["conf"].clone()
    for i in range(V):
        for j in range(V):
            if i == j:
                continue
            r, t, fx, fy = cams[j]
            p = (seen[i] - t) @ r
            u, v = (0.5 * (fx + fy) * p[..., k] / p[..., 2] + (W, H)[k] / 2 for k in (0, 1))
            u, v = ((a.abs() + 0.5).floor() * a.sign() for a in (u, v))
            ok = (s["fg"][i] > 0) & (p[..., 2] > 0) & (u >= 0) & (v >= 0) & (u < W) & (v < H)
            at = torch.where(ok, v * W + u, torch.zeros_like(u)).long()
            take = lambda m: m[j].reshape(-1)[at]  # noqa: E731
            conf[i][ok & (take(s["fg"]) > 0) & (p[..., 2] < 0.98 * take(s["depth"])) & (s["conf"][i] < take(s["conf"]))] = 0
    cam = torch.stack([torch.cat([r.reshape(9), t, torch.tensor([fx, fy, W / 2, H / 2], dtype=torch.float64, device=DEV)])
                       for r, t, fx, fy in cams])
    return {"cameras": cam, "points": points, "conf": conf}


def exact(case, seed):
    c, kind = case, case["kind"]
    with torch.no_grad():
        if kind == "da3":
            return _exact_da3(c, seed)
        if kind == "ma":
            return _exact_ma(c, seed)
        if kind == "block":
            return _exact_block(c, seed)
        if kind == "photos":
            return _exact_photos(c, seed)
        if kind == "geometry":
            return _exact_geometry(c, seed)
        s = {k: _d(v) for k, v in (_unit_inputs if kind == "unit" else _tail_inputs)(c, seed).items()}
        k3 = lambda w: w.reshape(w.shape[0], 3, 3, -1)  # noqa: E731
        if kind == "unit":
            mid = _conv3(s["x"].clamp(min=0), k3(s["w1"]), s["b1"])
            return {"mid": mid, "y": _conv3(mid.clamp(min=0), k3(s["w2"]), s["b2"]) + s["x"]}
        a = _conv3(s["x"], k3(s["w1"]), s["b1"])
        up = _resize(a, 14 * c["R"], 14 * c["Cc"])
        return {"a": a, "up": up, "y": _conv3(up, k3(s["w2"]), s["b2"]).clamp(min=0)}
