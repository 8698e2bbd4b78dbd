"""Performance cases of the framework: what a user's program has it do, through
the package's public entry points, with inputs already on the GPU (host
images for the whole inpainting call, which takes and returns host images).

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the state a program holds before the call
    run(state)           one pass and its outputs
    work(case)           the bytes and operations the path cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    the outputs in 64 bits, by plain torch

Models and contexts are made once per process and kept, as a program that
serves many calls keeps them; weights are random-initialised from fixed seeds
with the distributions the benchmark uses.
"""
from __future__ import annotations

import atexit
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from moebius_cpu_amd import engine as E
from moebius_cpu_amd import pipeline as PL
from moebius_cpu_amd import unet_params as UP
from moebius_cpu_amd import vae_params as VP

GROUPS = 32


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # The smallest call of the framework's kernel sweep: the 1x1 projection of
        # the deepest map. Launch latency counts as much as the product.
        {"name": "conv1x1_8x8_1280", "kind": "conv1x1", "n": 1, "h": 8, "w": 8, "ci": 1280, "co": 1280,
         "f16w": False, "residual": False, "fast": False},
        # The denoise step's most frequent GEMM (attention and resnet projections of
        # the 64x64 level, both guidance branches) on the f16-stored weights that
        # the converter writes, with the residual add.
        {"name": "conv1x1_64x64_320_f16w", "kind": "conv1x1", "n": 2, "h": 64, "w": 64, "ci": 320, "co": 320,
         "f16w": True, "residual": True, "fast": False},
        # A downsampling conv on a ragged map: no size a multiple of a tile, as the
        # region-of-interest encode of a small mask meets it.
        {"name": "conv3x3_s2_ragged", "kind": "conv3x3", "n": 1, "h": 75, "w": 53, "ci": 252, "co": 308, "stride": 2,
         "up": False, "winograd": False, "f16w": False, "fast": False},
        # The benchmark's first configuration: a 3x3 conv and the GroupNorm + SiLU
        # that follows it, at the UNet's widest map.
        {"name": "conv3x3_gn_silu_64x64_320", "kind": "conv_gn", "n": 1, "h": 64, "w": 64, "ci": 320, "co": 320},
        # A whole ResNet block with its time embedding and shortcut.
        {"name": "resnet_block_32x32_320_640", "kind": "resnet", "h": 32, "w": 32, "ci": 320, "co": 640},
        # GroupNorm + SiLU of the VAE's largest map: bound by memory alone.
        {"name": "gn_silu_512x512_128", "kind": "gn", "n": 1, "h": 512, "w": 512, "ci": 128},
        # The framework's headline: one denoise step with classifier-free guidance.
        {"name": "unet_step_cfg", "kind": "unet", "cfg": True, "fast": False},
        # The same step in the f16-product precision that a caller may choose.
        {"name": "unet_step_cfg_fast", "kind": "unet", "cfg": True, "fast": True},
        # The encode of an inpainting call: the image and the masked image.
        {"name": "vae_encode_pair_512", "kind": "encode", "n": 2, "h": 512, "w": 512},
        # The region-of-interest encode of a small mask: an odd number of latents.
        {"name": "vae_encode_roi_216x296", "kind": "encode", "n": 1, "h": 216, "w": 296},
        # The decode every call ends with.
        {"name": "vae_decode_64x64", "kind": "decode", "h": 64, "w": 64},
        # A whole call, host image in and out: crop, resample, encode, nine steps
        # (three guided), decode, resample back, feather paste.
        {"name": "inpaint_fast_1024x768", "kind": "inpaint", "iw": 1024, "ih": 768, "ch": 3, "mw": 400, "mh": 300},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv1x1", "conv1x1", "conv3x3", "conv3x3", "conv_gn", "resnet", "gn", "unet", "encode",
                       "encode", "decode", "decode", "inpaint"])
    if kind == "conv1x1":
        return {"kind": kind, "n": rng.choice([1, 2]), "h": _log(rng, 1, 80), "w": _log(rng, 1, 80),
                "ci": _log(rng, 64, 3200), "co": _log(rng, 64, 3200), "f16w": rng.random() < 0.5,
                "residual": rng.random() < 0.5, "fast": rng.random() < 0.3}
    if kind == "conv3x3":
        h, w = _log(rng, 7, 160), _log(rng, 7, 160)
        most = max(64, min(1280, int(640 * 64 / math.sqrt(h * w))))
        ci, co = _log(rng, 32, most), _log(rng, 32, most)
        form = rng.choice(["winograd", "direct", "stride2", "up"])
        if form == "winograd":
            ci, co = 4 * (ci // 4), 4 * (co // 4)
        return {"kind": kind, "n": rng.choice([1, 2]), "h": h, "w": w, "ci": ci, "co": co,
                "stride": 2 if form == "stride2" else 1, "up": form == "up", "winograd": form == "winograd",
                "f16w": rng.random() < 0.5, "fast": rng.random() < 0.3}
    if kind == "conv_gn":
        return {"kind": kind, "n": rng.choice([1, 2]), "h": _log(rng, 8, 128), "w": _log(rng, 8, 128),
                "ci": GROUPS * rng.randint(1, 16), "co": GROUPS * rng.randint(1, 16)}
    if kind == "resnet":
        return {"kind": kind, "h": _log(rng, 8, 96), "w": _log(rng, 8, 96), "ci": GROUPS * rng.randint(2, 20),
                "co": GROUPS * rng.randint(2, 20)}
    if kind == "gn":
        return {"kind": kind, "n": rng.choice([1, 2]), "h": _log(rng, 8, 360), "w": _log(rng, 8, 360),
                "ci": GROUPS * rng.randint(1, 16)}
    if kind == "unet":
        return {"kind": kind, "cfg": rng.random() < 0.5, "fast": rng.random() < 0.4, "t": rng.randint(1, 999)}
    if kind == "encode":
        return {"kind": kind, "n": rng.choice([1, 2]), "h": 8 * rng.randint(8, 64), "w": 8 * rng.randint(8, 64)}
    if kind == "decode":
        return {"kind": kind, "h": rng.randint(8, 64), "w": rng.randint(8, 64)}
    iw, ih = _log(rng, 400, 1024), _log(rng, 400, 768)
    return {"kind": "inpaint", "iw": iw, "ih": ih, "ch": rng.choice([3, 4]), "mw": rng.randint(24, min(400, iw // 2)),
            "mh": rng.randint(24, min(300, ih // 2))}


# ---------------------------------------------------------------- kept for the process

_kept: dict = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _context(fast: bool) -> E.Context:
    def make():
        c = E.Context(0)
        c.set_precision(fast)
        return c

    return _keep(("context", fast), make)


def _normals(seed: int, shape, std=1.0, mean=0.0) -> np.ndarray:
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return (torch.randn(tuple(shape), generator=g, device="cuda") * std + mean).cpu().numpy()


def _unet_params() -> dict:
    """Weights and biases N(0, 0.02), norm scales 1 + N(0, 0.02)."""
    return _keep("unet params", lambda: {
        s.name: _normals(4000 * 100003 + i, s.shape, 0.02, 1.0 if s.kind == "norm_w" else 0.0)
        for i, s in enumerate(UP.unet_specs())})


def _vae_params() -> dict:
    """Kaiming-normal weights; norm scales 1 + N(0, 0.05), shifts N(0, 0.05), biases N(0, 0.02)."""
    def std(s):
        if s.kind == "weight":
            return math.sqrt(2.0 / float(np.prod(s.shape[1:])))
        return 0.05 if s.kind in ("norm_w", "norm_b") else 0.02

    return _keep("vae params", lambda: {
        s.name: _normals(6000 * 100003 + i, s.shape, std(s), 1.0 if s.kind == "norm_w" else 0.0)
        for i, s in enumerate(VP.vae_specs())})


def _unet(fast: bool):
    from moebius_cpu_amd.unet import UNet

    # the f16-product precision is used with the f16-stored weights of the converter
    return _keep(("unet", fast), lambda: UNet(_context(fast), _unet_params(), f16_gemm=fast))


def _vae():
    from moebius_cpu_amd.vae import Vae

    return _keep("vae", lambda: Vae(_context(False), _vae_params()))


def _engine():
    """The engine over converter-format weight files, removed once they are loaded."""
    def make():
        from moebius_cpu_amd import weights_io as WIO

        d = tempfile.mkdtemp(prefix="moebius_weights_")
        atexit.register(shutil.rmtree, d, True)
        try:
            WIO.write_weights(os.path.join(d, "unet.safetensors"), _unet_params(),
                              [s.name for s in UP.unet_specs() if s.gemm], f16=True)
            WIO.write_weights(os.path.join(d, "vae.safetensors"), _vae_params(),
                              metadata={"scaling_factor": WIO.VAE_SCALING})
            return PL.Engine.load(d)
        finally:
            shutil.rmtree(d, ignore_errors=True)

    return _keep("engine", make)


class _View:
    """A device buffer of the framework as torch sees it (no copy)."""

    def __init__(self, d):
        self.keep = d
        self.__cuda_array_interface__ = {"shape": tuple(d.shape), "typestr": d.dtype.str, "data": (d.ptr, False),
                                         "version": 2}


def _torch(d) -> torch.Tensor:
    return torch.as_tensor(_View(d), device="cuda")


def _kaiming(seed, shape, fan_in):
    return _normals(seed, shape, math.sqrt(2.0 / fan_in))


# ---------------------------------------------------------------- inputs

def _inputs(c, seed) -> dict:
    """The arrays of one case, from the seed alone."""
    s = 64 * int(seed)
    k = c["kind"]
    if k == "conv1x1":
        d = {"x": _normals(s, (c["n"], c["h"], c["w"], c["ci"])), "w": _kaiming(s + 1, (c["co"], c["ci"]), c["ci"]),
             "b": _normals(s + 2, (c["co"],), 0.02)}
        if c["residual"]:
            d["r"] = _normals(s + 3, (c["n"], c["h"], c["w"], c["co"]))
    elif k in ("conv3x3", "conv_gn"):
        d = {"x": _normals(s, (c["n"], c["h"], c["w"], c["ci"])),
             "w": _kaiming(s + 1, (c["co"], 3, 3, c["ci"]), 9 * c["ci"]), "b": _normals(s + 2, (c["co"],), 0.02)}
        if k == "conv_gn":
            d["g"], d["be"] = _normals(s + 3, (c["co"],), 0.1, 1.0), _normals(s + 4, (c["co"],), 0.1)
    elif k == "gn":
        d = {"x": _normals(s, (c["n"], c["h"], c["w"], c["ci"]), 2.0, 0.3), "g": _normals(s + 1, (c["ci"],), 0.1, 1.0),
             "be": _normals(s + 2, (c["ci"],), 0.1)}
    elif k == "resnet":
        ci, co = c["ci"], c["co"]
        d = {"x": _normals(s, (1, c["h"], c["w"], ci)), "temb": _normals(s + 1, (1, 1, 1, 1280)),
             "g1": _normals(s + 2, (ci,), 0.1, 1.0), "b1": _normals(s + 3, (ci,), 0.1),
             "w1": _kaiming(s + 4, (co, 3, 3, ci), 9 * ci), "c1": _normals(s + 5, (co,), 0.02),
             "lw": _normals(s + 6, (co, 1280), 0.02), "lb": _normals(s + 7, (co,), 0.02),
             "g2": _normals(s + 8, (co,), 0.1, 1.0), "b2": _normals(s + 9, (co,), 0.1),
             "w2": _kaiming(s + 10, (co, 3, 3, co), 9 * co), "c2": _normals(s + 11, (co,), 0.02),
             "ws": _kaiming(s + 12, (co, ci), ci), "bs": _normals(s + 13, (co,), 0.02)}
    elif k == "unet":
        i = UP.unet_input(5000 + int(seed))
        d = {"x": i.x, "t": int(c.get("t", i.timestep))}
    elif k == "encode":
        g = torch.Generator(device="cuda").manual_seed(s)
        x = torch.rand((c["n"], c["h"], c["w"], 3), generator=g, device="cuda") * 2 - 1
        d = {"x": x.cpu().numpy(), "noise": _normals(s + 1, (c["n"], c["h"] // 8, c["w"] // 8, 4))}
    elif k == "decode":
        d = {"z": _normals(s, (1, c["h"], c["w"], 4))}
    else:
        r = np.random.RandomState(seed & 0x7FFFFFFF)
        img = r.randint(0, 256, (c["ih"], c["iw"], c["ch"])).astype(np.uint8)
        mask = np.zeros((c["ih"], c["iw"]), np.uint8)
        y, x = r.randint(0, c["ih"] - c["mh"] + 1), r.randint(0, c["iw"] - c["mw"] + 1)
        mask[y:y + c["mh"], x:x + c["mw"]] = 255
        d = {"img": img, "mask": mask, "seed": int(seed) + 1}
    if c.get("f16w"):  # stored in f16, as the converter writes GEMM weights
        d["w"] = d["w"].astype(np.float16)
    return d


# ---------------------------------------------------------------- the calls

def prepare(case, seed):
    d = _inputs(case, seed)
    k = case["kind"]
    if k == "inpaint":
        p = PL.Preset.FAST.params()
        p.seed = d["seed"]
        return {"kind": k, "engine": _engine(), "img": d["img"], "mask": d["mask"], "params": p}
    ctx = _context(bool(case.get("fast")))
    T = lambda a: E.Tensor.from_numpy(ctx, a)  # noqa: E731
    st = {"kind": k, "ctx": ctx}
    if k == "unet":
        st.update(net=_unet(bool(case["fast"])), x=E.DeviceArray.from_numpy(ctx, d["x"]), t=d["t"], cfg=case["cfg"],
                  out=E.DeviceArray(ctx, (2 if case["cfg"] else 1, 64, 64, 4)))
    elif k == "encode":
        st.update(vae=_vae(), x=E.DeviceArray.from_numpy(ctx, d["x"]), noise=E.DeviceArray.from_numpy(ctx, d["noise"]),
                  out=E.DeviceArray(ctx, d["noise"].shape))
    elif k == "decode":
        st.update(vae=_vae(), z=E.DeviceArray.from_numpy(ctx, d["z"]),
                  out=E.DeviceArray(ctx, (1, 8 * case["h"], 8 * case["w"], 3)))
    elif k == "conv1x1":
        w = E.Param(ctx, d["w"], f16=case["f16w"])
        st.update(op=E.Conv1x1(ctx, case["ci"], case["co"], w, d["b"]), x=T(d["x"]),
                  res=T(d["r"]) if case["residual"] else None,
                  out=E.Tensor(ctx, case["n"], case["h"], case["w"], case["co"]))
    elif k in ("conv3x3", "conv_gn"):
        stride, up = case.get("stride", 1), case.get("up", False)
        op = E.Conv3x3(ctx, case["ci"], case["co"], E.Param(ctx, d["w"], f16=case.get("f16w", False)), d["b"],
                       stride=stride, upsample2x=up, winograd=case.get("winograd", k == "conv_gn"))
        ho, wo = op.output_hw(case["h"], case["w"])
        shape = (case["n"], ho, wo, case["co"])
        st.update(op=op, x=T(d["x"]), out=E.Tensor(ctx, *shape))
        if k == "conv_gn":
            st.update(gn=E.GroupNorm(ctx, GROUPS, 1e-5, d["g"], d["be"]), norm=E.Tensor(ctx, *shape))
    elif k == "gn":
        st.update(gn=E.GroupNorm(ctx, GROUPS, 1e-5, d["g"], d["be"]), x=T(d["x"]), out=E.Tensor(ctx, *d["x"].shape))
    else:
        from types import SimpleNamespace

        from moebius_cpu_amd.workloads import ResnetBlockGpu

        wl = SimpleNamespace(x=d["x"], temb=d["temb"], gn1_g=d["g1"], gn1_b=d["b1"], w1=d["w1"], b1=d["c1"],
                             lin_w=d["lw"], lin_b=d["lb"], gn2_g=d["g2"], gn2_b=d["b2"], w2=d["w2"], b2=d["c2"],
                             ws=d["ws"], bs=d["bs"], eps=1e-5)
        st["block"] = ResnetBlockGpu(ctx, wl)
    ctx.synchronize()
    return st


def run(st):
    k = st["kind"]
    if k == "inpaint":
        img = st["img"].copy()  # the call edits the image in place
        p = st["params"]
        rect, lat = st["engine"].inpaint_traced(img, st["mask"], p, PL.NoiseSet.sample(p.seed), latents=True)
        return {"image": img, "latents": lat, "rect": [rect.x, rect.y, rect.w, rect.h]}
    if k == "unet":
        st["net"].forward(st["x"], st["t"], st["cfg"], st["out"])
    elif k == "encode":
        st["vae"].encode(st["x"], st["noise"], st["out"])
    elif k == "decode":
        st["vae"].decode(st["z"], st["out"])
    elif k == "conv1x1":
        st["op"].forward(st["x"], st["out"], st["res"])
    elif k == "conv3x3":
        st["op"].forward(st["x"], st["out"])
    elif k == "conv_gn":
        st["op"].forward(st["x"], st["out"])
        st["gn"].forward(st["out"], None, True, st["norm"])
        return {"conv": _torch(st["out"]), "norm": _torch(st["norm"])}
    elif k == "gn":
        st["gn"].forward(st["x"], None, True, st["out"])
    else:
        return {"out": _torch(st["block"].forward())}
    return {"out": _torch(st["out"])}


# ---------------------------------------------------------------- bytes and operations

def _out_hw(c):
    up = 2 if c.get("up") else 1
    return (c["h"] * up - 1) // c.get("stride", 1) + 1, (c["w"] * up - 1) // c.get("stride", 1) + 1


def _conv3_flops(px, ci, co, same):
    """A stride-1 conv of whole channel quads as F(2x2, 3x3) products, else direct."""
    return (8.0 if same and ci % 4 == 0 and co % 4 == 0 else 18.0) * px * ci * co


def work(case):
    c, k = case, case["kind"]
    wb = 2 if c.get("f16w") else 4
    if k == "conv1x1":
        px, ci, co = c["n"] * c["h"] * c["w"], c["ci"], c["co"]
        return {"bytes": 4.0 * px * (ci + co * (2 if c["residual"] else 1)) + wb * ci * co + 4 * co,
                "flops": 2.0 * px * ci * co}
    if k in ("conv3x3", "conv_gn"):
        ho, wo = _out_hw(c)
        px, ci, co = c["n"] * ho * wo, c["ci"], c["co"]
        out = 2 if k == "conv_gn" else 1
        return {"bytes": 4.0 * c["n"] * c["h"] * c["w"] * ci + 4.0 * px * co * out + wb * 9 * ci * co,
                "flops": _conv3_flops(px, ci, co, c.get("stride", 1) == 1)}
    if k == "gn":
        e = c["n"] * c["h"] * c["w"] * c["ci"]
        return {"bytes": 8.0 * e, "flops": 10.0 * e}
    if k == "resnet":
        px, ci, co = c["h"] * c["w"], c["ci"], c["co"]
        return {"bytes": 4.0 * (px * (ci + co) + 9 * co * (ci + co) + co * ci + 1280 * co),
                "flops": _conv3_flops(px, ci, co, True) + _conv3_flops(px, co, co, True) + 2.0 * px * ci * co}
    if k == "unet":
        b = 2 if c["cfg"] else 1
        return {"bytes": (2.0 if c["fast"] else 4.0) * UP.param_count() + 4.0 * 4096 * (9 + 4 * b),
                "flops": UP.step_flops(b, winograd=True, cfg_shared=True)["total"]}
    vae_bytes = 4.0 * VP.param_count() / 2
    if k == "encode":
        px = c["n"] * c["h"] * c["w"]
        return {"bytes": vae_bytes + 4.0 * px * 3 + 8.0 * px / 16,
                "flops": VP.encode_flops(c["n"], c["h"], c["w"], winograd=True)}
    if k == "decode":
        px = c["h"] * c["w"]
        return {"bytes": vae_bytes + 4.0 * px * (4 + 192), "flops": VP.decode_flops(c["h"], c["w"], winograd=True)}
    # The Fast preset: one region encode and one whole encode, three guided and six
    # plain steps, one decode. The region is the mask's, so at least its own size.
    b2, b1 = (UP.step_flops(b, winograd=True, cfg_shared=True)["total"] for b in (2, 1))
    return {"bytes": 9 * 2.0 * UP.param_count() + 2.0 * VP.param_count() + 2.0 * c["iw"] * c["ih"] * c["ch"],
            "flops": 3 * b2 + 6 * b1 + VP.encode_flops(1, winograd=True) + VP.decode_flops(winograd=True)}


def tolerance(case):
    k = case["kind"]
    if case.get("fast"):
        # f16 products: the operands' rounding (2^-11) decides, whatever the order of the sums
        return {"rel": 5e-3} if k == "unet" else {"rel": 1e-3, "max": 1e-2}
    if k == "inpaint":
        # nine steps and a decode over another order of the sums, then 8-bit rounding: ties of a level
        return {"rel": 2e-5, "max": 2e-3, "differ": 5e-3}
    if k in ("unet", "encode", "decode"):
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 4e-6, "max": 1e-4}


# ---------------------------------------------------------------- the same in 64 bits

def _d(a) -> torch.Tensor:
    return torch.as_tensor(np.asarray(a), device="cuda").double()


def _silu(x):
    return x * torch.sigmoid(x)


def _lin(x, w, b=None):
    y = (x.reshape(-1, x.shape[-1]) @ _d(w).t()).reshape(*x.shape[:-1], w.shape[0])
    return y if b is None else y + _d(b)


def _gnorm(x, eps, g, b):
    n, h, w, c = x.shape
    xs = x.reshape(n, h * w, GROUPS, c // GROUPS)
    mean = xs.mean(dim=(1, 3), keepdim=True)
    var = ((xs - mean) ** 2).mean(dim=(1, 3), keepdim=True)
    y = ((xs - mean) / torch.sqrt(var + float(np.float32(eps)))).reshape(n, h, w, c)
    return y * _d(g) + _d(b)


def _lnorm(x, g, b):
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + float(np.float32(1e-5))) * _d(g) + _d(b)


def _conv(x, w, b, stride=1, up=False, pad=(1, 1, 1, 1)):
    """A 3x3 conv as nine products; w [co, 3, 3, ci], pad top, left, bottom, right."""
    if up:
        x = x.repeat_interleave(2, 1).repeat_interleave(2, 2)
    n, h, wd, ci = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, pad[1], pad[3], pad[0], pad[2]))
    ho, wo = (h + pad[0] + pad[2] - 3) // stride + 1, (wd + pad[1] + pad[3] - 3) // stride + 1
    wt = _d(w)
    out = _d(b).expand(n * ho * wo, -1).clone()
    for ky in range(3):
        for kx in range(3):
            p = xp[:, ky:ky + stride * (ho - 1) + 1:stride, kx:kx + stride * (wo - 1) + 1:stride]
            out += p.reshape(-1, ci) @ wt[:, ky, kx].t()
    return out.reshape(n, ho, wo, -1)


def _depthwise(x, w, b):
    n, h, wd, c = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    wt = _d(w)
    out = _d(b).expand_as(x).clone()
    for ky in range(3):
        for kx in range(3):
            out += xp[:, ky:ky + h, kx:kx + wd] * wt[ky, kx]
    return out


def _exact_unet(x, t, cfg, fast):
    P = _unet_params()
    if fast:  # its GEMM weights are stored in f16
        gemm = {s.name for s in UP.unet_specs() if s.gemm}
        P = {name: v.astype(np.float16) if name in gemm else v for name, v in P.items()}
    branches = [0, 1] if cfg else [1]
    nb = len(branches)
    lin = lambda p, v, bias=True: _lin(v, P[p + ".weight"], P[p + ".bias"] if bias else None)  # noqa: E731

    def dwconv(p, v):
        mid = torch.relu(_depthwise(v, P[p + ".conv_dw.weight"], P[p + ".conv_dw.bias"]))
        y = lin(p + ".conv_pw", mid)
        return y + v if y.shape == v.shape else y

    def resnet(p, v, temb):
        h = dwconv(p + ".conv1", _silu(_gnorm(v, 1e-5, P[p + ".norm1.weight"], P[p + ".norm1.bias"])))
        h = h + lin(p + ".time_emb_proj", _silu(temb))[:, None, None, :]
        h = dwconv(p + ".conv2", _silu(_gnorm(h, 1e-5, P[p + ".norm2.weight"], P[p + ".norm2.bias"])))
        return h + (lin(p + ".conv_shortcut", v) if p + ".conv_shortcut.weight" in P else v)

    def self_lambda(p, v):
        n, hh, ww, c = v.shape
        k = c // 8
        q = lin(p + ".to_q", v).reshape(n, hh * ww, 8, k)
        keys, val = lin(p + ".to_k", v, False).reshape(n, hh * ww, k), lin(p + ".to_v", v)
        sk = torch.softmax(keys, 1)
        out = torch.matmul(q.reshape(n, -1, k), torch.matmul(sk.transpose(1, 2), val.reshape(n, hh * ww, k)))
        out = out.reshape(n, hh, ww, 8, k)
        coef = torch.matmul(q, _d(P[p + ".pos_conv.weight"])).reshape(n, hh, ww, 8, 225)
        out += torch.matmul(q, _d(P[p + ".pos_conv.bias"])).reshape(n, hh, ww, 8, 1)
        vp = torch.nn.functional.pad(val, (0, 0, 7, 7, 7, 7))
        for dy in range(15):
            for dx in range(15):
                out.addcmul_(coef[..., dy * 15 + dx, None], vp[:, dy:dy + hh, dx:dx + ww, None, :])
        return out.reshape(n, hh, ww, c)

    ehs = lin("diff_model.encoder_hid_proj", _d(P["embedding_layer.weight"]))
    ehs = [ehs[10:20], ehs[0:10]]  # without and with the text

    def cross_lambda(p, v):
        n, hh, ww, c = v.shape
        k = c // 8
        q = lin(p + ".to_q", v).reshape(n, hh * ww, 8, k)
        e = _d(P[p + ".rel_pos_emb"])
        out = torch.empty_like(q)
        for i, br in enumerate(branches):
            sk = torch.softmax(lin(p + ".to_k", ehs[br], False), 0)
            val = lin(p + ".to_v", ehs[br])
            out[i] = torch.matmul(q[i], sk.t() @ val) + torch.matmul(torch.matmul(q[i], e.transpose(1, 2)), val)
        return out.reshape(n, hh, ww, c)

    def transformer(p, v):
        b, c = p + ".transformer_blocks.0", v.shape[-1]
        norm = lambda i, u: _lnorm(u, P[f"{b}.norm{i}.weight"], P[f"{b}.norm{i}.bias"])  # noqa: E731
        h = lin(p + ".proj_in", _gnorm(v, 1e-6, P[p + ".norm.weight"], P[p + ".norm.bias"]))
        h = h + self_lambda(b + ".attn1", norm(1, h))
        h = h + cross_lambda(b + ".attn2", norm(2, h))
        a = _silu(lin(b + ".ff.inverted_conv.conv", norm(3, h)))
        a = _depthwise(a, P[b + ".ff.depth_conv.conv.weight"], P[b + ".ff.depth_conv.conv.bias"])
        hid = a.shape[-1] // 2
        return lin(p + ".proj_out", lin(b + ".ff.point_conv.conv", a[..., :hid] * _silu(a[..., hid:]), False) + h) + v

    m = "diff_model"
    # the reference's sinusoid: its angles are 32-bit values
    half = torch.arange(160, dtype=torch.float32)
    freq = torch.exp(-np.float32(math.log(10000.0)) * half / 160)
    arg = (np.float32(t) * freq).double()
    temb = torch.cat([torch.cos(arg), torch.sin(arg)])[None].cuda()
    temb = lin(m + ".time_embedding.linear_2", _silu(lin(m + ".time_embedding.linear_1", temb))).expand(nb, -1)
    skips = [dwconv(m + ".conv_in", _d(x).expand(nb, -1, -1, -1))]
    for i in range(3):
        for j in range(2):
            h = resnet(f"{m}.down_blocks.{i}.resnets.{j}", skips[-1], temb)
            skips.append(transformer(f"{m}.down_blocks.{i}.attentions.{j}", h))
        if i < 2:
            p = f"{m}.down_blocks.{i}.downsamplers.0.conv"
            skips.append(_conv(skips[-1], P[p + ".weight"], P[p + ".bias"], stride=2))
    h = skips[-1]
    for i in range(3):
        for j in range(3):
            h = resnet(f"{m}.up_blocks.{i}.resnets.{j}", torch.cat([h, skips.pop()], -1), temb)
            h = transformer(f"{m}.up_blocks.{i}.attentions.{j}", h)
        if i < 2:
            p = f"{m}.up_blocks.{i}.upsamplers.0.conv"
            h = _conv(h, P[p + ".weight"], P[p + ".bias"], up=True)
    h = _silu(_gnorm(h, 1e-5, P[m + ".conv_norm_out.weight"], P[m + ".conv_norm_out.bias"]))
    return dwconv(m + ".conv_out", h)


def _exact_vae():
    P = _vae_params()

    def conv(p, v, **kw):
        return _conv(v, P[p + ".weight"], P[p + ".bias"], **kw)

    def lin(p, v):
        return _lin(v, P[p + ".weight"], P[p + ".bias"])

    def norm(p, v):
        return _gnorm(v, 1e-6, P[p + ".weight"], P[p + ".bias"])

    def resnet(p, v):
        h = conv(p + ".conv1", _silu(norm(p + ".norm1", v)))
        h = conv(p + ".conv2", _silu(norm(p + ".norm2", h)))
        return h + (lin(p + ".conv_shortcut", v) if p + ".conv_shortcut.weight" in P else v)

    def mid(p, v):
        v = resnet(p + ".resnets.0", v)
        a = p + ".attentions.0"
        n, h, w, c = v.shape
        t = norm(a + ".group_norm", v).reshape(n, h * w, c)
        q, k, val = (lin(f"{a}.to_{x}", t) for x in "qkv")
        s = torch.softmax(torch.matmul(q, k.transpose(1, 2)) / math.sqrt(c), -1)
        v = lin(a + ".to_out.0", torch.matmul(s, val)).reshape(n, h, w, c) + v
        return resnet(p + ".resnets.1", v)

    return conv, lin, norm, resnet, mid


def _exact_encode(images, noise):
    conv, lin, norm, resnet, mid = _exact_vae()
    out = []
    for img, nz in zip(images, noise):
        x = conv("encoder.conv_in", _d(img)[None])
        for i in range(4):
            for j in range(2):
                x = resnet(f"encoder.down_blocks.{i}.resnets.{j}", x)
            if i < 3:
                x = conv(f"encoder.down_blocks.{i}.downsamplers.0.conv", x, stride=2, pad=(0, 0, 1, 1))
        x = mid("encoder.mid_block", x)
        x = lin("quant_conv", conv("encoder.conv_out", _silu(norm("encoder.conv_norm_out", x))))
        out.append((x[..., :4] + torch.exp(0.5 * x[..., 4:].clamp(-30, 20)) * _d(nz)[None]) * VP.SCALING)
    return torch.cat(out)


def _exact_decode(z):
    conv, lin, norm, resnet, mid = _exact_vae()
    x = conv("decoder.conv_in", lin("post_quant_conv", _d(z) / float(np.float32(VP.SCALING))))
    x = mid("decoder.mid_block", x)
    for i in range(4):
        for j in range(3):
            x = resnet(f"decoder.up_blocks.{i}.resnets.{j}", x)
        if i < 3:
            x = conv(f"decoder.up_blocks.{i}.upsamplers.0.conv", x, up=True)
    return (conv("decoder.conv_out", _silu(norm("decoder.conv_norm_out", x))) + 1) / 2


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "inpaint":
        return None  # host imaging and nine steps: its stages are cases of their own
    d = _inputs(c, seed)
    if k == "conv1x1":
        y = _lin(_d(d["x"]), d["w"], d["b"])
        return {"out": y + _d(d["r"]) if c["residual"] else y}
    if k == "conv3x3":
        return {"out": _conv(_d(d["x"]), d["w"], d["b"], c["stride"], c["up"])}
    if k == "conv_gn":
        y = _conv(_d(d["x"]), d["w"], d["b"])
        return {"conv": y, "norm": _silu(_gnorm(y, 1e-5, d["g"], d["be"]))}
    if k == "gn":
        return {"out": _silu(_gnorm(_d(d["x"]), 1e-5, d["g"], d["be"]))}
    if k == "resnet":
        x = _d(d["x"])
        h = _conv(_silu(_gnorm(x, 1e-5, d["g1"], d["b1"])), d["w1"], d["c1"])
        h = h + _lin(_silu(_d(d["temb"])), d["lw"], d["lb"])
        h = _conv(_silu(_gnorm(h, 1e-5, d["g2"], d["b2"])), d["w2"], d["c2"])
        return {"out": h + _lin(x, d["ws"], d["bs"])}
    if k == "unet":
        return {"out": _exact_unet(d["x"], d["t"], c["cfg"], c["fast"])}
    if k == "encode":
        return {"out": _exact_encode(d["x"], d["noise"])}
    return {"out": _exact_decode(d["z"])}
