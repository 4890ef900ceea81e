"""What is measured of this framework: the forwards and the binary-conv layers
as a program calls them.

The work is hyperspectral segmentation with a binary UNet.  A program loads a
blob once and then runs cubes through it: as batches of equal patches, as
scenes cut into patches, as whole images, and, where it was written for the
reference's C interface, one host patch at a time.  Three models share that
interface (the v1 UNet, the v2 model with a spectral stem, the v3 real-highway
model), and the binary conv can be called as a layer of its own.

Every output is defined bit for bit (the binary stages are whole numbers and
the float chains have one order), so the tolerance is "exact" throughout.
"""
from __future__ import annotations

import os
import tempfile

import numpy as np
import torch

from bnns_to_c_amd import blob, blob_react, engine, synth


def _forward(name, model, n, h, w, base=16, bands=120, via="device"):
    return {"name": name, "kind": "forward", "model": model, "base": base, "bands": bands,
            "n": n, "h": h, "w": w, "via": via}


def listed():
    return [
        # the reference's own use: one 32x32 patch from host memory (latency, launches)
        _forward("host_patch", "v1", 1, 32, 32, via="host"),
        # a small serving batch, too small to fill the GPU
        _forward("batch_64", "v1", 64, 32, 32),
        # the headline: a large batch of 32x32 patches already on the GPU
        _forward("batch_1024", "v1", 1024, 32, 32),
        # a scene cut into 32x32 patches, on the GPU; its last row and column of patches are partial
        {"name": "scene", "kind": "scene", "model": "v1", "base": 16, "bands": 120, "h": 956, "w": 684, "patch": 32},
        # a small scene of odd sides, so that no row but the first starts on a 16-byte boundary
        {"name": "scene_odd", "kind": "scene", "model": "v1", "base": 16, "bands": 120, "h": 301, "w": 217, "patch": 32},
        # one whole image without patches, at the size the reference quotes
        _forward("image_512", "v1", 1, 512, 512),
        # large tiles through the wide model (32 to 512 channels)
        _forward("tiles_256_wide", "v1", 64, 256, 256, base=32),
        # patches of odd sides, a band count of another sensor and a width between the two above
        _forward("odd_patches", "v1", 48, 45, 51, base=24, bands=103),
        # the spectral-stem model at the headline's batch
        _forward("stem_batch_1024", "v2", 1024, 32, 32),
        # the real-highway model at the headline's batch
        _forward("react_batch_1024", "v3", 1024, 32, 32),
        # one binary conv with its integer sums as the result
        {"name": "conv_sums", "kind": "conv", "cin": 64, "cout": 64, "n": 256, "h": 64, "w": 64, "pool": False},
        # one binary conv with both rules and the 2x2 pool, packed bits out
        {"name": "conv_pool", "kind": "conv", "cin": 128, "cout": 128, "n": 1024, "h": 32, "w": 32, "pool": True},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case: a batch, a scene, a host call or a layer, odd sizes among them."""
    kind = rng.choice(["batch", "batch", "batch", "image", "scene", "scene", "host", "conv", "conv"])
    model = rng.choice(["v1", "v1", "v1", "v2", "v3"])
    base = rng.choice([8, 16, 16, 16, 24, 32])
    bands = rng.choice([120, 120, 120, _log(rng, 16, 224)])
    # at most the headline's input, and of the wide models at most its work
    most = 503_000_000 // 4 // max(bands, 4 * base)
    if kind == "batch":
        if rng.random() < 0.5:
            h = w = 32
        else:
            h, w = _log(rng, 16, 128), _log(rng, 16, 128)
        return {"kind": "forward", "model": model, "base": base, "bands": bands,
                "n": _log(rng, 1, max(1, min(1536, most // (h * w)))), "h": h, "w": w, "via": "device"}
    if kind == "image":
        h, w = _log(rng, 96, 640), _log(rng, 96, 640)
        return {"kind": "forward", "model": model, "base": base, "bands": bands, "n": 1, "h": h, "w": w,
                "via": "device"}
    if kind == "scene":
        return {"kind": "scene", "model": model, "base": base, "bands": bands, "h": _log(rng, 65, 960),
                "w": _log(rng, 65, 960), "patch": rng.choice([32, 32, 64])}
    if kind == "host":
        return {"kind": "forward", "model": model, "base": base, "bands": bands, "n": _log(rng, 1, 16),
                "h": 32, "w": 32, "via": "host"}
    cin, cout = 8 * _log(rng, 2, 64), 8 * _log(rng, 2, 64)
    h, w = _log(rng, 4, 96), _log(rng, 4, 96)
    pool = rng.random() < 0.5
    # at most conv_pool's bit operations and conv_sums' output
    n = min(1024 * 1024 * 128 * 128 // (h * w * cin * cout), 256 * 4096 * 64 // (h * w * cout))
    return {"kind": "conv", "cin": cin, "cout": cout, "n": _log(rng, 1, max(1, n)), "h": h, "w": w, "pool": pool}


# ------------------------------------------------------------------ inputs --
def _blob(case, seed):
    base, bands = case["base"], case["bands"]
    if case["model"] == "v1":
        return synth.make_blob(seed=seed, base=base, n_bands=bands)
    if case["model"] == "v2":
        return synth.make_blob_v2(seed=seed, base=base, n_bands=bands)
    return synth.make_blob_react(seed=seed, base=base, n_bands=bands)


def _bytes(case, b):
    return blob_react.to_bytes(b) if case["model"] == "v3" else blob.to_bytes(b)


def _cube(case, seed):
    """Spectra ~ N(0,1) float32; a scene's bands have an offset ~ U(-0.5, 0.5) each."""
    if case.get("via") == "host":
        return synth.make_input(seed, case["n"], case["bands"], case["h"], case["w"])
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if case["kind"] == "scene":
        x = torch.randn((case["bands"], case["h"], case["w"]), generator=g, device="cuda")
        return x.add_(torch.rand((case["bands"], 1, 1), generator=g, device="cuda").sub_(0.5))
    return torch.randn((case["n"], case["bands"], case["h"], case["w"]), generator=g, device="cuda")


def _layer(case, seed):
    cin, cout = case["cin"], case["cout"]
    rules = ()
    if case["pool"]:
        rules = (synth.make_thresholds(seed + 1, cout, cin * 9 // 4), synth.make_thresholds(seed + 2, cout, cin * 9 // 4))
    return engine.ConvLayer(blob.pack_kidx(synth.make_signs(seed, cout, cin)), cin, cout, *rules)


def prepare(case, seed):
    if case["kind"] == "conv":
        n, h, w, cin, cout = case["n"], case["h"], case["w"], case["cin"], case["cout"]
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        act = torch.randint(-2**31, 2**31, (n, h, w, (cin + 31) // 32), generator=g, device="cuda",
                            dtype=torch.int64).to(torch.int32)
        if cin % 32:
            act[..., -1] &= (1 << cin % 32) - 1
        cwo = (cout + 31) // 32
        state = {"case": case, "layer": _layer(case, seed), "act": act}
        if case["pool"]:
            state["skip"] = torch.empty((n, h, w, cwo), dtype=torch.int32, device="cuda")
            state["down"] = torch.empty((n, h // 2, w // 2, cwo), dtype=torch.int32, device="cuda")
        else:
            state["sums"] = torch.empty((n, cout, h, w), dtype=torch.int32, device="cuda")
        return state
    b = _blob(case, seed)
    fd, path = tempfile.mkstemp(suffix=".blob")
    try:
        with os.fdopen(fd, "wb") as f:
            f.write(_bytes(case, b))
        model = {"v1": engine.Engine, "v2": engine.StemEngine, "v3": engine.ReactEngine}[case["model"]](path)
    finally:
        os.unlink(path)
    state = {"case": case, "model": model, "x": _cube(case, seed)}
    if case["kind"] == "scene":
        state["logits"] = torch.empty((3, case["h"], case["w"]), device="cuda")
    elif case["via"] == "device":
        state["logits"] = torch.empty((case["n"], 3, case["h"], case["w"]), device="cuda")
    return state


def run(state):
    case = state["case"]
    stream = torch.cuda.current_stream().cuda_stream
    if case["kind"] == "conv":
        n, h, w, act = case["n"], case["h"], case["w"], state["act"]
        if case["pool"]:
            state["layer"].fold_pool_device(act.data_ptr(), n, h, w, state["skip"].data_ptr(),
                                            state["down"].data_ptr(), stream)
            return state["skip"], state["down"]
        state["layer"].P_device(act.data_ptr(), n, h, w, state["sums"].data_ptr(), stream)
        return state["sums"]
    model, x = state["model"], state["x"]
    if case["kind"] == "scene":
        model.forward_patched_device(x.data_ptr(), case["h"], case["w"], state["logits"].data_ptr(), case["patch"],
                                     stream)
        return state["logits"]
    if case["via"] == "host":
        return model.forward_batch(x)
    model.forward_device(x.data_ptr(), case["n"], case["h"], case["w"], state["logits"].data_ptr(), stream)
    return state["logits"]


# ------------------------------------------------------------------ bounds --
def _pixels(case):
    """[(patches, h, w)] that the model runs."""
    if case["kind"] == "scene":
        p = case["patch"]
        return -(-case["h"] // p) * -(-case["w"] // p), p, p
    return case["n"], case["h"], case["w"]


def work(case):
    """Each input and output once; two operations per multiply-add, bits counted as the binary convs' terms."""
    if case["kind"] == "conv":
        n, h, w, cin, cout = case["n"], case["h"], case["w"], case["cin"], case["cout"]
        out = n * (h * w + (h // 2) * (w // 2)) * -(-cout // 32) * 4 if case["pool"] else n * h * w * cout * 4
        return {"bytes": n * h * w * -(-cin // 32) * 4 + cout * cin * 9 // 8 + out, "flops": 2 * 9 * n * h * w * cin * cout}
    n, h, w = _pixels(case)
    base, bands, v = case["base"], case["bands"], case["model"]
    macs, weights = 0, 0
    for i, (name, ci, co) in enumerate(synth.topology(base, bands)):
        level = 4 if name.startswith("bott") else int(name[3]) - 1
        px = (h >> level) * (w >> level)
        taps = 9 * ci
        if i == 0 and v == "v2":
            taps = bands + 9 * 16
        if v == "v3" and name.endswith("conv1"):
            taps += ci  # the real 1x1 projection beside it
            weights += 4 * ci * co
        macs += px * co * taps
        weights += 9 * ci * co // 8
    macs += h * w * base * 3
    px = case["n"] * h * w if case["kind"] == "forward" else case["h"] * case["w"]
    return {"bytes": px * (bands + 3) * 4 + weights, "flops": 2 * n * macs}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------- 64-bit results --
def _conv(x, w):
    """3x3 (zero padding) or 1x1 conv of [C, N, H, W] with [Cout, C, k, k], as one product per tap."""
    co, ci, k, _ = w.shape
    c, n, h, wd = x.shape
    out = torch.zeros((co, n, h, wd), dtype=x.dtype, device=x.device)
    r = k // 2
    xp = torch.nn.functional.pad(x, (r, r, r, r)) if r else x
    flat = xp.reshape(c, -1)
    for ky in range(k):
        for kx in range(k):
            y = (w[:, :, ky, kx].contiguous() @ flat).reshape(co, n, h + 2 * r, wd + 2 * r)
            out += y[:, :, ky:ky + h, kx:kx + wd]
    return out


def _sign(v):
    return torch.where(v > 0, 1.0, -1.0).to(torch.float64)


def _fold(a, v):
    """The activation of a record: the real chain, or the integer rule ge (1) or lt (2)."""
    def t(u, dt=torch.float64):
        return torch.from_numpy(np.ascontiguousarray(u)).to(v.device, dt).reshape(-1, 1, 1, 1)
    if a.kind == 1:
        z = t(a.A) * v + t(a.B)
        return _sign(torch.where(z < 0, t(a.slope) * z, z) + t(a.rsign))
    ge, lt = t(a.type) == blob.RULE_GE, t(a.type) == blob.RULE_LT
    return _sign(((ge & (v >= t(a.t))) | (lt & (v < t(a.t)))).to(torch.float64) - 0.5)


def _pool(v):
    c, n, h, w = v.shape
    v = v[:, :, :h // 2 * 2, :w // 2 * 2].reshape(c, n, h // 2, 2, w // 2, 2)
    return v.amax(dim=(3, 5))


def _cat(skip, x, fill):
    """The skip and the doubled x on channels; what the doubling does not cover holds `fill`."""
    c, n, h, w = skip.shape
    up = x.repeat_interleave(2, 2).repeat_interleave(2, 3)
    y = torch.full((x.shape[0], n, h, w), fill, dtype=x.dtype, device=x.device)
    dy, dx = (h - up.shape[2]) // 2, (w - up.shape[3]) // 2
    y[:, :, dy:dy + up.shape[2], dx:dx + up.shape[3]] = up
    return torch.cat([skip, y])


def _model_bits(b, x):
    dev = x.device

    def w(conv):
        return torch.from_numpy(conv.signs()).to(dev, torch.float64)

    def real(conv):
        return torch.from_numpy(conv.alpha).to(dev, torch.float64).reshape(-1, 1, 1, 1)
    if b.version == blob.VERSION_STEM:
        x = _fold(b.stem_act, _conv(x, w(b.stem_conv)) * real(b.stem_conv))
    skips = []
    for i in range(4):
        c1 = b.enc_conv1[i]
        v = _conv(x, w(c1))
        v = _fold(b.enc_act1[i], v * real(c1) if c1.tag == blob.TAG_CONV_REAL else v)
        v = _conv(v, w(b.enc_conv2[i]))
        skips.append(_fold(b.enc_act2_skip[i], v))
        x = _fold(b.enc_act2_down[i], _pool(v))
    x = _fold(b.bott_act1, _conv(x, w(b.bott_conv1)))
    x = _fold(b.bott_act2, _conv(x, w(b.bott_conv2)))
    for i in range(4):
        x = _fold(b.dec_act1[i], _conv(_cat(skips[3 - i], x, -1.0), w(b.dec_conv1[i])))
        x = _fold(b.dec_act2[i], _conv(x, w(b.dec_conv2[i])))
    return x


def _model_react(b, x):
    dev = x.device

    def t(u):
        return torch.from_numpy(np.ascontiguousarray(u)).to(dev, torch.float64)

    def epi(e, acc, res):
        c = (-1, 1, 1, 1)
        v = t(e.A).reshape(c) * acc + (t(e.B) + t(e.move1)).reshape(c) + res
        return torch.where(v >= 0, v, t(e.prelu_w).reshape(c) * v)

    def tap(p, v):
        return _sign(v + t(p.rsign).reshape(-1, 1, 1, 1))

    def unit1(k, v):
        res = _conv(v, t(k.proj1.W)[:, :, None, None])
        if k.input_real:
            acc = _conv(v, t(k.conv1.signs())) * t(k.conv1.alpha).reshape(-1, 1, 1, 1)
        else:
            acc = _conv(tap(k.tap1, v), t(k.conv1.signs()))
        return epi(k.epi1, acc, res)

    skips = []
    for k in b.enc:
        h1 = unit1(k, x)
        p = _conv(tap(k.tap2, h1), t(k.conv2.signs()))
        skips.append(epi(k.epi_a, p, h1))
        x = epi(k.epi_b, _pool(p), _pool(h1))
    for i, k in enumerate([b.bott] + b.dec):
        h1 = unit1(k, x if i == 0 else _cat(skips[4 - i], x, 0.0))
        x = epi(k.epi_a, _conv(tap(k.tap2, h1), t(k.conv2.signs())), h1)
    return x


def exact(case, seed):
    if case["kind"] == "conv":
        return None  # whole numbers
    b = _blob(case, seed)
    x = _cube(case, seed)
    host = case.get("via") == "host"
    x = torch.from_numpy(x) if host else x
    dev = torch.device("cuda")
    n, h, w = _pixels(case)
    if case["kind"] == "scene":
        rows, cols = -(-case["h"] // h), -(-case["w"] // w)
        x = torch.nn.functional.pad(x, (0, cols * w - case["w"], 0, rows * h - case["h"]))
        x = x.reshape(case["bands"], rows, h, cols, w).permute(1, 3, 0, 2, 4).reshape(n, case["bands"], h, w)
    out = torch.empty((n, 3, h, w), dtype=torch.float64, device=dev)
    wh = torch.from_numpy(b.head.W).to(dev, torch.float64)
    bias = torch.from_numpy(b.head.bias).to(dev, torch.float64)
    step = max(1, 300_000_000 // (h * w * max(case["bands"], 4 * case["base"])) // 2)
    for i in range(0, n, step):
        v = x[i:i + step].to(dev, torch.float64).transpose(0, 1).contiguous()
        v = _model_react(b, v) if case["model"] == "v3" else _model_bits(b, v)
        y = _conv(v, wh[:, :, None, None]) + bias.reshape(-1, 1, 1, 1)
        out[i:i + step] = y.transpose(0, 1)
    if case["kind"] == "scene":
        out = out.reshape(rows, cols, 3, h, w).permute(2, 0, 3, 1, 4).reshape(3, rows * h, cols * w)
        return out[:, :case["h"], :case["w"]].contiguous()
    return out.cpu().numpy() if host else out
