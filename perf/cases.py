"""Timing cases of the YOLO26 inference path on one MI355X.

Each case is one call that a program using this framework makes: a whole
network, one of its blocks (C3k2, C2PSA, the Detect head), a single
convolution, or a step around the network (letterbox, detection post-process,
deformable attention).  `listed()` holds the sizes that stand for these uses,
`draw()` further sizes of the same ranges.  Networks and blocks run as a
captured graph that is replayed, as a serving loop does, except the Detect
head, which runs as a plain forward call; single operations are plain calls
with the automatic tile choice.

`exact()` restates every operation in float64 with plain torch.
"""
import json
import math
import os
import sys
import zlib

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "vision-rs_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import vrs  # noqa: E402

DEV = "cuda"
EPS = 1e-3
VARIANTS = {"n": (0.5, 0.25, 1024), "s": (0.5, 0.50, 1024), "m": (0.5, 1.00, 512), "l": (1.0, 1.00, 512)}
STRIDES = (8, 16, 32)
TDT = {"f32": torch.float32, "bf16": torch.bfloat16}
VDT = {"f32": vrs.F32, "bf16": vrs.BF16, "fp8": vrs.FP8}
ES = {"f32": 4, "bf16": 2, "fp8": 1}

_ctx = None
_stream = None


def _context():
    """The context and stream that a program keeps for its whole life."""
    global _ctx, _stream
    if _ctx is None:
        torch.cuda.init()
        _ctx = vrs.Context(0)
        _stream = torch.cuda.Stream()
    return _ctx, _stream


# ---- the cases ----------------------------------------------------------------


def listed():
    return [
        # one camera frame through the smallest network in float32: the latency of the whole call
        {"name": "net-n-f32-b1", "kind": "net", "variant": "n", "dtype": "f32", "batch": 1, "h": 640, "w": 640},
        # the throughput configuration: a full batch through the medium network with its committed tile plan
        {"name": "net-m-bf16-b64", "kind": "net", "variant": "m", "dtype": "bf16", "batch": 64, "h": 640, "w": 640},
        # a C3k bottleneck conv of the medium network for one frame, float32: a small call
        {"name": "conv-f32-b1", "kind": "conv", "dtype": "f32", "batch": 1, "h": 40, "w": 40, "cin": 128,
         "cout": 128, "k": 3, "s": 1, "res": True},
        # a backbone conv at an ordinary batch
        {"name": "conv-bf16-b32", "kind": "conv", "dtype": "bf16", "batch": 32, "h": 80, "w": 80, "cin": 128,
         "cout": 128, "k": 3, "s": 1, "res": False},
        # a downsampling conv between two e4m3 tensors
        {"name": "conv-fp8-b32", "kind": "conv", "dtype": "fp8", "batch": 32, "h": 40, "w": 40, "cin": 256,
         "cout": 512, "k": 3, "s": 2, "res": False},
        # the depthwise conv of a class branch
        {"name": "dw-bf16-b32", "kind": "dw", "dtype": "bf16", "batch": 32, "h": 20, "w": 20, "c": 512, "s": 1},
        # the P4 block of the medium network for one frame in bfloat16
        {"name": "c3k2-bf16-b1", "kind": "c3k2", "dtype": "bf16", "batch": 1, "h": 40, "w": 40, "c": 512, "c3k": True,
         "e": 0.5},
        # the attention block of the medium network at an ordinary batch
        {"name": "c2psa-bf16-b32", "kind": "c2psa", "dtype": "bf16", "batch": 32, "h": 20, "w": 20, "c": 512},
        # the Detect head of the medium network for a few frames, as a plain forward call
        {"name": "detect-bf16-b8", "kind": "detect", "dtype": "bf16", "batch": 8, "h": 80, "w": 80, "c0": 256,
         "c1": 512, "c2": 512, "nc": 80, "one2one": True},
        # raw head outputs of a full batch to detections, at the evaluation threshold
        {"name": "post-b64", "kind": "post", "batch": 64, "h": 640, "w": 640, "nc": 80, "thr": 0.001, "max_det": 300},
        # the decoder's deformable attention at its usual size
        {"name": "msda-b8", "kind": "msda", "batch": 8, "q": 300, "heads": 8, "levels": 4, "points": 4, "h": 80,
         "w": 80},
        # HD video frames to network input
        {"name": "letterbox-b16", "kind": "letterbox", "batch": 16, "h": 720, "w": 1280, "size": 640},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng, kind):
    c = {"kind": kind}
    if kind == "net":
        c.update(variant=rng.choice("nsm"), dtype=rng.choice(("f32", "bf16", "bf16")), batch=_log(rng, 1, 32),
                 h=32 * rng.randint(10, 30), w=32 * rng.randint(10, 30))
    elif kind == "conv":
        dt = rng.choice(("f32", "bf16", "bf16", "fp8"))
        step = 64 if dt == "fp8" else 8
        c.update(dtype=dt, batch=_log(rng, 1, 64), h=_log(rng, 10, 160), w=_log(rng, 10, 160),
                 cin=step * max(1, _log(rng, 16, 1024) // step), cout=16 * max(1, _log(rng, 16, 1024) // 16),
                 k=rng.choice((1, 3, 3)))
        c["s"] = rng.choice((1, 1, 2)) if c["k"] == 3 else 1
        c["res"] = dt != "fp8" and c["s"] == 1 and rng.random() < 0.5
    elif kind == "dw":
        c.update(dtype=rng.choice(("f32", "bf16", "bf16")), batch=_log(rng, 1, 64), h=_log(rng, 10, 160),
                 w=_log(rng, 10, 160), c=8 * _log(rng, 4, 64), s=rng.choice((1, 1, 1, 2)))
    elif kind == "c3k2":
        c.update(dtype=rng.choice(("f32", "bf16", "bf16")), batch=_log(rng, 1, 32), h=_log(rng, 10, 160),
                 w=_log(rng, 10, 160), c=64 * rng.choice((1, 2, 4, 6, 8)), c3k=rng.random() < 0.5,
                 e=rng.choice((0.25, 0.5, 0.5)))
    elif kind == "c2psa":
        c.update(dtype=rng.choice(("f32", "bf16", "bf16")), batch=_log(rng, 1, 32), h=rng.randint(7, 40),
                 w=rng.randint(7, 40), c=128 * rng.choice((2, 4, 4, 6)))
    elif kind == "detect":
        wide = rng.choice(((64, 128, 256), (128, 256, 512), (256, 512, 512)))
        c.update(dtype=rng.choice(("f32", "bf16", "bf16")), batch=_log(rng, 1, 16), h=4 * rng.randint(10, 30),
                 w=4 * rng.randint(10, 30), c0=wide[0], c1=wide[1], c2=wide[2], nc=rng.choice((1, 20, 80, 80, 91)),
                 one2one=rng.random() < 0.7)
    elif kind == "post":
        c.update(batch=_log(rng, 1, 64), h=32 * rng.randint(10, 40), w=32 * rng.randint(10, 40),
                 nc=rng.choice((1, 20, 80, 80, 91)), thr=rng.choice((0.25, 0.001)),
                 max_det=rng.choice((100, 300, 300, 1000)))
    elif kind == "msda":
        c.update(batch=_log(rng, 1, 16), q=_log(rng, 100, 900), heads=8, levels=rng.choice((3, 4, 4)),
                 points=rng.choice((2, 4, 4)), h=rng.randint(40, 120), w=rng.randint(40, 120))
    else:
        c.update(batch=_log(rng, 1, 32), h=_log(rng, 240, 2400), w=_log(rng, 320, 3200),
                 size=32 * rng.randint(10, 40))
    return c


def draw(rng):
    kind = rng.choice(("net", "net", "conv", "conv", "conv", "dw", "c3k2", "c3k2", "c2psa", "detect", "post", "msda",
                       "letterbox"))
    while True:
        c = _draw_once(rng, kind)
        w = work(c)
        if w["flops"] <= 1.5e12 and _memory(c) <= 2e9 and (c.get("dtype") != "f32" or w["flops"] <= 2e11):
            return c


# ---- inputs --------------------------------------------------------------------


def _param(seed, name, shape):
    """A parameter of a trained-like network: Kaiming-normal conv weights, BN statistics near identity."""
    r = np.random.default_rng([seed, zlib.crc32(name.encode())])
    shape = tuple(int(v) for v in shape)
    if len(shape) == 4:
        w = r.standard_normal(shape, dtype=np.float32)
        w *= np.float32(math.sqrt(2.0 / (shape[1] * shape[2] * shape[3])))
        return w
    if name.endswith("bn.weight") or name.endswith("bn.running_var"):
        return r.uniform(0.7, 1.3, shape).astype(np.float32)
    return r.normal(0, 0.1, shape).astype(np.float32)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _features(g, *shape):
    """Activations as the network holds them: SiLU of a standard normal."""
    return torch.nn.functional.silu(torch.randn(*shape, generator=g, device=DEV))


def _net_input(c, seed):
    g = _gen(seed)
    if c["kind"] == "net":
        return torch.rand(c["batch"], 3, c["h"], c["w"], generator=g, device=DEV)
    if c["kind"] == "detect":
        return torch.cat([_features(g, c["batch"] * c["c%d" % i] * (c["h"] >> i) * (c["w"] >> i)) for i in range(3)])
    return _features(g, c["batch"], c["c"], c["h"], c["w"])


def _desc(c):
    if c["kind"] == "net":
        return vrs.block(vrs.BLOCK_YOLO26, 3, nc=80, variant=c["variant"], one2one=True)
    if c["kind"] == "c3k2":
        return vrs.block(vrs.BLOCK_C3K2, c["c"], c["c"], n=1, c3k=c["c3k"], shortcut=True, e=c["e"])
    if c["kind"] == "c2psa":
        return vrs.block(vrs.BLOCK_C2PSA, c["c"], c["c"], n=1, e=0.5)
    return vrs.block(vrs.BLOCK_DETECT, c["c0"], nc=c["nc"], one2one=c["one2one"], ch=(c["c0"], c["c1"], c["c2"]))


def _committed_plan(c, names):
    """The repository's tile plan of this network, if it holds one (as bench.py applies it)."""
    if c["kind"] != "net" or c["h"] != c["w"]:
        return None
    p = os.path.join(PKG, "plans", "yolo26%s_%s_bs%d_%d.json" % (c["variant"], c["dtype"], c["batch"], c["h"]))
    if not os.path.isfile(p):
        return None
    with open(p) as f:
        rows = json.load(f)["plan"]
    return [int(r[1]) for r in rows] if [r[0] for r in rows] == names else None


def _model_state(c, seed):
    ctx, stream = _context()
    x = _net_input(c, seed)
    m = vrs.Model(ctx, _desc(c), c["batch"], c["h"], c["w"], VDT[c["dtype"]], EPS)
    plan = _committed_plan(c, [n for n, _, _ in m.conv_info()])
    if plan is not None:
        m.set_plan(plan)
    m.load({n: _param(seed, n, s) for n, s in m.params()})
    outs = m.alloc_outputs(DEV)
    torch.cuda.synchronize()
    if c["kind"] != "detect":
        m.capture(x, outs, stream.cuda_stream)
    return {"kind": "model", "model": m, "x": x, "outs": outs, "replay": c["kind"] != "detect",
            "stream": stream.cuda_stream}


def _out_hw(c):
    return (c["h"] - 1) // c["s"] + 1, (c["w"] - 1) // c["s"] + 1


def _fp8_step(v):
    return 2.0 ** math.ceil(math.log2(float(v) / 448.0))


def _conv_inputs(c, seed):
    """x (NHWC), the float32 weights (OIHW), scale and shift, the residual (or None)."""
    g = _gen(seed)
    cin, cout, k = c.get("cin", c.get("c")), c.get("cout", c.get("c")), c.get("k", 3)
    x = _features(g, c["batch"], c["h"], c["w"], cin)
    w = _param(seed, "weight", (cout, 1 if c["kind"] == "dw" else cin, k, k))
    scale = torch.rand(cout, generator=g, device=DEV) * 0.6 + 0.7
    shift = torch.randn(cout, generator=g, device=DEV) * 0.1
    ho, wo = _out_hw(c)
    res = _features(g, c["batch"], ho, wo, cout) if c.get("res") else None
    if c["dtype"] == "fp8":
        step = _fp8_step(8.0)
        x = (x / step).clamp(-448, 448).to(torch.float8_e4m3fn)
        return x, w, scale, shift, res, step
    dt = TDT[c["dtype"]]
    return x.to(dt), w, scale, shift, None if res is None else res.to(dt), 1.0


def _conv_state(c, seed):
    ctx, _ = _context()
    x, w, scale, shift, res, step = _conv_inputs(c, seed)
    cout, dt = w.shape[0], c["dtype"]
    ho, wo = _out_hw(c)
    if dt == "fp8":
        packed, ws = vrs.pack_conv_weight_fp8(w)
        scale = scale * torch.from_numpy(ws).to(DEV) * step
        y = torch.empty(c["batch"], ho, wo, cout, dtype=torch.uint8, device=DEV)
        more = {"in_scale": step, "x_e4m3": True, "y_e4m3": True, "out_step": _fp8_step(8.0)}
    else:
        packed = vrs.pack_conv_weight(w, groups=cout if c["kind"] == "dw" else 1, dtype=VDT[dt])
        y = torch.empty(c["batch"], ho, wo, cout, dtype=TDT[dt], device=DEV)
        more = {}
    args = {"k": w.shape[2], "stride": c["s"], "groups": cout if c["kind"] == "dw" else 1, "act": vrs.ACT_SILU,
            "res": None if res is None else vrs.nhwc(res), "dtype": VDT[dt], **more}
    return {"kind": "conv", "ctx": ctx, "x": x, "w": torch.from_numpy(packed).to(DEV), "scale": scale, "shift": shift,
            "res": res, "y": y, "xv": vrs.nhwc(x), "yv": vrs.nhwc(y), "args": args}


def _post_inputs(c, seed):
    g = _gen(seed)
    a = sum((c["h"] // s) * (c["w"] // s) for s in STRIDES)
    boxes = torch.randn(c["batch"], 4 * a, generator=g, device=DEV) * 1.5 + 3.0
    scores = torch.randn(c["batch"], c["nc"] * a, generator=g, device=DEV) * 2.0 - 8.0
    return boxes, scores


def _msda_shapes(c):
    return [(max(1, c["h"] >> i), max(1, c["w"] >> i)) for i in range(c["levels"])]


def _msda_inputs(c, seed):
    g = _gen(seed)
    n, q, hd, lv, p = c["batch"], c["q"], c["heads"], c["levels"], c["points"]
    s = sum(h * w for h, w in _msda_shapes(c))
    value = torch.randn(n, s, hd, 32, generator=g, device=DEV)
    ref = torch.rand(n, q, 2, generator=g, device=DEV)
    off = torch.randn(n, q, hd, lv, p, 2, generator=g, device=DEV) * 0.05
    attw = torch.randn(n, q, hd, lv * p, generator=g, device=DEV).softmax(-1).reshape(n, q, hd, lv, p).contiguous()
    return value, ref, off, attw


def _letterbox_inputs(c, seed):
    """Frames of about the case's size (each a little different) in one flat buffer: smooth shapes with noise."""
    g = _gen(seed)
    r = np.random.default_rng([seed, 17])
    wh = [(c["w"] - int(r.integers(0, 1 + c["w"] // 16)), c["h"] - int(r.integers(0, 1 + c["h"] // 16)))
          for _ in range(c["batch"])]
    parts, offs, at = [], [], 0
    for w, h in wh:
        low = torch.rand(1, 3, 1 + h // 40, 1 + w // 40, generator=g, device=DEV)
        img = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear") * 235 + 20 * torch.rand(
            1, 3, h, w, generator=g, device=DEV)
        parts.append(img[0].permute(1, 2, 0).to(torch.uint8).reshape(-1))
        offs.append(at)
        at += 3 * w * h
    return torch.cat(parts), offs, wh


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("net", "c3k2", "c2psa", "detect"):
        return _model_state(case, seed)
    if kind in ("conv", "dw"):
        return _conv_state(case, seed)
    ctx, _ = _context()
    n = case["batch"]
    if kind == "post":
        boxes, scores = _post_inputs(case, seed)
        md = case["max_det"]
        st = (vrs.C.c_int32 * 4)(*STRIDES, 0)
        d = vrs.DetectDesc(n, case["nc"], case["h"], case["w"], 3, st, case["thr"], md)
        ws = torch.empty(vrs.lib().vrs_detect_workspace_size(vrs.C.byref(d)), dtype=torch.uint8, device=DEV)
        outs = tuple(torch.empty(*s, dtype=t, device=DEV) for s, t in (
            ((n,), torch.int32), ((n, md), torch.float32), ((n, md), torch.int32), ((n, md), torch.int32),
            ((n, md, 4), torch.float32)))
        return {"kind": kind, "ctx": ctx, "boxes": boxes, "scores": scores, "outs": outs, "ws": ws, "case": case}
    if kind == "msda":
        value, ref, off, attw = _msda_inputs(case, seed)
        out = torch.empty(n, case["q"], case["heads"] * 32, device=DEV)
        return {"kind": kind, "ctx": ctx, "value": value, "ref": ref, "off": off, "attw": attw, "out": out,
                "shapes": _msda_shapes(case)}
    rgb, offs, wh = _letterbox_inputs(case, seed)
    out = torch.empty(n, 3, case["size"], case["size"], device=DEV)
    return {"kind": kind, "ctx": ctx, "rgb": rgb, "offs": offs, "wh": wh, "size": case["size"], "out": out}


def run(s):
    kind = s["kind"]
    if kind == "model":
        if s["replay"]:
            s["model"].replay(s["stream"])
        else:
            s["model"].forward(s["x"], s["outs"])
        return s["outs"]
    if kind == "conv":
        s["ctx"].conv2d(s["xv"], s["w"], s["scale"], s["shift"], s["yv"], **s["args"])
        return s["y"]
    if kind == "post":
        c = s["case"]
        return s["ctx"].detect_postprocess(s["boxes"], s["scores"], c["nc"], c["h"], c["w"], STRIDES, c["thr"],
                                           c["max_det"], outs=s["outs"], workspace=s["ws"])
    if kind == "msda":
        s["ctx"].msda(s["value"], s["shapes"], s["ref"], s["off"], s["attw"], s["out"])
        return s["out"]
    return s["ctx"].letterbox(s["rgb"], s["offs"], s["wh"], s["size"], out=s["out"])


# ---- the same in float64 -------------------------------------------------------


class _Graph:
    """The layers in float64 (or, on the meta device, their operation counts)."""

    def __init__(self, seed, meta=False):
        self.seed, self.meta, self.flops, self.weights = seed, meta, 0.0, 0

    def conv(self, pre, x, cout, k=1, s=1, dw=False, plain=False, act=True):
        n, cin, h, w = x.shape
        ho, wo = (h - 1) // s + 1, (w - 1) // s + 1
        name = (pre + "." if pre else "") + ("weight" if plain else "conv.weight")
        shape = (cout, 1 if dw else cin, k, k)
        self.flops += 2.0 * n * ho * wo * math.prod(shape)
        self.weights += math.prod(shape)
        if self.meta:
            return torch.empty(n, cout, ho, wo, device="meta")
        wt = torch.from_numpy(_param(self.seed, name, shape)).to(DEV).double()
        if plain:
            sc, sh = torch.ones(cout, dtype=torch.float64, device=DEV), self._vec(pre + ".bias", cout)
        else:
            b = (pre + "." if pre else "") + "bn."
            sc = self._vec(b + "weight", cout) / torch.sqrt(self._vec(b + "running_var", cout) + EPS)
            sh = self._vec(b + "bias", cout) - sc * self._vec(b + "running_mean", cout)
        y = _conv64(x, wt, s, dw) * sc.view(1, -1, 1, 1) + sh.view(1, -1, 1, 1)
        return y * torch.sigmoid(y) if act and not plain else y

    def _vec(self, name, n):
        return torch.from_numpy(_param(self.seed, name, (n,))).to(DEV).double()

    def bottleneck(self, p, x, ch, shortcut):
        y = self.conv(p + ".cv2", self.conv(p + ".cv1", x, ch, 3), x.shape[1], 3)
        return x + y if shortcut else y

    def c3k(self, p, x, shortcut):
        ch = x.shape[1] // 2
        a = self.conv(p + ".cv1", x, ch)
        for i in range(2):
            a = self.bottleneck("%s.m.%d" % (p, i), a, ch, shortcut)
        return self.conv(p + ".cv3", torch.cat([a, self.conv(p + ".cv2", x, ch)], 1), x.shape[1])

    def c3k2(self, p, x, cout, n, c3k, shortcut, e):
        p = p + "." if p else ""
        c = int(cout * e)
        ys = list(self.conv(p + "cv1", x, 2 * c).split(c, 1))
        for i in range(n):
            b = "%sm.%d" % (p, i)
            ys.append(self.c3k(b, ys[-1], shortcut) if c3k else self.bottleneck(b, ys[-1], c // 2, shortcut))
        return self.conv(p + "cv2", torch.cat(ys, 1), cout)

    def attention(self, p, x):
        n, c, h, w = x.shape
        qkv = self.conv(p + ".qkv", x, 2 * c, act=False).reshape(n, c // 64, 128, h * w)
        self.flops += 2.0 * n * (c // 64) * (h * w) ** 2 * 96
        q, k, v = qkv.split((32, 32, 64), 2)
        if self.meta:
            o = v
        else:
            a = torch.matmul(q.transpose(2, 3).contiguous(), k.contiguous()) * 32 ** -0.5
            o = torch.matmul(v.contiguous(), a.softmax(-1).transpose(2, 3).contiguous())
        v = v.reshape(n, c, h, w)
        o = o.reshape(n, c, h, w) + self.conv(p + ".pe", v, c, 3, dw=True, act=False)
        return self.conv(p + ".proj", o, c, act=False)

    def psa(self, p, b):
        b = b + self.attention(p + ".attn", b)
        return b + self.conv(p + ".ffn.1", self.conv(p + ".ffn.0", b, 2 * b.shape[1]), b.shape[1], act=False)

    def c2psa(self, p, x, n):
        p = p + "." if p else ""
        a, b = self.conv(p + "cv1", x, x.shape[1]).chunk(2, 1)
        for i in range(n):
            b = self.psa("%sm.%d" % (p, i), b)
        return self.conv(p + "cv2", torch.cat([a, b], 1), x.shape[1])

    def c3k2_psa(self, p, x, cout):
        ys = list(self.conv(p + ".cv1", x, cout).chunk(2, 1))
        t = self.bottleneck(p + ".m.0.0", ys[-1], cout // 4, True)
        ys.append(self.psa(p + ".m.0.1", t))
        return self.conv(p + ".cv2", torch.cat(ys, 1), cout)

    def sppf(self, p, x):
        c = x.shape[1]
        ys = [self.conv(p + ".cv1", x, c // 2, act=False)]
        for _ in range(3):
            ys.append(ys[-1] if self.meta else torch.nn.functional.max_pool2d(ys[-1], 5, 1, 2))
        return x + self.conv(p + ".cv2", torch.cat(ys, 1), c)

    def detect(self, p, feats, nc, one2one):
        p = p + "." if p else ""
        head = "one2one_" if one2one else ""
        c2, c3 = max(16, feats[0].shape[1] // 4), max(feats[0].shape[1], min(nc, 100))
        boxes, scores = [], []
        for i, x in enumerate(feats):
            q = "%s%scv2.%d" % (p, head, i)
            t = self.conv(q + ".1", self.conv(q + ".0", x, c2, 3), c2, 3)
            boxes.append(self.conv(q + ".2", t, 4, plain=True).flatten(1))
            q = "%s%scv3.%d" % (p, head, i)
            t = self.conv(q + ".0.1", self.conv(q + ".0.0", x, x.shape[1], 3, dw=True), c3)
            t = self.conv(q + ".1.1", self.conv(q + ".1.0", t, c3, 3, dw=True), c3)
            scores.append(self.conv(q + ".2", t, nc, plain=True).flatten(1))
        return [torch.cat(boxes, 1), torch.cat(scores, 1)]

    def net(self, x, variant):
        dep, wid, mc = VARIANTS[variant]
        c = [int(math.floor(min(b, mc) * wid + 0.5)) for b in (64, 128, 256, 512, 1024)]
        n = int(math.floor(max(2 * dep, 1.0) + 0.5))
        up = (lambda t: t.repeat_interleave(2, 2).repeat_interleave(2, 3)) if not self.meta else (
            lambda t: torch.empty(t.shape[0], t.shape[1], 2 * t.shape[2], 2 * t.shape[3], device="meta"))
        x = self.conv("model.1", self.conv("model.0", x, c[0], 3, 2), c[1], 3, 2)
        x = self.conv("model.3", self.c3k2("model.2", x, c[2], n, False, True, 0.25), c[2], 3, 2)
        p3 = self.c3k2("model.4", x, c[3], n, False, True, 0.25)
        p4 = self.c3k2("model.6", self.conv("model.5", p3, c[3], 3, 2), c[3], n, True, True, 0.5)
        x = self.c3k2("model.8", self.conv("model.7", p4, c[4], 3, 2), c[4], n, True, True, 0.5)
        p5 = self.c2psa("model.10", self.sppf("model.9", x), n)
        n4 = self.c3k2("model.13", torch.cat([up(p5), p4], 1), c[3], n, True, True, 0.5)
        f0 = self.c3k2("model.16", torch.cat([up(n4), p3], 1), c[2], n, True, True, 0.5)
        f1 = self.c3k2("model.19", torch.cat([self.conv("model.17", f0, c[2], 3, 2), n4], 1), c[3], n, True, True, 0.5)
        f2 = self.c3k2_psa("model.22", torch.cat([self.conv("model.20", f1, c[3], 3, 2), p5], 1), c[4])
        return self.detect("model.23", [f0, f1, f2], 80, True)

    def forward(self, c, x):
        """The outputs for the images x (a list of three maps for the Detect head)."""
        if c["kind"] == "net":
            return self.net(x, c["variant"])
        if c["kind"] == "c3k2":
            return [self.c3k2("", x, c["c"], 1, c["c3k"], True, c["e"])]
        if c["kind"] == "c2psa":
            return [self.c2psa("", x, 1)]
        return self.detect("", x, c["nc"], c["one2one"])


def _conv64(x, w, s, dw):
    """A float64 convolution with 'same' padding, one product per tap."""
    k = w.shape[2]
    n, cin, h, wd = x.shape
    ho, wo = (h - 1) // s + 1, (wd - 1) // s + 1
    xp = torch.nn.functional.pad(x, (k // 2,) * 4) if k > 1 else x
    y = torch.zeros(n, w.shape[0], ho, wo, dtype=torch.float64, device=x.device)
    for ky in range(k):
        for kx in range(k):
            t = xp[:, :, ky:ky + (ho - 1) * s + 1:s, kx:kx + (wo - 1) * s + 1:s]
            if dw:
                y += t * w[:, 0, ky, kx].view(1, -1, 1, 1)
            else:
                for b in range(n):
                    y[b] += torch.mm(w[:, :, ky, kx].contiguous(), t[b].reshape(cin, ho * wo)).view(-1, ho, wo)
    return y


def _model_exact(c, seed):
    x = _net_input(c, seed)
    if c["kind"] == "detect":
        n, maps, at = c["batch"], [], 0
        for i in range(3):
            shape = (n, c["c%d" % i], c["h"] >> i, c["w"] >> i)
            maps.append(x[at:at + math.prod(shape)].view(shape))
            at += math.prod(shape)
    outs = []
    for b in range(c["batch"]):   # one image at a time: float64 maps are large
        one = [t[b:b + 1].double() for t in maps] if c["kind"] == "detect" else x[b:b + 1].double()
        outs.append(_Graph(seed).forward(c, one))
    return [torch.cat([o[i] for o in outs]) for i in range(len(outs[0]))]


def _conv_exact(c, seed):
    x, w, scale, shift, res, _ = _conv_inputs(c, seed)
    x = x.double().permute(0, 3, 1, 2)
    wt = torch.from_numpy(w).to(DEV)
    if c["dtype"] == "bf16":   # the weights in the type that the program hands over
        wt = wt.bfloat16()
    y = _conv64(x, wt.double(), c["s"], c["kind"] == "dw").permute(0, 2, 3, 1)
    y = y * scale.double() + shift.double()
    y = y * torch.sigmoid(y)
    return y if res is None else y + res.double()


def _msda_exact(c, seed):
    value, ref, off, attw = (t.double() for t in _msda_inputs(c, seed))
    n, q, hd = c["batch"], c["q"], c["heads"]
    out, at = 0, 0
    for i, (h, w) in enumerate(_msda_shapes(c)):
        v = value[:, at:at + h * w].permute(0, 2, 3, 1).reshape(n * hd, 32, h, w)
        at += h * w
        loc = (ref[:, :, None, None] + off[:, :, :, i]).permute(0, 2, 1, 3, 4).reshape(n * hd, q, -1, 2)
        s = torch.nn.functional.grid_sample(v, 2 * loc - 1, mode="bilinear", padding_mode="zeros",
                                            align_corners=False)
        out = out + (s * attw[:, :, :, i].permute(0, 2, 1, 3).reshape(n * hd, 1, q, -1)).sum(-1)
    return out.reshape(n, hd, 32, q).permute(0, 3, 1, 2).reshape(n, q, hd * 32)


def _post_exact(c, seed):
    """The sorted scores; the rest are whole numbers, or depend on the order of near-equal scores."""
    _, scores = _post_inputs(c, seed)
    best, at = [], 0
    for s in STRIDES:
        a = (c["h"] // s) * (c["w"] // s)
        best.append(scores[:, at:at + c["nc"] * a].view(-1, c["nc"], a).amax(1))
        at += c["nc"] * a
    p = torch.sigmoid(torch.cat(best, 1).double())
    p = torch.where(p > c["thr"], p, torch.zeros_like(p)).sort(1, descending=True).values[:, :c["max_det"]]
    p = torch.nn.functional.pad(p, (0, c["max_det"] - p.shape[1]))
    return (None, p, None, None, None)


def _letterbox_exact(c, seed):
    rgb, offs, wh = _letterbox_inputs(c, seed)
    size, out = c["size"], []
    for o, (w, h) in zip(offs, wh):
        img = rgb[o:o + 3 * w * h].view(h, w, 3).permute(2, 0, 1)[None].double()
        sc = size / max(w, h)
        nw, nh = (int(math.floor(v * sc + 0.5)) for v in (w, h))
        img = torch.nn.functional.interpolate(img, size=(nh, nw), mode="bilinear", antialias=True,
                                              align_corners=False)
        canvas = torch.full((3, size, size), 114.0, dtype=torch.float64, device=DEV)
        y0, x0 = (size - nh) // 2, (size - nw) // 2
        canvas[:, y0:y0 + nh, x0:x0 + nw] = torch.floor(img[0] + 0.5).clamp(0, 255)
        out.append(canvas / 255)
    return torch.stack(out)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("net", "c3k2", "c2psa", "detect"):
        return _model_exact(case, seed)
    if kind in ("conv", "dw"):
        return None if case["dtype"] == "fp8" else _conv_exact(case, seed)   # fp8: e4m3 bytes
    if kind == "post":
        return _post_exact(case, seed)
    if kind == "msda":
        return _msda_exact(case, seed)
    return _letterbox_exact(case, seed)


# ---- work and tolerance --------------------------------------------------------


def _counted(c):
    g = _Graph(0, meta=True)
    n, h, w = c["batch"], c["h"], c["w"]
    if c["kind"] == "detect":
        x = [torch.empty(n, c["c%d" % i], h >> i, w >> i, device="meta") for i in range(3)]
        read = sum(t.numel() for t in x)
    else:
        x = torch.empty(n, 3 if c["kind"] == "net" else c["c"], h, w, device="meta")
        read = x.numel()
    return g, read, sum(t.numel() for t in g.forward(c, x))


def work(case):
    c = case
    kind, n = c["kind"], c["batch"]
    if kind in ("net", "c3k2", "c2psa", "detect"):
        g, read, written = _counted(c)
        return {"bytes": 4.0 * (read + written) + ES[c["dtype"]] * g.weights, "flops": g.flops}
    if kind in ("conv", "dw"):
        ho, wo = _out_hw(c)
        cin, cout, k = c.get("cin", c.get("c")), c.get("cout", c.get("c")), c.get("k", 3)
        per = k * k * (1 if kind == "dw" else cin)
        elems = n * (c["h"] * c["w"] * cin + ho * wo * cout * (2 if c.get("res") else 1)) + cout * per
        return {"bytes": float(ES[c["dtype"]] * elems), "flops": 2.0 * n * ho * wo * cout * per}
    if kind == "post":
        a = sum((c["h"] // s) * (c["w"] // s) for s in STRIDES)
        return {"bytes": 4.0 * n * (a * (4 + c["nc"]) + 7 * c["max_det"]), "flops": 4.0 * n * a * c["nc"]}
    if kind == "msda":
        s = sum(h * w for h, w in _msda_shapes(c))
        lp = c["levels"] * c["points"]
        return {"bytes": 4.0 * n * (s * c["heads"] * 32 + c["q"] * (2 + c["heads"] * (3 * lp + 32))),
                "flops": 9.0 * n * c["q"] * c["heads"] * lp * 32}
    sc = c["size"] / max(c["h"], c["w"])
    taps = max(1.0, 1.0 / sc) * 4
    return {"bytes": n * (3.0 * c["h"] * c["w"] + 12.0 * c["size"] ** 2), "flops": 6.0 * n * c["size"] ** 2 * taps}


def _memory(c):
    """About the bytes of a case's largest tensors, intermediate maps included."""
    if c["kind"] == "net":
        return 900.0 * c["batch"] * c["h"] * c["w"] * VARIANTS[c["variant"]][1] * (2 if c["dtype"] == "f32" else 1) / 4
    return work(c)["bytes"]


def tolerance(case):
    """Relative errors of another correct implementation at the same precision:
    about four times what another summation order (another tile) gave.  A
    conv differed by 4e-5 (one bfloat16 step at worst), a block by 1e-4, the
    medium network, where one layer's rounding travels through all that
    follow, by 0.011.  Attention rounds its probabilities, so blocks that hold
    it are given more."""
    kind = case["kind"]
    if kind in ("post", "letterbox"):   # defined to the last bit: the same rounding steps in the same order
        return "exact"
    if kind == "msda":                  # float32 sampling positions: 2e-6 off float64
        return {"rel": 1e-5, "max": 1e-3}
    if kind in ("conv", "dw"):
        if case["dtype"] == "fp8":      # e4m3 bytes: ties of the rounding
            return {"rel": 0.0, "differ": 2e-3}
        return {"rel": 2e-6, "max": 1e-4} if case["dtype"] == "f32" else {"rel": 5e-4, "max": 2e-2}
    if case["dtype"] == "f32":
        return {"rel": 2e-5, "max": 2e-3}
    return {"rel": 3e-2, "max": 0.9} if kind == "net" else {"rel": 5e-3, "max": 0.1}
