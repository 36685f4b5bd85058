"""The workloads whose speed is tracked, each through the package's public
entry points on inputs that are resident on the GPU.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) the inputs (and plan) a program holds before the call
run(state)          one pass; returns every output, whole
work(case)          bytes and FLOPs one pass cannot do without
exact(case, seed)   the outputs in FP64 from plain torch

Sizes are given in af order (dim0 = width fastest); torch tensors hold the
same bytes with the dims reversed.
"""
from __future__ import annotations

import math
import random

import torch

import arrayfire_amd as af

_AF = {"f32": af.f32, "f16": af.f16, "bf16": af.bf16, "u8": af.u8, "b8": af.b8}
_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "u8": torch.uint8, "b8": torch.bool}
_TYPESTR = {"f32": "<f4", "f16": "<f2", "bf16": "<i2", "u8": "|u1", "b8": "|b1"}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "u8": 1, "b8": 1}


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one small image through a 5x5 smoothing: the smallest call, where
        # the launch and the host path count
        _conv2("conv2_512_5x5", 512, 512, 1, 5, 5),
        # a frame in colour planes as a camera delivers it: bytes, odd sides,
        # the full (EXPAND) result
        _conv2("conv2_u8_frame_5x5", 1919, 1079, 3, 5, 5, mode=1, dtype="u8"),
        # a large batch of images under one 7x7 filter: the largest call
        _conv2("conv2_batch_7x7", 1024, 1024, 256, 7, 7),
        # Gaussian smoothing of such a batch, 17 taps each way
        {"name": "sep_batch_17", "kind": "sep", "w": 1024, "h": 1024, "n": 256, "f": 17, "mode": 0},
        # a volume through a 3x3x3 stencil
        {"name": "conv3_128_3x3x3", "kind": "conv3", "w": 128, "h": 128, "d": 128, "f": 3, "mode": 0},
        # an image through a filter past the spatial limit: the frequency domain
        {"name": "fft_1024_31x31", "kind": "fft", "w": 1024, "h": 1024, "n": 1, "fw": 31, "fh": 31, "mode": 0},
        # many small images of different sizes and filters in one planned launch
        {"name": "ragged_60", "kind": "ragged", "count": 60, "lo": 64, "hi": 1024, "pick": 20261206},
        # edge detection: the separable path inside a whole pipeline
        {"name": "canny_1024", "kind": "canny", "w": 1024, "h": 1024, "n": 1, "otsu": False, "low": 0.1, "high": 0.3},
        # the training step of a convolution layer, forward and both
        # gradients: 16-bit operands, then the same layer in FP32
        _nn("nn_step_bf16", "step", "bf16", 56, 56, 64, 32, 128, 3, 1, 1),
        _nn("nn_step_f32", "step", "f32", 56, 56, 64, 32, 128, 3, 1, 1),
        # a small strided layer's step as a captured plan
        _nn("nn_plan_bf16_s2", "plan", "bf16", 28, 28, 128, 16, 128, 3, 2, 1),
        # inference through a layer of odd width and a 5x5 filter
        _nn("nn_fwd_f16_27_5x5", "fwd", "f16", 27, 27, 96, 16, 128, 5, 1, 2),
    ]


def _conv2(name, w, h, n, fw, fh, mode=0, dtype="f32"):
    return {"name": name, "kind": "conv2", "w": w, "h": h, "n": n, "fw": fw, "fh": fh, "mode": mode, "dtype": dtype}


def _nn(name, api, dtype, w, h, c, n, k, f, s, p):
    return {"name": name, "kind": "nn", "api": api, "dtype": dtype, "w": w, "h": h, "c": c, "n": n, "k": k, "f": f,
            "stride": s, "pad": p}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv2", "conv2", "sep", "conv3", "fft", "ragged", "canny", "nn", "nn", "nn"])
    if kind == "conv2":
        w, h, n = _log(rng, 48, 2048), _log(rng, 48, 2048), _log(rng, 1, 128)
        n = max(1, min(n, (1 << 27) // (w * h)))
        f = rng.choice([3, 5, 7, 9])
        c = _conv2("", w, h, n, f, f, rng.randrange(2), rng.choice(["f32", "f32", "f32", "u8"]))
        if c["dtype"] == "u8":  # pictures in bytes come as frames, not as thousands
            c["n"] = min(c["n"], 8)
    elif kind == "sep":
        w, h, n = _log(rng, 48, 2048), _log(rng, 48, 2048), _log(rng, 1, 128)
        n = max(1, min(n, (1 << 27) // (w * h)))
        c = {"kind": kind, "w": w, "h": h, "n": n, "f": rng.choice([3, 5, 9, 13, 17]), "mode": rng.randrange(2)}
    elif kind == "conv3":
        c = {"kind": kind, "w": _log(rng, 24, 192), "h": _log(rng, 24, 192), "d": _log(rng, 16, 128),
             "f": rng.choice([3, 3, 5]), "mode": rng.randrange(2)}
    elif kind == "fft":
        fw, fh = rng.randrange(19, 64), rng.randrange(19, 64)
        w, h = _log(rng, 150, 1900), _log(rng, 150, 1900)
        n = 1 if w * h > 300_000 else rng.randrange(1, 4)
        c = {"kind": kind, "w": w, "h": h, "n": n, "fw": fw, "fh": fh, "mode": rng.randrange(2)}
    elif kind == "ragged":
        c = {"kind": kind, "count": rng.randrange(12, 61), "lo": 64, "hi": 1024, "pick": rng.randrange(1 << 30)}
    elif kind == "canny":
        w, h = _log(rng, 100, 1024), _log(rng, 100, 1024)
        n = 1 if w * h > 200_000 else rng.randrange(1, 4)
        c = {"kind": kind, "w": w, "h": h, "n": n, "otsu": rng.random() < 0.25, "low": rng.choice([0.05, 0.1, 0.2]),
             "high": rng.choice([0.3, 0.4])}
    else:
        f = rng.choice([1, 3, 3, 3, 3, 5])
        c = _nn("", rng.choice(["step", "step", "plan", "fwd"]), rng.choice(["bf16", "bf16", "f32", "f16"]),
                rng.randrange(7, 81), rng.randrange(7, 81), rng.choice([3, 16, 32, 48, 64, 96, 128, 256]), 1,
                rng.choice([16, 32, 64, 96, 128, 256]), f, rng.choice([1, 1, 1, 2]), f // 2)
        c["n"] = min(_log(rng, 1, 32), max(1, int(4e9 / _nn_flops(c))))
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, shape):
    return torch.rand(shape, generator=g, device="cuda")


def _gauss(f):
    x = torch.arange(f, dtype=torch.float64) - (f - 1) / 2
    k = torch.exp(-0.5 * (x / (0.25 * (f - 1) / 2 + 0.75)) ** 2)
    return (k / k.sum()).float().cuda()


def _picture(g, n, h, w):
    """A picture in [0, 255]: soft shapes, a few hard-edged boxes, specks."""
    low = torch.nn.functional.interpolate(_rand(g, (n, 1, max(2, h // 12), max(2, w // 12))), size=(h, w),
                                          mode="bicubic", align_corners=False)[:, 0].clamp(0, 1) * 160
    box = torch.zeros(n, h, w, device="cuda")
    at = _rand(g, (12, 4)).tolist()
    for x0, y0, dx, dy in at:
        box[:, int(y0 * h):int((y0 + 0.3 * dy) * h), int(x0 * w):int((x0 + 0.3 * dx) * w)] += 30.0
    return (low + box + (_rand(g, (n, h, w)) > 0.997) * 50.0 + 2.0 * _rand(g, (n, h, w))).clamp(0, 255)


def _problems(case):
    r = random.Random(case["pick"])
    return [(_log(r, case["lo"], case["hi"]), _log(r, case["lo"], case["hi"]), r.randrange(3, 16, 2),
             r.randrange(3, 16, 2), r.randrange(2)) for _ in range(case["count"])]


def _nn_out(case):
    f, s, p = case["f"], case["stride"], case["pad"]
    return 1 + (case["w"] + 2 * p - f) // s, 1 + (case["h"] + 2 * p - f) // s


def _inputs(case, seed):
    """The case's input tensors (dims reversed from af order)."""
    g, k = _gen(seed), case["kind"]
    if k == "conv2":
        if case["dtype"] == "u8":
            t = _gauss(case["fw"])
            return [(_picture(g, case["n"], case["h"], case["w"])).to(torch.uint8), torch.outer(t, t)]
        return [_rand(g, (case["n"], case["h"], case["w"])), _rand(g, (case["fh"], case["fw"])) * 2 - 1]
    if k == "sep":
        return [_rand(g, (case["n"], case["h"], case["w"])), _gauss(case["f"])]
    if k == "conv3":
        return [_rand(g, (case["d"], case["h"], case["w"])), _rand(g, (case["f"],) * 3) * 2 - 1]
    if k == "fft":
        return [_rand(g, (case["n"], case["h"], case["w"])),
                torch.randn((case["fh"], case["fw"]), generator=g, device="cuda")]
    if k == "ragged":
        return [t for w, h, fw, fh, _ in _problems(case) for t in (_rand(g, (h, w)), _rand(g, (fh, fw)))]
    if k == "canny":
        return [_picture(g, case["n"], case["h"], case["w"])]
    ow, oh = _nn_out(case)
    dt, f = _TORCH[case["dtype"]], case["f"]
    x = torch.randn((case["n"], case["c"], case["h"], case["w"]), generator=g, device="cuda")
    w = torch.randn((case["k"], case["c"], f, f), generator=g, device="cuda") * math.sqrt(2.0 / (case["c"] * f * f))
    dy = torch.randn((case["n"], case["k"], oh, ow), generator=g, device="cuda")
    return [x.to(dt), w.to(dt), dy.to(dt)]


class _Memory:
    """An af array's device memory, as other GPU libraries take it."""

    def __init__(self, array, shape, dtype):
        self.array = array  # keeps the memory while a tensor looks at it
        self.__cuda_array_interface__ = {"shape": shape, "typestr": _TYPESTR[dtype],
                                         "data": (array.device_ptr(), False), "version": 3}


def _tensor(array, shape, dtype):
    t = torch.as_tensor(_Memory(array, shape, dtype), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def _array(t, dtype="f32"):
    """A new af array holding a copy of the device tensor t."""
    a = af.constant(0, tuple(reversed(t.shape)), _AF[dtype])
    af.sync()
    _tensor(a, tuple(t.shape), dtype).copy_(t)
    torch.cuda.synchronize()
    return a


# --------------------------------------------------------------------- run
def prepare(case, seed):
    k = case["kind"]
    t = _inputs(case, seed)
    s = {"case": case, "dtype": case.get("dtype", "f32"), "shape": _out_shape(case)}
    if k == "nn":
        s["in"] = [_array(v, case["dtype"]) for v in t]
        if case["api"] == "plan":
            s["plan"] = p = af.NNStepPlan(*s["in"], (case["stride"],) * 2, (case["pad"],) * 2, (1, 1))
            s["out"] = [_tensor(a, tuple(v.shape), case["dtype"]) for a, v in zip((p.dx, p.dw), t)]
            s["out"].insert(0, _tensor(p.y, tuple(t[2].shape), case["dtype"]))
        else:
            s["in_shapes"] = [tuple(v.shape) for v in t]
    elif k == "ragged":
        a = [_array(v) for v in t]
        probs = _problems(case)
        s["plan"] = af.RaggedPlan(a[0::2], a[1::2], [p[4] for p in probs])
        s["out"] = [_tensor(o, shape, "f32") for o, shape in zip(s["plan"].outputs, s["shape"])]
    else:
        s["in"] = [_array(t[0], s["dtype"])] + [_array(v) for v in t[1:]]
    return s


def _out_shape(case):
    k = case["kind"]
    if k == "ragged":
        return [(h + (fh - 1) * m, w + (fw - 1) * m) for w, h, fw, fh, m in _problems(case)]
    if k == "conv3":
        e = case["mode"] * (case["f"] - 1)
        return (case["d"] + e, case["h"] + e, case["w"] + e)
    if k == "nn":
        ow, oh = _nn_out(case)
        return (case["n"], case["k"], oh, ow)
    e = case.get("mode", 0)
    return (case["n"], case["h"] + e * (case.get("fh", case.get("f", 1)) - 1),
            case["w"] + e * (case.get("fw", case.get("f", 1)) - 1))


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "conv2":
        return _tensor(af.convolve2(*s["in"], c["mode"], af.AF_CONV_AUTO), s["shape"], c["dtype"])
    if k == "sep":
        x, f = s["in"]
        return _tensor(af.convolve_sep(f, f, x, c["mode"]), s["shape"], "f32")
    if k == "conv3":
        return _tensor(af.convolve3(*s["in"], c["mode"], af.AF_CONV_AUTO), s["shape"], "f32")
    if k == "fft":
        return _tensor(af.convolve2(*s["in"], c["mode"], af.AF_CONV_AUTO), s["shape"], "f32")
    if k == "canny":
        return _tensor(af.canny(s["in"][0], int(c["otsu"]), c["low"], c["high"]), s["shape"], "b8")
    if "plan" in s:  # the ragged list and the captured step
        s["plan"].run()
        return s["out"]
    x, w, dy = s["in"]
    geo = ((c["stride"],) * 2, (c["pad"],) * 2, (1, 1))
    y = af.convolve2NN(x, w, *geo)
    out = [_tensor(y, s["shape"], c["dtype"])]
    if c["api"] == "step":
        dx = af.convolve2GradientNN(dy, x, w, y, *geo, af.AF_CONV_GRADIENT_DATA)
        dw = af.convolve2GradientNN(dy, x, w, y, *geo, af.AF_CONV_GRADIENT_FILTER)
        out += [_tensor(dx, s["in_shapes"][0], c["dtype"]), _tensor(dw, s["in_shapes"][1], c["dtype"])]
    return out


# -------------------------------------------------------------------- work
def _nn_flops(case):
    ow, oh = _nn_out(case)
    return 2.0 * case["n"] * case["k"] * case["c"] * case["f"] ** 2 * ow * oh


def work(case):
    k = case["kind"]
    if k == "ragged":
        b = fl = 0.0
        for (w, h, fw, fh, _), (oh, ow) in zip(_problems(case), _out_shape(case)):
            b += 4.0 * (w * h + fw * fh + ow * oh)
            fl += 2.0 * fw * fh * ow * oh
        return {"bytes": b, "flops": fl}
    out = float(math.prod(_out_shape(case)))
    if k == "nn":
        e = _BYTES[case["dtype"]]
        x, w = case["n"] * case["c"] * case["h"] * case["w"], case["k"] * case["c"] * case["f"] ** 2
        one = case["api"] == "fwd"
        # the step reads x, w and dy and writes y, dx and dw
        return {"bytes": float(e * ((x + w + out) if one else 2 * (x + w + out))),
                "flops": _nn_flops(case) * (1 if one else 3)}
    src = float(case["w"] * case["h"] * case.get("d", case.get("n", 1)))
    if k == "conv3":
        return {"bytes": 4 * (src + out), "flops": 2.0 * case["f"] ** 3 * out}
    if k == "sep":
        return {"bytes": 4 * (src + out), "flops": 4.0 * case["f"] * out}
    if k == "canny":
        # 5-tap smoothing both ways, Sobel, magnitude, interpolation, thresholds
        return {"bytes": 5 * src, "flops": 60.0 * src}
    e = _BYTES[case.get("dtype", "f32")]
    if k == "fft":
        # a transform of the padded picture there and back, and the product
        L = math.prod(1 << (case[d] + case["f" + d] - 2).bit_length() for d in ("w", "h"))
        return {"bytes": 4 * (src + out), "flops": case["n"] * (5.0 * L * math.log2(L) + 3.0 * L)}
    return {"bytes": e * (src + out), "flops": 2.0 * case["fw"] * case["fh"] * out}


# ------------------------------------------------------------------- exact
def _conv_f64(x, f, expand):
    """True convolution over the trailing dims of x (as many as f has), in
    FP64: the full result, or the part of x's size that starts at f // 2."""
    r = f.dim()
    pads = [p for d in reversed(f.shape) for p in (d - 1, d - 1)]
    f = f.double()
    shape = [x.shape[x.dim() - r + i] + f.shape[i] - 1 for i in range(r)]
    lo = [0 if expand else f.shape[i] // 2 for i in range(r)]
    size = [shape[i] if expand else shape[i] - f.shape[i] + 1 for i in range(r)]
    xp = torch.nn.functional.pad(x.double(), pads)
    out = torch.zeros(list(x.shape[:x.dim() - r]) + size, dtype=torch.float64, device=x.device)
    for at, v in zip(torch.cartesian_prod(*[torch.arange(d) for d in f.shape]).reshape(-1, r).tolist(),
                     f.reshape(-1).tolist()):
        part = xp
        for i in range(r):
            part = part.narrow(x.dim() - r + i, lo[i] + f.shape[i] - 1 - at[i], size[i])
        out.add_(part, alpha=v)
    return out


def _nn_f64(case, x, w):
    ow, oh = _nn_out(case)
    s, p, f = case["stride"], case["pad"], case["f"]
    xp = torch.nn.functional.pad(x, (p, p, p, p))
    y = 0
    for b in range(f):
        for a in range(f):
            cut = xp[:, :, b:b + (oh - 1) * s + 1:s, a:a + (ow - 1) * s + 1:s].reshape(case["n"], case["c"], oh * ow)
            y = y + torch.matmul(w[:, :, f - 1 - b, f - 1 - a].contiguous(), cut)
    return y.reshape(case["n"], case["k"], oh, ow)


def exact(case, seed):
    k = case["kind"]
    if k == "canny" or case.get("dtype") == "u8":
        return None  # whole numbers
    t = _inputs(case, seed)
    if k == "conv2" or k == "fft" or k == "conv3":
        if k == "conv3":
            return _conv_f64(t[0], t[1], case["mode"])
        return torch.cat([_conv_f64(x, t[1], case["mode"]) for x in t[0].split(16)])
    if k == "sep":
        f = t[1]
        return torch.cat([_conv_f64(_conv_f64(x, f[None, :], case["mode"]), f[:, None], case["mode"])
                          for x in t[0].split(16)])
    if k == "ragged":
        return [_conv_f64(x, f, p[4]) for x, f, p in zip(t[0::2], t[1::2], _problems(case))]
    x, w, dy = (v.double() for v in t)
    if case["api"] == "fwd":
        return [_nn_f64(case, x, w)]
    x.requires_grad_(True)
    w.requires_grad_(True)
    y = _nn_f64(case, x, w)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    return [y.detach(), dx, dw]
