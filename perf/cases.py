"""The performance cases of the framework: what its users run, over the sizes they run it at.

A case is a dict of plain values.  Its "path" names the entry points a pass goes through:

  i8     qconv2d_nhwc_i8 and its _dequant / _acc32 forms: one layer of int8 inference
  qi32   launch_fprop_nhwc_qi32 and its blocked form: one layer on the float-code surface
  f32    launch_fprop_nhwc: one layer of fp32 inference
  step   launch_{fprop,bprop,grad}_nhwc: one layer of fp32 training, forward and backward
  bstep  launch_block_{fprop,bprop,grad}_nhwc with a bias: one blocked layer of fp32 training
  bmm    bmm_matmul_i32: the integer product

Convolution fields: n, h, w, c, k, r, s, pad, stride, dil, groups (square padding, stride and
dilation).  Layer sizes are those of the int8 workloads, of the fp32 and blocked suites and of
the integer products that bench.py runs, or generic ones of the same kind.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import my_own_cnn_amd as M
from my_own_cnn_amd.conv import BlockConv2DParams, Conv2DParams, DataType, qparams_array

IN_SCALE = 0.02


def _conv(name, path, n, h, w, c, k, r, s, pad, stride=1, dil=1, groups=1, **more):
    case = {"name": name, "path": path, "n": n, "h": h, "w": w, "c": c, "k": k, "r": r, "s": s, "pad": pad,
            "stride": stride, "dil": dil, "groups": groups, **more}
    if name is None:
        del case["name"]
    return case


def _bmm(name, batch, m, n, kdim, ta, tb, values):
    case = {"name": name, "path": "bmm", "batch": batch, "m": m, "n": n, "kdim": kdim, "ta": ta, "tb": tb,
            "values": values}
    if name is None:
        del case["name"]
    return case


def listed():
    return [
        # int8 inference, the five benchmark layers, two at their batch and three at a serving batch.
        # The smallest call: latency and launch cost.
        _conv("i8_tiny", "i8", 1, 32, 32, 16, 32, 3, 3, 1, relu=False, out="i8"),
        # the headline layer, the body of a residual network
        _conv("i8_3x3", "i8", 32, 56, 56, 64, 64, 3, 3, 1, relu=True, out="i8"),
        # an expanding pointwise layer: the output outweighs the input four to one
        _conv("i8_1x1", "i8", 256, 28, 28, 128, 512, 1, 1, 0, relu=False, out="i8"),
        # a down-sampling layer: the largest int8 work
        _conv("i8_down", "i8", 128, 56, 56, 128, 256, 3, 3, 1, stride=2, relu=True, out="i8"),
        # an image stem: three channels, 7x7
        _conv("i8_stem", "i8", 128, 224, 224, 3, 64, 7, 7, 3, stride=2, relu=True, out="i8"),
        # a layer of odd sizes whose result leaves the integer network as floats
        _conv("i8_ragged", "i8", 5, 37, 29, 48, 80, 3, 3, 1, relu=False, out="f32"),
        # the float-code surface on the headline layer
        _conv("qi32_3x3", "qi32", 32, 56, 56, 64, 64, 3, 3, 1, codes="u8", by=1, bx=1),
        # fp32 inference of one image
        _conv("f32_image", "f32", 1, 56, 56, 64, 64, 3, 3, 1),
        # fp32 training: the ordinary layer, a strided one, a blocked one
        _conv("step_3x3", "step", 32, 56, 56, 64, 64, 3, 3, 1),
        _conv("step_down", "step", 32, 112, 112, 32, 32, 3, 3, 1, stride=2),
        _conv("bstep_28x28", "bstep", 32, 28, 28, 128, 256, 3, 3, 1, by=2, bx=4),
        # the integer product of a lowered 3x3 layer: centred codes, tall and narrow
        _bmm("bmm_lowered", 1, 32 * 56 * 56, 64, 576, False, True, "codes"),
    ]


# ---- drawn cases ----------------------------------------------------------------------------

def _log(rng, lo, hi):
    """An integer spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _extent(h, r, pad, stride, dil):
    return (h + 2 * pad - dil * (r - 1) - 1) // stride + 1


def _macs(case):
    ho = _extent(case["h"], case["r"], case["pad"], case["stride"], case["dil"])
    wo = _extent(case["w"], case["s"], case["pad"], case["stride"], case["dil"])
    return case["n"] * ho * wo * case["k"] * case["r"] * case["s"] * (case["c"] // case["groups"])


def _capped(case, macs):
    """The case with its batch, then its image, cut until it does no more than `macs`."""
    while _macs(case) > macs and case["n"] > 1:
        case["n"] = max(1, min(case["n"] - 1, int(case["n"] * macs / _macs(case))))
    while _macs(case) > macs:
        case["h"], case["w"] = max(8, case["h"] * 3 // 4), max(8, case["w"] * 3 // 4)
    return case


def _image(rng, lo, hi):
    h = _log(rng, lo, hi)
    return h, h if rng.random() < 0.6 else max(lo, int(h * rng.uniform(0.6, 1.4)))


def _draw_i8(rng):
    out = rng.choice(["i8", "i8", "i8", "f32", "acc"])
    relu = out != "acc" and rng.random() < 0.6
    kind = rng.choice(["3x3", "3x3", "1x1", "1x1", "down", "stem", "grouped"])
    n = _log(rng, 1, 256)
    ch = [16, 32, 48, 64, 64, 96, 128, 128, 192, 256, 512]
    if kind == "stem":
        h, w = _image(rng, 64, 224)
        r = rng.choice([3, 5, 7, 7])
        case = _conv(None, "i8", n, h, w, 3, rng.choice([32, 64, 64, 96]), r, r, r // 2, stride=2, relu=relu, out=out)
        return _capped(case, 15e9)
    h, w = _image(rng, 7, 112)
    c, k = rng.choice(ch), rng.choice(ch + [40, 80, 1000])
    if kind == "1x1":
        case = _conv(None, "i8", n, h, w, c, k, 1, 1, 0, stride=rng.choice([1, 1, 1, 2]), relu=relu, out=out)
    elif kind == "down":
        case = _conv(None, "i8", n, h, w, c, k, 3, 3, 1, stride=2, relu=relu, out=out)
    elif kind == "grouped":
        g = rng.choice([2, 4])
        case = _conv(None, "i8", n, h, w, 64 * g, rng.choice([32, 64, 128]) * g, 3, 3, 1, groups=g, relu=relu, out=out)
    else:
        d = rng.choice([1, 1, 1, 2])
        case = _conv(None, "i8", n, h, w, c, k, 3, 3, d, dil=d, relu=relu, out=out)
    return _capped(case, 29e9)


def _draw_qi32(rng):
    n = _log(rng, 1, 32)
    codes = rng.choice(["u8", "u8", "s5"])
    kind = rng.choice(["3x3", "1x1", "down", "stem", "blocked"])
    c, k = rng.choice([32, 48, 64, 64, 128]), rng.choice([32, 64, 64, 96, 128, 256])
    if kind == "stem":
        h, w = _image(rng, 64, 224)
        return _capped(_conv(None, "qi32", n, h, w, 3, 64, 7, 7, 3, stride=2, codes=codes, by=1, bx=1), 3.7e9)
    if kind == "blocked":
        by, bx = rng.choice([(2, 2), (2, 4), (4, 4)])
        h, w = by * rng.randint(4, 14), bx * rng.randint(4, 14)
        case = _conv(None, "qi32", n, h, w, 64, 64, 3, 3, 1, codes=codes, by=by, bx=bx)
        while _macs(case) > 3.7e9:  # the image has to stay a multiple of the blocks
            case["n"] //= 2
        return case
    h, w = _image(rng, 7, 64)
    if kind == "1x1":
        case = _conv(None, "qi32", n, h, w, c, k, 1, 1, 0, codes=codes, by=1, bx=1)
    else:
        case = _conv(None, "qi32", n, h, w, c, k, 3, 3, 1, stride=2 if kind == "down" else 1, codes=codes, by=1, bx=1)
    return _capped(case, 3.7e9)


F32_CHANNELS = [16, 20, 32, 48, 64, 64, 96, 128, 256]


def _draw_f32(rng, path):
    n = _log(rng, 1, 32)
    h, w = _image(rng, 7, 112)
    kind = rng.choice(["3x3", "3x3", "1x1", "down", "dilated", "grouped", "depthwise"])
    c, k = rng.choice(F32_CHANNELS), rng.choice(F32_CHANNELS)
    if kind == "1x1":
        return _capped(_conv(None, path, n, h, w, c, k, 1, 1, 0), 3.7e9)
    if kind == "down":
        return _capped(_conv(None, path, n, h, w, c, k, 3, 3, 1, stride=2), 0.93e9)
    if kind == "dilated":
        return _capped(_conv(None, path, n, h, w, c, k, 3, 3, 2, dil=2), 3.7e9)
    if kind == "grouped":
        return _capped(_conv(None, path, n, h, w, 128, 128, 3, 3, 1, groups=4), 3.7e9)
    if kind == "depthwise":
        c = rng.choice([32, 64, 96, 128])
        return _capped(_conv(None, path, n, h, w, c, c, 3, 3, 1, groups=c), 0.11e9)
    return _capped(_conv(None, path, n, h, w, c, k, 3, 3, 1), 3.7e9)


def _draw_bstep(rng):
    by, bx = rng.choice([(2, 2), (2, 4), (4, 4)])
    bh, bw = rng.randint(6, 14), rng.randint(6, 14)
    c, k = rng.choice([32, 64, 64, 128]), rng.choice([32, 64, 96, 128])
    r = rng.choice([1, 3, 3])
    case = _conv(None, "bstep", _log(rng, 1, 32), by * bh, bx * bw, c, k, r, r, r // 2, by=by, bx=bx)
    while _macs(case) > 3.7e9:
        case["n"] //= 2
    return case


def _draw_bmm(rng):
    ta, tb = rng.random() < 0.5, rng.random() < 0.5
    values = rng.choice(["codes", "full"])
    if rng.random() < 0.4:  # a lowered layer
        return _bmm(None, 1, _log(rng, 196, 100352), rng.choice([32, 64, 64, 100, 128]), 9 * rng.choice([16, 32, 64]),
                    False, True, values)
    m, n, kdim = _log(rng, 33, 1024), _log(rng, 33, 1024), _log(rng, 33, 1024)
    batch = max(1, min(_log(rng, 1, 32), int(4e9 / (m * n * kdim))))
    return _bmm(None, batch, m, n, kdim, ta, tb, values)


def draw(rng):
    path = rng.choice(["i8"] * 5 + ["qi32"] * 2 + ["f32"] + ["step"] * 3 + ["bstep"] + ["bmm"])
    if path == "i8":
        return _draw_i8(rng)
    if path == "qi32":
        return _draw_qi32(rng)
    if path == "bstep":
        return _draw_bstep(rng)
    if path == "bmm":
        return _draw_bmm(rng)
    return _draw_f32(rng, path)


# ---- inputs -----------------------------------------------------------------------------------

def _params(case):
    return Conv2DParams(case["pad"], case["pad"], case["stride"], case["stride"], case["dil"], case["dil"],
                        case["groups"])


def _dims(case):
    return tuple(case[f] for f in ("n", "h", "w", "c", "r", "s", "k"))


def _out_hw(case):
    return (_extent(case["h"], case["r"], case["pad"], case["stride"], case["dil"]),
            _extent(case["w"], case["s"], case["pad"], case["stride"], case["dil"]))


def _w_shape(case):
    blocks = (case["by"], case["bx"]) if case["path"] == "bstep" or case.get("by", 1) * case.get("bx", 1) > 1 else ()
    return (case["k"], *blocks, case["r"], case["s"], case["c"] // case["groups"])


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def ints(shape, lo, hi, dtype):
        return torch.randint(lo, hi + 1, shape, generator=gen, device=dev, dtype=torch.int64).to(dtype)

    def normal(shape, scale=1.0):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32) * scale

    state = {"case": dict(case)}
    if case["path"] == "bmm":
        b, m, n, kd = case["batch"], case["m"], case["n"], case["kdim"]
        lo, hi = (-255, 255) if case["values"] == "codes" else (-2 ** 31, 2 ** 31 - 1)
        state["a"] = ints((b, kd, m) if case["ta"] else (b, m, kd), lo, hi, torch.int32)
        state["b"] = ints((b, n, kd) if case["tb"] else (b, kd, n), lo, hi, torch.int32)
        return state

    n, h, w, c, r, s, k = _dims(case)
    ho, wo = _out_hw(case)
    x_shape, w_shape, y_shape = (n, h, w, c), _w_shape(case), (n, ho, wo, k)
    if case["path"] == "i8":
        # the activations behind a ReLU are half zeros; an image or a linear layer's output is not
        if case["relu"] and c > 4:
            state["x"] = ints(x_shape, -127, 127, torch.int16).clamp_(min=0).to(torch.int8)
        else:
            state["x"] = ints(x_shape, -128, 127, torch.int8)
        state["w"] = ints(w_shape, -127, 127, torch.int8)
        state["bias"] = ints((k,), -1024, 1024, torch.int32)
        # scales that put the outputs' standard deviation at about a third of the int8 range
        std = 70.0 * 73.0 * math.sqrt(r * s * (c // case["groups"])) * IN_SCALE / 40.0
        state["w_scale"] = (torch.rand((k,), generator=gen, device=dev) * 1.5 + 0.5) / std
        return state
    if case["path"] == "qi32":
        tin = DataType.LinQuantU8 if case["codes"] == "u8" else DataType.LinQuantS5
        lo, hi = (0, 255) if case["codes"] == "u8" else (-16, 15)
        host = np.random.default_rng(seed)
        zps = host.integers(lo, hi + 1, n + 1)
        to_dev = lambda a: torch.from_numpy(a.view(np.uint8).copy()).to(dev)  # noqa: E731
        state.update(tin=tin, in_qp=to_dev(qparams_array(tin, zps[:n])), f_qp=to_dev(qparams_array(tin, zps[n:])),
                     x=ints(x_shape, lo, hi, torch.float32), w=ints(w_shape, lo, hi, torch.float32),
                     y=torch.empty(y_shape, dtype=torch.int32, device=dev))
        return state
    kdim = r * s * (c // case["groups"])
    state["x"] = normal(x_shape).clamp_(min=0)
    state["w"] = normal(w_shape, math.sqrt(2.0 / kdim))
    state["y"] = torch.empty(y_shape, dtype=torch.float32, device=dev)
    if case["path"] != "f32":
        state["dy"] = normal(y_shape, 1e-2)
        state["dx"] = torch.empty(x_shape, dtype=torch.float32, device=dev)
        state["dw"] = torch.empty(w_shape, dtype=torch.float32, device=dev)
    if case["path"] == "bstep":
        state["bias"] = normal((k, case["by"], case["bx"]), 0.1)
        state["dbias"] = torch.empty((k, case["by"], case["bx"]), dtype=torch.float32, device=dev)
    return state


# ---- one pass ---------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    path = case["path"]
    if path == "i8":
        conv = {"stride": case["stride"], "padding": case["pad"], "dilation": case["dil"], "groups": case["groups"]}
        if case["out"] == "acc":
            return M.qconv2d_nhwc_i8_acc32(state["x"], state["w"], **conv)
        op = M.qconv2d_nhwc_i8 if case["out"] == "i8" else M.qconv2d_nhwc_i8_dequant
        return op(state["x"], state["w"], state["bias"], state["w_scale"], relu=case["relu"], in_scale=IN_SCALE, **conv)
    if path == "bmm":
        return M.bmm_i32(state["a"], state["b"], trans_a=case["ta"], trans_b=case["tb"])
    dims = _dims(case)
    x, w, y = state["x"], state["w"], state["y"]
    if path == "qi32":
        if case["by"] * case["bx"] > 1:
            bp = BlockConv2DParams(_params(case), case["by"], case["bx"])
            M.launch_block_fprop_nhwc_qi32(state["tin"], x, w, y, *dims, bp, state["in_qp"], state["f_qp"])
        else:
            M.launch_fprop_nhwc_qi32(state["tin"], x, w, y, *dims, _params(case), state["in_qp"], state["f_qp"])
        return y
    if path == "f32":
        M.launch_fprop_nhwc(x, w, y, *dims, _params(case))
        return y
    dy, dx, dw = state["dy"], state["dx"], state["dw"]
    if path == "step":
        p = _params(case)
        M.launch_fprop_nhwc(x, w, y, *dims, p)
        M.launch_bprop_nhwc(dy, w, dx, *dims, p)
        M.launch_grad_nhwc(x, dy, dw, *dims, p)
        return {"y": y, "dx": dx, "dw": dw}
    bp = BlockConv2DParams(_params(case), case["by"], case["bx"])
    M.launch_block_fprop_nhwc(x, w, y, *dims, bp, state["bias"])
    M.launch_block_bprop_nhwc(dy, w, dx, *dims, bp)
    M.launch_block_grad_nhwc(x, dy, dw, *dims, bp, state["dbias"])
    return {"y": y, "dx": dx, "dw": dw, "dbias": state["dbias"]}


# ---- what a pass cannot do without --------------------------------------------------------------

def work(case):
    if case["path"] == "bmm":
        b, m, n, kd = case["batch"], case["m"], case["n"], case["kdim"]
        return {"bytes": 4 * b * (m * kd + kd * n + m * n), "flops": 2 * b * m * n * kd}
    n, h, w, c, r, s, k = _dims(case)
    ho, wo = _out_hw(case)
    xs, ws, ys = n * h * w * c, math.prod(_w_shape(case)), n * ho * wo * k
    flops = 2 * _macs(case)
    if case["path"] == "i8":
        out = 1 if case["out"] == "i8" else 4
        return {"bytes": xs + ws + out * ys + (0 if case["out"] == "acc" else 8 * k), "flops": flops}
    if case["path"] in ("qi32", "f32"):
        return {"bytes": 4 * (xs + ws + ys), "flops": flops}
    extra = 2 * 4 * k * case["by"] * case["bx"] if case["path"] == "bstep" else 0
    # reads x, w, dy once; writes y, dx, dw once
    return {"bytes": 4 * 2 * (xs + ws + ys) + extra, "flops": 3 * flops}


def tolerance(case):
    """int8, int32 and the integer product are exact.  The dequantized view is two fp32 roundings.
    An fp32 sum is off by its own rounding, which grows with the square root of its length; the
    longest is the filter gradient's, over every output position."""
    if case["path"] == "i8":
        return {"rel": 5e-7, "max": 2e-6} if case["out"] == "f32" else "exact"
    if case["path"] in ("qi32", "bmm"):
        return "exact"
    return {"rel": 4e-6, "max": 1e-4}


# ---- the same results in 64 bits ------------------------------------------------------------------

def _taps(case):
    """(r, s, rows, cols): each filter tap and the slices of the padded image its outputs read."""
    ho, wo = _out_hw(case)
    st, d = case["stride"], case["dil"]
    for i in range(case["r"]):
        for j in range(case["s"]):
            yield i, j, slice(i * d, i * d + (ho - 1) * st + 1, st), slice(j * d, j * d + (wo - 1) * st + 1, st)


def _blocks(case):
    """(index into the filter, output rows, output columns) of each filter block."""
    ho, wo = _out_hw(case)
    by, bx = case.get("by", 1), case.get("bx", 1)
    blocked = len(_w_shape(case)) == 6
    for i in range(by):
        for j in range(bx):
            idx = (slice(None), i, j) if blocked else (slice(None),)
            yield idx, slice(i * ho // by, (i + 1) * ho // by), slice(j * wo // bx, (j + 1) * wo // bx)


def _pad64(x, case):
    p = case["pad"]
    return torch.nn.functional.pad(x.double(), (0, 0, p, p, p, p))


def _mm(a, b):
    return torch.matmul(a.contiguous(), b.contiguous())


def _forward64(x, w, case):
    xp, wd = _pad64(x, case), w.double()
    ho, wo = _out_hw(case)
    n, g, k = case["n"], case["groups"], case["k"]
    cg, kg = case["c"] // g, k // g
    y = torch.zeros((n, ho, wo, k), dtype=torch.float64, device=x.device)
    for i, j, rows, cols in _taps(case):
        xs = xp[:, rows, cols, :]
        for idx, bh, bw in _blocks(case):
            part = xs[:, bh, bw, :]
            tap = wd[idx][:, i, j, :]
            if cg == 1 and kg == 1:
                y[:, bh, bw, :] += part * tap[:, 0]
                continue
            for q in range(g):
                o = _mm(part[..., q * cg:(q + 1) * cg].reshape(-1, cg), tap[q * kg:(q + 1) * kg].t())
                y[:, bh, bw, q * kg:(q + 1) * kg] += o.reshape(*part.shape[:3], kg)
    return y


def _backward64(x, w, dy, case):
    xp, wd, dyd = _pad64(x, case), w.double(), dy.double()
    n, h, wd_, c = x.shape
    g, p = case["groups"], case["pad"]
    cg, kg = c // g, case["k"] // g
    dxp = torch.zeros_like(xp)
    dw = torch.zeros_like(wd)
    for i, j, rows, cols in _taps(case):
        xs, dxs = xp[:, rows, cols, :], dxp[:, rows, cols, :]
        for idx, bh, bw in _blocks(case):
            d, part = dyd[:, bh, bw, :], xs[:, bh, bw, :]
            tap, dtap = wd[idx][:, i, j, :], dw[idx][:, i, j, :]
            if cg == 1 and kg == 1:
                dxs[:, bh, bw, :] += d * tap[:, 0]
                dtap[:, 0] = (d * part).sum(dim=(0, 1, 2))
                continue
            for q in range(g):
                dq = d[..., q * kg:(q + 1) * kg].reshape(-1, kg)
                o = _mm(dq, tap[q * kg:(q + 1) * kg])
                dxs[:, bh, bw, q * cg:(q + 1) * cg] += o.reshape(*d.shape[:3], cg)
                dtap[q * kg:(q + 1) * kg] = _mm(dq.t(), part[..., q * cg:(q + 1) * cg].reshape(-1, cg))
    return dxp[:, p:p + h, p:p + wd_, :], dw


def exact(case, seed):
    """The floating-point results in 64 bits; the integer paths are compared bit for bit instead."""
    if case["path"] in ("qi32", "bmm") or (case["path"] == "i8" and case["out"] != "f32"):
        return None
    state = prepare(case, seed)
    x, w = state["x"], state["w"]
    y = _forward64(x, w, case)
    if case["path"] == "i8":
        y = (y + state["bias"].double()) * (state["w_scale"].double() * IN_SCALE)
        return y.clamp(min=0) if case["relu"] else y
    if case["path"] == "f32":
        return y
    dx, dw = _backward64(x, w, state["dy"], case)
    if case["path"] == "step":
        return {"y": y, "dx": dx, "dw": dw}
    dbias = torch.empty(state["dbias"].shape, dtype=torch.float64, device=x.device)
    for (_, i, j), bh, bw in _blocks(case):
        y[:, bh, bw, :] += state["bias"][:, i, j].double()
        dbias[:, i, j] = state["dy"][:, bh, bw, :].double().sum(dim=(0, 1, 2))
    return {"y": y, "dx": dx, "dw": dw, "dbias": dbias}
