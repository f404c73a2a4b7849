"""Performance cases: the work a user of this framework has it do.

Each case is one call (or one short sequence of calls) through the C ABI that
`onnxsharp_amd.native` binds -- the surface a host program holds -- on device
buffers, with weights packed beforehand, as a loaded model keeps them; the
whole network goes through `onnxsharp_amd.yolo11n.Frame`.  The listed cases
stand for ranges that `draw` samples: any size of a range counts as much as
the listed one.

Inputs follow the distributions of the repository's benchmark: matrices
U(-1, 1); activations U(0, 1) with weights N(0, 0.05) and biases N(0, 0.01);
quantized products A N(0, 1) with 8-bit weights over their whole range and
per-column scales U(0.001, 0.02).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch
import torch.nn.functional as F

from onnxsharp_amd import native as N
from onnxsharp_amd import yolo11n
from onnxsharp_amd.layers import ConvLayer, DynamicQuantizeMatMulLayer

# The largest case's operation count bounds what a drawn matrix product may
# cost; convolutions and quantized products have their own.
_MATMUL_FLOPS = 2.0 * 4096 * 1024 * 4096
_CONV_FLOPS = 2.0e9
_DQM_OPS = 2.0 * 1028 * 1280 * 5120


def listed():
    return [
        # one token through a projection (autoregressive decoding): launch and latency
        dict(name="matmul_token", kind="matmul", m=1, k=768, n=768),
        # MatMul + Add(bias), the benchmark's FP32 GEMM
        dict(name="matmul_ffn", kind="matmul", m=1024, k=768, n=768),
        # a batch of sequences through a feed-forward layer: the throughput end
        dict(name="matmul_large", kind="matmul", m=4096, k=1024, n=4096),
        # attention core of an image transformer: 16 x 16 patches + 1 class
        # token, so rows of 257 (odd strides) in both products
        dict(name="attention_257", kind="attention", heads=12, rows=257, dim=64),
        # 3x3 conv + SiLU at 160 x 160, the benchmark's headline layer
        dict(name="conv3x3", kind="conv", n=1, c=64, h=160, w=160, m=64, k=3, s=1, group=1, act="Silu", res=False),
        # the same layer in a residual block over a batch of small maps
        dict(name="conv3x3_batch", kind="conv", n=8, c=64, h=56, w=56, m=64, k=3, s=1, group=1, act="Silu",
             res=True),
        # 1x1 conv + SiLU, the benchmark's pointwise layer
        dict(name="conv1x1", kind="conv", n=1, c=256, h=80, w=80, m=128, k=1, s=1, group=1, act="Silu", res=False),
        # a classifier's first layer: 7x7 stride 2 over an RGB batch
        dict(name="conv_stem", kind="conv", n=4, c=3, h=224, w=224, m=64, k=7, s=2, group=1, act="Relu", res=False),
        # depthwise 3x3 over a batch of large maps: memory-bound
        dict(name="depthwise", kind="conv", n=4, c=128, h=112, w=112, m=128, k=3, s=1, group=128, act="Silu",
             res=False),
        # DynamicQuantizeMatMul, the benchmark's encoder feed-forward shape
        dict(name="dqm_ffn", kind="dqm", m=512, k=512, n=2048, wt="s8"),
        # the same for a long ragged sequence and a wider model
        dict(name="dqm_long", kind="dqm", m=1028, k=1280, n=5120, wt="s8"),
        # a whole detection network: YOLO11n at 640 x 640, one frame
        dict(name="yolo_frame", kind="frame", size=640),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "attention", "conv3x3", "conv3x3", "conv1x1", "stem", "depthwise", "dqm",
                       "dqm", "frame"])
    while True:
        if kind == "matmul":
            c = dict(kind="matmul", m=_log_int(rng, 1, 4096), k=_log_int(rng, 32, 4096), n=_log_int(rng, 32, 8192))
            if rng.random() < 0.5:  # half of them at the round widths of real models
                c["k"], c["n"] = (c["k"] + 31) // 32 * 32, (c["n"] + 31) // 32 * 32
            if 2.0 * c["m"] * c["k"] * c["n"] <= _MATMUL_FLOPS:
                return c
        elif kind == "attention":
            return dict(kind="attention", heads=rng.randint(1, 16), rows=_log_int(rng, 16, 512),
                        dim=rng.choice([32, 64, 80, 128]))
        elif kind == "dqm":
            c = dict(kind="dqm", m=_log_int(rng, 1, 2048), k=_log_int(rng, 64, 2048), n=_log_int(rng, 64, 8192),
                     wt=rng.choice(["s8", "s8", "u8"]))
            if rng.random() < 0.5:
                c["k"], c["n"] = (c["k"] + 31) // 32 * 32, (c["n"] + 31) // 32 * 32
            if 2.0 * c["m"] * c["k"] * c["n"] <= _DQM_OPS:
                return c
        elif kind == "frame":
            return dict(kind="frame", size=32 * rng.randint(4, 20))
        else:
            n, act = rng.choice([1, 1, 1, 2, 4, 8]), rng.choice([None, "Relu", "Silu", "Silu"])
            h, w = _log_int(rng, 10, 160), _log_int(rng, 10, 160)
            if kind == "conv3x3":
                cc, m = 8 * _log_int(rng, 1, 32), 8 * _log_int(rng, 1, 32)
                s = rng.choice([1, 1, 2])
                c = dict(kind="conv", n=n, c=cc, h=h, w=w, m=m, k=3, s=s, group=1, act=act, res=rng.random() < 0.3)
            elif kind == "conv1x1":
                c = dict(kind="conv", n=n, c=8 * _log_int(rng, 2, 64), h=h, w=w, m=8 * _log_int(rng, 2, 64), k=1, s=1,
                         group=1, act=act, res=rng.random() < 0.3)
            elif kind == "stem":
                c = dict(kind="conv", n=n, c=3, h=rng.randint(96, 320), w=rng.randint(96, 320),
                         m=rng.choice([16, 24, 32, 48, 64]), k=rng.choice([3, 5, 7]), s=2, group=1, act=act, res=False)
            else:  # depthwise
                cc = 8 * _log_int(rng, 2, 32)
                c = dict(kind="conv", n=n, c=cc, h=h, w=w, m=cc, k=rng.choice([3, 3, 3, 5]), s=rng.choice([1, 1, 2]),
                         group=cc, act=act, res=rng.random() < 0.3)
            wk = work(c)
            if wk["flops"] <= _CONV_FLOPS and wk["bytes"] <= 6.0e7:
                return c


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _normal(g, shape, std):
    return torch.randn(shape, generator=g, device="cuda") * std


def _out_hw(case):
    p = case["k"] // 2
    return tuple((v + 2 * p - case["k"]) // case["s"] + 1 for v in (case["h"], case["w"]))


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "matmul":
        return dict(a=_uniform(g, (case["m"], case["k"]), -1, 1), b=_uniform(g, (case["k"], case["n"]), -1, 1),
                    bias=_uniform(g, (case["n"],), -1, 1))
    if kind == "attention":
        h, r, d = case["heads"], case["rows"], case["dim"]
        # K comes transposed, [heads, dim, rows], as an exported graph's MatMul takes it
        return dict(q=_normal(g, (h, r, d), 1.0), kt=_normal(g, (h, d, r), 1.0), v=_normal(g, (h, r, d), 1.0))
    if kind == "dqm":
        m, k, n = case["m"], case["k"], case["n"]
        if case["wt"] == "s8":
            w = torch.randint(-127, 128, (k, n), generator=g, device="cuda", dtype=torch.int8)
        else:
            w = torch.randint(0, 256, (k, n), generator=g, device="cuda", dtype=torch.uint8)
        return dict(a=_normal(g, (m, k), 1.0), w=w, ws=_uniform(g, (n,), 0.001, 0.02), bias=_normal(g, (n,), 0.01),
                    zp=None if case["wt"] == "s8" else [131])
    if kind == "conv":
        oh, ow = _out_hw(case)
        return dict(x=_uniform(g, (case["n"], case["c"], case["h"], case["w"]), 0, 1),
                    w=_normal(g, (case["m"], case["c"] // case["group"], case["k"], case["k"]), 0.05),
                    bias=_normal(g, (case["m"],), 0.01),
                    res=_uniform(g, (case["n"], case["m"], oh, ow), 0, 1) if case["res"] else None)
    return dict(x=_uniform(g, (1, 3, case["size"], case["size"]), 0, 1))


# ------------------------------------------------------------------ the path

def _p(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def prepare(case, seed):
    """Device buffers, packed weights and call arguments, as a loaded model holds them."""
    lib = N.lib()
    t = _inputs(case, seed)
    kind = case["kind"]
    new = lambda *shape: torch.empty(shape, dtype=torch.float32, device="cuda")
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        y = new(m, n)
        calls = [(lib.osh_gemm_f32, (m, n, k, _p(t["a"]), k, _p(t["b"]), n, _p(t["bias"]), None, None, N.ACT_NONE,
                                     _p(y), n))]
        return dict(calls=calls, out=y, keep=t)
    if kind == "attention":
        h, r, d = case["heads"], case["rows"], case["dim"]
        sc, pr, y = new(h, r, r), new(h, r, r), new(h, r, d)
        calls = [(lib.osh_gemm_f32_batched, (h, r, r, d, _p(t["q"]), d, r * d, _p(t["kt"]), r, d * r, None,
                                             N.ACT_NONE, _p(sc), r, r * r)),
                 (lib.osh_softmax_f32, (h * r, r, C.c_float(d ** -0.5), _p(sc), _p(pr))),
                 (lib.osh_gemm_f32_batched, (h, r, d, r, _p(pr), r, r * r, _p(t["v"]), d, r * d, None, N.ACT_NONE,
                                             _p(y), d, r * d))]
        return dict(calls=calls, out=(pr, y), keep=(t, sc))
    if kind == "dqm":
        m, k, n = case["m"], case["k"], case["n"]
        layer = DynamicQuantizeMatMulLayer()
        packed = layer.prepack_weights(t["w"], t["zp"])
        nbytes = C.c_size_t()
        N.call("osh_dqmm_scratch_bytes", m, k, C.byref(nbytes))
        scratch = torch.empty(nbytes.value, dtype=torch.uint8, device="cuda")
        y = new(m, n)
        calls = [(lib.osh_dqmm_u8s8, (m, k, n, _p(t["a"]), _p(packed), _p(t["ws"]), n, _p(t["bias"]), _p(y), None,
                                      None, _p(scratch)))]
        return dict(calls=calls, out=y, keep=(t, layer, packed, scratch))
    if kind == "conv":
        pad = case["k"] // 2
        layer = ConvLayer(group=case["group"], strides=[case["s"]] * 2, pads=[pad] * 4, fused_activation=case["act"])
        p, packed = layer.prepack_weights(tuple(t["x"].shape), t["w"])
        y = new(p.n, p.m, p.oh, p.ow)
        act = N.ACTIVATIONS[case["act"]]
        if t["res"] is None:
            calls = [(lib.osh_conv2d_f32, (C.byref(p), _p(t["x"]), _p(packed), _p(t["bias"]), act, _p(y)))]
        else:
            calls = [(lib.osh_conv2d_add_f32, (C.byref(p), _p(t["x"]), _p(packed), _p(t["bias"]), act, _p(t["res"]),
                                               _p(y)))]
        return dict(calls=calls, out=y, keep=(t, layer, p, packed))
    frame = yolo11n.Frame(yolo11n.build(case["size"]), torch.device("cuda"), nstreams=1)
    frame.set_input(t["x"])
    frame.run()  # first-use tile choices
    frame.sync()
    frame.capture()
    return dict(frame=frame, out=tuple(frame.outputs()))


def run(state):
    frame = state.get("frame")
    if frame is not None:
        frame.launch()
        return state["out"]
    stream = _stream()
    for fn, args in state["calls"]:
        N.check(fn(*args, stream))
    return state["out"]


# ------------------------------------------------------------ cost and error

def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4.0 * (m * k + k * n + n + m * n), flops=2.0 * m * k * n)
    if kind == "attention":
        h, r, d = case["heads"], case["rows"], case["dim"]
        # q, k, v in; the probabilities (an output) and the result out
        return dict(bytes=4.0 * h * (4 * r * d + r * r), flops=4.0 * h * r * r * d)
    if kind == "dqm":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4.0 * m * k + k * n + 8.0 * n + 4.0 * m * n, flops=2.0 * m * k * n)
    if kind == "conv":
        oh, ow = _out_hw(case)
        cg = case["c"] // case["group"]
        y = case["n"] * case["m"] * oh * ow
        x = case["n"] * case["c"] * case["h"] * case["w"]
        taps = cg * case["k"] * case["k"]
        return dict(bytes=4.0 * (x + case["m"] * taps + case["m"] + (2 if case["res"] else 1) * y),
                    flops=2.0 * y * taps)
    model = yolo11n.build(case["size"])
    weights = sum(o.w.size + o.b.size for o in model.convs)
    return dict(bytes=4.0 * (model.input.numel + weights + sum(b.numel for b in model.outputs)),
                flops=float(model.flops))


def tolerance(case):
    """About four times the error against 64 bits measured over the ranges:
    32-bit sums of up to 4096 products 1.2e-6, two chained products of an
    attention 5.6e-7, convolutions (up to 2300 products) 9e-7, one rounded
    dequantization of an exact integer 4e-8, a whole network 2.7e-7."""
    kind = case["kind"]
    if kind == "matmul":
        return {"rel": 5e-6, "max": 5e-5}
    if kind == "attention":
        return {"rel": 2.5e-6, "max": 3e-5}
    if kind == "conv":
        return {"rel": 4e-6, "max": 4e-5}
    if kind == "dqm":
        return {"rel": 2.5e-7, "max": 1e-6}
    return {"rel": 1.5e-6, "max": 1e-5}


def _conv64(x, w, b, s, group, act):
    """act(conv2d(x, w) + b) with "same" pads, in 64 bits (im2col and matrix products)."""
    n, c, h, wd = x.shape
    m, cg, k, _ = w.shape
    pad = k // 2
    oh, ow = (h + 2 * pad - k) // s + 1, (wd + 2 * pad - k) // s + 1
    y = torch.empty((n, m, oh, ow), dtype=torch.float64, device=x.device)
    for i in range(n):
        if cg == 1 and group == c == m:
            acc = torch.zeros((m, oh, ow), dtype=torch.float64, device=x.device)
            xp = F.pad(x[i], (pad, pad, pad, pad))
            for ky in range(k):
                for kx in range(k):
                    acc += w[:, 0, ky, kx, None, None] * xp[:, ky:ky + (oh - 1) * s + 1:s, kx:kx + (ow - 1) * s + 1:s]
            y[i] = acc
        else:
            cols = F.unfold(x[i:i + 1], k, padding=pad, stride=s)[0]
            y[i] = (w.reshape(m, -1) @ cols).reshape(m, oh, ow)
    y += b[None, :, None, None]
    if act == "Silu":
        return y * torch.sigmoid(y)
    return y.clamp_min(0.0) if act == "Relu" else y


def _frame64(case, x):
    """The network's op list (convs, adds, pools, upsampling, attention) in 64 bits."""
    model = yolo11n.build(case["size"])
    mem = {id(b): torch.zeros((b.c, b.h, b.w), dtype=torch.float64, device="cuda") for b in model.bufs}
    mem[id(model.input)][:] = x[0].double()
    view = lambda s: mem[id(s.buf)][s.c0:s.c0 + s.c]
    dev = lambda v: torch.from_numpy(np.asarray(v)).to("cuda").double()
    for op in model.ops:
        if isinstance(op, yolo11n.ConvOp):
            y = _conv64(view(op.x)[None], dev(op.w), dev(op.b), op.s, op.group, op.act)[0]
        elif isinstance(op, yolo11n.AddOp):
            y = view(op.a) + view(op.b)
        elif isinstance(op, yolo11n.MaxPoolOp):
            y = F.max_pool2d(view(op.x)[None], op.k, op.s, op.p)[0]
        elif isinstance(op, yolo11n.UpsampleOp):
            y = view(op.x).repeat_interleave(op.f, 1).repeat_interleave(op.f, 2)
        elif isinstance(op, yolo11n.AttentionOp):
            n, kd = op.qkv.h * op.qkv.w, op.key_dim
            heads = view(op.qkv).reshape(op.heads, 2 * kd + op.head_dim, n)
            parts = []
            for hd in heads:
                p = torch.softmax(op.scale * (hd[:kd].t() @ hd[kd:2 * kd]), -1)
                parts.append(hd[2 * kd:] @ p.t())
            y = torch.cat(parts).reshape(op.y.c, op.y.h, op.y.w)
        else:
            raise TypeError(op)
        view(op.y).copy_(y)
    return tuple(mem[id(b)][None] for b in model.outputs)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "matmul":
        return t["a"].double() @ t["b"].double() + t["bias"].double()
    if kind == "attention":
        q, kt, v = t["q"].double(), t["kt"].double(), t["v"].double()
        p = torch.stack([torch.softmax((q[i] @ kt[i]) * case["dim"] ** -0.5, -1) for i in range(case["heads"])])
        return p, torch.stack([p[i] @ v[i] for i in range(case["heads"])])
    if kind == "dqm":
        # The quantization is part of the operator's definition and is stated
        # in 32-bit arithmetic (scale, zero point, x * (1 / scale), ties to
        # even); the product and the dequantization are what 64 bits check.
        a, one = t["a"], torch.ones((), device="cuda")
        lo, hi = a.min().clamp_max(0.0), a.max().clamp_min(0.0)
        scale = (hi - lo) / (255.0 * one)
        zp = torch.round(-lo / scale).clamp(0, 255)
        q = (torch.round(a * (one / scale)) + zp).clamp(0, 255)
        wz = 0.0 if t["zp"] is None else float(t["zp"][0])
        acc = (q - zp).double() @ (t["w"].double() - wz)
        return acc * (scale.double() * t["ws"].double()) + t["bias"].double()
    if kind == "conv":
        y = _conv64(t["x"].double(), t["w"].double(), t["bias"].double(), case["s"], case["group"], case["act"])
        return y if t["res"] is None else y + t["res"].double()
    return _frame64(case, t["x"])
