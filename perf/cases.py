"""Workloads of the W8A8 convolution path, as a program that uses this package runs them.

Single layers and blocks go through the op-level entry points on NHWC fp16 device tensors (the
fp32 conv and the Detect-head postprocess on the layouts they take); the two whole networks go
through the session and the model object.  Sizes are those of the benchmark configurations
(``aexrt_amd.workloads``), of YOLOv8n at 160-640 pixels (``aexrt_amd.yolov8``), and ragged ones.

A case is a dict of plain values; ``kind`` names the path:

* ``int8``: the whole int8 conv command on a plain fp16 tensor (amax, then the conv), per tensor or
  with per-16-channel scales (``pg16``); below 4096 input elements it is the dynamic conv;
* ``int8_slots``: one int8 conv inside a network, the input's amax known from its producer;
* ``bottleneck``: a C2f bottleneck, two int8 3x3 convs with the amax handed on and a residual;
* ``fp16`` / ``winograd``: fp16 convs, direct and F(2x2,3x3);
* ``fp32``: the fp32 NCHW direct conv;
* ``detect``: sigmoid + DFL decode, NMS and top-k of one raw Detect head;
* ``net``: YOLOv8n W8A8 with its fp16 head, images to raw head output.
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
from pathlib import Path

import numpy as np
import torch

import aexrt_amd
from aexrt_amd import _lib
from aexrt_amd import engine as E
from aexrt_amd import kernels as K
from aexrt_amd.runtime import NativeHipYoloModel
from aexrt_amd.session import InferenceSession
from aexrt_amd.yolov8 import build_yolov8n

DEV = "cuda"
STRIPES = 16  # slot copies of a tensor, as the network runtime keeps them


def _conv(kind, n, c, h, w, oc, k, s=1, **more):
    return dict(kind=kind, n=n, c=c, h=h, w=w, oc=oc, k=k, s=s, **more)


def listed():
    return [
        # a 3x3 conv on the last map of a 160-pixel image: under 4096 elements, all latency
        dict(_conv("int8", 1, 128, 5, 5, 128, 3), name="int8_3x3_5px_bs1"),
        # the 1x1 benchmark configuration on one image: a service answering single requests
        dict(_conv("int8", 1, 128, 40, 40, 256, 1), name="int8_1x1_40px_bs1"),
        # the stride-2 benchmark configuration on a batch of 32: offline throughput
        dict(_conv("int8", 32, 64, 160, 160, 128, 3, 2), name="int8_3x3s2_160px_bs32"),
        # per-16-channel activation scales on a map that no tile divides, odd batch
        dict(_conv("int8", 5, 96, 27, 35, 48, 3, pg16=True), name="int8_pg16_3x3_27x35_bs5"),
        # the neck's 1x1 over a concat at the benchmark batch
        dict(_conv("int8_slots", 64, 384, 20, 20, 128, 1), name="int8_cat_1x1_20px_bs64"),
        # one bottleneck of the C2f benchmark block, a medium batch
        dict(kind="bottleneck", n=16, c=64, h=40, w=40, name="bottleneck_64_40px_bs16"),
        # a class-branch 3x3 of the fp16 detect head at the benchmark batch
        dict(_conv("fp16", 64, 80, 40, 40, 80, 3), name="fp16_head_3x3_40px_bs64"),
        # the reference's Winograd conv of an fp16 engine, a small batch
        dict(_conv("winograd", 8, 64, 40, 40, 64, 3), name="winograd_40px_bs8"),
        # the fp32 benchmark configuration
        dict(_conv("fp32", 1, 64, 80, 80, 64, 3, groups=1), name="fp32_3x3_80px_bs1"),
        # the postprocess of a 640-pixel image
        dict(kind="detect", size=640, classes=80, objects=48, name="detect_640px"),
        # one host image to the raw head output through the session, the committed kernel plan
        dict(kind="net", n=1, size=320, session=True, name="net_320px_bs1"),
        # a device-resident batch to the raw head output, the committed kernel plan
        dict(kind="net", n=64, size=320, session=False, name="net_320px_bs64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same paths: maps of 4-160 pixels a side (not always square), 16-512 channels,
    batches of 1-64, within the work of the largest listed cases."""
    kind = rng.choice(["int8", "int8", "int8", "int8_slots", "int8_slots", "bottleneck", "fp16", "fp16", "winograd",
                       "fp32", "detect", "net"])
    if kind == "detect":
        return dict(kind=kind, size=32 * rng.randint(5, 20), classes=rng.choice([1, 20, 80, rng.randint(2, 91)]),
                    objects=_log(rng, 2, 80))
    if kind == "net":
        return dict(kind=kind, n=_log(rng, 1, 16), size=32 * rng.randint(2, 10), session=rng.random() < 0.5)
    # flops and bytes a drawn case may ask of its path
    flops, elements = {"fp32": (2e9, 2e7), "winograd": (8e9, 4e7)}.get(kind, (30e9, 8e7))
    while True:
        h = _log(rng, 4, 160)
        w = h if rng.random() < 0.5 else max(4, min(160, int(h * rng.uniform(0.6, 1.7))))
        n = _log(rng, 1, 64)
        if kind == "bottleneck":
            case = dict(kind=kind, n=n, c=32 * rng.randint(1, 4), h=h, w=w)
        elif kind == "fp32":
            g = rng.choice([1, 1, 1, 2])
            case = _conv(kind, n, g * _log(rng, 1, 96), h, w, g * _log(rng, 2, 96), rng.choice([1, 3, 3]),
                         rng.choice([1, 1, 2]), groups=g)
        else:
            step = 8 if kind == "fp16" else 16
            c, oc = (step * _log(rng, 1, 512 // step) for _ in range(2))
            k = 3 if kind == "winograd" else rng.choice([1, 3])
            s = rng.choice([1, 1, 2]) if k == 3 and kind != "winograd" else 1
            case = _conv(kind, n, c, h, w, oc, k, s)
            if kind == "winograd":
                case["h"], case["w"] = h + h % 2, w + w % 2
            if kind == "int8" and rng.random() < 0.25:
                case["pg16"] = True
        if kind == "bottleneck" and n * h * w * case["c"] < 4096:
            continue
        done = work(case)
        limit = flops / 8 if case.get("pg16") else flops
        if done["flops"] <= limit and done["bytes"] <= 4 * elements:
            return case


def _out_hw(case):
    p, k, s = case["k"] // 2, case["k"], case["s"]
    return (case["h"] + 2 * p - k) // s + 1, (case["w"] + 2 * p - k) // s + 1


def _params(n, c, h, w, oc, oh, ow, k, s, groups=1):
    p = k // 2
    return [n, c, h, w, oc, oh, ow, k, k, s, s, p, p, 1, 1, groups]


def _anchors(size):
    return sum((size // st) ** 2 for st in (8, 16, 32))


# multiply-adds per image of YOLOv8n grow with its area: 1.093 G at 320 pixels
NET_MACS_320 = 1.093e9
NET_WEIGHT_BYTES = 3.5e6


def work(case):
    kind = case["kind"]
    if kind == "detect":
        a = _anchors(case["size"])
        return {"bytes": 4.0 * a * (64 + case["classes"]), "flops": 0.0}
    if kind == "net":
        area = (case["size"] / 320.0) ** 2
        return {"bytes": 4.0 * case["n"] * (3 * case["size"] ** 2 + 144 * _anchors(case["size"])) + NET_WEIGHT_BYTES,
                "flops": 2.0 * NET_MACS_320 * area * case["n"]}
    if kind == "bottleneck":
        m, c = case["n"] * case["h"] * case["w"], case["c"]
        return {"bytes": 2.0 * m * c * 3 + 2 * 9.0 * c * c, "flops": 2.0 * 2 * m * c * c * 9}
    oh, ow = _out_hw(case)
    g = case.get("groups", 1)
    kk = case["k"] ** 2
    esz, wsz = (4, 4) if kind == "fp32" else (2, 1 if kind.startswith("int8") else 2)
    x = case["n"] * case["c"] * case["h"] * case["w"]
    y = case["n"] * case["oc"] * oh * ow
    return {"bytes": float(esz * (x + y) + wsz * kk * case["c"] * case["oc"] // g),
            "flops": 2.0 * y * kk * case["c"] / g}


def tolerance(case):
    return {"detect": {"rel": 1e-6},
            "fp32": {"rel": 2e-6},
            "winograd": {"rel": 2e-3},
            "net": {"rel": 4e-2}}.get(case["kind"], {"rel": 1e-3})


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _uniform(g, lo, hi, *shape):
    return torch.rand(*shape, generator=g, device=DEV) * (hi - lo) + lo


def _activation(g, n, h, w, c):
    """fp16 NHWC, what a SiLU layer hands on; channels of different strength."""
    x = _randn(g, n, h, w, c) * _uniform(g, 0.5, 2.0, c)
    return torch.nn.functional.silu(x).half()


def _weight(g, oc, ic, k):
    return _randn(g, oc, ic, k, k) * math.sqrt(2.0 / (ic * k * k))


def _int8_weight(g, oc, ic, k):
    w = _weight(g, oc, ic, k).reshape(oc, -1)
    scale = w.abs().amax(1) / 127.0
    return torch.round(w / scale[:, None]).to(torch.int8).reshape(oc, ic, k, k), scale


def _int8_conv(params, q, scale, bias):
    payload = q.cpu().numpy().tobytes() + scale.cpu().numpy().astype(np.float32).tobytes()
    algorithm = 51 if params[7] == 1 else 51 + params[9]
    return K.prepare_conv(params, algorithm, K.SRC_LAYOUT_INT8, payload, bias.cpu().numpy(), device=DEV)


def _conv_inputs(case, seed):
    """(x, weight, weight scale or None, bias) of one conv, everything from the seed."""
    g = _gen(seed)
    n, c, h, w, oc, k = (case[v] for v in ("n", "c", "h", "w", "oc", "k"))
    bias = _uniform(g, -0.1, 0.1, oc)
    if case["kind"] == "fp32":
        return _randn(g, n, c, h, w), _weight(g, oc, c // case["groups"], k), None, bias
    x = _activation(g, n, h, w, c)
    if case["kind"].startswith("int8"):
        return x, *_int8_weight(g, oc, c, k), bias
    return x, _weight(g, oc, c, k).half(), None, bias


def _bottleneck_inputs(case, seed):
    g = _gen(seed)
    n, c, h, w = (case[v] for v in ("n", "c", "h", "w"))
    x = _activation(g, n, h, w, c)
    return x, [(*_int8_weight(g, c, c, 3), _uniform(g, -0.1, 0.1, c)) for _ in range(2)]


def _producer_slots(x):
    """x's amax slots as its producer leaves them: the groups' maxima spread over the copies."""
    groups = x.shape[3] // 16
    m = x.float().abs().reshape(-1, groups, 16).amax(2)
    slots = K.new_slots(x.shape[3], DEV, STRIPES)
    rows = torch.arange(m.shape[0], device=DEV) % STRIPES
    slots.view(torch.float32).scatter_reduce_(0, rows[:, None].expand(-1, groups), m, "amax")
    return slots


def _detect_inputs(case, seed):
    """A raw Detect head [64 + classes][anchors]: background logits far below the threshold, and
    objects that lift the anchors around their centre on the level of their size."""
    rng = np.random.default_rng(seed)
    size, classes = case["size"], case["classes"]
    levels = [(size // st, size // st, float(st)) for st in (8, 16, 32)]
    logits = rng.normal(-7.0, 1.0, (classes, _anchors(size))).astype(np.float32)
    bins = rng.normal(0.0, 1.0, (4, 16, _anchors(size))).astype(np.float32)
    offs = np.cumsum([0] + [h * w for h, w, _ in levels])
    for _ in range(case["objects"]):
        lv = int(rng.integers(0, 3))
        n = levels[lv][0]
        cy, cx, cls = int(rng.integers(0, n)), int(rng.integers(0, n)), int(rng.integers(0, classes))
        half = rng.uniform(2.0, 8.0, 2)
        for y in range(max(0, cy - 1), min(n, cy + 2)):
            for x in range(max(0, cx - 1), min(n, cx + 2)):
                a = offs[lv] + y * n + x
                logits[cls, a] = rng.normal(2.0 - abs(y - cy) - abs(x - cx), 0.7)
                side = (half[0] + x - cx, half[1] + y - cy, half[0] - x + cx, half[1] - y + cy)
                for d in range(4):
                    bins[d, :, a] -= 2.0 * np.abs(np.arange(16) - np.clip(side[d], 0.0, 15.0))
    head = np.concatenate([bins.reshape(64, -1), logits])
    return torch.from_numpy(np.ascontiguousarray(head)).to(DEV), levels


@functools.lru_cache(maxsize=2)
def _net(n, size):
    """The seeded YOLOv8n graph and its W8A8 engine, compiled once by the program."""
    graph = build_yolov8n(batch=n, imgsz=size, seed=4)
    algo = E.w8a8_algo_map(E.lower_graph(graph), graph.metadata["int8_convs"].split(","))
    return graph, algo, E.build_aexrt_engine(graph, precision="fp16", algo_overrides=algo, classes=80)


def _use_committed_plan():
    """Kernel choices from the committed plan, the automatic ones where it has none; nothing is
    measured at load."""
    os.environ["AEXRT_HIP_AUTOTUNE"] = "0"
    os.environ["AEXRT_HIP_TUNE_CACHE"] = str(Path(aexrt_amd.__file__).resolve().parent / "tuned" / "yolov8n320.tune")


# ---- one pass -------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "net":
        _use_committed_plan()
        graph, algo, data = _net(case["n"], case["size"])
        images = torch.rand(case["n"], 3, case["size"], case["size"], generator=_gen(seed), device=DEV)
        if case["session"]:
            return dict(kind="session", session=InferenceSession(graph, backend="hip", algo_map=algo),
                        images=images.cpu().numpy())
        torch.cuda.synchronize()
        return dict(kind=kind, model=NativeHipYoloModel(data), images=images)
    if kind == "detect":
        head, levels = _detect_inputs(case, seed)
        return dict(kind=kind, head=head, levels=levels, classes=case["classes"])
    if kind == "bottleneck":
        x, convs = _bottleneck_inputs(case, seed)
        n, c, h, w = (case[v] for v in ("n", "c", "h", "w"))
        params = _params(n, c, h, w, c, h, w, 3, 1)
        return dict(kind=kind, x=x, x_slots=_producer_slots(x), t=torch.empty_like(x), y=torch.empty_like(x),
                    t_slots=K.new_slots(c, DEV, STRIPES), convs=[_int8_conv(params, *v) for v in convs])
    x, w, scale, bias = _conv_inputs(case, seed)
    oh, ow = _out_hw(case)
    params = _params(case["n"], case["c"], case["h"], case["w"], case["oc"], oh, ow, case["k"], case["s"],
                     case.get("groups", 1))
    if kind == "fp32":
        return dict(kind=kind, desc=_lib.ConvDesc.from_params(params), x=x, w=w.contiguous(), bias=bias,
                    y=torch.empty(case["n"], case["oc"], oh, ow, device=DEV))
    y = torch.empty(case["n"], oh, ow, case["oc"], dtype=torch.float16, device=DEV)
    state = dict(kind=kind, x=x, y=y, flags=K.SILU | (K.INT8_PG16 if case.get("pg16") else 0))
    if kind.startswith("int8"):
        state["conv"] = _int8_conv(params, w, scale, bias)
        if kind == "int8_slots":
            state["x_slots"] = _producer_slots(x)
    elif kind == "winograd":
        state["conv"] = K.prepare_conv(params, 40, K.SRC_LAYOUT_WINO_F16, _winograd_weight(w), bias.cpu().numpy(),
                                       device=DEV)
    else:
        state["conv"] = K.prepare_conv(params, 5, K.SRC_RAW_F16, w.cpu().numpy(), bias.cpu().numpy(), device=DEV)
    return state


def _winograd_weight(w):
    """U = G g G^T of the fp16 filters, [oc][ic][4][4] fp16 (the engine's packed layout)."""
    g = torch.tensor([[1, 0, 0], [0.5, 0.5, 0.5], [0.5, -0.5, 0.5], [0, 0, 1]], dtype=torch.float64, device=DEV)
    return (g @ w.double() @ g.T).half().cpu().numpy()


def run(state):
    kind = state["kind"]
    if kind == "int8":
        K.conv2d_int8(state["conv"], state["x"], state["y"], flags=state["flags"])
        return state["y"]
    if kind == "int8_slots":
        K.conv2d(state["conv"], state["x"], state["y"], flags=state["flags"], x_slots=state["x_slots"])
        return state["y"]
    if kind in ("fp16", "winograd"):
        K.conv2d(state["conv"], state["x"], state["y"], flags=state["flags"])
        return state["y"]
    if kind == "bottleneck":
        a, b = state["convs"]
        x, t, y, t_slots = state["x"], state["t"], state["y"], state["t_slots"]
        K.fill_u32(t_slots)
        K.conv2d(a, x, t, x_slots=state["x_slots"], y_slots=t_slots)
        K.conv2d(b, t, y, flags=K.SILU | K.RESIDUAL, x_slots=t_slots, residual=x)
        return t, y
    if kind == "fp32":
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        _lib.check(_lib.lib().aexrt_hip_conv2d_f32(
            ctypes.byref(state["desc"]), K.SILU, state["x"].data_ptr(), state["w"].data_ptr(),
            state["bias"].data_ptr(), state["y"].data_ptr(), stream), "conv2d_f32")
        return state["y"]
    if kind == "detect":
        return K.yolo_dfl_decode_nms_topk(state["head"], state["levels"], classes=state["classes"])
    if kind == "session":
        return state["session"].run({"images": state["images"]})["output0"]
    state["model"].run_device(state["images"].data_ptr())
    return state["model"].output()


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------

def _conv64(x, w, s):
    """NHWC conv in 64 bits: x [N, H, W, C], w [OC, C, K, K], padding K // 2."""
    k = w.shape[2]
    p = k // 2
    x = torch.nn.functional.pad(x, (0, 0, p, p, p, p))
    oh, ow = (x.shape[1] - k) // s + 1, (x.shape[2] - k) // s + 1
    y = 0
    for i in range(k):
        for j in range(k):
            v = x[:, i:i + s * (oh - 1) + 1:s, j:j + s * (ow - 1) + 1:s]
            y = y + v @ w[:, :, i, j].T
    return y


def _silu64(v):
    return v / (1.0 + torch.exp(-v))


def _quantized64(x, amax):
    """The path's integers for x and what one step of them is worth: the scale 127 / amax and the
    product with it are fp32 by definition."""
    amax = amax.float()
    step = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    q = torch.round(x.float() * step).double()
    # a byte: at more than one image a strip's amax is not the amax of its channel group, and larger
    # values wrap
    return torch.remainder(q + 128.0, 256.0) - 128.0, amax.double() / 127.0


def _int8_conv64(x, q, scale, bias, s, pg16=False):
    c = x.shape[3]
    if pg16:
        # strips of 16 * N * H * W elements of the NCHW tensor, scale s for channel group s
        strips = x.permute(0, 3, 1, 2).reshape(c // 16, -1).float().abs().amax(1)
        xi, step = _quantized64(x, strips.repeat_interleave(16))
        return _silu64(_conv64(xi * step, q.double(), s) * scale.double() + bias.double())
    xi, step = _quantized64(x, x.float().abs().amax())
    return _silu64(_conv64(xi, q.double(), s) * step * scale.double() + bias.double())


def _dynamic_conv64(x, q, scale, bias, s):
    """A scale per output position and 4 input channels over the taps."""
    n, h, w, c = x.shape
    oc, _, k, _ = q.shape
    p = k // 2
    xp = torch.nn.functional.pad(x.float(), (0, 0, p, p, p, p))
    oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    taps = torch.stack([xp[:, i:i + s * (oh - 1) + 1:s, j:j + s * (ow - 1) + 1:s] for i in range(k)
                        for j in range(k)], 3).reshape(n, oh, ow, k * k, c // 4, 4)
    xi, step = _quantized64(taps, taps.abs().amax((3, 5), keepdim=True))
    wt = q.double().reshape(oc, c // 4, 4, k * k).permute(3, 1, 2, 0).reshape(-1, oc)
    return _silu64((xi * step).reshape(n, oh, ow, -1) @ wt * scale.double() + bias.double())


def _detect64(case, seed):
    head, levels = _detect_inputs(case, seed)
    head = head.cpu().numpy().astype(np.float64)
    scores = 1.0 / (1.0 + np.exp(-head[64:]))
    cls, best = scores.argmax(0), scores.max(0)
    keep = np.flatnonzero(~(best < 0.25))[:512]
    bins = head[:64].reshape(4, 16, -1)[:, :, keep]
    e = np.exp(bins - bins.max(1, keepdims=True))
    dist = (e * np.arange(16)[None, :, None]).sum(1) / e.sum(1)
    grid = np.concatenate([np.stack([np.tile(np.arange(w), h) + 0.5, np.repeat(np.arange(h), w) + 0.5,
                                     np.full(h * w, st)]) for h, w, st in levels], 1)[:, keep]
    x, y, st = grid
    box = np.stack([(x - dist[0]) * st, (y - dist[1]) * st, (x + dist[2]) * st, (y + dist[3]) * st], 1)
    cls, best = cls[keep], best[keep]
    lo = np.maximum(box[:, None, :2], box[None, :, :2])
    hi = np.minimum(box[:, None, 2:], box[None, :, 2:])
    inter = np.maximum(hi - lo, 0.0).prod(2)
    area = np.maximum(box[:, 2:] - box[:, :2], 0.0).prod(1)
    iou = inter / np.maximum(area[:, None] + area[None] - inter, 1e-7)
    drop = ((best[None] > best[:, None]) & (cls[None] == cls[:, None]) & (iou > 0.45)).any(1)
    order = [i for i in np.argsort(-best, kind="stable") if not drop[i]][:100]
    return torch.from_numpy(np.concatenate([box, best[:, None], cls[:, None]], 1)[order])


def exact(case, seed):
    kind = case["kind"]
    if kind == "net":
        # every layer quantizes with the amax of what the one before it rounded to fp16: the
        # integers, and so the outputs, have no 64-bit value of their own
        return None
    if kind == "detect":
        return _detect64(case, seed)
    if kind == "bottleneck":
        x, ((qa, sa, ba), (qb, sb, bb)) = _bottleneck_inputs(case, seed)
        t = _int8_conv64(x, qa, sa, ba, 1)
        # the second conv quantizes the fp16 tensor that the first one stores
        return t, _int8_conv64(t.half(), qb, sb, bb, 1) + x.double()
    x, w, scale, bias = _conv_inputs(case, seed)
    if kind == "fp32":
        y = torch.nn.functional.conv2d(x.double().cpu(), w.double().cpu(), bias.double().cpu(), stride=case["s"],
                                       padding=case["k"] // 2, groups=case["groups"])
        return _silu64(y)
    if kind.startswith("int8"):
        if kind == "int8" and x.numel() < 4096:
            return _dynamic_conv64(x, w, scale, bias, case["s"])
        return _int8_conv64(x, w, scale, bias, case["s"], bool(case.get("pg16")))
    return _silu64(_conv64(x.double(), w.double(), case["s"]) + bias.double())
