"""The work that is timed when the kernels or the host path change: the calls a program makes
through infvino_amd's public entry points, from one image to full batches.

Shapes are those of the plans infvino_amd.planwriter writes (YOLOv8n-pose, YOLO11n-pose and
MobileNetV3-small), of the benchmark's conv sweep and of the tests; draw() gives further sizes
of the same ranges.  Activations are SiLU outputs of normal values (what a layer inside these
models reads), weights He-normal, both fp16.  Channels-last tensors hold pixels of
round8(C) channels, as include/ivh.h states.
"""
import math
import os
import tempfile

import numpy as np
import torch
import torch.nn.functional as F

import infvino_amd as ia
from infvino_amd import ops
from infvino_amd import planwriter as pw

ACTS = {"none": ops.ACT_NONE, "silu": ops.ACT_SILU, "relu": ops.ACT_RELU, "hswish": ops.ACT_HSWISH}


def conv(name=None, *, cin, cout, h, w, k, s, batch, act="silu", res=False, nhwc=True, dw=False):
    c = {"kind": "conv", "cin": cin, "cout": cout, "h": h, "w": w, "k": k, "s": s, "batch": batch, "act": act,
         "res": res, "nhwc": nhwc, "dw": dw}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one camera frame, host floats in and out: the reference's ClBackend::infer call, where
        # latency counts
        {"name": "pose_infer_b1", "kind": "pose", "imgsz": 640, "batch": 1, "call": "infer"},
        # the throughput benchmark's step: 64 frames already on the card, the heads read back
        {"name": "pose_run_b64", "kind": "pose", "imgsz": 640, "batch": 64, "call": "run"},
        # the plan's conv1x1 op on graph tensors (NCHW planes), one image: the smallest call
        conv("pointwise_planes_b1", cin=64, cout=128, h=80, w=80, k=1, s=1, batch=1, nhwc=False),
        # C2f bottleneck conv with its residual at the finest head level, full batch
        conv("conv3_64_80_b64", cin=64, cout=64, h=80, w=80, k=3, s=1, batch=64, res=True),
        # downsample between the 80x80 and 40x40 levels, full batch
        conv("down_64_128_80_b64", cin=64, cout=128, h=80, w=80, k=3, s=2, batch=64),
        # neck pointwise conv over a concat, full batch
        conv("pointwise_384_128_40_b64", cin=384, cout=128, h=40, w=40, k=1, s=1, batch=64),
        # the deepest 3x3 conv of the backbone for one image: few pixels, a long sum
        conv("conv3_256_20_b1", cin=256, cout=256, h=20, w=20, k=3, s=1, batch=1),
        # keypoint branch (51 channels) of a 624-pixel frame's middle level, a small batch
        conv("conv3_128_51_39_b6", cin=128, cout=51, h=39, w=39, k=3, s=1, batch=6),
        # MobileNetV3-small's strided 5x5 depthwise, classification batch
        conv("dw5_72_28_b256", cin=72, cout=72, h=28, w=28, k=5, s=2, batch=256, act="hswish", dw=True),
        # C2PSA attention core: 4 heads of 64 channels over 20x20 tokens, full batch
        {"name": "attention_400_b64", "kind": "attention", "heads": 4, "tokens": 400, "dim": 64, "batch": 64},
        # MobileNetV3-small's classifier for one image
        {"name": "classifier_b1", "kind": "classifier", "n_in": 576, "hidden": 1024, "classes": 1000, "batch": 1},
        # SPPF's three chained max pools, full batch
        {"name": "sppf_128_20_b64", "kind": "sppf", "c": 128, "h": 20, "w": 20, "batch": 64},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """Mostly whole groups of 8 or 16 channels, as the models have; now and then an odd count."""
    c = _log(rng, lo, hi)
    return c if rng.random() < 0.2 else max(8, c // (16 if c >= 64 else 8) * (16 if c >= 64 else 8))


def draw(rng):
    kind = rng.choice(("pointwise", "planes", "conv3", "conv3", "down", "stem", "dw", "attention", "classifier",
                       "sppf", "pose"))
    while True:
        batch, h = _log(rng, 1, 64), _log(rng, 7, 160)
        w = h if rng.random() < 0.7 else _log(rng, 7, 160)
        if kind == "pose":
            size = 32 * rng.randint(5, 20)
            call = rng.choice(("infer", "run"))
            batch = _log(rng, 1, 8 if call == "infer" else 48)
            return {"kind": "pose", "imgsz": size, "batch": batch, "call": call}
        if kind == "attention":
            side = rng.randint(7, 24)
            c = {"kind": kind, "heads": rng.choice((2, 4, 8)), "tokens": side * rng.randint(7, 24), "dim": 64,
                 "batch": batch}
        elif kind == "classifier":
            c = {"kind": kind, "n_in": 8 * _log(rng, 12, 160), "hidden": 8 * _log(rng, 16, 160),
                 "classes": _log(rng, 10, 1200), "batch": batch}
        elif kind == "sppf":
            c = {"kind": kind, "c": _channels(rng, 32, 256), "h": min(h, 40), "w": min(w, 40), "batch": batch}
        elif kind == "stem":
            c = conv(cin=3, cout=16, h=4 * h, w=4 * w, k=3, s=2, batch=batch,
                     act=rng.choice(("silu", "hswish")), nhwc=False)
        elif kind == "dw":
            ch = _channels(rng, 16, 576)
            c = conv(cin=ch, cout=ch, h=h, w=w, k=rng.choice((3, 5)), s=rng.choice((1, 2)), batch=_log(rng, 1, 256),
                     act=rng.choice(("silu", "relu", "hswish")), dw=True)
        else:
            # a level's channels grow as its map shrinks, as they do in the models
            most = 512 if h * w <= 1600 else (256 if h * w <= 6400 else 96)
            cin, cout = _channels(rng, 16, most), _channels(rng, 16, most)
            if kind == "planes":  # whole 16-byte pieces of a plane, as the plan's graph tensors have
                h, w = h // 4 * 4 or 4, w // 4 * 4 or 4
            k, s = (1, 1) if kind in ("pointwise", "planes") else (3, 2 if kind == "down" else 1)
            res = kind == "conv3" and rng.random() < 0.3
            c = conv(cin=cin, cout=cin if res else cout, h=h, w=w, k=k, s=s, batch=batch, res=res,
                     nhwc=kind != "planes", act="silu" if rng.random() < 0.8 else rng.choice(("none", "hswish")))
        need = work(c)
        if need["bytes"] < 5e8 and need["flops"] < 1.5e11:
            return c


def _round8(c):
    return (c + 7) // 8 * 8


def _out(c, n):
    pad = c["k"] // 2
    return (n + 2 * pad - c["k"]) // c["s"] + 1


# ---------------------------------------------------------------- inputs, the same for both sides

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(g, *shape):
    return F.silu(torch.randn(*shape, device="cuda", generator=g)).half()


def _weights(seed, *shape):
    """He-normal fp16 weights [out][in...] and a small bias, on the host as a plan's files hold them."""
    r = np.random.default_rng(seed)
    fan = int(np.prod(shape[1:]))
    w = (r.standard_normal(shape, dtype=np.float32) * np.float32(math.sqrt(2.0 / fan))).astype(np.float16)
    b = (r.standard_normal(shape[0], dtype=np.float32) * np.float32(0.1)).astype(np.float16)
    return w, b


def _conv_inputs(c, seed):
    g = _gen(seed)
    ho, wo = _out(c, c["h"]), _out(c, c["w"])
    x = _activations(g, c["batch"], c["cin"], c["h"], c["w"])
    r = _activations(g, c["batch"], c["cout"], ho, wo) if c["res"] else None
    w, b = _weights(seed, c["cout"], 1 if c["dw"] else c["cin"], c["k"], c["k"])
    return x, r, w, b


def _attention_inputs(c, seed):
    """q^T scaled by 1/sqrt(dim) [heads][tokens][dim], k [heads][dim][tokens], v^T [heads][tokens][dim]."""
    g = _gen(seed)
    shape = (c["batch"], c["heads"])
    q = torch.randn(*shape, c["tokens"], c["dim"], device="cuda", generator=g) / math.sqrt(c["dim"])
    k = torch.randn(*shape, c["dim"], c["tokens"], device="cuda", generator=g)
    v = torch.randn(*shape, c["tokens"], c["dim"], device="cuda", generator=g)
    return q.half(), k.half(), v.half()


def _frames(c, seed):
    n = c["batch"] * 3 * c["imgsz"] ** 2
    return np.random.default_rng(seed).random(n, dtype=np.float32).astype(np.float16)


def _layout(t, nhwc):
    """NCHW values as the entry points take them: planes, or pixels of round8(C) channels."""
    if not nhwc:
        return t.contiguous()
    b, c, h, w = t.shape
    y = torch.zeros(b, h, w, _round8(c), dtype=t.dtype, device=t.device)
    y[..., :c] = t.permute(0, 2, 3, 1)
    return y


def _packed(d, w, b):
    buf = torch.empty(ops.conv_packed_bytes(d), dtype=torch.uint8, device="cuda")
    ops.pack_conv_weights(d, w.view(np.uint16), b.view(np.uint16), buf.data_ptr())
    return buf


def prepare(case, seed):
    c = case
    if c["kind"] == "pose":
        with tempfile.TemporaryDirectory() as d:
            path, _ = pw.yolov8n_pose(d, seed=seed, imgsz=c["imgsz"])
            x = _frames(c, seed)
            if c["call"] == "infer":
                return {"case": c, "backend": ia.HipBackend(path, 0, c["batch"]), "x": x.astype(np.float32)}
            m = ia.PlanModel(path, 0, c["batch"])
        m.setInput(x, c["batch"])
        return {"case": c, "model": m}
    if c["kind"] == "conv":
        x, r, w, b = _conv_inputs(c, seed)
        d = ops.conv_desc(c["cin"], c["cout"], c["h"], c["w"], c["k"], c["s"], c["k"] // 2,
                          c["cin"] if c["dw"] else 1, ACTS[c["act"]], True, c["nhwc"])
        ho, wo, bt, co = _out(c, c["h"]), _out(c, c["w"]), c["batch"], c["cout"]
        y = torch.zeros((bt, ho, wo, _round8(co)) if c["nhwc"] else (bt, co, ho, wo), dtype=torch.float16,
                        device="cuda")
        return {"case": c, "desc": d, "x": _layout(x, c["nhwc"]), "res": None if r is None else _layout(r, c["nhwc"]),
                "packed": _packed(d, w, b), "y": y, "out": y[..., :co] if c["nhwc"] else y}
    if c["kind"] == "attention":
        q, k, v = _attention_inputs(c, seed)
        s = torch.empty(c["batch"], c["heads"], c["tokens"], c["tokens"], dtype=torch.float16, device="cuda")
        return {"case": c, "q": q, "k": k, "v": v, "s": s, "p": torch.empty_like(s), "y": torch.empty_like(v)}
    if c["kind"] == "classifier":
        x = _activations(_gen(seed), c["batch"], c["n_in"])
        d1 = ops.conv_desc(c["n_in"], c["hidden"], 1, 1, act=ops.ACT_HSWISH, channels_last=False)
        d2 = ops.conv_desc(c["hidden"], c["classes"], 1, 1, act=ops.ACT_NONE, channels_last=False)
        return {"case": c, "x": x, "d1": d1, "d2": d2,
                "w1": _packed(d1, *_weights(seed, c["hidden"], c["n_in"], 1, 1)),
                "w2": _packed(d2, *_weights(seed + 1, c["classes"], c["hidden"], 1, 1)),
                "h": torch.empty(c["batch"], c["hidden"], dtype=torch.float16, device="cuda"),
                "y": torch.empty(c["batch"], c["classes"], dtype=torch.float16, device="cuda")}
    x = _activations(_gen(seed), c["batch"], c["c"], c["h"], c["w"])
    return {"case": c, "x": x, "y": [torch.empty_like(x) for _ in range(3)]}


def run(state):
    c = state["case"]
    if c["kind"] == "pose":
        if c["call"] == "infer":
            return [t.data for t in state["backend"].infer(state["x"])]
        m = state["model"]
        m.run(c["batch"])
        return [m.readOutput(0, c["batch"]).view(np.float16)]
    if c["kind"] == "conv":
        r = state["res"]
        (ops.dwconv if c["dw"] else ops.conv2d)(state["desc"], state["x"].data_ptr(), state["packed"].data_ptr(),
                                                None if r is None else r.data_ptr(), state["y"].data_ptr(), c["batch"])
        return state["out"]
    if c["kind"] == "attention":
        n, t, d, b = c["heads"], c["tokens"], c["dim"], c["batch"]
        s, p, y = state["s"], state["p"], state["y"]
        ops.bmm(state["q"].data_ptr(), state["k"].data_ptr(), s.data_ptr(), n, t, d, t, b)
        ops.softmax(s.data_ptr(), p.data_ptr(), n * t, t, 1, b)
        ops.bmm(p.data_ptr(), state["v"].data_ptr(), y.data_ptr(), n, t, t, d, b)
        return y
    if c["kind"] == "classifier":
        ops.gemv(state["d1"], state["x"].data_ptr(), state["w1"].data_ptr(), state["h"].data_ptr(), c["batch"])
        ops.gemv(state["d2"], state["h"].data_ptr(), state["w2"].data_ptr(), state["y"].data_ptr(), c["batch"])
        return state["y"]
    x = state["x"]
    for y in state["y"]:
        ops.pool(ops.POOL_MAX, x.data_ptr(), y.data_ptr(), c["c"], c["h"], c["w"], 5, 1, 2, c["batch"])
        x = y
    return state["y"]


def work(case):
    c, b = case, case["batch"]
    if c["kind"] == "pose":
        area = (c["imgsz"] / 640.0) ** 2
        # 9.178 GFLOP of convs an image; the frame in, the 56-row head out (fp16), the 3.3 M weights
        # read once, and each layer's output written and read once (about 20 MB an image)
        f = 4 if c["call"] == "infer" else 2
        return {"bytes": b * area * (3 * 640 * 640 * f + 56 * 8400 * f + 40e6) + 6.6e6, "flops": b * area * 9.178e9}
    if c["kind"] == "conv":
        px, po = c["h"] * c["w"], _out(c, c["h"]) * _out(c, c["w"])
        macs = c["cout"] * (1 if c["dw"] else c["cin"]) * c["k"] ** 2
        return {"bytes": 2 * (b * (c["cin"] * px + c["cout"] * po * (2 if c["res"] else 1)) + macs + c["cout"]),
                "flops": 2 * b * po * macs}
    if c["kind"] == "attention":
        n, t, d = c["heads"], c["tokens"], c["dim"]
        # q, k and v in, the result out, and the scores and probabilities the three calls return
        return {"bytes": 2 * b * n * (4 * t * d + 4 * t * t), "flops": 4 * b * n * t * t * d}
    if c["kind"] == "classifier":
        n = c["n_in"] * c["hidden"] + c["hidden"] * c["classes"]
        return {"bytes": 2 * (n + b * (c["n_in"] + 2 * c["hidden"] + c["classes"])), "flops": 2 * b * n}
    n = b * c["c"] * c["h"] * c["w"]
    return {"bytes": 2 * n * 6, "flops": 3 * 24 * n}


def tolerance(case):
    # fp16 results of fp32 sums: one rounding of the result (2e-4 in norm, 1 ulp = 1e-3 of a
    # value), two with a residual.  The attention core rounds its scores and probabilities too,
    # and a model every layer's output.
    k = case["kind"]
    if k == "sppf":
        return "exact"
    if k == "pose":
        return {"rel": 1e-3, "max": 5e-2}
    if k == "attention":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-3, "max": 5e-3}


# ---------------------------------------------------------------- the same in 64 bits

def _act64(x, code):
    if code == ops.ACT_SILU:
        return x * torch.sigmoid(x)
    if code == ops.ACT_RELU:
        return x.clamp(min=0)
    if code == ops.ACT_HSWISH:
        return x * ((x + 3).clamp(0, 6) / 6)
    if code == ops.ACT_HSIGMOID:
        return (x + 3).clamp(0, 6) / 6
    return torch.sigmoid(x) if code == ops.ACT_SIGMOID else x


def _conv64(x, w, b, s, p, dw):
    """x [B][Cin][H][W], w [Cout][Cin or 1][K][K], fp64: image by image, as one product of the
    unfolded pixels (or one shifted product a tap)."""
    k = w.shape[2]
    ho, wo = (x.shape[2] + 2 * p - k) // s + 1, (x.shape[3] + 2 * p - k) // s + 1
    out = []
    for img in x:
        if dw:
            z, y = F.pad(img, (p, p, p, p)), 0
            for i in range(k):
                for j in range(k):
                    y = y + z[:, i:i + (ho - 1) * s + 1:s, j:j + (wo - 1) * s + 1:s] * w[:, 0, i, j, None, None]
        else:
            cols = img.reshape(img.shape[0], -1) if k == 1 and s == 1 else F.unfold(img[None], k, 1, p, s)[0]
            y = (w.reshape(w.shape[0], -1) @ cols).reshape(-1, ho, wo)
        out.append(y if b is None else y + b[:, None, None])
    return torch.stack(out)


def _pose64(path, x, batch):
    """The written plan's nodes, one by one, on fp64 tensors."""
    T, dims, inits, out = {}, {}, set(), []

    def d64(a):
        return torch.from_numpy(np.asarray(a, np.float64)).cuda()

    with open(path) as f:
        lines = [ln.split() for ln in f if ln.strip() and not ln.startswith("#")]
    for tok in lines:
        if tok[0] in ("input", "tensor"):
            dims[tok[1]] = [int(v) for v in tok[2:]]
            if tok[0] == "input":
                T[tok[1]] = d64(x).reshape([batch] + dims[tok[1]][1:])
        elif tok[0] == "init":
            inits.add(tok[1])
            dims[tok[1]] = [int(v) for v in tok[3:]]
            T[tok[1]] = d64(np.fromfile(os.path.join(os.path.dirname(path), tok[2]), np.float16)).reshape(dims[tok[1]])
        elif tok[0] == "output":
            out.append(T[tok[1]])
        if tok[0] != "node":
            continue
        op, ins, o = tok[1], tok[2].split(","), tok[3]
        at = dict(kv.split("=", 1) for kv in tok[4:] if "=" in kv)
        n = {k: int(v) for k, v in at.items() if "," not in v}
        v = [None if i == "-" else T[i] for i in ins]
        if op in ("conv3x3", "conv1x1"):
            a, w = (v[0], v[1]) if op == "conv3x3" else (v[1], v[0])
            a = a.reshape(batch, w.shape[1], *([-1, 1] if a.dim() < 4 else a.shape[2:]))
            y = _act64(_conv64(a, w.reshape(*w.shape[:2], *([3, 3] if op == "conv3x3" else [1, 1])), v[2],
                               n.get("stride", 1), 1 if op == "conv3x3" else 0, False), n.get("act", 0))
            y = y if len(v) < 4 or v[3] is None else y + v[3].reshape(y.shape)
        elif op == "copy_c":
            y = v[0][:, n["c0"]:n["c0"] + n["cnt"]]
        elif op == "concat4":
            cs = [n["ca"], n["cb"], n["cc"], n["cd"]]
            y = torch.cat([a.reshape(batch * n["outer"], c, n["inner"]) for a, c in zip(v, cs) if c], 1)
        elif op == "ew_binary":
            a, b = v
            if n.get("b_scalar") == 1 or b.numel() == 1:
                b = b.reshape(())
            else:  # right-aligned shapes; an init holds one set of values for all images
                r = max(len(dims[ins[0]]), len(dims[ins[1]]))
                a, b = (t.reshape([1] * (r - t.dim()) + list(t.shape)) if i in inits else
                        t.reshape([batch] + [1] * (r - t.dim()) + list(t.shape[1:])) for i, t in zip(ins, (a, b)))
            y = (a + b, a - b, a * b, a / b)[n["op"]]
        elif op == "ew_unary":
            y = torch.sigmoid(v[0]) if n["op"] == 0 else v[0].clamp(min=0)
        elif op == "maxpool":
            y = F.max_pool2d(v[0].reshape(batch, n["C"], n["H"], n["W"]), n["K"], n["S"], n["P"])
        elif op == "resize_nn":
            y = v[0].repeat_interleave(n["S"], 2).repeat_interleave(n["S"], 3)
        elif op == "permute_0213":
            a = v[0].reshape(batch, n["D1"], n["D2"], n["I"])
            y = a.permute(0, 2, 1, 3) if n["mode"] == 0 else a.permute(0, 1, 3, 2)
        elif op == "softmax_axis":
            y = torch.softmax(v[0].reshape(batch * n["outer"], n["axdim"], n["inner"]), 1)
        elif op == "slice_axis":
            y = v[0].reshape(batch * n["outer"], n["axdim"], n["inner"])[:, n["start"]:n["start"] + n["len"]]
        elif op == "reshape":
            y = v[0]
        else:
            raise RuntimeError("no fp64 form of " + op)
        T[o] = y.reshape([batch] + dims[o][1:])
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "pose":
        if c["batch"] > 4:
            return None
        with tempfile.TemporaryDirectory() as d:
            path, _ = pw.yolov8n_pose(d, seed=seed, imgsz=c["imgsz"])
            out = _pose64(path, _frames(c, seed), c["batch"])
        return [o if c["call"] == "infer" else o.reshape(-1) for o in out]
    if c["kind"] == "conv":
        x, r, w, b = _conv_inputs(c, seed)
        w, b = torch.from_numpy(w).cuda().double(), torch.from_numpy(b).cuda().double()
        y = _act64(_conv64(x.double(), w, b, c["s"], c["k"] // 2, c["dw"]), ACTS[c["act"]])
        y = y if r is None else y + r.double()
        return y.permute(0, 2, 3, 1) if c["nhwc"] else y
    if c["kind"] == "attention":
        q, k, v = (t.double() for t in _attention_inputs(c, seed))
        out = []
        for i in range(c["batch"]):
            out.append(torch.stack([torch.softmax(q[i, j] @ k[i, j], -1) @ v[i, j] for j in range(c["heads"])]))
        return torch.stack(out)
    if c["kind"] == "classifier":
        x = _activations(_gen(seed), c["batch"], c["n_in"]).double()
        for n, (o, i, act) in enumerate(((c["hidden"], c["n_in"], ops.ACT_HSWISH),
                                         (c["classes"], c["hidden"], ops.ACT_NONE))):
            w, b = (torch.from_numpy(a).cuda().double() for a in _weights(seed + n, o, i, 1, 1))
            x = _act64(x @ w.reshape(o, i).T + b, act)
        return x
    x, out = _activations(_gen(seed), c["batch"], c["c"], c["h"], c["w"]).double(), []
    for _ in range(3):
        x = F.max_pool2d(x, 5, 1, 2)
        out.append(x)
    return out
