"""The work whose time this repository's changes are judged by.

A page recogniser runs, per page: resize and normalise the scan, one det
forward, the DB mask, pack the text lines' crops, classify their orientation
(cls), and read them (rec).  The cases are those calls through the public
sessions and operators, from the smallest (one short line, a small crop's
det) to the largest (a 1536 px page, 50 long lines), with the inputs where a
page pipeline has them: in device memory, except where a program passes host
arrays.  All arithmetic is float32 (and u8 images), the only types the
framework has.
"""
import functools
import math
import random

import numpy as np
import torch

from qppocr_amd import _lib, nets, ops, pipeline, plan

GPU = "cuda:0"
# most work of a drawn rec case: steps = lines * width / 8 of the largest listed one
MAX_STEPS = 6800


def listed():
    return [
        # det of a cropped region (a label, a receipt's header): latency
        dict(name="det_crop", kind="det", h=160, w=416),
        # det of a page at the detector's usual input size
        dict(name="det_page", kind="det", h=640, w=640),
        # det of a large scan
        dict(name="det_scan", kind="det", h=1536, w=1536),
        # one short line through the engine's rec session, host arrays in and out
        dict(name="rec_line", kind="rec_host", lines=1, width=192),
        # a page's batch of lines at the usual width
        dict(name="rec_batch", kind="rec", lines=32, cap=32, width=320, head="fused"),
        # a ragged batch of long lines: 50 real lines on the engine's 64-line session
        dict(name="rec_long", kind="rec", lines=50, cap=64, width=1088, head="fused"),
        # lines whose whole probability rows are exported (rescoring, beam search)
        dict(name="rec_probs", kind="rec", lines=19, cap=19, width=488, head="probs"),
        # orientation of a batch of lines
        dict(name="cls_batch", kind="cls", lines=32, cap=32),
        # the det and rec graphs as GraphPlans (the reference's GPU plan model)
        dict(name="plan_det", kind="plan_det", h=640, w=640),
        dict(name="plan_rec", kind="plan_rec", lines=32, width=320),
        # the steps around the nets: page resize, det input, DB mask, crop packing
        dict(name="page_steps", kind="page", sh=2339, sw=1654, h=1344, w=960, lines=24, width=448),
        # one dense conv layer through the operator API
        dict(name="conv_layer", kind="conv", n=1, c=32, m=32, h=160, w=160, k=3, s=1, dw=False,
             act="relu"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grain(v, g, lo):
    return max(lo, (v + g // 2) // g * g)


def draw(rng):
    kind = rng.choice(["det", "det", "rec", "rec", "rec", "rec_host", "cls", "plan_det", "plan_rec",
                       "page", "conv", "conv"])
    if kind in ("det", "plan_det"):
        # any multiple of 32, pages and strips
        top = 1536 if kind == "det" else 960
        return dict(kind=kind, h=_grain(_log(rng, 96, top), 32, 96),
                    w=_grain(_log(rng, 96, top), 32, 96))
    if kind in ("rec", "rec_host", "plan_rec"):
        # the engine rounds widths to 64; other programs run tight widths (multiples of 8)
        width = _grain(_log(rng, 80, 1280), rng.choice([8, 64]), 80)
        most = {"rec": 64, "rec_host": 8, "plan_rec": 32}[kind]
        steps = MAX_STEPS if kind == "rec" else 1600
        lines = max(1, min(_log(rng, 1, most), steps * 8 // width))
        if kind != "rec":
            return dict(kind=kind, lines=lines, width=width)
        cap = 64 if rng.random() < 0.5 else lines
        head = rng.choice(["fused", "fused", "probs", "pairs"])
        if head != "fused":
            lines = min(lines, max(1, 2400 * 8 // width))
        return dict(kind=kind, lines=lines, cap=max(cap, lines), width=width, head=head)
    if kind == "cls":
        lines = _log(rng, 1, 32)
        return dict(kind=kind, lines=lines, cap=rng.choice([32, lines]))
    if kind == "page":
        return dict(kind=kind, sh=_log(rng, 200, 3000), sw=_log(rng, 200, 3000),
                    h=_grain(_log(rng, 96, 1536), 32, 96), w=_grain(_log(rng, 96, 1536), 32, 96),
                    lines=_log(rng, 1, 64), width=_grain(_log(rng, 80, 1280), 8, 80))
    # conv layers of the nets' kinds: dense 3x3, pointwise, depthwise 3x3 / 5x5
    form = rng.choice(["3x3", "3x3", "1x1", "dw"])
    k = 1 if form == "1x1" else rng.choice([3, 5]) if form == "dw" else 3
    c = _grain(_log(rng, 3, 256), rng.choice([1, 8]), 3)
    m = c if form == "dw" else _grain(_log(rng, 8, 256), rng.choice([1, 8]), 8)
    h, w = _log(rng, 10, 320), _log(rng, 10, 320)
    n = rng.choice([1, 1, 4])
    # no layer past 6 GFLOP or 16 M input values
    while n * c * h * w > 1 << 24 or 2 * n * m * (1 if form == "dw" else c) * k * k * h * w > 6e9:
        h, w, n = max(10, h // 2), max(10, w // 2), 1
    return dict(kind="conv", n=n, c=c, m=m, h=h, w=w, k=k, s=1 if k == 1 else rng.choice([1, 1, 2]),
                dw=form == "dw", act=rng.choice(["relu", "hardswish"]))


# ---------------------------------------------------------------- the user's side

class _Region:
    """Device memory of a session as an array that torch can view.  A view
    holds its region and so the session: the memory outlives every view."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(int(v) for v in shape), typestr="<f4",
                                             data=(int(ptr), False), version=2)


def _view(owner, ptr, shape):
    return torch.as_tensor(_Region(owner, ptr, shape), device=GPU)


def _tensor(sess, tid, lines=None):
    shape = sess.graph.lshapes[tid]
    v = _view(sess, sess.tensor_ptr(tid)[0], shape)
    return v if lines is None else v[:lines]


def _pairs(p):
    """(value, class id) of a rec exit's pairs: the ids are the bits of the second word."""
    return {"value": p[..., 0], "ids": p.view(torch.int32)[..., 1]}


@functools.lru_cache(maxsize=4)
def _det_graph(h, w):
    return nets.build_det(2, h, w)[0]


@functools.lru_cache(maxsize=1)
def _rec_weights():
    return nets.rec_weights(nets.WeightRng(3))


@functools.lru_cache(maxsize=1)
def _cls_weights():
    return nets.cls_weights(nets.WeightRng(5))


def _rec_graph(case, batch):
    head = case.get("head", "fused")
    return nets.build_rec_graph(_rec_weights(), batch, case["width"], probs=head == "probs",
                                fused_head=head == "fused")


def _gen(seed):
    return torch.Generator(device=GPU).manual_seed(seed)


def _uniform(seed, shape, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=_gen(seed), device=GPU) * (hi - lo) + lo


def _image(seed, h, w):
    """A u8 page: dark strokes on a bright, uneven ground with sensor noise."""
    g = _gen(seed)
    low = torch.rand((1, 3, max(2, h // 64), max(2, w // 64)), generator=g, device=GPU)
    ink = torch.rand((1, 1, max(2, h // 4), max(2, w // 4)), generator=g, device=GPU)
    size = dict(size=(h, w), mode="bilinear", align_corners=False)
    f = torch.nn.functional.interpolate
    v = 180.0 + 60.0 * f(low, **size) - 170.0 * (f(ink, **size) > 0.62)
    v = v + 8.0 * torch.randn((1, 3, h, w), generator=g, device=GPU)
    return v.clamp(0, 255).to(torch.uint8)[0].permute(1, 2, 0).contiguous()


def _prob_map(seed, h, w):
    """A det output: text blobs near 1 on a ground near 0."""
    t = torch.rand((1, 1, max(2, h // 12), max(2, w // 24)), generator=_gen(seed), device=GPU)
    t = torch.nn.functional.interpolate(t, size=(h, w), mode="bilinear", align_corners=False)
    return torch.sigmoid(14.0 * (t - 0.6)).contiguous()


def _crop_sizes(case):
    r = random.Random(case["lines"] * 7919 + case["width"])
    return [(r.randint(18, 72), r.randint(case["width"] // 3, case["width"] * 5 // 4))
            for _ in range(case["lines"])]


def _conv_weights(case, seed):
    c, m, k = case["c"], case["m"], case["k"]
    cg = 1 if case["dw"] else c
    g = _gen(seed + 1)
    w = torch.randn((m, cg, k, k), generator=g, device=GPU) * math.sqrt(2.0 / (cg * k * k))
    b = torch.randn((m,), generator=g, device=GPU) * 0.1
    return w, b


def _inputs(case, seed):
    kind = case["kind"]
    if kind in ("det", "plan_det"):
        return _uniform(seed, (1, 3, case["h"], case["w"]))
    if kind in ("rec", "rec_host", "plan_rec"):
        return _uniform(seed, (case["lines"], 3, pipeline.REC_H, case["width"]))
    if kind == "cls":
        return _uniform(seed, (case["lines"], 3, nets.CLS_H, nets.CLS_W))
    return _uniform(seed, (case["n"], case["c"], case["h"], case["w"]), 0.0, 1.0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "page":
        return dict(kind=kind, case=case, src=_image(seed, case["sh"], case["sw"]),
                    pred=_prob_map(seed + 1, case["h"], case["w"]),
                    crops=[_image(seed + 2 + i, ch, cw)
                           for i, (ch, cw) in enumerate(_crop_sizes(case))])
    x = _inputs(case, seed)
    if kind == "conv":
        w, b = _conv_weights(case, seed)
        c, k, s = case["c"], case["k"], case["s"]
        params = ops.conv_params(s, s, k // 2, k // 2, group=c if case["dw"] else 1)
        act = _lib.ACT_RELU if case["act"] == "relu" else _lib.ACT_HARDSWISH
        return dict(kind=kind, x=x, w=w, b=b, params=params, act=act)
    if kind == "rec_host":
        sess = pipeline.HipRecSession(_rec_weights())
        host = x.cpu().numpy()
        sess.run(host)           # the net of this shape is made on its first run
        return dict(kind=kind, sess=sess, x=host)
    if kind in ("plan_det", "plan_rec"):
        g = _det_graph(case["h"], case["w"]) if kind == "plan_det" else \
            nets.build_rec_graph(_rec_weights(), case["lines"], case["width"], probs=False)
        sess = plan.HipPlanSession(plan.build_plan(g))
        sess.run(x.cpu().numpy())    # leaves the input in the plan's arena
        base = sess.arena()[0]
        outs = [_view(sess, base + 4 * off, shape) for off, _, shape in sess.plan.outputs]
        return dict(kind=kind, sess=sess,
                    out={"map": outs[0]} if kind == "plan_det" else _pairs(outs[0]))
    if kind == "det":
        sess = nets.HipSession(_det_graph(case["h"], case["w"]))
        out = {"map": _tensor(sess, sess.graph.outputs[0])}
    elif kind == "cls":
        sess = nets.HipSession(nets.build_cls_graph(_cls_weights(), case["cap"]))
        sess.set_real_n(case["lines"])
        out = {"probs": _tensor(sess, sess.graph.outputs[0], case["lines"]),
               "hidden": _tensor(sess, sess.graph.nodes[-2]["inp"], case["lines"])}
    else:
        g = _rec_graph(case, case["cap"])
        sess = nets.HipSession(g)
        sess.set_real_n(case["lines"])
        out = _pairs(_tensor(sess, g.outputs[-1], case["lines"]))
        out["hidden"] = _tensor(sess, g.nodes[-2]["inp"], case["lines"])
        if case["head"] == "probs":
            out["probs"] = _tensor(sess, g.outputs[0], case["lines"])
    torch.cuda.synchronize()     # the session's stream does not wait for torch's
    return dict(kind=kind, sess=sess, x=x, out=out)


def run(state):
    kind = state["kind"]
    if kind in ("det", "rec", "cls"):
        state["sess"].run(state["x"].data_ptr(), outputs=False)
        return state["out"]
    if kind == "rec_host":
        p = state["sess"].run(state["x"])
        return {"value": p[..., 0], "ids": p.view(np.int32)[..., 1]}
    if kind in ("plan_det", "plan_rec"):
        state["sess"].run(None, outputs=False)
        return state["out"]
    if kind == "conv":
        return ops.conv2d(state["x"], state["w"], state["b"], state["params"], state["act"])
    case = state["case"]
    page = ops.resize_bilinear_rgb_u8(state["src"], case["w"], case["h"])
    x = ops.det_normalize_u8(page)
    mask = ops.db_mask(state["pred"], 0.3)
    lines = ops.pack_crops(state["crops"], pipeline.REC_H, case["width"])
    return {"page": page, "x": x, "mask": mask, "lines": lines}


# ---------------------------------------------------------------- what a pass needs

def work(case):
    kind = case["kind"]
    if kind == "page":
        px = case["h"] * case["w"]
        # a resize reads at most the pixels it samples (four a target pixel, 3 bytes each)
        crops = sum(min(ch * cw, 4 * 48 * max(1, 48 * cw // ch)) for ch, cw in _crop_sizes(case))
        read = 3 * min(case["sh"] * case["sw"], 4 * px) + 4 * px + 3 * crops
        wrote = 3 * px + 12 * px + px + 4 * 3 * 48 * case["width"] * case["lines"]
        return {"bytes": read + wrote, "flops": 0}
    if kind == "conv":
        n, c, m, k, s = case["n"], case["c"], case["m"], case["k"], case["s"]
        oh, ow = (case["h"] - 1) // s + 1, (case["w"] - 1) // s + 1
        cg = 1 if case["dw"] else c
        words = n * c * case["h"] * case["w"] + m * cg * k * k + m + n * m * oh * ow
        return {"bytes": 4 * words, "flops": 2 * n * m * cg * k * k * oh * ow}
    if kind in ("det", "plan_det"):
        g = _det_graph(case["h"], case["w"])
        outs = case["h"] * case["w"]
    elif kind == "cls":
        g = nets.build_cls_graph(_cls_weights(), case["lines"])
        outs = 2 * case["lines"]
    else:
        g = _rec_graph(dict(case, head=case.get("head", "fused")), case["lines"])
        steps = case["lines"] * case["width"] // 8
        outs = steps * (2 + (nets.REC_CLASSES if case.get("head") == "probs" else 0))
    words = g.numel(0) + sum(w.size for w in g.weights) + outs
    return {"bytes": 4 * words, "flops": nets.flops(g)}


def tolerance(case):
    if case["kind"] == "page":
        return "exact"              # u8 images, and floats that are functions of a byte
    # float32 sums: about four times the distance of the results from float64 (det
    # 1e-7, conv layers 3e-7 to 1e-6, rec probabilities 5e-6; ids may differ at ties)
    if case["kind"] in ("rec", "rec_host", "plan_rec"):
        return {"rel": 2e-5, "max": 1e-3, "differ": 2e-3}
    return {"rel": 4e-6 if case["kind"] == "conv" else 1e-6, "max": 1e-4}


# ---------------------------------------------------------------- the same in 64 bits

def _w64(weights):
    return iter([torch.from_numpy(np.asarray(w, np.float64)).to(GPU) for w in weights])


def _hswish64(x):
    return x * torch.clamp(x / 6.0 + 0.5, 0.0, 1.0)


def _conv64(x, w, b, stride=(1, 1), pad=(0, 0, 0, 0)):
    """Dense or depthwise conv, one tap at a time; pad = (top, left, bottom, right)."""
    x = torch.nn.functional.pad(x, (pad[1], pad[3], pad[0], pad[2]))
    n, c, h, wd = x.shape
    m, cg, kh, kw = w.shape
    oh, ow = (h - kh) // stride[0] + 1, (wd - kw) // stride[1] + 1
    y = b.reshape(1, m, 1, 1).expand(n, m, oh, ow).clone()
    for i in range(kh):
        for j in range(kw):
            t = x[:, :, i:i + (oh - 1) * stride[0] + 1:stride[0],
                  j:j + (ow - 1) * stride[1] + 1:stride[1]]
            if cg == 1 and c > 1:
                y += t * w[:, 0, i, j].reshape(1, m, 1, 1)
            else:
                t = t.permute(1, 0, 2, 3).reshape(c, -1)
                y += (w[:, :, i, j] @ t).reshape(m, n, oh, ow).permute(1, 0, 2, 3)
    return y


def _convt64(x, w):
    """2x2 stride-2 transposed conv, no bias."""
    n, c, h, wd = x.shape
    m = w.shape[1]
    y = torch.zeros((n, m, 2 * h, 2 * wd), dtype=x.dtype, device=x.device)
    t = x.permute(1, 0, 2, 3).reshape(c, -1)
    for i in range(2):
        for j in range(2):
            y[:, :, i::2, j::2] = (w[:, :, i, j].T @ t).reshape(m, n, h, wd).permute(1, 0, 2, 3)
    return y


def _ln64(x, g, b):
    mu = x.mean(-1, keepdim=True)
    var = ((x - mu) ** 2).mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(var + 1e-6) * g + b


def _det64(weights, x):
    it = _w64(weights)
    w = lambda: next(it)  # noqa: E731
    h = _hswish64(_conv64(x, w(), w(), (2, 2), (1,) * 4))
    feats = []
    strides = [2, 1, 2, 1, 2, 1, 1, 1, 1, 1, 2]
    for s in strides:
        wd = w()
        h = _hswish64(_conv64(h, wd, w(), (s, s), (wd.shape[2] // 2,) * 4))
        h = _hswish64(_conv64(h, w(), w()))
        feats.append(h)
    up = lambda t, f: t.repeat_interleave(f, 2).repeat_interleave(f, 3)  # noqa: E731
    tops = [_conv64(feats[10], w(), w())]
    for f in (feats[9], feats[3], feats[1]):
        tops.append(_conv64(f, w(), w()) + up(tops[-1], 2))
    maps = [up(_conv64(t, w(), w(), pad=(1,) * 4), f) for t, f in zip(tops, (8, 4, 2, 1))]
    h = torch.relu(_conv64(torch.cat(maps, 1), w(), w(), pad=(1,) * 4))
    return torch.sigmoid(_convt64(_convt64(h, w()), w()))


def _rec64(weights, x):
    it = _w64(weights)
    w = lambda: next(it)  # noqa: E731
    h = _hswish64(_conv64(x, w(), w(), (2, 2), (1,) * 4))
    for st, pad in [((2, 2), (1,) * 4), ((2, 2), (1,) * 4), ((2, 1), (1,) * 4), ((3, 1), (0, 1, 0, 1))]:
        h = _hswish64(_conv64(h, w(), w(), st, pad))
        h = _hswish64(_conv64(h, w(), w()))
    b, c, _, t = h.shape
    x = h.reshape(b, c, t).transpose(1, 2).contiguous()
    for _ in range(2):
        a = _ln64(x, w(), w())
        qkv = (a @ w() + w()).reshape(b, t, 3, 8, 32).permute(2, 0, 3, 1, 4).contiguous()
        p = torch.softmax((qkv[0] / math.sqrt(32)) @ qkv[1].transpose(-1, -2).contiguous(), -1)
        x = x + (p @ qkv[2]).transpose(1, 2).reshape(b, t, c) @ w() + w()
        m = _ln64(x, w(), w()) @ w() + w()
        m = 0.5 * m * (1.0 + torch.erf(m / math.sqrt(2.0)))
        x = x + m @ w() + w()
    return x, torch.softmax(x @ w() + w(), -1)


def _cls64(weights, x):
    it = _w64(weights)
    w = lambda: next(it)  # noqa: E731
    h = _hswish64(_conv64(x, w(), w(), (2, 2), (1,) * 4))
    for s, se in [(1, 0), (2, 0), (1, 0), (2, 0), (1, 0), (2, 1), (1, 1)]:
        wd = w()
        h = _hswish64(_conv64(h, wd, w(), (s, s), (wd.shape[2] // 2,) * 4))
        if se:
            gate = torch.relu(_conv64(h.mean((2, 3), keepdim=True), w(), w()))
            h = h * torch.clamp(_conv64(gate, w(), w()) / 6.0 + 0.5, 0.0, 1.0)
        h = _hswish64(_conv64(h, w(), w()))
    h = _hswish64(_conv64(h.mean((2, 3), keepdim=True), w(), w()))
    return h, torch.softmax(h.flatten(1) @ w() + w(), -1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "page":
        return None                 # bytes, and float32 functions of single bytes
    x = _inputs(case, seed).double()
    if kind == "conv":
        w, b = _conv_weights(case, seed)
        k, s = case["k"], case["s"]
        y = _conv64(x, w.double(), b.double(), (s, s), (k // 2,) * 4)
        return torch.relu(y) if case["act"] == "relu" else _hswish64(y)
    if kind in ("det", "plan_det"):
        return {"map": _det64(_det_graph(case["h"], case["w"]).weights, x)}
    if kind == "cls":
        hidden, probs = _cls64(_cls_weights(), x)
        return {"probs": probs, "hidden": hidden}
    hidden, probs = _rec64(_rec_weights(), x)
    out = {"value": probs.max(-1).values, "ids": None}
    if kind == "rec":
        out["hidden"] = hidden
        if case["head"] == "probs":
            out["probs"] = probs
    return out
