"""The work this framework is measured on: graphs replayed through the session, detection from
host images, and single operators through the C ABI, each over the range of sizes, types and
options a program uses.

A case is a dict of plain values; `kind` names the path:

  ssd       a MobileNet-v1 SSD graph (.dlx) in a session, one replayed pass on resident inputs
  detect    Session.detect: host images in, final detections out (upload, pass, decode + score
            filter, top-k + NMS, readback)
  classify  a residual classification graph (stem, max pool, residual blocks, global average
            pool, Gemm) in a session, one replayed pass
  block     a depthwise-separable block: in a session (fp32) or through the C ABI (fp16 storage)
  conv      one convolution through the C ABI: dense, depthwise, pointwise or grouped, fp32 or
            fp16 storage
  heads     the twelve SSD head convolutions as one grouped call, the two concatenations and the
            decode + score filter, through the C ABI

Weights and inputs are synthetic, drawn from the seed alone.
"""
import ctypes
import math

import numpy as np
import torch

from ogle_amd import dlx, hip, models, session

F32, F16 = "f32", "f16"

# feature maps of the SSD heads: (size, channels, anchors per cell)
HEAD_MAPS = [(19, 512, 3), (10, 1024, 6), (5, 512, 6), (3, 256, 6), (2, 256, 6), (1, 128, 6)]
PRIORS = sum(m * m * a for m, _, a in HEAD_MAPS)


def conv_case(name, dtype, n, h, w, c, o, k=1, s=1, p=0, g=1, act="relu", bias=True):
    case = dict(kind="conv", dtype=dtype, n=n, h=h, w=w, c=c, o=o, k=k, s=s, p=p, g=g, act=act, bias=bias)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one camera, one frame at a time: latency of the whole network, resident input
        dict(name="ssd_b1", kind="ssd", batch=1, image=300, classes=21),
        # the headline workload: a server's batch
        dict(name="ssd_b16", kind="ssd", batch=16, image=300, classes=21),
        # offline processing: the largest batch of the batch sweep
        dict(name="ssd_b64", kind="ssd", batch=64, image=300, classes=21),
        # the detector as an application calls it, from a host image to the list of boxes
        dict(name="detect_b1", kind="detect", batch=1, image=300, classes=21),
        # a residual classifier with its elementwise ops, pools and final Gemm
        dict(name="classify_b16", kind="classify", batch=16, image=224, width=64, classes=1000),
        # depthwise-separable block on 38x38x256, batch 8
        dict(name="block_f32_b8", kind="block", dtype=F32, batch=8, size=38, c=256, o=512, s=1),
        # the same operators with fp16 storage, on an early, large and odd-sized map with stride 2
        dict(name="block_f16_ragged", kind="block", dtype=F16, batch=12, size=113, c=88, o=168, s=2),
        # pointwise convolution as a GEMM, M = 11552, K = 512, N = 1024, in both storage types
        conv_case("pw_f32", F32, 32, 19, 19, 512, 1024),
        conv_case("pw_f16", F16, 32, 19, 19, 512, 1024),
        # one small dense convolution: launch latency counts
        conv_case("dense3x3_b1", F32, 1, 112, 112, 32, 64, 3, 1, 1),
        # grouped convolution, ragged map, channel counts that are no power of two
        conv_case("grouped_ragged", F32, 4, 57, 43, 96, 144, 3, 1, 1, g=12),
        # SSD heads, concatenation and score filter of 64 images, operator by operator
        dict(name="heads_b64", kind="heads", batch=64, classes=21),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_conv(rng):
    """One convolution of any of the four forms; at most about 40 GFLOP and 250 MB."""
    dtype = rng.choice([F32, F32, F16])
    form = rng.choice(["pw", "pw", "dense", "dense", "dw", "grouped", "odd"])
    while True:
        n = _log_int(rng, 1, 64)
        h = _log_int(rng, 1, 160)
        w = max(1, int(round(h * rng.uniform(0.7, 1.4))))
        step = 8 if dtype == F16 else 4
        c, o = (step * _log_int(rng, 16 // step, 1024 // step) for _ in range(2))
        k, s, g = 1, 1, 1
        if form == "dense":
            k, s = rng.choice([3, 3, 3, 5]), rng.choice([1, 1, 2])
        elif form == "dw":
            o = g = c
            k, s = 3, rng.choice([1, 1, 2])
        elif form == "grouped":
            g = rng.choice([2, 3, 4, 8, 12, 16, 32])
            c, o = g * _log_int(rng, 2, 32), g * _log_int(rng, 2, 32)
            k, s = rng.choice([1, 3, 3]), rng.choice([1, 1, 2])
        elif form == "odd":   # channel counts that fill no vector
            c, o = 2 * _log_int(rng, 2, 90) + 1, 2 * _log_int(rng, 2, 90) + 1
            k, s = rng.choice([1, 3]), rng.choice([1, 1, 2])
        p = k // 2
        if h + 2 * p < k or w + 2 * p < k:
            continue
        case = conv_case(None, dtype, n, h, w, c, o, k, s, p, g, rng.choice(["relu", "clip", "none"]),
                         rng.random() < 0.8)
        todo = work(case)
        most = 4e10 if form not in ("grouped", "odd") else 4e9
        if todo["flops"] <= most and todo["bytes"] <= 2.5e8:
            return case


def draw(rng):
    kind = rng.choice(["ssd", "ssd", "detect", "classify", "block", "block", "conv", "conv", "conv", "conv", "heads"])
    if kind == "ssd":
        return dict(kind=kind, batch=_log_int(rng, 1, 56), image=rng.randint(289, 304), classes=rng.randint(2, 40))
    if kind == "detect":
        return dict(kind=kind, batch=_log_int(rng, 1, 12), image=rng.randint(289, 304), classes=rng.randint(2, 40))
    if kind == "classify":
        return dict(kind=kind, batch=_log_int(rng, 1, 24), image=rng.randint(64, 240),
                    width=8 * rng.randint(2, 8), classes=rng.randint(10, 1000))
    if kind == "block":
        while True:
            case = dict(kind=kind, dtype=rng.choice([F32, F16]), batch=_log_int(rng, 1, 32),
                        size=_log_int(rng, 5, 160), c=8 * _log_int(rng, 4, 128), o=8 * _log_int(rng, 4, 128),
                        s=rng.choice([1, 1, 2]))
            todo = work(case)
            if todo["flops"] <= 4e10 and todo["bytes"] <= 2.5e8:
                return case
    if kind == "conv":
        return _draw_conv(rng)
    return dict(kind=kind, batch=_log_int(rng, 1, 64), classes=rng.randint(2, 40))


# ------------------------------------------------------------------------- inputs --
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _torch_dtype(dtype):
    return torch.float16 if dtype == F16 else torch.float32


class _SessionTensor:
    """A session's device tensor, for torch; it keeps the session (and its memory) alive."""

    def __init__(self, sess, name):
        self.session = sess
        self.__cuda_array_interface__ = dict(
            shape=sess.tensor_shape(name), typestr="<f4", version=2, strides=None,
            data=(sess.tensor_device_ptr(name), False))


def _session_tensor(sess, name):
    return torch.as_tensor(_SessionTensor(sess, name), device="cuda")


class _Conv:
    """One convolution through the C ABI: packed filter, bias, output and workspace."""

    ENTRY = {"dw": "ogle_hip_dwconv2d", "pw": "ogle_hip_pwconv_gemm", "dense": "ogle_hip_conv2d"}

    def __init__(self, gen, x, o, k, s, p, g, act, bias, dtype, std=None):
        lib, tdt = hip.lib(), _torch_dtype(dtype)
        hd = hip.F16 if dtype == F16 else hip.F32
        n, h, w, c = x.shape
        form = "dw" if g == c == o and g != 1 else "pw" if k == 1 and s == 1 and p == 0 and g == 1 else "dense"
        std = math.sqrt(2.0 / (c // g * k * k)) if std is None else std
        oihw = torch.randn(o, c // g, k, k, device="cuda", generator=gen) * std
        self.x = x
        self.weight = torch.empty(oihw.numel(), dtype=tdt, device="cuda")
        stream = torch.cuda.current_stream().cuda_stream
        hip.check(lib.ogle_hip_pack_filter(oihw.data_ptr(), self.weight.data_ptr(),
                                           hip.FILTER_HWC if form == "dw" else hip.FILTER_OHWI, hd, o,
                                           c // g, k, k, stream))
        self.bias = torch.rand(o, device="cuda", generator=gen) * 0.2 - 0.1 if bias else None
        self.y = torch.empty(n, hip.out_size(h, k, s, p), hip.out_size(w, k, s, p), o, dtype=tdt, device="cuda")
        self.args = hip.conv_args(
            x.data_ptr(), self.weight.data_ptr(), self.bias.data_ptr() if bias else None, self.y.data_ptr(),
            n, h, w, c, o, k, s, p, 1, g, {"none": hip.ACT_NONE, "clip": hip.ACT_CLIP, "relu": hip.ACT_RELU}[act],
            0.0, 6.0 if act == "clip" else 0.0, hip.VARIANT_PW if form == "pw" else hip.VARIANT_NHWC4, hd)
        need = lib.ogle_hip_conv_workspace_bytes(ctypes.byref(self.args)) if form != "dw" else 0
        self.workspace = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
        if need:
            self.args.workspace_dev, self.args.workspace_bytes = self.workspace.data_ptr(), need
        self.entry = getattr(lib, self.ENTRY[form])
        torch.cuda.current_stream().synchronize()   # oihw is read until here

    def __call__(self, stream):
        hip.check(self.entry(ctypes.byref(self.args), stream))
        return self.y


def _features(gen, shape, dtype):
    """Activations behind a ReLU6: U(0, 6)."""
    return (torch.rand(shape, device="cuda", generator=gen) * 6).to(_torch_dtype(dtype))


def _images(seed, batch, size):
    return np.random.Generator(np.random.PCG64(seed + 1)).uniform(-1, 1, (batch, size, size, 3)).astype(np.float32)


def _residual_classifier(seed, batch, image, width, classes):
    """7x7 stride-2 stem, 3x3 max pool, four residual blocks (width .. 8 * width, stride 2 from
    the second on, 1x1 stride-2 shortcut), global average pool, Gemm; batch norm folded."""
    r = np.random.Generator(np.random.PCG64(seed))
    g = dlx.GraphBuilder()

    def conv(name, x, cin, cout, k, s, act):
        w = r.standard_normal((cout, cin, k, k), np.float32) * np.float32(math.sqrt(2.0 / (cin * k * k)))
        b = r.uniform(-0.1, 0.1, cout).astype(np.float32)
        return g.add_conv(name, x, g.add_filter(name + ".w", w), g.add_const(name + ".b", b), k, s, k // 2, 1, 1, act)

    x = g.add_input("input", [batch, 3, image, image])
    x = conv("stem", x, 3, width, 7, 2, "Relu")
    x = g.add_pool("pool", x, "MaxPool", 3, 2, 1)
    cin = width
    for i in range(4):
        cout, s = width << i, 1 if i == 0 else 2
        y = conv("b%d.c1" % i, x, cin, cout, 3, s, "Relu")
        y = conv("b%d.c2" % i, y, cout, cout, 3, 1, "")
        short = x if s == 1 else conv("b%d.short" % i, x, cin, cout, 1, s, "")
        x = g.add_relu("b%d" % i, g.add_add("b%d.add" % i, y, short))
        cin = cout
    x = g.add_flatten("flat", g.add_pool("gap", x, "GlobalAveragePool"))
    w = r.standard_normal((classes, cin), np.float32) * np.float32(math.sqrt(1.0 / cin))
    g.add_gemm("scores", x, g.add_const("fc.w", w), g.add_const("fc.b", r.uniform(-0.1, 0.1, classes).astype(np.float32)))
    g.add_output_name("scores")
    return g


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("ssd", "detect"):
        # heads spread wide enough that scores pass the threshold, as a trained detector's do
        g, _ = models.mobilenet_v1_ssd(case["batch"], seed=seed, num_classes=case["classes"], image=case["image"],
                                       head_std=0.05 if kind == "detect" else 0.01)
        images = _images(seed, case["batch"], case["image"])
        s = session.Session()
        s.load_graph(g)
        s.run({"input": images})
        if kind == "detect":
            s.sync()
            return dict(case=case, session=s, images=images)
        s.compute(graph=True)
        s.sync()
        return dict(case=case, session=s, outputs=[_session_tensor(s, n) for n in ("cls_logits", "box_preds")])
    if kind == "classify" or (kind == "block" and case["dtype"] == F32):
        s = session.Session()
        if kind == "classify":
            s.load_graph(_residual_classifier(seed, case["batch"], case["image"], case["width"], case["classes"]))
            x, names = _images(seed, case["batch"], case["image"]), ["scores"]
        else:
            r = np.random.Generator(np.random.PCG64(seed))
            g = dlx.GraphBuilder()
            b, n, c, o = case["batch"], case["size"], case["c"], case["o"]
            t = g.add_input("input", [b, c, n, n])
            for name, ci, co, k, st, grp in (("dw", c, c, 3, case["s"], c), ("pw", c, o, 1, 1, 1)):
                w = r.standard_normal((co, ci // grp, k, k), np.float32) * np.float32(math.sqrt(2.0 / (ci // grp * k * k)))
                bias = r.uniform(-0.1, 0.1, co).astype(np.float32)
                t = g.add_conv(name, t, g.add_filter(name + ".w", w), g.add_const(name + ".b", bias), k, st, k // 2, 1,
                               grp, "Clip", 0.0, 6.0)
            g.add_output_name("pw")
            s.load_graph(g)
            x, names = r.random((b, n, n, c), np.float32) * np.float32(6), ["pw"]
        s.run({"input": x})
        s.compute(graph=True)
        s.sync()
        return dict(case=case, session=s, outputs=[_session_tensor(s, n) for n in names])
    gen = _generator(seed)
    if kind == "block":
        n, c, o = case["size"], case["c"], case["o"]
        dw = _Conv(gen, _features(gen, (case["batch"], n, n, c), F16), c, 3, case["s"], 1, c, "clip", True, F16)
        pw = _Conv(gen, dw.y, o, 1, 1, 0, 1, "clip", True, F16)
        return dict(case=case, convs=[dw, pw])
    if kind == "conv":
        x = _features(gen, (case["n"], case["h"], case["w"], case["c"]), case["dtype"])
        return dict(case=case, convs=[_Conv(gen, x, case["o"], case["k"], case["s"], case["p"], case["g"], case["act"],
                                            case["bias"], case["dtype"])])
    batch, classes = case["batch"], case["classes"]
    heads = {4: [], classes + 100: []}   # keyed by output: boxes, class scores
    for m, c, a in HEAD_MAPS:
        x = _features(gen, (batch, m, m, c), F32)
        for key, last in ((4, 4), (classes + 100, classes)):
            heads[key].append(_Conv(gen, x, a * last, 3, 1, 1, 1, "none", True, F32, std=0.01))
    loc, conf = heads[4], heads[classes + 100]
    state = dict(case=case, heads=loc + conf, args=(hip.ConvArgs * 12)(*[h.args for h in loc + conf]), concats=[])
    for group, last in ((loc, 4), (conf, classes)):
        out = torch.empty(batch, PRIORS, last, device="cuda")
        ca = hip.ConcatArgs()
        for i, (h, (m, _, a)) in enumerate(zip(group, HEAD_MAPS)):
            ca.inputs_dev[i], ca.axis_len[i] = h.y.data_ptr(), m * m * a
        ca.output_dev, ca.n_inputs, ca.outer, ca.inner, ca.dtype = out.data_ptr(), 6, batch, last, hip.F32
        state["concats"].append((ca, out))
    anchors = torch.from_numpy(models.ssd_anchors()).cuda()
    f = lambda *s: torch.zeros(*s, device="cuda")                       # noqa: E731
    i = lambda *s: torch.zeros(*s, dtype=torch.int32, device="cuda")    # noqa: E731
    lists = [i(batch, PRIORS), i(batch, PRIORS), f(batch, PRIORS), f(batch, PRIORS, 4), i(batch, PRIORS, 4)]
    boxes = f(batch, PRIORS, 4)
    (_, preds), (_, logits) = state["concats"]
    state["detect"] = hip.DetectArgs(
        logits.data_ptr(), preds.data_ptr(), anchors.data_ptr(), boxes.data_ptr(), batch, PRIORS, classes, 0,
        (ctypes.c_float * 4)(0.1, 0.1, 0.2, 0.2), 0.3, 300.0, 300.0, None, *[t.data_ptr() for t in lists])
    state.update(lists=lists, boxes=boxes, anchors=anchors)
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------------------- run --
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "detect":
        s, batch = state["session"], case["batch"]
        found = s.detect(state["images"], 640, 480, score_threshold=0.3, nms_threshold=0.45, topk=100)
        classes = np.zeros((batch, PRIORS), np.int32)   # class of every prior that is reported, else 0
        for b, items in enumerate(found):
            for d in items:
                classes[b, d["prior"]] = d["cls"]
        return dict(classes=classes, logits=_session_tensor(s, "cls_logits"), boxes=_session_tensor(s, "box_preds"))
    if "session" in state:
        state["session"].compute(graph=True)
        return state["outputs"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "heads":
        lib = hip.lib()
        hip.check(lib.ogle_hip_conv2d_batch(state["args"], 12, stream))
        for ca, _ in state["concats"]:
            hip.check(lib.ogle_hip_concat(ctypes.byref(ca), stream))
        hip.check(lib.ogle_hip_ssd_detect(ctypes.byref(state["detect"]), stream))
        return [out for _, out in state["concats"]] + state["lists"] + [state["boxes"]]
    for conv in state["convs"]:
        y = conv(stream)
    return y


# --------------------------------------------------------------------------- work --
def _conv_work(n, h, w, c, o, k, s, p, g=1, esz=4, bias=True):
    oh, ow = hip.out_size(h, k, s, p), hip.out_size(w, k, s, p)
    return dict(flops=2.0 * n * oh * ow * o * (c // g) * k * k,
                bytes=float(esz * (n * h * w * c + o * (c // g) * k * k + n * oh * ow * o) + (4 * o if bias else 0)))


def _total(parts, extra_bytes=0.0):
    """Work of a chain of operators: every product; of the tensors between them nothing has to
    reach memory, so the bytes are given by the caller."""
    return dict(flops=sum(q["flops"] for q in parts), bytes=extra_bytes)


def work(case):
    kind = case["kind"]
    if kind in ("ssd", "detect"):
        b, n, c = case["batch"], case["image"], 32
        parts, weights, size = [_conv_work(b, n, n, 3, 32, 3, 2, 1)], 27 * 32 + 32, (n - 1) // 2 + 1
        for o, s in models.MOBILENET_V1_BLOCKS:
            parts.append(_conv_work(b, size, size, c, c, 3, s, 1, c))
            size = (size - 1) // s + 1
            parts.append(_conv_work(b, size, size, c, o, 1, 1, 0))
            weights += 10 * c + c * o + o
            c = o
        for m, (c1, c2) in zip((10, 5, 3, 2), models.SSD_EXTRAS):
            parts += [_conv_work(b, m, m, c, c1, 1, 1, 0), _conv_work(b, m, m, c1, c2, 3, 2, 1)]
            weights += c * c1 + c1 + 9 * c1 * c2 + c2
            c = c2
        for m, ch, a in HEAD_MAPS:
            parts.append(_conv_work(b, m, m, ch, a * (4 + case["classes"]), 3, 1, 1))
            weights += 9 * ch * a * (4 + case["classes"])
        return _total(parts, 4.0 * (b * n * n * 3 + weights + b * PRIORS * (4 + case["classes"])))
    if kind == "classify":
        b, n, wd = case["batch"], case["image"], case["width"]
        parts, weights, size = [_conv_work(b, n, n, 3, wd, 7, 2, 3)], 148 * wd, (n - 1) // 2 + 1
        size, c = (size - 1) // 2 + 1, wd
        for i in range(4):
            o, s = wd << i, 1 if i == 0 else 2
            parts.append(_conv_work(b, size, size, c, o, 3, s, 1))
            if s == 2:
                parts.append(_conv_work(b, size, size, c, o, 1, 2, 0))
                weights += c * o + o
            size = (size - 1) // s + 1
            parts.append(_conv_work(b, size, size, o, o, 3, 1, 1))
            weights += 9 * c * o + 9 * o * o + 2 * o
            c = o
        parts.append(_conv_work(b, 1, 1, c, case["classes"], 1, 1, 0))
        weights += (c + 1) * case["classes"]
        return _total(parts, 4.0 * (b * n * n * 3 + weights + b * case["classes"]))
    if kind == "block":
        b, n, c, o, s = (case[k] for k in ("batch", "size", "c", "o", "s"))
        m, esz = (n - 1) // s + 1, 4 if case["dtype"] == F32 else 2
        parts = [_conv_work(b, n, n, c, c, 3, s, 1, c), _conv_work(b, m, m, c, o, 1, 1, 0)]
        return _total(parts, float(esz * (b * n * n * c + 9 * c + c * o + b * m * m * o) + 4 * (c + o)))
    if kind == "conv":
        return _conv_work(case["n"], case["h"], case["w"], case["c"], case["o"], case["k"], case["s"], case["p"],
                          case["g"], 4 if case["dtype"] == F32 else 2, case["bias"])
    b, classes = case["batch"], case["classes"]
    parts = [_conv_work(b, m, m, c, a * (4 + classes), 3, 1, 1) for m, c, a in HEAD_MAPS]
    features = sum(b * m * m * c for m, c, _ in HEAD_MAPS)
    weights = sum((9 * c + 1) * a * (4 + classes) for _, c, a in HEAD_MAPS)
    # out: box predictions, class scores, decoded boxes, and per prior index, class, score, box, rectangle
    return _total(parts, 4.0 * (features + weights + 4 * PRIORS + b * PRIORS * (4 + classes + 4 + 11)))


def tolerance(case):
    """About four times what these paths were measured to differ from the same case in 64-bit
    arithmetic (2-norm): a whole SSD pass 1.6e-6, a single fp32 operator up to 1.0e-6 (sums of
    25,600 products), the SSD heads 2.4e-7, the classifier 2.2e-7, fp16 storage 2.1e-4."""
    if case.get("dtype") == F16:
        return {"rel": 8e-4}            # outputs rounded to fp16
    if case["kind"] in ("conv", "block"):
        return {"rel": 4e-6}
    if case["kind"] == "heads":
        return {"rel": 1e-6, "differ": 2e-4}    # rectangles are truncated to whole pixels
    if case["kind"] == "detect":
        return {"rel": 6e-6, "differ": 2e-3}    # scores at the threshold, equal scores
    return {"rel": 1e-6 if case["kind"] == "classify" else 6e-6}
