"""Performance cases: the work that programs built on this package have it do, through its public entry points.

A case is a dict of plain values.  `listed()` gives a fixed set over the whole range, `draw(rng)` one more case of the same ranges,
`prepare(case, seed)` what a program holds before the call (tensors on the device, operators, packed weights, workspace), `run(state)` one
pass, `work(case)` the bytes and operations a pass cannot do without, `tolerance(case)` how far a correct result may be off, `exact(case, seed)`
the same results in 64 bits.

Kinds of case:
  network     a ResNet forward pass: graphs.GraphRunner on one batch of images (image sizes and batches as they are served: one image where
              latency counts, 16 and 64 as the published benchmarks have it, 128 for throughput)
  train       one convolution of a training step: forward, then the gradients of input, filter and bias
  block       the inverted residual block of MobileNet-v2 at inference: 1x1 expansion, 3x3 depthwise, 1x1 projection
  train_block the depthwise + pointwise pair of such a block in a training step
  head        the fully connected classifier of AlexNet / VGG with softmax and the validation loss
  decoder     an upsampling stage of a segmentation or generator network: transposed convolution, then bilinear interpolation by two
"""
import math

import torch

import dlprimitives_amd as dlp
from dlprimitives_amd import graphs
from dlprimitives_amd.capi import BFLOAT16_DATA, FLOAT_DATA

DEVICE = "cuda:0"
CLASSES = 1000


def listed():
    return [
        # throughput serving: the repository's own ResNet-50 configuration, bfloat16, batch 128, everything fused
        dict(name="resnet50_bf16_b128", kind="network", net="resnet50", dtype="bfloat16", batch=128, size=224, algo="", deployed=True),
        # latency serving: one image; some 55 dependent launches
        dict(name="resnet50_bf16_b1", kind="network", net="resnet50", dtype="bfloat16", batch=1, size=224, algo="", deployed=True),
        # float inference at the batch of the published benchmark tables
        dict(name="resnet50_f32_b16", kind="network", net="resnet50", dtype="float32", batch=16, size=224, algo="", deployed=True),
        # the repository's headline workload: algorithm gemm, filters handed over raw in every call, sums as operators of their own
        dict(name="resnet18_f32_b64_gemm", kind="network", net="resnet18", dtype="float32", batch=64, size=224, algo="gemm", deployed=False),
        # training, the layer most convolutional networks spend their time in: 3x3, stride 1, a middle stage
        dict(name="train_3x3_128_at28_b64", kind="train", batch=64, cin=128, cout=128, h=28, w=28, k=3, s=1, p=1, d=1, g=1, algo=""),
        # training, the layer that opens a stage: 3x3, stride 2, twice the channels
        dict(name="train_3x3s2_128to256_at28_b32", kind="train", batch=32, cin=128, cout=256, h=28, w=28, k=3, s=2, p=1, d=1, g=1, algo=""),
        # training on ragged sizes: odd image, odd batch, channels off every tile, 5x5
        dict(name="train_5x5_48to80_at35x27_b9", kind="train", batch=9, cin=48, cout=80, h=35, w=27, k=5, s=1, p=2, d=1, g=1, algo="gemm"),
        # mobile inference, large images: bound by memory
        dict(name="block_f32_24x6_at56_b64", kind="block", dtype="float32", batch=64, cin=24, hidden=144, cout=24, h=56, w=56, s=1),
        # mobile inference, small images in bfloat16: bound by launches
        dict(name="block_bf16_96x6_at14s2_b24", kind="block", dtype="bfloat16", batch=24, cin=96, hidden=576, cout=160, h=14, w=14, s=2),
        # training of the depthwise + pointwise pair
        dict(name="train_block_192_at28_b32", kind="train_block", batch=32, c=192, cout=32, h=28, w=28, s=1),
        # the VGG classifier at a serving batch: 0.5 GB of weights read once
        dict(name="head_f32_25088_b16", kind="head", dtype="float32", batch=16, inputs=25088, hidden=4096),
        # one decoder stage
        dict(name="decoder_256to128_at14_b16", kind="decoder", batch=16, cin=256, cout=128, h=14, w=14, k=4, s=2, p=1, op=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng, lo, hi):
    """mostly multiples of 16 and 32, as networks have them; one in five anything"""
    c = _log(rng, lo, hi)
    return c if rng.random() < 0.2 else max(16, (c + 8) // 16 * 16)


def draw(rng):
    kind = rng.choice(["network", "network", "train", "train", "train", "block", "block", "train_block", "head", "decoder"])
    if kind == "network":
        net = rng.choice(["resnet18", "resnet50"])
        dtype = rng.choice(["bfloat16", "float32"])
        case = dict(kind=kind, net=net, dtype=dtype, batch=_log(rng, 1, 128), size=rng.choice([128, 160, 192, 224, 224, 224, 256, rng.randint(120, 260)]),
                    algo=rng.choice(["", "", "gemm"]), deployed=rng.random() < 0.75)
        limit = 1.0e12 if dtype == "bfloat16" else 1.8e11
        while case["batch"] > 1 and work(case)["flops"] > limit:
            case["batch"] = max(1, case["batch"] * 3 // 4)
        return case
    if kind == "train":
        k = rng.choice([3, 3, 3, 1, 1, 5, 7])
        h = _log(rng, 7, 112)
        w = h if rng.random() < 0.7 else max(5, int(h * rng.uniform(0.6, 1.6)))
        g = rng.choice([1, 1, 1, 1, 1, 2, 4])
        cin, cout = (max(1, _channels(rng, 16, 512) // g) * g for _ in range(2))
        d = 2 if k == 3 and rng.random() < 0.1 else 1
        case = dict(kind=kind, batch=_log(rng, 1, 64), cin=cin, cout=cout, h=h, w=w, k=k, s=rng.choice([1, 1, 1, 2]), p=d * (k // 2), d=d, g=g,
                    algo=rng.choice(["", "", "gemm"]))
        while case["batch"] > 1 and (work(case)["flops"] > 8e10 or work(case)["bytes"] > 1.5e9):
            case["batch"] = max(1, case["batch"] * 3 // 4)
        while case["cin"] > 2 * g and work(case)["flops"] > 8e10:
            case["cin"] = case["cin"] // (2 * g) * g
        return case
    if kind == "block":
        h = _log(rng, 7, 112)
        s = rng.choice([1, 1, 2])
        cin = max(8, int(1200 / h * rng.uniform(0.5, 2.0)) // 8 * 8)
        cin = min(cin, 160)
        cout = cin if s == 1 and rng.random() < 0.6 else max(8, int(cin * rng.uniform(0.7, 2.0)) // 8 * 8)
        case = dict(kind=kind, dtype=rng.choice(["float32", "bfloat16"]), batch=_log(rng, 1, 96), cin=cin, hidden=cin * 6, cout=cout, h=h,
                    w=h if rng.random() < 0.8 else h + rng.randint(1, 6), s=s)
        while case["batch"] > 1 and case["batch"] * case["hidden"] * case["h"] * case["w"] > 3.2e7:
            case["batch"] = max(1, case["batch"] * 3 // 4)
        return case
    if kind == "train_block":
        h = _log(rng, 7, 56)
        c = max(16, int(5000 / h * rng.uniform(0.5, 1.5)) // 8 * 8)
        c = min(c, 960)
        case = dict(kind=kind, batch=_log(rng, 1, 64), c=c, cout=max(8, int(c * rng.uniform(0.15, 0.5)) // 8 * 8), h=h,
                    w=h if rng.random() < 0.8 else h + rng.randint(1, 6), s=rng.choice([1, 1, 2]))
        while case["batch"] > 1 and case["batch"] * case["c"] * case["h"] * case["w"] > 2.0e7:
            case["batch"] = max(1, case["batch"] * 3 // 4)
        return case
    if kind == "head":
        return dict(kind=kind, dtype=rng.choice(["float32", "bfloat16"]), batch=_log(rng, 1, 128), inputs=rng.choice([512, 1280, 2048, 9216, 25088, _log(rng, 500, 25000)]),
                    hidden=rng.choice([1024, 4096, _log(rng, 256, 4096)]))
    k, s, p, op = rng.choice([(4, 2, 1, 0), (3, 2, 1, 1), (2, 2, 0, 0), (3, 1, 1, 0), (5, 2, 2, 1)])
    h = _log(rng, 7, 56)
    case = dict(kind="decoder", batch=_log(rng, 1, 32), cin=_channels(rng, 16, 512), cout=_channels(rng, 16, 256), h=h,
                w=h if rng.random() < 0.7 else max(5, int(h * rng.uniform(0.6, 1.6))), k=k, s=s, p=p, op=op)
    while case["batch"] > 1 and (work(case)["flops"] > 8e10 or work(case)["bytes"] > 1.0e9):
        case["batch"] = max(1, case["batch"] * 3 // 4)
    return case


class _Made:
    """Random tensors of one seed, made on the device: activations behind a ReLU, Kaiming-normal filters, small gradients."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * std).to(dtype)

    def activations(self, *shape, dtype=torch.float32):
        return torch.randn(shape, generator=self.gen, device=DEVICE).relu_().to(dtype)

    def filters(self, cout, cin_g, k, dtype=torch.float32):
        return self.normal(cout, cin_g, k, k, std=math.sqrt(2.0 / (cin_g * k * k)), dtype=dtype)

    def bias(self, n):
        return torch.rand((n,), generator=self.gen, device=DEVICE) * 0.2 - 0.1


def _types(case):
    return (torch.bfloat16, BFLOAT16_DATA) if case.get("dtype") == "bfloat16" else (torch.float32, FLOAT_DATA)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEVICE)


def _out(n, k, s, p, d=1):
    return (n + 2 * p - d * (k - 1) - 1) // s + 1


def _tconv_out(n, case):
    return (n - 1) * case["s"] - 2 * case["p"] + case["k"] - 1 + case["op"] + 1


def _workspace(*ops):
    return torch.empty(max([1] + [op.workspace() for op in ops]), dtype=torch.uint8, device=DEVICE)


def _packed(op, w):
    buf = torch.empty(max(op.packed_size(), 1), dtype=torch.uint8, device=DEVICE)
    op.pack(w, buf)
    return buf


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed, _Made(seed))


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---- network: what a serving program does with a batch of images ----
def _prepare_network(case, seed, made):
    ops = getattr(graphs, case["net"])()
    shape = (case["batch"], 3, case["size"], case["size"])
    on = bool(case["deployed"])
    runner = graphs.GraphRunner(ops, graphs.random_parameters(ops, seed), shape, algo=case["algo"], dtype=case["dtype"], fuse_residual=on, prepack=on,
                                channels_last=on, fuse_stem_pool=on)
    return dict(kind="network", runner=runner, x=made.normal(*shape, dtype=_types(case)[0]))


def _run_network(st):
    return st["runner"].forward(st["x"])


# ---- train: forward and the three gradients of one convolution ----
def _prepare_train(case, seed, made):
    b, cin, cout, h, w, k = (case[n] for n in ("batch", "cin", "cout", "h", "w", "k"))
    oh, ow = (_out(n, k, case["s"], case["p"], case["d"]) for n in (h, w))
    settings = dlp.Conv2DSettings(cin, cout, k, case["s"], case["d"], case["p"], case["g"], (b, cin, h, w))
    st = dict(kind="train", x=made.activations(b, cin, h, w), w=made.filters(cout, cin // case["g"], k), b=made.bias(cout),
              dy=made.normal(b, cout, oh, ow, std=1e-2), y=_empty(b, cout, oh, ow), dx=_empty(b, cin, h, w), dw=_empty(cout, cin // case["g"], k, k), db=_empty(cout),
              fwd=dlp.Conv2DForward.create(settings, True, "identity", case["algo"]), data=dlp.Conv2DBackwardData.create(settings, case["algo"]),
              filter=dlp.Conv2DBackwardFilter.create(settings, case["algo"]))
    st["ws"] = _workspace(st["fwd"], st["data"], st["filter"])
    return st


def _run_train(st):
    st["fwd"].enqueue(st["x"], st["w"], st["b"], st["y"], st["ws"])
    st["data"].enqueue(st["dx"], st["w"], st["dy"], st["ws"])
    st["filter"].enqueue(st["x"], st["dw"], st["dy"], st["ws"])
    dlp.bias_backward(st["dy"], st["db"])
    return {n: st[n] for n in ("y", "dx", "dw", "db")}


# ---- block: inverted residual at inference, constant filters ----
def _prepare_block(case, seed, made):
    tdt, code = _types(case)
    b, cin, hid, cout, h, w, s = (case[n] for n in ("batch", "cin", "hidden", "cout", "h", "w", "s"))
    oh, ow = _out(h, 3, s, 1), _out(w, 3, s, 1)
    st = dict(kind="block", x=made.normal(b, cin, h, w, dtype=tdt), skip=s == 1 and cin == cout,
              w1=made.filters(hid, cin, 1, tdt), b1=made.bias(hid), wd=made.filters(hid, 1, 3, tdt), bd=made.bias(hid), w2=made.filters(cout, hid, 1, tdt), b2=made.bias(cout),
              t1=_empty(b, hid, h, w, dtype=tdt), y=_empty(b, cout, oh, ow, dtype=tdt), sum=_empty(b, cout, oh, ow, dtype=tdt))
    st["expand"] = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, hid, 1, 1, 1, 0, 1, (b, cin, h, w), dtype=code), True, "relu6")
    st["p1"] = _packed(st["expand"], st["w1"])
    depthwise = dlp.Conv2DSettings(hid, hid, 3, s, 1, 1, hid, (b, hid, h, w), dtype=code)
    if dlp.DepthwisePointwiseForward.supported(depthwise, "relu6", cout, "identity"):
        st["pair"] = dlp.DepthwisePointwiseForward.create(depthwise, True, "relu6", cout, True, "identity")
        st["ws"] = _workspace(st["expand"])
    else:
        st["t2"] = _empty(b, hid, oh, ow, dtype=tdt)
        st["depthwise"] = dlp.Conv2DForward.create(depthwise, True, "relu6")
        st["pd"] = _packed(st["depthwise"], st["wd"])
        st["project"] = dlp.Conv2DForward.create(dlp.Conv2DSettings(hid, cout, 1, 1, 1, 0, 1, (b, hid, oh, ow), dtype=code), True, "identity")
        st["p2"] = _packed(st["project"], st["w2"])
        st["ws"] = _workspace(st["expand"], st["depthwise"], st["project"])
    return st


def _run_block(st):
    st["expand"].enqueue_packed(st["x"], st["w1"], st["p1"], st["b1"], st["t1"], st["ws"])
    if "pair" in st:
        st["pair"].enqueue(st["t1"], st["wd"], st["bd"], st["w2"], st["b2"], st["y"])
    else:
        st["depthwise"].enqueue_packed(st["t1"], st["wd"], st["pd"], st["bd"], st["t2"], st["ws"])
        st["project"].enqueue_packed(st["t2"], st["w2"], st["p2"], st["b2"], st["y"], st["ws"])
    if not st["skip"]:
        return st["y"]
    dlp.eltwise_forward(st["y"], st["x"], st["sum"])
    return st["sum"]


# ---- train_block: depthwise + pointwise, forward and all gradients ----
def _prepare_train_block(case, seed, made):
    b, c, cout, h, w, s = (case[n] for n in ("batch", "c", "cout", "h", "w", "s"))
    oh, ow = _out(h, 3, s, 1), _out(w, 3, s, 1)
    deep = dlp.Conv2DSettings(c, c, 3, s, 1, 1, c, (b, c, h, w))
    point = dlp.Conv2DSettings(c, cout, 1, 1, 1, 0, 1, (b, c, oh, ow))
    st = dict(kind="train_block", x=made.activations(b, c, h, w), wd=made.filters(c, 1, 3), bd=made.bias(c), wp=made.filters(cout, c, 1), bp=made.bias(cout),
              dy=made.normal(b, cout, oh, ow, std=1e-2), t=_empty(b, c, oh, ow), y=_empty(b, cout, oh, ow), dt=_empty(b, c, oh, ow), dx=_empty(b, c, h, w),
              dwd=_empty(c, 1, 3, 3), dbd=_empty(c), dwp=_empty(cout, c, 1, 1), dbp=_empty(cout),
              ops=[(dlp.Conv2DForward.create(x, True, "identity"), dlp.Conv2DBackwardData.create(x), dlp.Conv2DBackwardFilter.create(x)) for x in (deep, point)])
    st["ws"] = _workspace(*[op for three in st["ops"] for op in three])
    return st


def _run_train_block(st):
    (deep, deep_data, deep_filter), (point, point_data, point_filter) = st["ops"]
    ws = st["ws"]
    deep.enqueue(st["x"], st["wd"], st["bd"], st["t"], ws)
    point.enqueue(st["t"], st["wp"], st["bp"], st["y"], ws)
    point_filter.enqueue(st["t"], st["dwp"], st["dy"], ws)
    dlp.bias_backward(st["dy"], st["dbp"])
    point_data.enqueue(st["dt"], st["wp"], st["dy"], ws)
    deep_filter.enqueue(st["x"], st["dwd"], st["dt"], ws)
    dlp.bias_backward(st["dt"], st["dbd"])
    deep_data.enqueue(st["dx"], st["wd"], st["dt"], ws)
    return {n: st[n] for n in ("y", "dx", "dwd", "dbd", "dwp", "dbp")}


# ---- head: three fully connected layers, softmax, loss ----
def _prepare_head(case, seed, made):
    tdt, code = _types(case)
    b = case["batch"]
    sizes = [case["inputs"], case["hidden"], case["hidden"], CLASSES]
    st = dict(kind="head", x=made.activations(b, sizes[0], dtype=tdt), layers=[], prob=_empty(b, CLASSES, dtype=tdt), loss=_empty(1, dtype=tdt),
              labels=torch.randint(0, CLASSES, (b,), generator=made.gen, device=DEVICE, dtype=torch.int32))
    for i in range(3):
        op = dlp.IPForward.create(dlp.IPSettings(sizes[i], sizes[i + 1], b, dtype=code), True, "relu" if i < 2 else "identity")
        st["layers"].append((op, made.normal(sizes[i + 1], sizes[i], std=math.sqrt(2.0 / sizes[i]), dtype=tdt), made.bias(sizes[i + 1]), _empty(b, sizes[i + 1], dtype=tdt)))
    return st


def _run_head(st):
    t = st["x"]
    for op, w, bias, y in st["layers"]:
        op.enqueue(t, w, bias, y)
        t = y
    dlp.softmax_forward(t, st["prob"])
    dlp.softmax_loss_forward(t, st["labels"], st["loss"])
    return t, st["prob"], st["loss"]


# ---- decoder: transposed convolution, bilinear interpolation by two ----
def _prepare_decoder(case, seed, made):
    b, cin, cout, h, w, k = (case[n] for n in ("batch", "cin", "cout", "h", "w", "k"))
    oh, ow = _tconv_out(h, case), _tconv_out(w, case)
    op = dlp.TransposedConv2DForward.create(dlp.Conv2DSettings(cin, cout, k, case["s"], 1, case["p"], 1, (b, cin, h, w)), (case["op"], case["op"]), True, "relu")
    return dict(kind="decoder", op=op, x=made.activations(b, cin, h, w), w=made.normal(cin, cout, k, k, std=math.sqrt(2.0 * case["s"] ** 2 / (cin * k * k))), b=made.bias(cout),
                t=_empty(b, cout, oh, ow), y=_empty(b, cout, 2 * oh, 2 * ow), ws=_workspace(op))


def _run_decoder(st):
    st["op"].enqueue(st["x"], st["w"], st["b"], st["t"], st["ws"])
    dlp.interpolate2d_forward(st["t"], st["y"], "bilinear", 2.0, 2.0)
    return st["t"], st["y"]


# ---- what a pass cannot do without: every input read once, every output written once, every product of the definition ----
def work(case):
    e = 2 if case.get("dtype") == "bfloat16" else 4
    b = case["batch"]
    kind = case["kind"]
    if kind == "network":
        nbytes, flops, size = 3.0 * b * case["size"] ** 2 * e + b * CLASSES * e, 0.0, {"data": case["size"]}
        for o in getattr(graphs, case["net"])():
            src = o["src"] if isinstance(o["src"], str) else o["src"][0]
            if o["op"] == "conv":
                size[o["dst"]] = _out(size[src], o["k"], o["s"], o["p"])
                per = o["cin"] * o["k"] ** 2
                flops += 2.0 * b * o["cout"] * size[o["dst"]] ** 2 * per
                nbytes += o["cout"] * (per * e + 4)
            elif o["op"] == "maxpool":
                size[o["dst"]] = _out(size[src], o["k"], o["s"], o["p"])
            elif o["op"] == "ip":
                flops += 2.0 * b * o["inputs"] * o["outputs"]
                nbytes += o["outputs"] * (o["inputs"] * e + 4)
            else:
                size[o["dst"]] = size[src]
        return {"bytes": nbytes, "flops": flops}
    if kind == "train":
        oh, ow = (_out(case[n], case["k"], case["s"], case["p"], case["d"]) for n in ("h", "w"))
        per = case["cin"] // case["g"] * case["k"] ** 2
        x, y, w = b * case["cin"] * case["h"] * case["w"], b * case["cout"] * oh * ow, case["cout"] * per
        return {"bytes": 4.0 * (2 * x + 2 * y + 2 * w + 2 * case["cout"]), "flops": 6.0 * y * per + y}
    if kind == "block":
        oh, ow = _out(case["h"], 3, case["s"], 1), _out(case["w"], 3, case["s"], 1)
        t1, t2 = b * case["hidden"] * case["h"] * case["w"], b * case["hidden"] * oh * ow
        weights = case["hidden"] * (case["cin"] + 9 + case["cout"])
        return {"bytes": float(e * (b * case["cin"] * case["h"] * case["w"] + b * case["cout"] * oh * ow + weights) + 4 * (2 * case["hidden"] + case["cout"])),
                "flops": 2.0 * t1 * case["cin"] + 18.0 * t2 + 2.0 * t2 * case["cout"]}
    if kind == "train_block":
        oh, ow = _out(case["h"], 3, case["s"], 1), _out(case["w"], 3, case["s"], 1)
        x, t, y = b * case["c"] * case["h"] * case["w"], b * case["c"] * oh * ow, b * case["cout"] * oh * ow
        return {"bytes": 4.0 * (2 * x + 2 * y + 2 * case["c"] * (9 + case["cout"])), "flops": 54.0 * t + 6.0 * t * case["cout"] + t + y}
    if kind == "head":
        n = case["inputs"] * case["hidden"] + case["hidden"] ** 2 + case["hidden"] * CLASSES
        return {"bytes": float(e * (n + b * (case["inputs"] + 2 * CLASSES)) + 4 * b), "flops": 2.0 * b * n}
    oh, ow = _tconv_out(case["h"], case), _tconv_out(case["w"], case)
    x, t, w = b * case["cin"] * case["h"] * case["w"], b * case["cout"] * oh * ow, case["cin"] * case["cout"] * case["k"] ** 2
    return {"bytes": 4.0 * (x + w + t + 4 * t), "flops": 2.0 * x * case["cout"] * case["k"] ** 2 + 4.0 * t * 8}


def tolerance(case):
    # four times what the paths differ from a 64-bit evaluation of the same tensors, over the listed and some fifty drawn cases: float at most
    # 1.0e-6 (2-norm) and 8e-6 (single values), bfloat16 2.8e-3 and 1.1e-2 for the networks, 4.9e-3 and 1.3e-2 for the rest
    if case.get("dtype") == "bfloat16":
        return {"rel": 1.2e-2, "max": 5e-2} if case["kind"] == "network" else {"rel": 1.5e-2, "max": 6e-2}
    return {"rel": 4e-6, "max": 4e-5}


# ---- the same results in 64 bits, from torch alone ----
def _conv64(x, w, s=1, p=0, d=1, g=1):
    """convolution as one product of matrices per filter tap and group"""
    b, c, h, wd = x.shape
    cout, cin_g, k, _ = w.shape
    oh, ow = _out(h, k, s, p, d), _out(wd, k, s, p, d)
    x = torch.nn.functional.pad(x, (p, p, p, p))
    if cin_g == 1 and cout == g:
        y = torch.zeros((b, cout, oh, ow), dtype=x.dtype, device=x.device)
        for i in range(k):
            for j in range(k):
                y += w[:, 0, i, j].view(1, -1, 1, 1) * x[:, :, i * d:i * d + (oh - 1) * s + 1:s, j * d:j * d + (ow - 1) * s + 1:s]
        return y
    y = torch.zeros((b, g, cout // g, oh * ow), dtype=x.dtype, device=x.device)
    for i in range(k):
        for j in range(k):
            taps = x[:, :, i * d:i * d + (oh - 1) * s + 1:s, j * d:j * d + (ow - 1) * s + 1:s].reshape(b, g, cin_g, oh * ow)
            y += torch.matmul(w[:, :, i, j].reshape(1, g, cout // g, cin_g), taps)
    return y.view(b, cout, oh, ow)


def _conv64_gradients(x, w, dy, s, p, d=1, g=1):
    b, c, h, wd = x.shape
    cout, cin_g, k, _ = w.shape
    oh, ow = dy.shape[2:]
    x = torch.nn.functional.pad(x, (p, p, p, p))
    dx, dw = torch.zeros_like(x), torch.zeros_like(w)
    dyg = dy.reshape(b, g, cout // g, oh * ow)
    for i in range(k):
        for j in range(k):
            rows, cols = slice(i * d, i * d + (oh - 1) * s + 1, s), slice(j * d, j * d + (ow - 1) * s + 1, s)
            if cin_g == 1 and cout == g:
                dw[:, 0, i, j] = (x[:, :, rows, cols] * dy).sum((0, 2, 3))
                dx[:, :, rows, cols] += w[:, 0, i, j].view(1, -1, 1, 1) * dy
                continue
            taps = x[:, :, rows, cols].reshape(b, g, cin_g, oh * ow)
            dw[:, :, i, j] = torch.matmul(dyg, taps.transpose(2, 3).contiguous()).sum(0).reshape(cout, cin_g)
            wt = w[:, :, i, j].reshape(1, g, cout // g, cin_g).transpose(2, 3).contiguous()
            dx[:, :, rows, cols] += torch.matmul(wt, dyg).reshape(b, c, oh, ow)
    return dx[:, :, p:p + h, p:p + wd].contiguous(), dw


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    f64 = lambda n: st[n].double()
    chan = lambda t: t.double().view(1, -1, 1, 1)
    if kind == "network":
        runner = st["runner"]
        ops = getattr(graphs, case["net"])()
        parts = []
        for x in st["x"].split(8):
            t = {"data": x.double()}
            for o in ops:
                if o["op"] == "conv":
                    w, bias = runner.p[o["dst"]]
                    v = _conv64(t[o["src"]], w.double(), o["s"], o["p"]) + chan(bias)
                    t[o["dst"]] = v.relu() if o["act"] == "relu" else v
                elif o["op"] == "maxpool":
                    t[o["dst"]] = torch.nn.functional.max_pool2d(t[o["src"]], o["k"], o["s"], o["p"])
                elif o["op"] == "add":
                    t[o["dst"]] = (t[o["src"][0]] + t[o["src"][1]]).relu()
                elif o["op"] == "gap":
                    t[o["dst"]] = t[o["src"]].mean((2, 3))
                else:
                    w, bias = runner.p[o["dst"]]
                    t[o["dst"]] = t[o["src"]] @ w.double().t().contiguous() + bias.double()
            parts.append(t["logits"])
        return torch.cat(parts)
    if kind == "train":
        s, p, d, g = (case[n] for n in ("s", "p", "d", "g"))
        dx, dw = _conv64_gradients(f64("x"), f64("w"), f64("dy"), s, p, d, g)
        return {"y": _conv64(f64("x"), f64("w"), s, p, d, g) + chan(st["b"]), "dx": dx, "dw": dw, "db": f64("dy").sum((0, 2, 3))}
    if kind == "block":
        t = (_conv64(f64("x"), f64("w1")) + chan(st["b1"])).clamp(0, 6)
        t = (_conv64(t, f64("wd"), case["s"], 1, 1, case["hidden"]) + chan(st["bd"])).clamp(0, 6)
        y = _conv64(t, f64("w2")) + chan(st["b2"])
        return y + f64("x") if st["skip"] else y
    if kind == "train_block":
        c, s = case["c"], case["s"]
        t = _conv64(f64("x"), f64("wd"), s, 1, 1, c) + chan(st["bd"])
        dt, dwp = _conv64_gradients(t, f64("wp"), f64("dy"), 1, 0)
        dx, dwd = _conv64_gradients(f64("x"), f64("wd"), dt, s, 1, 1, c)
        return {"y": _conv64(t, f64("wp")) + chan(st["bp"]), "dx": dx, "dwd": dwd, "dbd": dt.sum((0, 2, 3)), "dwp": dwp, "dbp": f64("dy").sum((0, 2, 3))}
    if kind == "head":
        t = f64("x")
        for i, (_, w, bias, _) in enumerate(st["layers"]):
            t = t @ w.double().t().contiguous() + bias.double()
            t = t.relu() if i < 2 else t
        return t, torch.softmax(t, 1), torch.nn.functional.cross_entropy(t, st["labels"].long()).reshape(1)
    k, s, p = case["k"], case["s"], case["p"]
    x, w = f64("x"), f64("w")
    b, _, h, wd = x.shape
    oh, ow = _tconv_out(h, case), _tconv_out(wd, case)
    full = torch.zeros((b, case["cout"], max((h - 1) * s + k, oh + p), max((wd - 1) * s + k, ow + p)), dtype=x.dtype, device=x.device)
    for i in range(k):
        for j in range(k):
            tap = torch.matmul(w[:, :, i, j].t().contiguous().unsqueeze(0), x.reshape(b, -1, h * wd)).view(b, -1, h, wd)
            full[:, :, i:i + (h - 1) * s + 1:s, j:j + (wd - 1) * s + 1:s] += tap
    t = (full[:, :, p:p + oh, p:p + ow] + chan(st["b"])).relu()
    return t, torch.nn.functional.interpolate(t, scale_factor=2, mode="bilinear", align_corners=False)
