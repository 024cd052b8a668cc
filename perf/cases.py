"""The work whose speed counts in this library, through its public entry points (mindspore_amd/kernels.py).

Six kinds of case, each over the sizes it is used at:
  fc        one FullConnection / MatMul on device tensors, int8 in and out
  layer     the MatMuls of one transformer layer: QKV, output projection, the feed-forward pair (gated: gate and up,
            which share their input, as a group) and the down projection.  rows is the batch of a decode step, the
            length of a prompt, or all tokens of an encoder batch.  quant says how activations are quantised:
              static   full-quant int8 in and out, parameters fixed in the model
              tensor   DynamicQuant per tensor, its parameters handed on in device memory
              fetched  DynamicQuant per tensor, its parameters fetched to the host and passed by value
              row      DynamicQuant with one scale per row
  block     inverted-residual image block (configuration 2): strided stem on three channels, 1x1 expand, depthwise,
            1x1 project, each layer reading what the one before it wrote
  residual  residual-network stage: 7x7 stem on the image, then at a quarter of its extent a 3x3, a strided 3x3 and
            a strided 1x1 shortcut
  host      one FullConnection on host (NumPy) tensors, as a CPU-arch provider kernel receives them
Weights, bias and quant parameters go into the kernel objects in prepare(), as a program does once when it loads its
model; run() is what it does for every input.
"""
import math

import numpy as np
import torch

from mindspore_amd import kernels as K

QP = K.QuantParam


def listed():
    return [
        # the smallest call in common use: one FullConnection of a small encoder at batch 1 (configuration 1)
        dict(name="fc_128x768", kind="fc", rows=128, k=768, n=768, zw=False, act=0),
        # a classifier head with nothing aligned: K % 16 != 0, N % 4 != 0, asymmetric weights
        dict(name="fc_ragged", kind="fc", rows=333, k=1000, n=1001, zw=True, act=1),
        # the headline GEMM (configuration 5)
        dict(name="fc_4096", kind="fc", rows=4096, k=4096, n=4096, zw=False, act=0),
        # one decode step of one sequence (configuration 4)
        dict(name="decode_1", kind="layer", rows=1, hidden=4096, ffn=11008, gated=True, quant="static"),
        # one decode step of a small serving batch, activations quantised on the fly
        dict(name="decode_8_dynamic", kind="layer", rows=8, hidden=4096, ffn=11008, gated=True, quant="tensor"),
        # an ordinary prompt
        dict(name="prefill_512", kind="layer", rows=512, hidden=4096, ffn=11008, gated=True, quant="static"),
        # a long prompt with one activation scale per token: the most work of all
        dict(name="prefill_2048_rows", kind="layer", rows=2048, hidden=4096, ffn=11008, gated=True, quant="row"),
        # encoder batch (configuration 3)
        dict(name="encoder_4096", kind="layer", rows=4096, hidden=768, ffn=3072, gated=False, quant="tensor"),
        # one sentence through the same encoder, parameters by value as the reference's kernels pass them
        dict(name="encoder_197", kind="layer", rows=197, hidden=768, ffn=3072, gated=False, quant="fetched"),
        # one image (configuration 2)
        dict(name="block_1x224", kind="block", batch=1, image=224, stem=32, expand=6, taps=3),
        # a batch of images
        dict(name="residual_32x224", kind="residual", batch=32, image=224, channels=64),
        # host tensors in and out
        dict(name="host_1024", kind="host", rows=1024, k=4096, n=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi):
    """An extent between lo and hi: three in four a multiple of 16, as most models have them, the others anything."""
    x = _log_int(rng, lo, hi)
    return max(lo, x // 16 * 16) if rng.random() < 0.75 else x


def draw(rng):
    kind = rng.choice(["fc", "fc", "decode", "decode", "prefill", "prefill", "encoder", "block", "residual", "host"])
    if kind == "fc":
        while True:
            rows, k, n = _log_int(rng, 1, 8192), _extent(rng, 64, 8192), _extent(rng, 64, 8192)
            if rows * k * n <= 1 << 37:
                return dict(kind="fc", rows=rows, k=k, n=n, zw=rng.random() < 0.25, act=rng.choice([0, 1, 3]))
    if kind in ("decode", "prefill"):
        hidden = 128 * _log_int(rng, 8, 32)
        rows = _log_int(rng, 1, 64) if kind == "decode" else _log_int(rng, 65, 2048)
        return dict(kind="layer", rows=rows, hidden=hidden, ffn=_extent(rng, 2 * hidden, int(2.68 * hidden)), gated=True,
                    quant=rng.choice(["static", "static", "tensor", "fetched", "row"]))
    if kind == "encoder":
        hidden = 64 * _log_int(rng, 4, 24)
        return dict(kind="layer", rows=_log_int(rng, 16, 6144), hidden=hidden, ffn=4 * hidden, gated=False,
                    quant=rng.choice(["static", "tensor", "fetched", "row"]))
    if kind == "block":
        return dict(kind="block", batch=_log_int(rng, 1, 32), image=rng.randint(96, 256), stem=8 * rng.randint(2, 5),
                    expand=rng.choice([3, 4, 6]), taps=rng.choice([3, 3, 5]))
    if kind == "residual":
        return dict(kind="residual", batch=_log_int(rng, 1, 32), image=rng.randint(112, 256),
                    channels=16 * rng.randint(2, 6))
    return dict(kind="host", rows=_log_int(rng, 1, 2048), k=_extent(rng, 256, 4096), n=_extent(rng, 256, 4096))


# ---- shapes of what a case holds ------------------------------------------------------------------------------------

def _matmuls(case):
    """The layer's MatMuls as (name, N, K), grouped by the input they share."""
    h, f = case["hidden"], case["ffn"]
    up = [("gate", f, h), ("up", f, h)] if case["gated"] else [("up", f, h)]
    return [[("qkv", 3 * h, h)], [("out", h, h)], up, [("down", h, f)]]


def _out(extent, taps, stride, pad_before, pad_after):
    return (extent + pad_before + pad_after - taps) // stride + 1


def _convs(case):
    """The convolutions of a block or stage: dicts of input, channels, taps, stride, pad and output extent."""
    if case["kind"] == "block":
        b, i, c, t = case["batch"], case["image"], case["stem"], case["taps"]
        o = _out(i, 3, 2, 0, 1)
        mid = c * case["expand"]
        spec = [(i, 3, c, 3, 2, (0, 1, 0, 1), False, 3), (o, c, mid, 1, 1, (0,) * 4, False, 3),
                (o, mid, mid, t, 1, (t // 2,) * 4, True, 3), (o, mid, c, 1, 1, (0,) * 4, False, 0)]
    else:
        b, i, c = case["batch"], case["image"], case["channels"]
        q = i // 4
        spec = [(i, 3, c, 7, 2, (3,) * 4, False, 1), (q, c, c, 3, 1, (1,) * 4, False, 1),
                (q, c, 2 * c, 3, 2, (1,) * 4, False, 1), (q, c, 2 * c, 1, 2, (0,) * 4, False, 0)]
    return [dict(batch=b, size=s, ic=ic, oc=oc, taps=t, stride=st, pad=p, dw=dw, act=act,
                 out=_out(s, t, st, p[0], p[1])) for s, ic, oc, t, st, p, dw, act in spec]


# ---- inputs ---------------------------------------------------------------------------------------------------------

class _Random:
    def __init__(self, seed):
        self.gpu = torch.Generator(device="cuda")
        self.gpu.manual_seed(seed)
        self.host = np.random.default_rng(seed)

    def int8(self, *shape):  # uniform, as in configurations 1, 2 and 5
        return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=self.gpu)

    def weight(self, *shape):  # bell-shaped, as in configuration 4
        x = torch.randn(shape, dtype=torch.float32, device="cuda", generator=self.gpu)
        return x.mul_(32.0).round_().clamp_(-127.0, 127.0).to(torch.int8)

    def activation(self, *shape):  # normal with one value in a hundred at +-8, as in configuration 3
        x = torch.randn(shape, dtype=torch.float32, device="cuda", generator=self.gpu)
        u = torch.rand(shape, dtype=torch.float32, device="cuda", generator=self.gpu)
        return torch.where(u < 0.01, x.sign() * 8.0, x)

    def channel_scales(self, n):
        return self.host.uniform(0.001, 0.01, n).astype(np.float32).astype(np.float64)

    def bias(self, n):
        return self.host.integers(-5000, 5001, n).astype(np.int32)


def _int8_matmul(r, weight, act=0, zw=False, zx=7):
    """A full-quant MatMul against `weight` [N, K] whose outputs spread over the int8 range."""
    n, k = weight.shape
    sw = r.channel_scales(n)
    zps = r.host.integers(-8, 9, n) if zw else np.zeros(n, np.int64)
    spread = float(weight[: min(n, 256)].float().std())
    so = float(np.float32(0.02 * float(np.mean(sw)) * math.sqrt(k) * 74.0 * spread / 40.0))
    return K.MatmulInt8Kernel(weight.cpu().numpy(), r.bias(n), QP(0.02, zx), [QP(float(s), int(z)) for s, z in zip(sw, zps)],
                              QP(so, 0), True, act)


def _dynamic_matmul(r, weight):
    n, _ = weight.shape
    return K.MatmulDynamicInt8Kernel(weight.cpu().numpy(), (r.host.standard_normal(n) * 0.1).astype(np.float32),
                                     [QP(float(s), 0) for s in r.channel_scales(n)])


def _conv(r, c, sx, zx):
    """Returns the kernel and the quantisation of its output (a ReLU6 bound inside the int8 range)."""
    shape = (c["oc"], c["taps"], c["taps"]) if c["dw"] else (c["oc"], c["taps"], c["taps"], c["ic"])
    w, sw = r.int8(*shape).cpu().numpy(), r.channel_scales(c["oc"])
    depth = c["taps"] ** 2 * (1 if c["dw"] else c["ic"])
    so = 6.0 / 140.0 if c["act"] == 3 else float(np.float32(sx * float(np.mean(sw)) * math.sqrt(depth) * 74.0 * 2.0))
    zo = int(r.host.integers(-20, 21))
    kern = K.ConvolutionInt8Kernel(w, r.bias(c["oc"]), QP(sx, zx), [QP(float(s), 0) for s in sw], QP(so, zo),
                                   (c["stride"],) * 2, (1, 1), c["pad"], c["oc"] if c["dw"] else 1, c["act"],
                                   exact_3x3=True)
    return kern, so, zo


def prepare(case, seed):
    r = _Random(seed)
    state = dict(case=case)
    if case["kind"] in ("fc", "host"):
        state["kernel"] = _int8_matmul(r, r.int8(case["n"], case["k"]), case.get("act", 0), case.get("zw", False))
        x = r.int8(case["rows"], case["k"])
        state["x"] = x.cpu().numpy() if case["kind"] == "host" else x
    elif case["kind"] == "layer":
        make = _int8_matmul if case["quant"] == "static" else _dynamic_matmul
        value = r.int8 if case["quant"] == "static" else r.activation
        state["steps"] = []
        for group in _matmuls(case):
            kernels = [make(r, r.weight(n, k)) for _, n, k in group]
            quant = None if case["quant"] == "static" else K.DynamicQuantKernel(case["quant"] == "row")
            state["steps"].append((quant, kernels, value(case["rows"], group[0][2])))
    else:
        sx, zx = 0.02, int(r.host.integers(-20, 21))
        convs = _convs(case)
        first = convs[0]
        state["x"] = r.int8(first["batch"], first["size"], first["size"], first["ic"])
        if case["kind"] == "residual":  # what the pooled stem hands on
            state["y"] = r.int8(first["batch"], convs[1]["size"], convs[1]["size"], convs[1]["ic"])
        state["kernels"] = []
        for c in convs:
            kern, so, zo = _conv(r, c, sx, zx)
            state["kernels"].append(kern)
            if case["kind"] == "block":
                sx, zx = so, zo
    return state


# ---- one pass -------------------------------------------------------------------------------------------------------

def _run_static(kernels, x):
    return K.matmul_run_group(kernels, x) if len(kernels) > 1 else [kernels[0].run(x)]


def _run_dynamic(quant, kernels, x, how):
    if how == "row":
        q, params = quant.run_rows(x)
        given = dict(row_params=params)
    elif how == "tensor":
        q, _ = quant.run(x, fetch_params=False)
        given = dict(params_dev=quant.device_params())
    else:
        q, param = quant.run(x)
        given = dict(in_quant=param)
    if len(kernels) > 1:
        return [q] + K.dynmm_run_group(kernels, q, **given)
    return [q, kernels[0].run(q, **given)]


def run(state):
    case = state["case"]
    if case["kind"] in ("fc", "host"):
        return state["kernel"].run(state["x"])
    if case["kind"] == "layer":
        outs = []
        for quant, kernels, x in state["steps"]:
            outs += _run_static(kernels, x) if quant is None else _run_dynamic(quant, kernels, x, case["quant"])
        return outs
    if case["kind"] == "block":
        outs, cur = [], state["x"]
        for kern in state["kernels"]:
            cur = kern.run(cur)
            outs.append(cur)
        return outs
    stem, *rest = state["kernels"]
    return [stem.run(state["x"])] + [kern.run(state["y"]) for kern in rest]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def work(case):
    """Every input and weight read once, every output written once (16 bytes of parameters per channel); two operations
    per multiply-add."""
    if case["kind"] in ("fc", "host"):
        m, k, n = case["rows"], case["k"], case["n"]
        return dict(bytes=m * k + n * k + m * n + 16 * n, flops=2 * m * n * k)
    total = dict(bytes=0, flops=0)
    if case["kind"] == "layer":
        m = case["rows"]
        for group in _matmuls(case):
            k = group[0][2]
            # a dynamically quantised input is read as fp32, written as int8 (it is an output) and read again
            total["bytes"] += m * k if case["quant"] == "static" else 6 * m * k
            for _, n, _ in group:
                total["bytes"] += n * k + 16 * n + m * n * (1 if case["quant"] == "static" else 4)
                total["flops"] += 2 * m * n * k
        return total
    convs = _convs(case)
    for i, c in enumerate(convs):
        depth = c["taps"] ** 2 * (1 if c["dw"] else c["ic"])
        pixels = c["batch"] * c["out"] ** 2
        total["bytes"] += pixels * c["oc"] + c["oc"] * (depth + 16)
        if case["kind"] == "block" or i < 2:  # (the residual stage's three convolutions share one input)
            total["bytes"] += c["batch"] * c["size"] ** 2 * c["ic"]
        total["flops"] += 2 * pixels * c["oc"] * depth
    return total


def tolerance(case):
    """int8 results are integer arithmetic; fp32 results are an exact integer sum put through a fixed sequence of
    separately rounded products and sums.  Nothing is left to an implementation's choice."""
    return "exact"
