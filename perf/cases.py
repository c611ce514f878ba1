"""What an InferenceSession is asked to do in earnest, as cases that can be timed and compared.

A case is one compiled model and one batch.  The models are the four families
of rustgears_amd/configs.py:

  mlp    Linear -> BatchNorm -> ReLU, repeated, and a Linear head (the
         quickstart and the deep MLP)
  cnn    conv3x3 -> BatchNorm -> ReLU -> MaxPool(2), twice, Flatten,
         Linear -> ReLU, Linear
  stack  depth x (square Linear -> activation), the 4096-wide GELU stack
  gemv   Linear(d, h) -> SiLU -> Linear(h, d) on 1 to 8 rows, one decode step

in the three precisions a session can be built with: "i8" and "f16"
(ExecutionProvider.Mi355x) and "f32" (ExecutionProvider.Gpu).  Calls are
device-resident (`run_device` on buffers the program already holds) or, with
"host" set, `run` on host arrays with both copies.

A program loads its model once and then runs it on new inputs, so the weights
and the session belong to the case (prepare() keeps the one it made last) and
the seed makes the inputs.  Results are whole model outputs.
"""
import json
import math

import numpy as np
import torch

import rustgears_amd as rg
from rustgears_amd.inference import Activation, LayerSpec

_ACTS = {"gelu": Activation.GELU, "relu": Activation.RELU, "silu": Activation.SILU, "tanh": Activation.TANH,
         "sigmoid": Activation.SIGMOID}
_WEIGHT_BYTES = {"i8": 1, "f16": 2, "f32": 4}
_MODEL_KEYS = {
    "mlp": ("d_in", "hidden", "depth", "d_out"),
    "cnn": ("hw", "c1", "c2", "fc", "classes"),
    "stack": ("width", "depth", "act"),
    "gemv": ("d", "h"),
}


def _mlp(name, precision, rows, d_in, hidden, depth, d_out, host=False):
    return {"name": name, "model": "mlp", "precision": precision, "rows": rows, "host": host, "d_in": d_in,
            "hidden": hidden, "depth": depth, "d_out": d_out}


def _cnn(name, precision, rows, hw=32, c1=32, c2=64, fc=256, classes=10, host=False):
    return {"name": name, "model": "cnn", "precision": precision, "rows": rows, "host": host, "hw": hw, "c1": c1,
            "c2": c2, "fc": fc, "classes": classes}


def _stack(name, precision, rows, width, depth, act, host=False):
    return {"name": name, "model": "stack", "precision": precision, "rows": rows, "host": host, "width": width,
            "depth": depth, "act": act}


def _gemv(name, precision, rows, d, h, host=False):
    return {"name": name, "model": "gemv", "precision": precision, "rows": rows, "host": host, "d": d, "h": h}


def listed():
    return [
        # The quickstart example's model on its 64 rows: nothing but latency.
        _mlp("quickstart_i8", "i8", 64, 4, 32, 1, 3),
        # The deep MLP benchmark: a large batch through a narrow classifier.
        _mlp("mlp_i8_4096", "i8", 4096, 784, 1024, 2, 10),
        # The same model as a service meets it: an odd batch, binary16.
        _mlp("mlp_f16_1000", "f16", 1000, 784, 1024, 2, 10),
        # And in full precision, the reference everybody compares against.
        _mlp("mlp_f32_777", "f32", 777, 784, 1024, 2, 10),
        # The image classifier benchmark: one full batch.
        _cnn("cnn_i8_256", "i8", 256),
        # The classifier in binary16 on a batch that fills no power of two.
        _cnn("cnn_f16_100", "f16", 100),
        # The classifier as the reference's own run() is called: host tensor in, host tensor out.
        _cnn("cnn_i8_host_256", "i8", 256, host=True),
        # The headline benchmark: the 4096-wide GELU stack on 8192 rows, the largest call.
        _stack("stack_i8_8192", "i8", 8192, 4096, 4, "gelu"),
        # Two of its layers in binary16 on a ragged batch.
        _stack("stack_f16_3000", "f16", 3000, 4096, 2, "gelu"),
        # The stack behind a batching server: too many rows for a GEMV, too few to fill the chip with tiles.
        _stack("stack_i8_100", "i8", 100, 4096, 4, "gelu"),
        # The decode benchmark: one row through two 235 MB matrices.
        _gemv("gemv_i8_1", "i8", 1, 8192, 28672),
        # Decode for a few concurrent requests, binary16 weights.
        _gemv("gemv_f16_5", "f16", 5, 4096, 14336),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    precision = rng.choice(("i8", "i8", "i8", "f16", "f16", "f32"))
    host = rng.random() < 0.1
    model = rng.choice(("mlp", "cnn", "stack", "gemv"))
    if model == "mlp":
        case = _mlp("", precision, _log_int(rng, 1, 8192), _log_int(rng, 4, 2048), _log_int(rng, 16, 2048),
                    rng.randint(1, 3), _log_int(rng, 2, 1000), host)
    elif model == "cnn":
        case = _cnn("", precision, _log_int(rng, 1, 256), rng.randint(12, 48), _log_int(rng, 8, 64),
                    _log_int(rng, 16, 128), _log_int(rng, 32, 512), _log_int(rng, 2, 100), host)
    elif model == "stack":
        case = _stack("", precision, _log_int(rng, 9, 8192), _log_int(rng, 256, 4096), rng.randint(1, 4),
                      rng.choice(sorted(_ACTS)), host)
    else:
        case = _gemv("", precision, rng.randint(1, 8), _log_int(rng, 512, 8192), _log_int(rng, 1024, 28672), host)
    del case["name"]
    # The f32 and f16 matrix rates are a sixteenth and a half of the i8 one.
    most = 1.09e12 / {"i8": 1, "f16": 2, "f32": 16}[precision]
    while work(case)["flops"] > most:
        case["rows"] = case["rows"] * 2 // 3
    return case


# ---- the model: plain layers, from which both the session and exact() are built ----


def _uniform(g, shape, bound):
    return (torch.rand(shape, generator=g, device="cuda") * 2 - 1).mul_(bound).cpu().numpy()


def _linear(g, n_in, n_out, xavier=False):
    bound = math.sqrt(6.0 / (n_in + n_out if xavier else n_in))
    return ("linear", n_in, n_out, _uniform(g, (n_in, n_out), bound), _uniform(g, (n_out,), 1 / math.sqrt(n_in)))


def _conv(g, c_in, c_out):
    n = c_in * 9
    return ("conv", c_in, c_out, _uniform(g, (c_out, c_in, 3, 3), math.sqrt(6.0 / n)),
            _uniform(g, (c_out,), 1 / math.sqrt(n)))


def _batch_norm(g, n):
    mean = torch.randn(n, generator=g, device="cuda").mul(0.1)
    scale = torch.rsqrt(torch.rand(n, generator=g, device="cuda") + 0.5 + 1e-5)
    return ("affine", scale.cpu().numpy(), (-mean * scale).cpu().numpy())


def _layers(case):
    g = torch.Generator(device="cuda").manual_seed(42)
    if case["model"] == "mlp":
        out, n = [], case["d_in"]
        for _ in range(case["depth"]):
            out += [_linear(g, n, case["hidden"]), _batch_norm(g, case["hidden"]), ("act", "relu")]
            n = case["hidden"]
        return out + [_linear(g, n, case["d_out"])]
    if case["model"] == "cnn":
        c1, c2, flat = case["c1"], case["c2"], case["c2"] * (case["hw"] // 2 // 2) ** 2
        return [_conv(g, 3, c1), _batch_norm(g, c1), ("act", "relu"), ("pool",),
                _conv(g, c1, c2), _batch_norm(g, c2), ("act", "relu"), ("pool",), ("flatten",),
                _linear(g, flat, case["fc"]), ("act", "relu"), _linear(g, case["fc"], case["classes"])]
    if case["model"] == "stack":
        out = []
        for _ in range(case["depth"]):
            out += [_linear(g, case["width"], case["width"], xavier=True), ("act", case["act"])]
        return out
    return [_linear(g, case["d"], case["h"], xavier=True), ("act", "silu"),
            _linear(g, case["h"], case["d"], xavier=True)]


def _spec(layer):
    kind = layer[0]
    if kind == "linear":
        return LayerSpec.Linear(*layer[1:])
    if kind == "conv":
        return LayerSpec.Conv2d(layer[1], layer[2], 3, 1, 1, layer[3], layer[4])
    if kind == "affine":
        return LayerSpec.ChannelAffine(*layer[1:])
    if kind == "pool":
        return LayerSpec.MaxPool2d(2, 2)
    if kind == "flatten":
        return LayerSpec.Flatten()
    return LayerSpec.Activation(_ACTS[layer[1]])


_last = {}


def _session(case):
    """The case's session; the one made last is kept, as a program keeps its model."""
    key = json.dumps([case["model"], case["precision"]] + [case[k] for k in _MODEL_KEYS[case["model"]]])
    if key not in _last:
        _last.clear()
        provider = {"i8": rg.ExecutionProvider.mi355x_int8, "f16": rg.ExecutionProvider.mi355x_fp16,
                    "f32": rg.ExecutionProvider.Gpu}[case["precision"]]()
        _last[key] = rg.InferenceSession.from_layers([_spec(layer) for layer in _layers(case)], provider)
    return _last[key]


class _Buffer:
    """A device tensor as run_device takes it: its address and its size."""

    def __init__(self, t):
        self.tensor, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _in_shape(case):
    if case["model"] == "cnn":
        return (case["rows"], 3, case["hw"], case["hw"])
    return (case["rows"], case[{"mlp": "d_in", "stack": "width", "gemv": "d"}[case["model"]]])


def _out_shape(case):
    return (case["rows"], case[{"mlp": "d_out", "cnn": "classes", "stack": "width", "gemv": "d"}[case["model"]]])


def _input(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["model"] == "mlp":  # pixel values and other features scaled to 0..1
        return torch.rand(_in_shape(case), generator=g, device="cuda")
    return torch.randn(_in_shape(case), generator=g, device="cuda")  # normalised images, hidden states


def prepare(case, seed):
    session = _session(case)
    x = _input(case, seed)
    if case["host"]:
        return {"session": session, "x": x.cpu().numpy()}
    return {"session": session, "x": _Buffer(x), "shape": _in_shape(case),
            "y": _Buffer(torch.empty(_out_shape(case), device="cuda"))}


def run(state):
    if "y" not in state:
        return state["session"].run(state["x"])
    state["session"].run_device(state["x"], state["shape"], state["y"])
    return state["y"].tensor


def work(case):
    rows, wide = case["rows"], _WEIGHT_BYTES[case["precision"]]
    if case["model"] == "mlp":
        sizes = [(case["d_in"], case["hidden"])] + [(case["hidden"],) * 2] * (case["depth"] - 1)
        sizes += [(case["hidden"], case["d_out"])]
    elif case["model"] == "cnn":
        sizes = [(case["c2"] * (case["hw"] // 2 // 2) ** 2, case["fc"]), (case["fc"], case["classes"])]
    elif case["model"] == "stack":
        sizes = [(case["width"],) * 2] * case["depth"]
    else:
        sizes = [(case["d"], case["h"]), (case["h"], case["d"])]
    macs = sum(a * b for a, b in sizes) * rows
    moved = sum(a * b * wide + 4 * b for a, b in sizes)
    if case["model"] == "cnn":
        hw, c1, c2 = case["hw"], case["c1"], case["c2"]
        macs += rows * (27 * c1 * hw * hw + 9 * c1 * c2 * (hw // 2) ** 2)
        moved += wide * (27 * c1 + 9 * c1 * c2) + 4 * (c1 + c2)
    return {"bytes": moved + 4 * (math.prod(_in_shape(case)) + math.prod(_out_shape(case))), "flops": 2 * macs}


def tolerance(case):
    # The INT8 provider's contract is the reference's bits: integer sums, one
    # f32 rounding per step in a fixed order.  The others sum in f32 in any
    # order; f16 rounds every layer's sum to binary16 besides, where another
    # order moves a value by a unit in the last place now and then.  Against
    # exact() the listed and some drawn cases differ by up to 2.2e-4 (f16) and
    # 4.1e-7 (f32); the limits are about four times that.
    if case["precision"] == "i8":
        return "exact"
    return {"rel": 8e-4, "max": 2e-2} if case["precision"] == "f16" else {"rel": 2e-6, "max": 1e-4}


# ---- the same models in 64 bits ----


def _half_away(v):
    return torch.sign(v) * torch.floor(torch.abs(v) + 0.5)


def _binary16(v):
    """Nearest value of 11 significant bits, ties away from zero; below the normal range 0, above it the largest."""
    e = torch.frexp(v)[1] - 11
    r = torch.ldexp(_half_away(torch.ldexp(v, -e)), e)
    r = torch.where(torch.abs(v) < 2.0 ** -14, torch.zeros_like(r), r)
    return torch.clamp(r, -65504.0, 65504.0)


def _quantized(v, per_image=False):
    """(whole values, scale): one symmetric 8-bit scale per tensor, or one per image."""
    most = v.abs().amax(dim=tuple(range(1, v.dim())), keepdim=True) if per_image else v.abs().max()
    scale = most / 127
    return torch.clamp(_half_away(v / scale), -127, 127), scale


def _operand(v, precision, per_image=False):
    if precision == "i8":
        return _quantized(v, per_image)
    return (_binary16(v) if precision == "f16" else v), 1.0


def _act64(v, act):
    if act == "relu":
        return torch.relu(v)
    if act == "gelu":
        return 0.5 * v * (1 + torch.tanh(0.7978846 * (v + 0.044715 * v ** 3)))
    if act == "silu":
        return v * torch.sigmoid(v)
    return torch.tanh(v) if act == "tanh" else torch.sigmoid(v)


def exact(case, seed):
    precision, v = case["precision"], _input(case, seed).double()
    layers = [list(layer) for layer in _layers(case)]
    for i, layer in enumerate(layers):
        if layer[0] in ("linear", "conv"):
            w = torch.from_numpy(layer[3]).cuda().double()
            w = w.t() if layer[0] == "linear" else w.reshape(layer[2], -1)
            b = torch.from_numpy(layer[4]).cuda().double()
            if i + 1 < len(layers) and layers[i + 1][0] == "affine":
                scale, shift = (torch.from_numpy(t).cuda().double() for t in layers[i + 1][1:])
                w, b = w * scale[:, None], b * scale + shift
            w, w_scale = _operand(w, precision)
            x, x_scale = _operand(v, precision, per_image=layer[0] == "conv")
            if layer[0] == "linear":
                v = torch.matmul(x, w.t()) * (x_scale * w_scale) + b
            else:
                n, _, h, width = x.shape
                cols = torch.nn.functional.unfold(x, 3, padding=1)
                v = torch.matmul(w, cols).reshape(n, -1, h, width) * (x_scale * w_scale) + b[:, None, None]
            if precision == "f16":
                v = _binary16(v)
        elif layer[0] == "act":
            v = _act64(v, layer[1])
        elif layer[0] == "pool":
            n, c, h, width = v.shape
            v = v[:, :, :h // 2 * 2, :width // 2 * 2].reshape(n, c, h // 2, 2, width // 2, 2).amax(dim=(3, 5))
        elif layer[0] == "flatten":
            v = v.reshape(v.shape[0], -1)
    return v.cpu().numpy() if case["host"] else v
