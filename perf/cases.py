"""Timing cases: the work a program built on this package has it do, through the public entry points.

Kinds of case (``"kind"``):

``mm``      the drop-in ``int8mm_cuda.int8_mm``: int8 x int8 -> int32, operands row-major, any extents
``sp_conv`` the drop-in ``cutlassconv_cuda.sp_conv``: int8 convolution with int32 result, any filter, stride and padding
``linear``  one ``TiLinear`` layer: forward, then backward (data gradient, weight gradient, update of the weights)
``conv``    one ``TiConv2d`` layer: forward, then backward
``pool``    one ``TiMaxpool2d`` layer: forward, then backward
``eval``    a ``TiVGG_cifar`` network in evaluation: float images -> logits
``train``   a training step of such a network: float images -> loss gradient -> updated weights; ``graph`` says whether
            the step runs through ``train.StepGraph`` (what the epoch driver does by default) or layer by layer

Everything the entry points return is integer and exactly defined, except the display metrics of ``train.StepGraph``."""
import math

import torch

from niti_amd import ti_torch, train
from niti_amd.shims import cutlassconv_cuda, int8mm_cuda
from niti_amd.ti_vgg import TiVGG_cifar, cifar_cfg

DEVICE = "cuda"


def listed():
    return [
        # the last product of a small classifier, the shortest call there is: launch latency and host cost
        {"name": "mm_small", "kind": "mm", "m": 16, "k": 512, "n": 10},
        # a product none of whose extents fits a tile or a 16-byte row
        {"name": "mm_ragged", "kind": "mm", "m": 333, "k": 1000, "n": 777},
        # the wide fully connected layer, every rounding stochastic on supplied integers
        {"name": "linear_fc", "kind": "linear", "n": 128, "f": 8192, "o": 1024, "rounding": "sto"},
        # a hidden layer whose widths and batch are no multiples of anything, the default roundings
        {"name": "linear_ragged", "kind": "linear", "n": 100, "f": 1000, "o": 300, "rounding": "default"},
        # BASELINE configs[0] as a layer: the second convolution of the VGG stack at batch 128
        {"name": "conv_vgg", "kind": "conv", "n": 128, "h": 32, "w": 32, "c": 128, "k": 128, "filter": 3},
        # an odd batch on a map that is no power of two, widths between the tile sizes
        {"name": "conv_ragged", "kind": "conv", "n": 37, "h": 14, "w": 14, "c": 96, "k": 160, "filter": 3},
        # a down-sampling convolution through the drop-in extension
        {"name": "sp_conv_stride2", "kind": "sp_conv", "n": 50, "h": 28, "w": 28, "c": 64, "k": 128, "filter": 3, "stride": 2, "padding": 1},
        # the first pooling of the VGG stack at batch 128
        {"name": "pool_vgg", "kind": "pool", "n": 128, "h": 32, "w": 32, "c": 128, "window": 2},
        # one image through the network: serving, where every launch counts
        {"name": "eval_one", "kind": "eval", "depth": 7, "n": 1},
        # the last batch of an epoch (50000 mod 256 = 80 images), stepped layer by layer
        {"name": "train_tail", "kind": "train", "depth": 7, "n": 80, "graph": False},
        # VGG-small at batch 128, as the epoch driver runs it
        {"name": "train_vgg7", "kind": "train", "depth": 7, "n": 128, "graph": True},
        # the deepest network of the reference at its default batch
        {"name": "train_vgg9", "kind": "train", "depth": 9, "n": 256, "graph": True},
    ]


def _log(rng, lo, hi):
    """Uniform over the logarithm, any whole number."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A channel count: a multiple of 16 (every layer's kernels work on 16-channel groups of int8)."""
    return 16 * _log(rng, lo // 16, hi // 16)


def _draw_any(rng):
    kind = rng.choice(["mm", "mm", "linear", "linear", "conv", "conv", "sp_conv", "pool", "eval", "eval", "train", "train", "train"])
    if kind == "mm":
        return {"kind": kind, "m": _log(rng, 1, 2048), "k": _log(rng, 16, 8192), "n": _log(rng, 1, 4096)}
    if kind == "linear":
        return {"kind": kind, "n": _log(rng, 1, 1024), "f": _log(rng, 32, 8192), "o": _log(rng, 2, 2048),
                "rounding": rng.choice(["default", "sto"])}
    if kind == "conv":
        h = _log(rng, 4, 48)
        w = h if rng.random() < 0.75 else _log(rng, 4, 48)
        return {"kind": kind, "n": _log(rng, 1, 256), "h": h, "w": w, "c": _width(rng, 16, 512), "k": _width(rng, 16, 512),
                "filter": rng.choice([1, 3, 3, 3, 5])}
    if kind == "sp_conv":
        h = _log(rng, 7, 64)
        f = rng.choice([1, 3, 3, 5])
        return {"kind": kind, "n": _log(rng, 1, 256), "h": h, "w": h, "c": _width(rng, 16, 512), "k": _log(rng, 16, 512), "filter": f,
                "stride": rng.choice([1, 2]), "padding": rng.choice([0, f // 2])}
    if kind == "pool":
        h = _log(rng, 4, 64)
        return {"kind": kind, "n": _log(rng, 1, 256), "h": h, "w": h, "c": _width(rng, 16, 512), "window": rng.choice([2, 2, 3])}
    if kind == "eval":
        return {"kind": kind, "depth": rng.choice(sorted(cifar_cfg)), "n": _log(rng, 1, 512)}
    return {"kind": kind, "depth": rng.choice(sorted(cifar_cfg)), "n": _log(rng, 8, 256), "graph": rng.choice([False, True])}


def draw(rng):
    # no drawn case is larger than the largest listed one; single layers and products stay at a quarter of a network's work
    top = work(listed()[-1])["flops"]
    while True:
        case = _draw_any(rng)
        w = work(case)
        if w["flops"] <= (top if case["kind"] in ("eval", "train") else top / 4) and w["bytes"] <= 400e6:
            return case


# ------------------------------------------------------------------------------------------------------------------
def _uniform(g, *shape):
    return torch.randint(-127, 128, shape, generator=g, dtype=torch.int8, device=DEVICE)


def _errors(g, *shape):
    """Errors as back-propagation delivers them: Laplace-distributed around zero."""
    u = torch.rand(shape, generator=g, device=DEVICE) - 0.5
    return (-16.0 * torch.sign(u) * torch.log1p(-2.0 * u.abs().clamp(max=0.499999))).round_().clamp_(-127, 127).to(torch.int8)


def _random_integers(g, *shape):
    return torch.randint(0, 1 << 20, shape, generator=g, dtype=torch.int32, device=DEVICE)


def _settings(training, rounding="default"):
    ti_torch.TRAINING = training
    ti_torch.GRAD_BITWIDTH = 5
    sto = rounding == "sto"
    ti_torch.ACT_ROUND_METHOD = ti_torch.StoShift if sto else ti_torch.RoundShift
    ti_torch.ERROR_ROUND_METHOD = ti_torch.StoShift if sto else ti_torch.RoundShift
    ti_torch.GRAD_ROUND_METHOD = ti_torch.StoShift if sto else ti_torch.PstoShift


def _out_side(size, case):
    return (size + 2 * case["padding"] - case["filter"]) // case["stride"] + 1


def prepare(case, seed):
    torch.manual_seed(seed)
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind == "mm":
        return {"kind": kind, "lhs": _uniform(g, case["m"], case["k"]), "rhs": _uniform(g, case["k"], case["n"])}
    if kind == "sp_conv":
        return {"kind": kind, "x": _uniform(g, case["n"], case["h"], case["w"], case["c"]),
                "w": _uniform(g, case["k"], case["filter"], case["filter"], case["c"]), "stride": case["stride"], "padding": case["padding"]}
    if kind == "linear":
        _settings(True, case["rounding"])
        n, f, o = case["n"], case["f"], case["o"]
        state = {"kind": kind, "layer": ti_torch.TiLinear(f, o), "x": _uniform(g, n, f), "err": _errors(g, n, o), "rand": (None, None, None)}
        if case["rounding"] == "sto":
            state["rand"] = (_random_integers(g, n, o), _random_integers(g, n, f), _random_integers(g, o, f))
        return state
    if kind == "conv":
        _settings(True)
        f = case["filter"]
        return {"kind": kind, "layer": ti_torch.TiConv2d(case["c"], case["k"], kernel_size=f, stride=1, padding=f // 2),
                "x": _uniform(g, case["n"], case["h"], case["w"], case["c"]), "err": _errors(g, case["n"], case["h"], case["w"], case["k"])}
    if kind == "pool":
        _settings(True)
        pad = case["window"] // 3
        p, q = ((case[s] + 2 * pad - case["window"]) // 2 + 1 for s in ("h", "w"))
        return {"kind": kind, "layer": ti_torch.TiMaxpool2d(case["window"], 2, pad), "x": _uniform(g, case["n"], case["h"], case["w"], case["c"]),
                "err": _errors(g, case["n"], p, q, case["c"])}
    x = torch.randn((case["n"], 3, 32, 32), generator=g, device=DEVICE)
    net = TiVGG_cifar(case["depth"])
    if kind == "eval":
        _settings(False)
        return {"kind": kind, "net": net, "x": x}
    _settings(True)
    target = torch.randint(0, 10, (case["n"],), generator=g, device=DEVICE)
    state = {"kind": kind, "net": net, "x": x, "target": target, "runner": None}
    if case["graph"]:
        # the epoch driver's runner: the first steps of a training run are eager, then the step is captured
        state["runner"] = train.StepGraph(net, True, x, target)
        state["sums"] = torch.zeros(3, dtype=torch.float64, device=DEVICE)
        for _ in range(5):
            state["runner"](x, target, state["sums"])
    else:
        net(x, target)
        net.backward(target)
    return state


def run(state):
    kind = state["kind"]
    if kind == "mm":
        return int8mm_cuda.int8_mm(state["lhs"], state["rhs"])
    if kind == "sp_conv":
        return cutlassconv_cuda.sp_conv(state["x"], state["w"], state["stride"], state["padding"])
    if kind == "linear":
        layer = state["layer"]
        fwd, err, grad = state["rand"]
        y, y_exp = layer.forward((state["x"], 0), rand=fwd)
        dx, dx_exp = layer.backward((state["err"], -4), rand=err, grad_rand=grad)
        return y, y_exp, dx, dx_exp, layer.weight
    if kind == "conv":
        layer = state["layer"]
        y, y_exp = layer.forward((state["x"], 0))
        dx, dx_exp = layer.backward((state["err"], -4))
        return y, y_exp, dx, dx_exp, layer.weight
    if kind == "pool":
        layer = state["layer"]
        y, _ = layer.forward((state["x"], 0))
        dx, _ = layer.backward((state["err"], -4))
        return y, dx
    net = state["net"]
    if kind == "eval":
        return net(state["x"])
    if state["runner"] is not None:
        state["runner"](state["x"], state["target"], state["sums"])
        return [net.out, net.out_exp, state["sums"]] + _weights(net)
    out, out_exp = net(state["x"], state["target"])
    net.backward(state["target"])
    return [out, out_exp] + _weights(net)


def _weights(net):
    return [layer.weight for layer in net.forward_layers if hasattr(layer, "weight")]


# ------------------------------------------------------------------------------------------------------------------
def _net_layers(depth):
    """(map side, input channels, filters) of the convolutions, (features, outputs) of the classifier."""
    side, c, convs = 32, 3, []
    for v in cifar_cfg[depth]:
        if v == "M":
            side //= 2
        else:
            convs.append((side, c, v))
            c = v
    return convs, (c * side * side, 10)


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "mm":
        m, k = case["m"], case["k"]
        return {"bytes": m * k + k * n + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "sp_conv":
        out = n * _out_side(case["h"], case) * _out_side(case["w"], case) * case["k"]
        taps = case["filter"] ** 2 * case["c"]
        return {"bytes": n * case["h"] * case["w"] * case["c"] + case["k"] * taps + 4 * out, "flops": 2 * out * taps}
    if kind == "linear":
        f, o = case["f"], case["o"]
        values = n * f + o * f + n * o       # activations, weights, errors in; as many results out; a random integer for each result
        return {"bytes": values * (6 if case["rounding"] == "sto" else 2), "flops": 6 * n * f * o}
    if kind == "conv":
        pixels, filters = n * case["h"] * case["w"], case["k"] * case["filter"] ** 2 * case["c"]
        return {"bytes": 2 * (pixels * (case["c"] + case["k"]) + filters), "flops": 6 * pixels * filters}
    if kind == "pool":
        big = n * case["h"] * case["w"] * case["c"]
        return {"bytes": 2 * (big + big // 4), "flops": 0}
    convs, (f, o) = _net_layers(case["depth"])
    weights = sum(9 * c * k for _, c, k in convs) + f * o
    forward = [2 * n * s * s * 9 * c * k for s, c, k in convs] + [2 * n * f * o]
    images = 4 * n * 3 * 32 * 32
    if kind == "eval":
        return {"bytes": images + weights + n * o, "flops": sum(forward)}
    # the first layer has no data gradient
    return {"bytes": images + 2 * weights + n * o, "flops": 3 * sum(forward) - forward[0]}


def tolerance(case):
    if case["kind"] == "train" and case["graph"]:
        # float32 display loss and accuracy summed in float64; every integer result exact
        return {"rel": 1e-5, "differ": 0.0}
    return "exact"

