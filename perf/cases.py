"""Performance cases: training and inference work on the xdna device, through the entry points a user calls.

Single layers and blocks at the sizes of the repository's workloads (the 3x3 conv sweep, the one-layer conv step, the
MLP, ResNet-18, the style-transfer network and its perceptual loss), ragged sizes beside them, and one whole forward.
Layers whose kernels are long run eagerly, as a training script calls them; chains of short kernels run as a captured
graph's replay, with the batch copied into the graph's input first, as a training loop does.

A case is a dict: "kind" says which of the builders below takes it, the rest are its sizes and options.
"""
import math
import sys
from pathlib import Path

import torch
from torch import nn
from torch.nn import functional as F

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "pytorch-xdna2_amd"))

import xdna_train  # noqa: E402,F401  (registers the device)
from xdna_train import regions  # noqa: E402

XDNA = "xdna"
BF16 = torch.bfloat16


def listed():
    return [
        # the whole training step of one conv layer (conv, MSE, Adam) as a captured step: what a small model's step costs
        {"name": "conv step 128ch B16 36x36", "kind": "conv_step", "n": 16, "c": 128, "h": 36, "w": 36},
        # a layer of a small custom net, called eagerly: odd sizes everywhere, nothing a multiple of a tile
        {"name": "conv ragged 48-80 B7 29x43", "kind": "conv", "n": 7, "cin": 48, "cout": 80, "h": 29, "w": 43, "k": 3, "stride": 1,
         "bias": True, "replay": False},
        # the middle of the conv sweep: forward, input, weight and bias gradients of a VGG-like layer
        {"name": "conv 256ch B40 36x36", "kind": "conv", "n": 40, "cin": 256, "cout": 256, "h": 36, "w": 36, "k": 3, "stride": 1,
         "bias": True, "replay": False},
        # its largest shape
        {"name": "conv 512ch B64 72x72", "kind": "conv", "n": 64, "cin": 512, "cout": 512, "h": 72, "w": 72, "k": 3, "stride": 1,
         "bias": True, "replay": False},
        # the style generator's 9x9 output layer: few outputs, a large kernel
        {"name": "conv 9x9 32-3 B40 36x36", "kind": "conv", "n": 40, "cin": 32, "cout": 3, "h": 36, "w": 36, "k": 9, "stride": 1,
         "bias": True, "replay": True},
        # ResNet-18's first strided block (3x3 stride 2, 3x3, 1x1 shortcut, three batch norms), forward and backward
        {"name": "resnet block 64-128 B128 64x64", "kind": "block", "n": 128, "cin": 64, "cout": 128, "stride": 2, "h": 64, "w": 64,
         "replay": False},
        # the MLP of 25.2M parameters, forward and backward
        {"name": "mlp 1024-4096-4096-1024 M8192", "kind": "mlp", "m": 8192, "k": 1024, "hidden": 4096, "n": 1024},
        # a classifier head: ResNet-18's fully connected layer, forward and backward, the smallest call here
        {"name": "linear 512-1000 M128", "kind": "linear", "m": 128, "k": 512, "n": 1000, "replay": False},
        # one optimizer step over the MLP's parameters
        {"name": "adam 25.2M bf16", "kind": "adam", "params": 25175040, "tensors": 6, "dtype": "bf16", "weight_decay": 0.0},
        # the style transfer's perceptual loss (frozen VGG, content and Gram terms) and its gradient in the image
        {"name": "perceptual loss B40 36x36", "kind": "loss", "n": 40, "h": 36, "w": 36},
        # one residual block of the style generator on its 9x9 grid, forward and backward
        {"name": "style residual 128ch B40 9x9", "kind": "residual", "n": 40, "c": 128, "h": 9, "w": 9},
        # a whole call: stylising a batch with the generator, without gradients
        {"name": "stylise B40 36x36", "kind": "stylise", "n": 40, "h": 36, "w": 36},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv_step", "conv", "conv", "conv", "conv9", "block", "mlp", "linear", "adam", "loss", "residual", "stylise"])
    if kind == "conv_step":
        return {"kind": kind, "n": _log_int(rng, 4, 40), "c": _log_int(rng, 32, 256), "h": rng.randint(12, 48), "w": rng.randint(12, 48)}
    if kind == "conv":
        while True:
            ch = [rng.choice([64, 128, 256, 512]) if rng.random() < 0.6 else _log_int(rng, 16, 512) for _ in range(2)]
            h = rng.randint(9, 72)
            c = {"kind": kind, "n": _log_int(rng, 4, 64), "cin": ch[0], "cout": ch[0] if rng.random() < 0.5 else ch[1], "h": h,
                 "w": h if rng.random() < 0.5 else rng.randint(9, 72), "k": 3, "stride": rng.choice([1, 1, 1, 2]),
                 "bias": rng.random() < 0.7, "replay": False}
            if 5e8 <= work(c)["flops"]:
                break
        c["replay"] = work(c)["flops"] < 3e10 and rng.random() < 0.5  # long kernels gain nothing from a capture
        return c
    if kind == "conv9":
        few = rng.random() < 0.5
        wide = _log_int(rng, 16, 64)
        return {"kind": "conv", "n": _log_int(rng, 8, 64), "cin": wide if few else 3, "cout": 3 if few else wide, "h": rng.randint(24, 72),
                "w": rng.randint(24, 72), "k": rng.choice([5, 7, 9, 9]), "stride": 1, "bias": True, "replay": True}
    if kind == "block":
        cin = rng.choice([64, 128, 256])
        stride = rng.choice([1, 2])
        size = {64: 64, 128: 32, 256: 16}[cin]
        return {"kind": kind, "n": _log_int(rng, 24, 128), "cin": cin, "cout": cin * stride, "stride": stride, "h": size + rng.choice([-3, 0, 0, 1]),
                "w": size + rng.choice([-2, 0, 0, 3]), "replay": False}
    if kind == "mlp":
        return {"kind": kind, "m": _log_int(rng, 512, 8192), "k": _log_int(rng, 256, 1024), "hidden": _log_int(rng, 512, 4096),
                "n": _log_int(rng, 256, 1024)}
    if kind == "linear":
        return {"kind": kind, "m": _log_int(rng, 16, 8192), "k": _log_int(rng, 64, 4096), "n": _log_int(rng, 64, 4096), "replay": rng.random() < 0.5}
    if kind == "adam":
        return {"kind": kind, "params": _log_int(rng, 1000000, 25000000), "tensors": rng.randint(4, 20), "dtype": rng.choice(["bf16", "bf16", "fp32"]),
                "weight_decay": rng.choice([0.0, 1e-5])}
    if kind == "residual":
        return {"kind": kind, "n": _log_int(rng, 8, 64), "c": rng.choice([64, 128, 128, 256]), "h": rng.randint(8, 24), "w": rng.randint(8, 24)}
    return {"kind": kind, "n": _log_int(rng, 8, 40), "h": 4 * rng.randint(6, 16), "w": 4 * rng.randint(6, 16)}


# ---------------------------------------------------------------------------------------
# Values: activations of unit variance, weights and biases of PyTorch's default init bounds
# ---------------------------------------------------------------------------------------
class _Values:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda").to(BF16)

    def unit(self, *shape):
        return torch.rand(shape, generator=self.g, device="cuda").to(BF16)

    def uniform(self, bound, *shape):
        return ((torch.rand(shape, generator=self.g, device="cuda") * 2 - 1) * bound).to(BF16)

    def conv(self, cout, cin, k, bias=True):
        bound = 1 / math.sqrt(cin * k * k)
        p = {"weight": self.uniform(bound, cout, cin, k, k)}
        return {**p, "bias": self.uniform(bound, cout)} if bias else p

    def linear(self, k, n):
        bound = 1 / math.sqrt(k)
        return {"weight": self.uniform(bound, n, k), "bias": self.uniform(bound, n)}

    def norm(self, c):
        return {"weight": (1 + 0.1 * self.normal(c).float()).to(BF16), "bias": (0.1 * self.normal(c).float()).to(BF16)}


def _named(prefix, params):
    return {"%s.%s" % (prefix, k): v for k, v in params.items()}


GENERATOR = ((3, 32, 9, 1), (32, 64, 3, 2), (64, 128, 3, 2)), 5, ((128, 64), (64, 32)), (32, 3, 9)
# VGG19's conv stack through relu4_1; the taps of the style terms and of the content term are relu1_1, relu2_1, relu3_1,
# relu4_1 and relu2_2
VGG = ((3, 64), (64, 64), "M", (64, 128), (128, 128), "M", (128, 256), (256, 256), (256, 256), (256, 256), "M", (256, 512))
STYLE_TAPS, CONTENT_TAP = (1, 6, 11, 20), 8


def _values(case, seed):
    """The tensors a program has in hand (on the GPU): "x" and "dy" where the kind has them, and "p", the parameters by name."""
    v, k = _Values(seed), case["kind"]
    if k == "conv_step":
        n, c, h, w = case["n"], case["c"], case["h"], case["w"]
        return {"x": v.normal(n, c, h, w), "p": v.conv(c, c, 3)}
    if k == "conv":
        ho, wo = _conv_out(case)
        return {"x": v.normal(case["n"], case["cin"], case["h"], case["w"]), "dy": v.normal(case["n"], case["cout"], ho, wo),
                "p": v.conv(case["cout"], case["cin"], case["k"], case["bias"])}
    if k == "block":
        cin, cout, s = case["cin"], case["cout"], case["stride"]
        p = {**_named("c1", v.conv(cout, cin, 3, False)), **_named("b1", v.norm(cout)), **_named("c2", v.conv(cout, cout, 3, False)),
             **_named("b2", v.norm(cout))}
        if s != 1 or cin != cout:
            p.update({**_named("down.0", v.conv(cout, cin, 1, False)), **_named("down.1", v.norm(cout))})
        ho, wo = (case["h"] - 1) // s + 1, (case["w"] - 1) // s + 1
        return {"x": F.relu(v.normal(case["n"], cin, case["h"], case["w"])), "dy": v.normal(case["n"], cout, ho, wo), "p": p}
    if k == "mlp":
        p = {**_named("0", v.linear(case["k"], case["hidden"])), **_named("2", v.linear(case["hidden"], case["hidden"])),
             **_named("4", v.linear(case["hidden"], case["n"]))}
        return {"x": v.normal(case["m"], case["k"]), "dy": v.normal(case["m"], case["n"]), "p": p}
    if k == "linear":
        return {"x": v.normal(case["m"], case["k"]), "dy": v.normal(case["m"], case["n"]), "p": v.linear(case["k"], case["n"])}
    if k == "adam":
        dtype = {"bf16": BF16, "fp32": torch.float32}[case["dtype"]]
        sizes = _adam_sizes(case)
        p = [0.02 * torch.randn(s, generator=v.g, device="cuda") for s in sizes]
        g = [0.01 * torch.randn(s, generator=v.g, device="cuda") for s in sizes]
        m = [0.005 * torch.randn(s, generator=v.g, device="cuda") for s in sizes]
        q = [1e-4 * torch.rand(s, generator=v.g, device="cuda") for s in sizes]
        return {n: [t.to(dtype) for t in ts] for n, ts in (("param", p), ("grad", g), ("exp_avg", m), ("exp_avg_sq", q))}
    if k == "residual":
        n, c, h, w = case["n"], case["c"], case["h"], case["w"]
        p = {**_named("body.0.0", v.conv(c, c, 3)), **_named("body.0.1", v.norm(c)), **_named("body.1.0", v.conv(c, c, 3)),
             **_named("body.1.1", v.norm(c))}
        return {"x": v.normal(n, c, h, w), "dy": v.normal(n, c, h, w), "p": p}
    if k == "stylise":
        down, blocks, up, (cin, cout, ks) = GENERATOR
        p, i = {}, 0
        for a, b, kk, _ in down:
            p.update({**_named("%d.0" % i, v.conv(b, a, kk)), **_named("%d.1" % i, v.norm(b))})
            i += 1
        for _ in range(blocks):
            for j in range(2):
                p.update({**_named("%d.body.%d.0" % (i, j), v.conv(128, 128, 3)), **_named("%d.body.%d.1" % (i, j), v.norm(128))})
            i += 1
        for a, b in up:
            p.update({**_named("%d.1.0" % i, v.conv(b, a, 3)), **_named("%d.1.1" % i, v.norm(b))})
            i += 1
        p.update(_named(str(i), v.conv(cout, cin, ks)))
        return {"x": v.unit(case["n"], 3, case["h"], case["w"]), "p": p}
    if k == "loss":
        n, h, w = case["n"], case["h"], case["w"]
        p = [v.conv(c[1], c[0], 3) for c in VGG if c != "M"]
        # a frozen feature net keeps its activations' scale from layer to layer
        p = [{"weight": (q["weight"].float() * math.sqrt(6)).to(BF16), "bias": q["bias"]} for q in p]
        grams = []
        for tap in STYLE_TAPS:
            c = [q["weight"].shape[0] for q in p][{1: 0, 6: 2, 11: 4, 20: 8}[tap]]
            a = torch.randn(c, 2 * c, generator=v.g, device="cuda")
            grams.append((a @ a.t() / (2 * c) * 0.002).contiguous())
        return {"x": v.unit(n, 3, h, w), "target": v.unit(n, 3, h, w), "p": p, "grams": grams}
    raise ValueError(k)


def _conv_out(c):
    return (c["h"] - 1) // c["stride"] + 1, (c["w"] - 1) // c["stride"] + 1


def _adam_sizes(case):
    """A few large weights and the rest small ones, as a network's parameters are."""
    n, t = case["params"], case["tensors"]
    if n == 25175040 and t == 6:
        return [4096 * 1024, 4096, 4096 * 4096, 4096, 1024 * 4096, 1024]
    share = [0.5 ** (i // 2 + 1) for i in range(t)]
    return [max(1, int(n * s / sum(share))) for s in share]


# ---------------------------------------------------------------------------------------
# Modules
# ---------------------------------------------------------------------------------------
class _ConvIN(nn.Sequential):
    def __init__(self, cin, cout, k, stride=1, relu=True):
        layers = [nn.Conv2d(cin, cout, k, stride=stride, padding=k // 2), nn.InstanceNorm2d(cout, affine=True)]
        super().__init__(*layers, *([nn.ReLU()] if relu else []))


class _Residual(nn.Module):
    def __init__(self, c):
        super().__init__()
        self.body = nn.Sequential(_ConvIN(c, c, 3), _ConvIN(c, c, 3, relu=False))

    def forward(self, x):
        return x + self.body(x)


class _UpConv(nn.Sequential):
    def __init__(self, cin, cout):
        super().__init__(nn.Upsample(scale_factor=2, mode="nearest"), _ConvIN(cin, cout, 3))


class _Block(nn.Module):
    def __init__(self, cin, cout, stride):
        super().__init__()
        self.c1 = nn.Conv2d(cin, cout, 3, stride, 1, bias=False)
        self.b1 = nn.BatchNorm2d(cout)
        self.c2 = nn.Conv2d(cout, cout, 3, 1, 1, bias=False)
        self.b2 = nn.BatchNorm2d(cout)
        self.down = None
        if stride != 1 or cin != cout:
            self.down = nn.Sequential(nn.Conv2d(cin, cout, 1, stride, bias=False), nn.BatchNorm2d(cout))

    def forward(self, x):
        y = torch.relu(self.b1(self.c1(x)))
        y = self.b2(self.c2(y))
        return torch.relu(y + (x if self.down is None else self.down(x)))


def _module(case):
    k = case["kind"]
    if k == "conv_step":
        return nn.Conv2d(case["c"], case["c"], 3, padding=1)
    if k == "conv":
        return nn.Conv2d(case["cin"], case["cout"], case["k"], case["stride"], case["k"] // 2, bias=case["bias"])
    if k == "block":
        return _Block(case["cin"], case["cout"], case["stride"])
    if k == "mlp":
        return nn.Sequential(nn.Linear(case["k"], case["hidden"]), nn.GELU(), nn.Linear(case["hidden"], case["hidden"]), nn.GELU(),
                             nn.Linear(case["hidden"], case["n"]))
    if k == "linear":
        return nn.Linear(case["k"], case["n"])
    if k == "residual":
        return _Residual(case["c"])
    if k == "stylise":
        down, blocks, up, (cin, cout, ks) = GENERATOR
        return nn.Sequential(*[_ConvIN(*d) for d in down], *[_Residual(128) for _ in range(blocks)], *[_UpConv(*u) for u in up],
                             nn.Conv2d(cin, cout, ks, padding=ks // 2))
    raise ValueError(k)


def _on_xdna(module, params):
    """The module on the device, with these parameters and fresh buffers."""
    with torch.no_grad():
        m = module.to(BF16).to_empty(device=XDNA)
        for name, t in m.named_parameters():
            t.copy_(params[name])
        for name, t in m.named_buffers():
            t.fill_(1 if name.endswith("running_var") else 0)
    return m.train()


def _captured(fn, x):
    """A program's captured step: `fn`'s work as one graph with `x` its input; returns (graph, outputs)."""
    for _ in range(2):
        fn()
    g = torch.xdna.Graph()
    with torch.xdna.graph(g):
        out = fn()
    return g, out


# ---------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------
def prepare(case, seed):
    v = _values(case, seed)
    kind = case["kind"]
    if kind == "adam":
        ps = [nn.Parameter(t.to(XDNA)) for t in v["param"]]
        for p, g in zip(ps, v["grad"]):
            p.grad = g.to(XDNA)
        opt = torch.optim.Adam(ps, lr=1e-3, weight_decay=case["weight_decay"], fused=True)
        for p, m, q in zip(ps, v["exp_avg"], v["exp_avg_sq"]):
            opt.state[p] = {"step": torch.full((), 100.0, device=XDNA), "exp_avg": m.to(XDNA), "exp_avg_sq": q.to(XDNA)}
        return {"kind": kind, "opt": opt, "params": ps}
    if kind == "loss":
        return _prepare_loss(case, v)
    x = v["x"].to(XDNA)
    if kind == "stylise":
        return _prepare_stylise(case, v, x)
    m = _on_xdna(_module(case), v["p"])
    if kind == "conv_step":
        return _prepare_conv_step(case, v, m, x)
    names = [n for n, _ in m.named_parameters()]
    if kind == "residual":
        regions.fuse_norm_activations(m)
        names = [n for n in names if not n.endswith("0.bias")]  # a bias before an instance norm has no gradient, only its rounding
    params = [p for n, p in m.named_parameters() if n in names]
    x.requires_grad_()
    dy = v["dy"].to(XDNA)
    s = {"kind": kind, "module": m, "params": params, "x": x, "dy": dy, "graph": None}
    if kind == "residual" or case.get("replay"):
        s["batch"] = v["x"].to(XDNA)
        s["graph"], s["out"] = _captured(lambda: _forward_backward(s), x)
    return s


def _prepare_loss(case, v):
    layers, i = [], 0
    for c in VGG:
        if c == "M":
            layers.append(nn.MaxPool2d(2))
            continue
        conv = _on_xdna(nn.Conv2d(c[0], c[1], 3, padding=1), v["p"][i])
        conv.requires_grad_(False)
        layers += [conv, nn.ReLU()]
        i += 1
    chain = regions.FrozenFeatureChain.from_sequential(layers, STYLE_TAPS + (CONTENT_TAP,))
    style = {t: (g.to(XDNA), 1e5) for t, g in zip(STYLE_TAPS, v["grams"])}
    x, target = v["x"].to(XDNA).requires_grad_(), v["target"].to(XDNA)

    def step():
        loss = regions.frozen_feature_loss(chain, x, target, mse_taps=(CONTENT_TAP,), style=style)
        return [loss.detach(), *torch.autograd.grad(loss, [x])]

    s = {"kind": "loss", "chain": chain, "x": x, "batch": v["x"].to(XDNA)}
    s["graph"], s["out"] = _captured(step, x)
    return s


def _prepare_stylise(case, v, x):
    m = _on_xdna(_module(case), v["p"])
    regions.fuse_norm_activations(m)

    def step():
        with torch.no_grad():
            return [m(x)]

    s = {"kind": "stylise", "module": m, "x": x, "batch": v["x"].to(XDNA)}
    s["graph"], s["out"] = _captured(step, x)
    return s


def _prepare_conv_step(case, v, m, x):
    opt = torch.optim.Adam(m.parameters(), lr=1e-3, fused=True, capturable=True)
    target = torch.zeros(x.shape, device=XDNA)

    def step():
        opt.zero_grad(set_to_none=True)
        loss = F.mse_loss(m(x).float(), target)
        loss.backward()
        opt.step()
        return [loss.detach(), m.weight.grad, m.bias.grad, m.weight, m.bias]

    s = {"kind": "conv_step", "module": m, "opt": opt, "x": x, "batch": v["x"].to(XDNA)}
    s["graph"], s["out"] = _captured(step, x)
    with torch.no_grad():  # back to where training begins
        for n, p in m.named_parameters():
            p.copy_(v["p"][n])
            for t in opt.state[p].values():
                t.zero_()
    return s


def _forward_backward(s):
    y = s["module"](s["x"])
    out = [y.detach(), *torch.autograd.grad(y, [s["x"], *s["params"]], s["dy"])]
    if s["kind"] == "block":
        out += [b for n, b in s["module"].named_buffers() if "running" in n]
    return out


def run(state):
    if state["kind"] == "adam":
        state["opt"].step()
        st = [state["opt"].state[p] for p in state["params"]]
        return [state["params"], [t["exp_avg"] for t in st], [t["exp_avg_sq"] for t in st]]
    if state.get("graph") is None:
        return _forward_backward(state)
    with torch.no_grad():
        state["x"].copy_(state["batch"])
    state["graph"].replay()
    return state["out"]


# ---------------------------------------------------------------------------------------
# Work, tolerances, and the same outputs in 64 bits
# ---------------------------------------------------------------------------------------
def _conv_work(n, cin, cout, h, w, k, stride=1, grads=3):
    """(bytes, flops) of a conv layer; grads 3: x, w and dy read, y, dx and dw written; 1: forward only; 2: no dx."""
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    x, y, p = n * cin * h * w, n * cout * ho * wo, cin * cout * k * k
    nbytes = {1: x + y + p, 2: x + 2 * y + 2 * p, 3: 2 * x + 2 * y + 2 * p}[grads] * 2
    return nbytes, 2.0 * grads * y * cin * k * k


def work(case):
    k = case["kind"]
    if k == "conv_step":
        n, c, h, w = case["n"], case["c"], case["h"], case["w"]
        # x read; the weight, its two moments read and written, its gradient written; y need not leave the step
        return {"bytes": 2.0 * n * c * h * w + 14.0 * (9 * c * c + c), "flops": _conv_work(n, c, c, h, w, 3, 1, 2)[1]}
    if k == "conv":
        b, f = _conv_work(case["n"], case["cin"], case["cout"], case["h"], case["w"], case["k"], case["stride"])
        return {"bytes": b, "flops": f}
    if k == "block":
        n, cin, cout, s, h, w = (case[i] for i in ("n", "cin", "cout", "stride", "h", "w"))
        ho, wo = (h - 1) // s + 1, (w - 1) // s + 1
        f = _conv_work(n, cin, cout, h, w, 3, s)[1] + _conv_work(n, cout, cout, ho, wo, 3)[1]
        p = 9 * cin * cout + 9 * cout * cout
        if s != 1 or cin != cout:
            f += _conv_work(n, cin, cout, h, w, 1, s)[1]
            p += cin * cout
        return {"bytes": 2.0 * (2 * n * cin * h * w + 2 * n * cout * ho * wo + 2 * p), "flops": f}
    if k == "mlp":
        m, a, h, b = case["m"], case["k"], case["hidden"], case["n"]
        p = a * h + h * h + h * b
        return {"bytes": 2.0 * (2 * m * a + 2 * m * b + 2 * p), "flops": 6.0 * m * p}
    if k == "linear":
        m, a, b = case["m"], case["k"], case["n"]
        return {"bytes": 2.0 * (2 * m * a + 2 * m * b + 2 * a * b), "flops": 6.0 * m * a * b}
    if k == "adam":
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": 7.0 * size * sum(_adam_sizes(case)), "flops": 14.0 * sum(_adam_sizes(case))}
    if k == "residual":
        n, c, h, w = case["n"], case["c"], case["h"], case["w"]
        return {"bytes": 2.0 * (4 * n * c * h * w + 4 * 9 * c * c), "flops": 2 * _conv_work(n, c, c, h, w, 3)[1]}
    n, h, w = case["n"], case["h"], case["w"]
    if k == "stylise":
        down, blocks, up, (cin, cout, ks) = GENERATOR
        f, p, s = 0.0, 0, 1
        for a, b, kk, st in down:
            f += _conv_work(n, a, b, h // s, w // s, kk, st, 1)[1]
            p += a * b * kk * kk
            s *= st
        f += 2 * blocks * _conv_work(n, 128, 128, h // s, w // s, 3, 1, 1)[1]
        p += 2 * blocks * 9 * 128 * 128
        for a, b in up:
            s //= 2
            f += _conv_work(n, a, b, h // s, w // s, 3, 1, 1)[1]
            p += 9 * a * b
        f += _conv_work(n, cin, cout, h, w, ks, 1, 1)[1]
        return {"bytes": 2.0 * (6 * n * h * w + p + cin * cout * ks * ks), "flops": f}
    # loss: the image's features and their gradient, the target's features through the content tap
    f, p, s, target = 0.0, 0, 1, True
    for i, c in enumerate(VGG):
        if c == "M":
            s *= 2
            continue
        one = _conv_work(n, c[0], c[1], h // s, w // s, 3, 1, 1)[1]
        f += one * (3 if i <= 4 else 2)
        p += 9 * c[0] * c[1]
        if i in (0, 3, 6, 11):  # a style tap's Gram matrix and its product in the gradient
            f += 2 * 2.0 * n * c[1] * c[1] * (h // s) * (w // s)
    return {"bytes": 2.0 * (3 * 3 * n * h * w + p), "flops": f}


def tolerance(case):
    k = case["kind"]
    # about four times the distance to 64 bits: 1.7e-3 for 32-bit sums rounded once to bf16, 4e-3 through the MLP
    if k == "adam" and case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if k in ("adam", "conv", "conv_step", "linear"):
        return {"rel": 7e-3}
    if k == "mlp":
        return {"rel": 1.6e-2}
    return {"rel": 3e-2}  # chains in bf16 (1.4e-2 to 5e-2): a rounding travels, and ReLU's masks turn over near zero


# Outputs in 64 bits. Gradients are written out: the autograd engine takes no plain GPU tensors once the xdna device is
# registered.
def _taps(xp, k, ho, wo, stride):
    """The padded input as each kernel tap sees it, and where that is."""
    for i in range(k):
        for j in range(k):
            at = (slice(None), slice(None), slice(i, i + stride * (ho - 1) + 1, stride), slice(j, j + stride * (wo - 1) + 1, stride))
            yield i, j, at, xp[at].reshape(xp.shape[0], xp.shape[1], ho * wo)


def _conv64(x, w, b=None, stride=1):
    """A convolution with padding k // 2, as one matrix product per kernel tap."""
    k, n = w.shape[2], x.shape[0]
    ho, wo = (x.shape[2] - 1) // stride + 1, (x.shape[3] - 1) // stride + 1
    y = 0
    for i, j, _, s in _taps(F.pad(x, [k // 2] * 4), k, ho, wo, stride):
        y = y + torch.matmul(w[:, :, i, j], s)
    y = y.view(n, w.shape[0], ho, wo)
    return y if b is None else y + b.view(1, -1, 1, 1)


def _conv64_grads(x, w, dy, stride=1):
    """(dx, dw, db)."""
    k, (n, cout, ho, wo) = w.shape[2], dy.shape
    d = dy.reshape(n, cout, ho * wo)
    xp = F.pad(x, [k // 2] * 4)
    dxp, dw = torch.zeros_like(xp), torch.zeros_like(w)
    for i, j, at, s in _taps(xp, k, ho, wo, stride):
        dxp[at] += torch.matmul(w[:, :, i, j].t().contiguous(), d).view(n, -1, ho, wo)
        dw[:, :, i, j] = torch.matmul(d, s.transpose(1, 2).contiguous()).sum(0)
    p = k // 2
    return dxp[:, :, p:p + x.shape[2], p:p + x.shape[3]], dw, dy.sum((0, 2, 3))


def _norm64(x, g, b, dims):
    """Batch norm (dims 0, 2, 3) or instance norm (dims 2, 3); returns the output and what the gradients take."""
    inv = 1 / torch.sqrt(x.var(dims, unbiased=False, keepdim=True) + 1e-5)
    xn = (x - x.mean(dims, keepdim=True)) * inv
    return xn * g.view(1, -1, 1, 1) + b.view(1, -1, 1, 1), (xn, inv, g, dims)


def _norm64_grads(kept, dy):
    xn, inv, g, dims = kept
    d = dy * g.view(1, -1, 1, 1)
    dx = inv * (d - d.mean(dims, keepdim=True) - xn * (d * xn).mean(dims, keepdim=True))
    return dx, (dy * xn).sum((0, 2, 3)), dy.sum((0, 2, 3))


def exact(case, seed):
    v, kind = _values(case, seed), case["kind"]
    if kind == "adam":
        return _exact_adam(case, v)
    if kind == "loss":
        return _exact_loss(v)
    p = {n: t.double() for n, t in v["p"].items()}
    x = v["x"].double()
    if kind == "stylise":
        return [_stylise64(x, p)]
    if kind == "conv_step":
        y = _conv64(x, p["weight"], p["bias"])
        _, gw, gb = _conv64_grads(x, p["weight"], y * (2 / y.numel()))
        # the first Adam step: both bias corrections cancel
        w, b = (t - 1e-3 * g / (g.abs() + 1e-8) for t, g in ((p["weight"], gw), (p["bias"], gb)))
        return [y.square().mean(), gw, gb, w, b]
    dy = v["dy"].double()
    if kind == "conv":
        y = _conv64(x, p["weight"], p.get("bias"), case["stride"])
        return [y, *_conv64_grads(x, p["weight"], dy, case["stride"])[:3 if case["bias"] else 2]]
    if kind in ("linear", "mlp"):
        return _exact_linears(x, dy, [p] if kind == "linear" else [{n: p["%d.%s" % (i, n)] for n in ("weight", "bias")} for i in (0, 2, 4)])
    return _exact_residual(x, dy, p) if kind == "residual" else _exact_block(case, x, dy, p)


def _exact_adam(case, v):
    out = [[], [], []]
    for p, g, m, q in zip(*(v[i] for i in ("param", "grad", "exp_avg", "exp_avg_sq"))):
        p, g, m, q = (t.double() for t in (p, g, m, q))
        g = g + case["weight_decay"] * p
        m, q = 0.9 * m + 0.1 * g, 0.999 * q + 0.001 * g * g
        denom = q.sqrt() / math.sqrt(1 - 0.999 ** 101) + 1e-8
        for o, t in zip(out, (p - 1e-3 / (1 - 0.9 ** 101) * m / denom, m, q)):
            o.append(t)
    return out


def _exact_linears(x, dy, layers):
    """Linear layers with GELU between them: the output, dx, then each layer's dw and db."""
    ins, pre = [x], []
    for i, q in enumerate(layers):
        pre.append(ins[-1] @ q["weight"].t() + q["bias"])
        if i + 1 < len(layers):
            ins.append(F.gelu(pre[-1]))
    grads, d = [], dy
    for i in reversed(range(len(layers))):
        grads = [d.t() @ ins[i], d.sum(0), *grads]
        d = d @ layers[i]["weight"]
        if i:
            z = pre[i - 1]
            d = d * (0.5 * (1 + torch.erf(z / math.sqrt(2))) + z * torch.exp(-z * z / 2) / math.sqrt(2 * math.pi))
    return [pre[-1], d, *grads]


def _exact_residual(x, dy, p):
    a = _conv64(x, p["body.0.0.weight"], p["body.0.0.bias"])
    z, ka = _norm64(a, p["body.0.1.weight"], p["body.0.1.bias"], (2, 3))
    r = F.relu(z)
    b = _conv64(r, p["body.1.0.weight"], p["body.1.0.bias"])
    y, kb = _norm64(b, p["body.1.1.weight"], p["body.1.1.bias"], (2, 3))
    db, g2, b2 = _norm64_grads(kb, dy)
    dr, w2, _ = _conv64_grads(r, p["body.1.0.weight"], db)
    da, g1, b1 = _norm64_grads(ka, dr * (z > 0))
    dx, w1, _ = _conv64_grads(x, p["body.0.0.weight"], da)
    return [x + y, dy + dx, w1, g1, b1, w2, g2, b2]


def _exact_block(case, x, dy, p):
    s, dims = case["stride"], (0, 2, 3)
    a = _conv64(x, p["c1.weight"], None, s)
    z, ka = _norm64(a, p["b1.weight"], p["b1.bias"], dims)
    r = F.relu(z)
    b = _conv64(r, p["c2.weight"])
    y, kb = _norm64(b, p["b2.weight"], p["b2.bias"], dims)
    stats, down = [a, b], "down.0.weight" in p
    if down:
        c = _conv64(x, p["down.0.weight"], None, s)
        t, kc = _norm64(c, p["down.1.weight"], p["down.1.bias"], dims)
        stats.append(c)
    y = y + (t if down else x)
    d = dy * (y > 0)
    db, g2, b2 = _norm64_grads(kb, d)
    dr, w2, _ = _conv64_grads(r, p["c2.weight"], db)
    da, g1, b1 = _norm64_grads(ka, dr * (z > 0))
    dx, w1, _ = _conv64_grads(x, p["c1.weight"], da, s)
    grads = [w1, g1, b1, w2, g2, b2]
    if down:
        dc, g3, b3 = _norm64_grads(kc, d)
        dt, w3, _ = _conv64_grads(x, p["down.0.weight"], dc, s)
        dx, grads = dx + dt, grads + [w3, g3, b3]
    else:
        dx = dx + d
    running = []
    for t in stats:
        running += [0.1 * t.mean(dims), 0.9 + 0.1 * t.var(dims, unbiased=True)]
    return [F.relu(y), dx, *grads, *running]


def _conv_in64(x, p, prefix, stride=1, relu=True):
    y = _conv64(x, p[prefix + ".0.weight"], p[prefix + ".0.bias"], stride)
    y = _norm64(y, p[prefix + ".1.weight"], p[prefix + ".1.bias"], (2, 3))[0]
    return F.relu(y) if relu else y


def _stylise64(x, p):
    down, blocks, up, _ = GENERATOR
    i = 0
    for _, _, _, s in down:
        x = _conv_in64(x, p, str(i), s)
        i += 1
    for _ in range(blocks):
        x = x + _conv_in64(_conv_in64(x, p, "%d.body.0" % i), p, "%d.body.1" % i, relu=False)
        i += 1
    for _ in up:
        x = _conv_in64(x.repeat_interleave(2, 2).repeat_interleave(2, 3), p, "%d.1" % i)
        i += 1
    return _conv64(x, p["%d.weight" % i], p["%d.bias" % i])


def _features64(x, p):
    """The output of every layer of the feature net, by its index."""
    out, i = [], 0
    for c in VGG:
        if c == "M":
            out.append(F.max_pool2d(out[-1], 2))
            continue
        out.append(_conv64(out[-1] if out else x, p[i]["weight"].double(), p[i]["bias"].double()))
        out.append(F.relu(out[-1]))
        i += 1
    return out


def _exact_loss(v):
    x, p = v["x"].double(), v["p"]
    f = _features64(x, p)
    t = _features64(v["target"].double(), p)[CONTENT_TAP]
    off = f[CONTENT_TAP] - t
    loss, seeds = off.square().mean(), {CONTENT_TAP: 2 * off / off.numel()}
    for tap, g in zip(STYLE_TAPS, v["grams"]):
        a, chw = f[tap].flatten(2), f[tap][0].numel()
        e = torch.matmul(a, a.transpose(1, 2).contiguous()) / chw - g.double()
        loss = loss + 1e5 * e.square().mean()
        seeds[tap] = torch.matmul(e + e.transpose(1, 2), a).view_as(f[tap]) * (2e5 / e.numel() / chw)
    d, i, k = 0, len(p), len(f) - 1
    for c in reversed(VGG):
        if c == "M":  # the gradient goes to each window's maximum
            _, at = F.max_pool2d(f[k - 1], 2, return_indices=True)
            d = F.max_unpool2d(d + seeds.get(k, 0), at, 2, output_size=f[k - 1].shape[2:])
            k -= 1
            continue
        i -= 1
        d = (d + seeds.get(k, 0)) * (f[k] > 0)
        d = _conv64_grads(f[k - 2] if k >= 2 else x, p[i]["weight"].double(), d)[0]
        k -= 2
    return [loss, d]
