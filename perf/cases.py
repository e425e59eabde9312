"""The work that a program hands to the MoE layer, as cases that can be timed.

listed() holds one case per way the layer is used: the steps of a sampling
loop (one token, a full context, bf16 and fp8 weights, the engine's fp32
tensors over fp8 weights), the engine's default fp32 block, prompts and
batches in bf16 and fp8, the fused transformer half-block, many experts, and
training steps in fp32 and bf16.  Sizes are those of mgpt_amd.workload's
configurations and of the tests, with a few odd ones; draw() spreads more
cases over the ranges between them.

A training step is what a trainer asks of the layer around its optimizer:
load the parameters as the optimizer left them, zero_grad, the training
forward, the backward, and the gradients added into the caller's tensors.
"""
from __future__ import annotations

import ctypes
import math

import torch

from mgpt_amd import capi
from mgpt_amd.moe import MoELayer

_DT = {"f32": torch.float32, "bf16": torch.bfloat16}
_WBYTES = {"f32": 4, "bf16": 2, "fp8": 1}
EPS = 1e-5


def _case(name, op, act, weights, N, C, E, k, H, bias="zero"):
    return {"name": name, "op": op, "act": act, "weights": weights, "N": N, "C": C, "E": E, "k": k,
            "H": H, "bias": bias}


def listed():
    return [
        # the first step of a sampling loop: one token, its k experts' weights
        _case("decode_first_fp8", "forward", "bf16", "fp8", 1, 2048, 64, 8, 1408),
        # the loop's steady step: the whole 64-token context (cfg5)
        _case("decode_full_fp8", "forward", "bf16", "fp8", 64, 2048, 64, 8, 1408),
        # a step of a bf16 model: the headline layer on a short context
        _case("decode_bf16", "forward", "bf16", "bf16", 24, 1024, 16, 2, 2816, "normal"),
        # a step through the engine's fp32 tensors over fp8 weights
        _case("decode_f32_rows_fp8", "forward", "f32", "fp8", 37, 1024, 16, 2, 2816),
        # the engine's default block on a batch of 16 x 64 tokens (cfg1)
        _case("default_f32", "forward", "f32", "f32", 1024, 128, 8, 2, 512),
        # the MoE half of a transformer block, mid size (cfg2)
        _case("block_bf16", "block", "bf16", "bf16", 8192, 512, 8, 2, 1376),
        # the headline layer (cfg3)
        _case("headline_bf16", "forward", "bf16", "bf16", 16384, 1024, 16, 2, 2816, "normal"),
        # fine-grained experts under a Zipf load (cfg4)
        _case("fine_grained_bf16", "forward", "bf16", "bf16", 32768, 2048, 64, 6, 1408, "zipf"),
        # more experts than a wave has lanes, an odd number of tokens
        _case("wide_bf16", "forward", "bf16", "bf16", 8191, 1024, 128, 8, 704),
        # a prompt through the fp8 handle of the sampling loop
        _case("prompt_fp8", "forward", "bf16", "fp8", 1999, 2048, 64, 8, 1408),
        # the engine's default training step (fp32)
        _case("train_f32", "train", "f32", "f32", 1024, 128, 8, 2, 512),
        # the headline training step, through the fused block
        _case("train_block_bf16", "train_block", "bf16", "bf16", 16384, 1024, 16, 2, 2816, "normal"),
    ]


# The ranges that the listed cases stand for: (op choices, act, weights, N, C,
# E choices, k, H); C and H are drawn as multiples of the last two numbers
# (8 leaves widths that the library pads).
_RANGES = [
    (("forward",), "bf16", "fp8", (1, 64), (512, 2048), (16, 32, 64), (1, 8), (704, 2816), 128, 32),
    (("forward",), "f32", "fp8", (1, 64), (512, 2048), (16, 32, 64), (1, 8), (704, 2816), 128, 32),
    (("forward", "block"), "bf16", "bf16", (1, 64), (512, 2048), (8, 16, 64), (1, 8), (704, 2816), 64, 32),
    (("forward", "block"), "f32", "f32", (16, 4096), (96, 512), (4, 6, 8), (1, 2), (256, 2048), 8, 8),
    (("forward", "block"), "bf16", "bf16", (256, 32768), (256, 2048), (8, 12, 16, 60, 64), (1, 8),
     (512, 2816), 8, 32),
    (("forward", "block"), "bf16", "bf16", (1024, 16384), (512, 1024), (96, 128, 256), (2, 8), (256, 1024), 64, 32),
    (("forward",), "bf16", "fp8", (256, 4096), (512, 2048), (16, 32, 64), (1, 8), (704, 2816), 128, 32),
    (("train", "train_block"), "f32", "f32", (64, 2048), (96, 512), (4, 6, 8), (1, 2), (256, 1376), 8, 8),
    (("train", "train_block"), "bf16", "bf16", (1024, 16384), (256, 1024), (8, 12, 16, 32), (1, 6),
     (512, 2816), 8, 32),
]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """A pass's rough cost in bf16-flop equivalents: fp32 products run at a
    sixteenth of the bf16 rate, a byte takes the time of about 300, and a
    training step moves every parameter and gradient several times, tensor by
    tensor."""
    w = work(case)
    cost = w["flops"] * (16 if case["weights"] == "f32" else 1) + 300 * w["bytes"]
    return 1.5 * cost + 6e10 * case["E"] if case["op"].startswith("train") else cost


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        ops, act, weights, n, c, es, ks, h, cstep, hstep = rng.choice(_RANGES)
        E = rng.choice(es)
        case = {
            "op": rng.choice(ops), "act": act, "weights": weights,
            "N": min(n[1], max(n[0], _log_int(rng, *n))),
            "C": min(c[1], max(c[0], _log_int(rng, *c) // cstep * cstep)),
            "E": E,
            "k": min(E, rng.randint(*ks)),
            "H": min(h[1], max(h[0], _log_int(rng, *h) // hstep * hstep)),
            "bias": rng.choice(("zero", "zero", "normal", "zipf")),
        }
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ inputs
def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda").mul_(std)


def _router_bias(case, gen):
    E = case["E"]
    if case["bias"] == "normal":
        return _normal(gen, 1, E)
    if case["bias"] == "zipf":
        rank = torch.randperm(E, generator=gen, device="cuda").float() + 1
        w = rank.pow(-1.1)
        return torch.log(w / w.sum()).view(1, E)
    return torch.zeros(1, E, device="cuda")


def _inputs(case, seed):
    """Parameters, rows and upstream gradient, from the seed alone.  Weights
    ~ N(0, 0.02^2), small expert biases; inference weights come from a
    checkpoint in the layer's dtype (bf16 values; fp32 ones that the layer
    quantises for fp8), training weights are an optimizer's fp32 masters.
    Rows are RMS-normalised, as ln2 leaves them, or for the fused block the
    residual stream before it."""
    N, C, E, H = case["N"], case["C"], case["E"], case["H"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    train = case["op"].startswith("train")

    def weight(*shape):
        w = _normal(gen, *shape, std=0.02)
        return w if train or case["weights"] != "bf16" else w.bfloat16().float()

    p = {"Wr": _normal(gen, C, E, std=0.02)}
    if case["act"] == "bf16" and not train:
        p["Wr"] = p["Wr"].bfloat16().float()
    p["br"] = _router_bias(case, gen)
    p["Wg"], p["Wu"], p["Wd"] = weight(E, C, H), weight(E, C, H), weight(E, H, C)
    p["bg"], p["bu"], p["bd"] = weight(E, H), weight(E, H), weight(E, C)
    x = _normal(gen, N, C)
    gamma = None
    if case["op"] in ("block", "train_block"):
        x.mul_(1.5)
        gamma = _normal(gen, C, std=0.1).add_(1.0)
    else:
        x.mul_(torch.rsqrt(x.pow(2).mean(dim=1, keepdim=True) + EPS))
    x = x.to(_DT[case["act"]])
    dy = _normal(gen, N, C).to(_DT[case["act"]]) if train else None
    return p, x, gamma, dy


def _parameter_list(p):
    """The 2 + 6E tensors in the layer's order."""
    out = [p["Wr"], p["br"]]
    for e in range(p["Wg"].shape[0]):
        out += [p[n][e] for n in ("Wg", "bg", "Wu", "bu", "Wd", "bd")]
    return out


def prepare(case, seed):
    p, x, gamma, dy = _inputs(case, seed)
    layer = MoELayer(case["C"], case["H"], case["E"], case["k"], act=case["act"],
                     weights=case["weights"])
    params = _parameter_list(p)
    layer.load_parameters(params)
    train = case["op"].startswith("train")
    layer.reserve(case["N"], train=train)
    state = {"case": case, "layer": layer, "x": x, "gamma": gamma}
    if train:
        # the caller's gradient tensors, one flat buffer behind them so that
        # a trainer's zero_grad is one fill
        flat = torch.zeros(sum(t.numel() for t in p.values()), device="cuda")
        grads, off = {}, 0
        for n, t in p.items():
            grads[n] = flat[off:off + t.numel()].view(t.shape)
            off += t.numel()
        views = _parameter_list(grads)
        state.update(dy=dy, params=params, keep=p, flat=flat, grads=grads, views=views,
                     ptrs=(ctypes.c_void_p * len(views))(*[v.data_ptr() for v in views]))
    return state


def run(state):
    op, layer, x = state["case"]["op"], state["layer"], state["x"]
    if op == "forward":
        return layer.forward(x)
    if op == "block":
        return layer.forward_block(x, state["gamma"], EPS)
    layer.load_parameters(state["params"])
    layer.zero_grad()
    state["flat"].zero_()
    out = {}
    if op == "train":
        out["y"] = layer.forward(x, train=True)
        out["dx"] = layer.backward(state["dy"])
    else:
        y = torch.empty_like(x)
        layer.forward_block_into(x, state["gamma"], EPS, y, train=True)
        out["y"] = y
        out["dx"], out["dgamma"] = layer.backward_block(state["dy"])
    capi.check(capi.lib().mgpt_moe_accumulate_gradients(
        layer._h, state["ptrs"], len(state["views"]), 1, torch.cuda.current_stream().cuda_stream))
    for n, g in state["grads"].items():
        out["d" + n] = g
    return out


def work(case):
    N, C, E, k, H = case["N"], case["C"], case["E"], case["k"], case["H"]
    a = 4 if case["act"] == "f32" else 2
    train = case["op"].startswith("train")
    flops = 6.0 * N * k * C * H + 2.0 * N * C * E
    expert = 3 * C * H + 2 * H + C
    if train:
        # rows, output, upstream and input gradient; fp32 parameters in,
        # their gradients out
        return {"bytes": 4 * N * C * a + 8 * (E * expert + C * E + E), "flops": 3 * flops}
    # the experts that N tokens of k choices reach, were they spread evenly
    reached = E * (1.0 - (1.0 - k / E) ** N)
    return {"bytes": int(2 * N * C * a + reached * expert * _WBYTES[case["weights"]] + 4 * C * E),
            "flops": flops}


def tolerance(case):
    """About four times the distance from exact() measured on MI355X: fp32
    outputs 2e-7, fp32 gradients up to 1.4e-6, bf16 outputs 3e-3, bf16
    gradients up to 8e-3 (the router bias's, a sum of terms of both signs)."""
    train = case["op"].startswith("train")
    if case["weights"] == "f32":
        return {"rel": 6e-6 if train else 1e-6}
    return {"rel": 3e-2 if train else 1.2e-2}


# ---------------------------------------------------------------- in 64 bits
def _rows(case, x, gamma):
    """The rows that the router sees, in the layer's own fp32 steps: the sum
    of squares in column order, r = 1/sqrt(ms/C + eps), (x*r)*gamma."""
    x = x.float()
    if gamma is None:
        return x
    ms = torch.zeros(x.shape[0], device=x.device)
    for c in range(x.shape[1]):
        ms = ms + x[:, c] * x[:, c]
    r = torch.sqrt(ms.double() / x.shape[1] + EPS).reciprocal()
    return (x * r.float()[:, None]) * gamma[None, :]


def _choices(case, p, rows):
    """The experts each token chooses: logits as fp32 sums in column order
    and then the bias (the layer's contract), the k largest, the lower id
    first among equals."""
    acc = torch.zeros(rows.shape[0], case["E"], device=rows.device)
    cols = rows.t().contiguous()
    for c in range(case["C"]):
        acc = acc + cols[c][:, None] * p["Wr"][c][None, :]
    logits = acc + p["br"]
    return torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :case["k"]]


def _as_held(case, w):
    """A weight [E, in, out] as the layer holds it, in 64 bits."""
    if case["weights"] == "bf16":
        return w.bfloat16().double()
    if case["weights"] == "fp8":
        amax = w.abs().amax(dim=1, keepdim=True)
        scale = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
        return (w / scale).to(torch.float8_e4m3fn).double() * scale.double()
    return w.double()


def exact(case, seed):
    if case["op"].startswith("train") and 18.0 * case["N"] * case["k"] * case["C"] * case["H"] > 4e12:
        return None
    p, x, gamma, dy = _inputs(case, seed)
    N, E, k = case["N"], case["E"], case["k"]
    idx = _choices(case, p, _rows(case, x, gamma))
    xd = x.double()
    r = torch.rsqrt(xd.pow(2).mean(dim=1) + EPS)
    xn = xd if gamma is None else xd * r[:, None] * gamma.double()[None, :]
    P = torch.softmax(xn @ p["Wr"].double() + p["br"].double(), dim=1).clamp(1e-7, 1.0)
    y = xd.clone() if gamma is not None else torch.zeros_like(xd)
    train = case["op"].startswith("train")
    if train:
        dyd = dy.double()
        dxn = torch.zeros_like(xd)
        dP = torch.zeros_like(P)
        g = {n: torch.zeros(t.shape, dtype=torch.float64, device="cuda") for n, t in p.items()}
    for e in range(E):
        hit = (idx == e).any(dim=1).nonzero().flatten()
        if train:
            dP[:, e] += 0.01 * E * (hit.numel() / N) / N
        if hit.numel() == 0:
            continue
        Wg, Wu, Wd = (_as_held(case, p[n][e:e + 1])[0] for n in ("Wg", "Wu", "Wd"))
        xe = xn[hit]
        gate = xe @ Wg + p["bg"][e].double()
        up = xe @ Wu + p["bu"][e].double()
        sig = torch.sigmoid(gate)
        h = gate * sig * up
        o = h @ Wd + p["bd"][e].double()
        pe = P[hit, e][:, None]
        y[hit] += pe * o
        if not train:
            continue
        dye = dyd[hit]
        dP[hit, e] += (o * dye).sum(dim=1)
        do = dye * pe
        dh = do @ Wd.t()
        du = dh * gate * sig
        dg = dh * up * sig * (1 + gate * (1 - sig))
        g["Wd"][e], g["bd"][e] = h.t() @ do, do.sum(dim=0)
        g["Wg"][e], g["bg"][e] = xe.t() @ dg, dg.sum(dim=0)
        g["Wu"][e], g["bu"][e] = xe.t() @ du, du.sum(dim=0)
        dxn[hit] += dg @ Wg.t() + du @ Wu.t()
    if not train:
        return y
    dL = P * (dP - (dP * P).sum(dim=1, keepdim=True))
    g["Wr"], g["br"] = xn.t() @ dL, dL.sum(dim=0, keepdim=True)
    dxn += dL @ p["Wr"].double().t()
    out = {"y": y, "dx": dxn}
    if gamma is not None:
        xhat = xd * r[:, None]
        dh = dxn * gamma.double()[None, :]
        s = (dh * xhat).sum(dim=1, keepdim=True)
        out["dgamma"] = (dxn * xhat).sum(dim=0)
        out["dx"] = dyd + r[:, None] * (dh - xhat * s / case["C"])
    for n, t in g.items():
        out["d" + n] = t
    return out
