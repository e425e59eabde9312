"""Loading parameters again: every layout that a load writes (the forward's
operands, the padded biases, the router's copies and, once a backward has run,
the backward's operands) must hold the new parameters and nothing of the old.

A handle that trained on other parameters and then loaded these computes what
a fresh handle computes, bit for bit: the kernels and their order are the same,
only the way the weights got into place differs.  Widths at the edges of the
64-wide tiles, hidden sizes that rule out 16-byte loads, device pointers that
are only 4-byte aligned, more experts than one launch takes, and host sources.
"""
import numpy as np
import pytest
import torch

from mgpt_amd import workload as wl
from mgpt_amd.moe import MoELayer

pytestmark = pytest.mark.gpu

# (C, H, E, k, act): edges of the 64 x 64 and 64 x 128 tiles, odd H and C
SHAPES = [
    (64, 32, 2, 1, "f32"), (16, 7, 4, 2, "f32"), (65, 65, 3, 2, "f32"), (200, 129, 5, 2, "bf16"),
    (128, 64, 8, 2, "bf16"), (192, 100, 17, 3, "bf16"), (64, 40, 130, 2, "bf16"),
]


def _inputs(C, H, E, k, act, seed):
    cfg = wl.MoEConfig("repack", 96, C, E, k, H, act, act, "normal")
    return wl.make_inputs(cfg, seed=seed, bias_std=0.05)


def _device(params, misalign):
    out = []
    for p in params:
        p = np.ascontiguousarray(p, np.float32)
        buf = torch.empty(p.size + 1, device="cuda")
        v = buf[1:] if misalign else buf[:-1]
        v.copy_(torch.from_numpy(p.reshape(-1)))
        out.append(v.view(p.shape))
    return out


def _step(layer, inp, dy):
    x = torch.from_numpy(inp.x).to("cuda").to(layer.dtype)
    layer.zero_grad()
    y = layer.forward(x, train=True)
    dx = layer.backward(dy)
    return [y, dx] + layer.get_gradients()


@pytest.mark.parametrize("source", ["device", "device_misaligned", "host"])
@pytest.mark.parametrize("C,H,E,k,act", SHAPES)
def test_reload_equals_a_fresh_handle(C, H, E, k, act, source):
    old, new = _inputs(C, H, E, k, act, 3), _inputs(C, H, E, k, act, 4)
    dtype = torch.float32 if act == "f32" else torch.bfloat16
    dy = torch.from_numpy(wl.normal_f32(9, 1, 96 * C).reshape(96, C)).to("cuda").to(dtype)
    load = (lambda inp: inp.params()) if source == "host" else (
        lambda inp: _device(inp.params(), source == "device_misaligned"))

    fresh = MoELayer(C, H, E, k, act=act)
    fresh.load_parameters(new.params())
    want = _step(fresh, new, dy)

    layer = MoELayer(C, H, E, k, act=act)
    layer.load_parameters(load(old))
    _step(layer, old, dy)
    for _ in range(2):   # the second load finds the backward's layouts in place
        layer.load_parameters(load(new))
        got = _step(layer, new, dy)
        torch.cuda.synchronize()
        for i, (a, b) in enumerate(zip(got, want)):
            assert torch.equal(a, b), f"output {i} of {len(want)}"


def _fresh(params, x, dy, shape):
    layer = MoELayer(*shape, act="bf16")
    layer.load_parameters(params)
    return _train(layer, x, dy)


def _train(layer, x, dy):
    layer.zero_grad()
    y = layer.forward(x, train=True)
    dx = layer.backward(dy)
    return [y, dx] + layer.get_gradients()


def _three(C, H, E, k, N, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    def normal(*s):
        return torch.randn(*s, generator=gen, device="cuda") * 0.05
    sets = []
    for _ in range(2):
        p = [normal(C, E), normal(1, E)]
        for _ in range(E):
            p += [normal(C, H), normal(1, H), normal(C, H), normal(1, H), normal(H, C), normal(1, C)]
        sets.append(p)
    return sets, normal(N, C).bfloat16(), normal(N, C).bfloat16()


def test_load_beside_a_running_backward():
    """A load on a second stream, ordered after the forward only, leaves the backward
    that still runs its own weights; the next step has the new ones."""
    shape, N = (512, 1024, 8, 2), 8192
    (old, new), x, dy = _three(*shape, N, 1)
    want_old, want_new = _fresh(old, x, dy, shape), _fresh(new, x, dy, shape)
    layer = MoELayer(*shape, act="bf16")
    layer.load_parameters(old)
    _train(layer, x, dy)      # a backward has filled its layouts
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        layer.load_parameters(old)
        layer.zero_grad()
        y = layer.forward(x, train=True)
        fwd = torch.cuda.Event()
        fwd.record(s1)
        dx = layer.backward(dy)
    with torch.cuda.stream(s2):
        s2.wait_event(fwd)
        layer.load_parameters(new)
    torch.cuda.synchronize()
    got = [y, dx] + layer.get_gradients()
    assert all(torch.equal(a, b) for a, b in zip(got, want_old))
    assert all(torch.equal(a, b) for a, b in zip(_train(layer, x, dy), want_new))


@pytest.mark.parametrize("load_in_graph", [False, True])
def test_loads_and_captured_backwards(load_in_graph):
    """A graph's backward, and an eager one after a graph's load, see the parameters
    loaded last, whichever was captured first."""
    shape, N = (128, 192, 6, 2), 700
    (old, new), x, dy = _three(*shape, N, 2)
    want_old, want_new = _fresh(old, x, dy, shape), _fresh(new, x, dy, shape)
    layer = MoELayer(*shape, act="bf16")
    layer.reserve(N, train=True)
    held = [p.clone() for p in old]
    layer.load_parameters(held)
    _train(layer, x, dy)
    torch.cuda.synchronize()
    out = torch.empty_like(x), torch.empty_like(x)
    step, load = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(step):
        layer.zero_grad()
        layer.forward_into(x, out[0], train=True)
        layer.backward_into(dy, out[1])
    if load_in_graph:
        with torch.cuda.graph(load):
            layer.load_parameters(held)
    for params, want in ((new, want_new), (old, want_old), (new, want_new)):
        for h, p in zip(held, params):
            h.copy_(p)
        if load_in_graph:
            load.replay()
        else:
            layer.load_parameters(held)
        step.replay()
        torch.cuda.synchronize()
        got = list(out) + layer.get_gradients()
        assert all(torch.equal(a, b) for a, b in zip(got, want)), "replayed step"
        assert all(torch.equal(a, b) for a, b in zip(_train(layer, x, dy), want)), "eager step"
