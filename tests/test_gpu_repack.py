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
