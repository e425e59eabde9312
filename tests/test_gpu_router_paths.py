"""Every way the router forms its logits routes bit for bit like the oracle:
the one-launch kernel at 1 to 64 experts, separate product and chain waves, an
expert per lane (1, 2 and 4 tokens a wave, 1 to 8 groups of 64 experts) and the
fused kernel, on both sides of each line between them, with token counts that
leave blocks and waves partly filled, training (router probabilities) included.
"""
import numpy as np
import pytest
import torch

import oracle_lib as O
from mgpt_amd import workload as wl
from mgpt_amd.moe import MoELayer

pytestmark = pytest.mark.gpu

# (N, C, E, k, act)
SHAPES = [
    # one launch: up to 64 tokens, any width that is a multiple of 64
    (1, 64, 1, 1, "f32"), (64, 64, 2, 2, "bf16"), (63, 128, 8, 2, "f32"), (17, 1024, 16, 2, "bf16"),
    (64, 576, 9, 8, "bf16"), (5, 2048, 33, 3, "f32"),
    # product and chain waves, from 17 experts on at every width
    (895, 128, 64, 6, "bf16"), (1791, 64, 32, 2, "f32"),
    # ... up to 16 experts by width and tokens, both sides (the second of each fused)
    (1023, 256, 16, 2, "bf16"), (1024, 256, 16, 2, "bf16"), (1025, 320, 16, 2, "f32"), (1281, 320, 16, 2, "f32"),
    (3583, 1024, 16, 2, "bf16"), (3584, 1024, 16, 2, "bf16"), (2559, 1024, 16, 2, "f32"), (2560, 1024, 16, 2, "f32"),
    (4095, 512, 8, 2, "bf16"), (4096, 512, 8, 2, "bf16"), (3583, 512, 8, 2, "f32"), (3584, 512, 8, 2, "f32"),
    (1819, 320, 10, 3, "bf16"), (65, 512, 5, 2, "bf16"),
    # ... up to 32 experts of wide rows, and an expert per lane past them (E = 32)
    (2047, 1088, 32, 2, "bf16"), (2049, 1088, 32, 2, "bf16"), (1793, 1088, 32, 2, "f32"),
    # the fused kernel: few or narrow
    (65, 128, 8, 2, "bf16"), (65, 192, 9, 2, "bf16"), (3583, 64, 16, 2, "bf16"), (3584, 64, 16, 2, "f32"),
    (900, 192, 9, 2, "bf16"), (65, 512, 4, 2, "bf16"),
    # an expert per lane, 1 and 2 tokens a wave
    (896, 128, 64, 6, "bf16"), (2048, 128, 40, 2, "bf16"), (2049, 192, 60, 4, "bf16"), (2049, 64, 64, 1, "f32"),
    # ... from 4096 tokens on by price, with the logits where the expert outputs come
    # later: 2 and 4 tokens a wave (fp32 rows: 2), and fused past it
    (4097, 512, 64, 2, "bf16"), (6147, 1024, 64, 2, "bf16"), (6147, 1024, 57, 2, "f32"),
    (16383, 256, 64, 2, "bf16"), (4097, 64, 32, 2, "bf16"), (9001, 64, 32, 2, "f32"), (16385, 64, 40, 2, "bf16"),
    # ids counted by the permute (up to 256 tokens) and by a launch of its own
    (190, 64, 33, 8, "bf16"), (256, 256, 16, 2, "bf16"), (256, 64, 512, 8, "f32"), (257, 64, 17, 8, "bf16"),
    # more than 64 experts: product and chain waves, an expert per lane (1, 2 and 4
    # tokens a wave), and past the widest rows of the lane layout the grouped kernel
    (511, 64, 65, 4, "bf16"), (513, 128, 70, 4, "bf16"), (1030, 64, 128, 8, "f32"),
    (3075, 64, 100, 3, "bf16"), (1025, 64, 512, 8, "bf16"), (127, 64, 300, 8, "bf16"),
]


def path(N, C, E, act, norm=False):
    """The launch rule, restated: which kernel forms a call's logits, where the
    workspace has room for them and for normalised rows (`norm`: they are asked for)."""
    C = -(-C // 64) * 64   # the library pads
    if E <= 64 and N <= 64 and C <= 8192:
        return "one launch"
    groups, nb, quads = -(-E // 64), -(-N // 64), C <= 8192
    f32 = act == "f32"

    def lane(pairs):
        return "lane 1" if pairs <= 2048 else "lane 2" if pairs <= 6144 or (f32 and groups == 1) else "lane 4"

    if E > 64:
        if norm and C <= 4096 and (C <= 2048 or N < 4096):
            return "rows, " + path(N, C, E, "f32")
        if not norm and quads and N * groups >= 1024:
            return lane(N * groups)
        if nb * groups >= 256:
            return "grouped"
        return "split" if norm else "product and chain"
    wide, NE = f32 or norm, N * E
    many = NE > (65536 if E <= 32 and C > 1024 and not wide else 57343)
    lane_us = 10 + N * (0.9e-3 + (4.1e-6 if f32 else 3.6e-6) * C)
    fused_us = (10 + C * (0.011 + 0.73e-3 * E)) * -(-nb // 256)
    by_lane = quads and many and E > 16 and (N < 4096 or lane_us < fused_us)
    if E > 16:
        pc = N < 4096
    elif E > 8:
        pc = C >= 256 and NE < min(40960 if wide else 57344, 64 * C)
    else:
        pc = E > 4 and C >= 512 and NE < (28672 if wide else 32768)
    if norm:
        rows = (by_lane or pc) and C <= 4096
        if E <= 16:
            rows = rows and NE < (48 if E > 8 else 40) * min(C, 1024)
        elif N < 4096:
            rows = rows and C >= 256 and (nb * -(-E // 4) > 256 or N <= (2048 if C >= 512 else 1024))
        else:
            rows = rows and E * C >= 30000 and N <= (6144 if E > 32 else 4096)
        if rows:
            return "rows, " + path(N, C, E, "f32")
        return "split" if E > 16 and N < 4096 else "fused"
    if by_lane:
        return lane(N)
    return "product and chain" if pc else "fused"


def test_shapes_reach_every_path():
    got = {path(N, C, E, act) for N, C, E, k, act in SHAPES}
    assert got >= {"one launch", "product and chain", "fused", "lane 1", "lane 2", "lane 4"}
    for big in (False, True):
        assert {"lane 2", "lane 4"} <= {path(N, C, E, act) for N, C, E, k, act in SHAPES if (E > 64) == big}
    assert {"lane 2", "lane 4"} <= {path(N, C, E, act) for N, C, E, k, act in SHAPES if N >= 4096 and E <= 64}
    norm = {path(N, C, E, act, norm=True) for N, C, E, k, act, H in NORM_SHAPES}
    assert norm >= {"one launch", "fused", "split", "grouped", "rows, product and chain", "rows, lane 1",
                    "rows, lane 2", "rows, lane 4"}


@pytest.mark.parametrize("N,C,E,k,act", SHAPES)
@pytest.mark.parametrize("train", [False, True])
def test_routing_bit_exact(N, C, E, k, act, train):
    cfg = wl.MoEConfig("paths", N, C, E, k, 8, act, act, "normal")
    inp = wl.make_inputs(cfg, seed=N + E, bias_std=0.02)
    # a router of ordinary fp32 weights: products that do round
    inp.Wr[:] = wl.normal_f32(7, 3, C * E, std=0.05).reshape(C, E)
    inp.x[min(3, N - 1), :] = 0.0   # equal logits up to the bias
    layer = MoELayer(C, 8, E, k, act=act)
    layer.load_parameters(inp.params())
    x = torch.from_numpy(inp.x).to("cuda").to(layer.dtype)
    layer.forward(x, train=train)
    torch.cuda.synchronize()
    r = {n: t.cpu().numpy() for n, t in layer.routing().items()}
    ref = O.forward(inp, with_y=False)
    assert np.array_equal(r["topk_idx"], ref["idx"])
    assert np.array_equal(r["topk_p"], ref["topp"])
    assert np.array_equal(r["counts"], ref["counts"])
    assert np.array_equal(r["perm"], ref["perm"])


# (N, C, E, k, act, H): normalised rows
NORM_SHAPES = [
    # one launch, the block's own 1/rms (the widest rows: every product buffer holds squares)
    (1, 64, 1, 1, "f32", 8), (64, 1024, 16, 2, "bf16", 8), (33, 4160, 8, 2, "bf16", 8), (64, 192, 64, 8, "f32", 8),
    (17, 8192, 16, 2, "bf16", 8), (3, 8192, 33, 2, "f32", 8),
    # rows normalised once, on both sides of the lines of its rule
    (65, 1024, 16, 2, "bf16", 8), (2559, 1024, 16, 2, "bf16", 8), (2560, 1024, 16, 2, "bf16", 8),
    (258, 512, 8, 2, "f32", 8), (2559, 512, 8, 2, "bf16", 8), (2560, 512, 8, 2, "bf16", 8),
    (1025, 256, 20, 2, "bf16", 8), (2049, 512, 64, 6, "bf16", 8),
    (4095, 512, 60, 2, "bf16", 8), (4097, 576, 64, 2, "bf16", 8), (6145, 512, 64, 2, "bf16", 8),
    # the widest rows that are normalised once
    (70, 4096, 16, 2, "bf16", 8), (66, 4096, 70, 2, "f32", 8),
    # no room for the rows (top-1, few hidden units), rows too wide for their kernel
    (300, 2048, 16, 1, "bf16", 8), (100, 4160, 16, 2, "bf16", 8),
    # more than 64 experts
    (65, 64, 65, 4, "bf16", 8), (513, 128, 128, 8, "f32", 8), (1030, 64, 300, 3, "bf16", 8),
    (3075, 64, 100, 3, "bf16", 8),
    # ... in groups of 64 where the rows cannot be normalised once: too wide, no room
    (8193, 4160, 70, 2, "bf16", 8), (2049, 320, 500, 1, "bf16", 8),
    # a width that the library pads
    (70, 200, 16, 2, "bf16", 8), (20, 200, 16, 2, "f32", 8),
]


@pytest.mark.parametrize("N,C,E,k,act,H", NORM_SHAPES)
def test_normalised_routing_bit_exact(N, C, E, k, act, H):
    """The same for the fused block's routing on RMSNorm(x) * gamma, with its
    1/rms, from a gamma that is only 4-byte aligned."""
    cfg = wl.MoEConfig("paths", N, C, E, k, H, act, act, "normal")
    inp = wl.make_inputs(cfg, seed=N + E, bias_std=0.02)
    inp.Wr[:] = wl.normal_f32(7, 3, C * E, std=0.05).reshape(C, E)
    inp.x[min(3, N - 1), :] = 0.0
    layer = MoELayer(C, H, E, k, act=act)
    layer.load_parameters(inp.params())
    x1 = inp.x.copy()
    gamma = (np.float32(1.0) + wl.normal_f32(9, 5, C, std=0.2)).astype(np.float32)
    g = torch.zeros(C + 1, device="cuda")[1:].copy_(torch.from_numpy(gamma))
    layer.forward_block(torch.from_numpy(x1).to("cuda").to(layer.dtype), g, 1e-5)
    torch.cuda.synchronize()
    r = {n: t.cpu().numpy() for n, t in layer.routing().items()}
    xn, rstd = O.rmsnorm_scaled(x1, gamma, 1e-5)
    inp.x[:] = xn
    ref = O.forward(inp, with_y=False)
    assert np.array_equal(layer.rstd().cpu().numpy(), rstd.reshape(-1))
    assert np.array_equal(r["topk_idx"], ref["idx"])
    assert np.array_equal(r["topk_p"], ref["topp"])
    assert np.array_equal(r["counts"], ref["counts"])
    assert np.array_equal(r["perm"], ref["perm"])


def test_grouped_logits_of_plain_rows():
    """Past the width of the expert-per-lane layout, more than 64 experts form plain
    rows' logits in groups of 64 (the last one of six)."""
    N, C, E, k = 8150, 8256, 70, 1
    assert path(N, C, E, "bf16") == "grouped"
    cfg = wl.MoEConfig("paths", N, C, E, k, 8, "bf16", "bf16", "normal")
    inp = wl.make_inputs(cfg, seed=5, bias_std=0.02)
    inp.Wr[:] = wl.normal_f32(7, 3, C * E, std=0.01).reshape(C, E)
    layer = MoELayer(C, 8, E, k, act="bf16")
    layer.load_parameters(inp.params())
    layer.forward(torch.from_numpy(inp.x).to("cuda").bfloat16())
    r = layer.routing()
    ref = O.forward(inp, with_y=False)
    assert np.array_equal(r["topk_idx"].cpu().numpy(), ref["idx"])
    assert np.array_equal(r["topk_p"].cpu().numpy(), ref["topp"])
    assert np.array_equal(r["counts"].cpu().numpy(), ref["counts"])
