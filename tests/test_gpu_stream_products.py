"""The weight-streaming expert products (gemm_stream.hip) at the edges of what
they take: bf16 weights under 64 rows per expert (and narrow down products
above), fp8 weights outside the decode kernel's range.  Segments that end
inside, at and one past a 64- or 256-row tile, one token, contractions of one
slab and of 64, widths that are not a multiple of 128, more experts than a wave
has lanes, and training through the 64-row tiles.  Against the oracle at the
layer's bars (bf16 2e-2, fp8 6e-2 of the fp32 path, which rounds the rows and
products in between), against the same rows one token at a time, which other
tiles compute, at a few bf16 roundings, and bit for bit against the 128 x 128 tiles.
"""
import numpy as np
import pytest
import torch

import oracle_lib as O
from mgpt_amd import workload as wl
from mgpt_amd.moe import MoELayer

pytestmark = pytest.mark.gpu

# (N, C, E, k, H, weights)
SHAPES = [
    (1, 64, 4, 2, 64, "bf16"), (1, 1024, 16, 2, 2816, "bf16"), (24, 1024, 4, 2, 2112, "bf16"),
    (63, 192, 3, 1, 96, "bf16"), (130, 320, 2, 1, 4096, "bf16"), (257, 256, 4, 2, 2560, "bf16"),
    (900, 128, 4, 2, 3000, "bf16"), (70, 64, 70, 2, 40, "bf16"),
    (255, 128, 1, 1, 128, "fp8"), (257, 128, 1, 1, 192, "fp8"), (300, 192, 3, 2, 160, "fp8"),
    (40, 192, 3, 2, 160, "fp8"), (600, 256, 8, 3, 1408, "fp8"), (260, 128, 80, 3, 96, "fp8"),
    (9, 128, 70, 2, 96, "fp8"),
    # groups of 64 experts as rows of one grid: 64- and 256-row tiles
    (2, 64, 130, 2, 2112, "bf16"), (700, 64, 130, 1, 64, "bf16"), (2400, 64, 70, 2, 96, "bf16"),
    (4300, 128, 130, 2, 64, "bf16"), (2500, 128, 70, 2, 96, "fp8"),
    # enough tiles for 256 x 256 fp8 ones in both products, with and without groups
    (2100, 576, 6, 4, 160, "fp8"), (2400, 576, 70, 4, 160, "fp8"),
]


@pytest.mark.parametrize("N,C,E,k,H,weights", SHAPES)
def test_forward_against_the_oracle(N, C, E, k, H, weights):
    cfg = wl.MoEConfig("stream", N, C, E, k, H, "bf16", weights, "normal")
    inp = wl.make_inputs(cfg, seed=N + C, bias_std=0.05)
    layer = MoELayer(C, H, E, k, act="bf16", weights=weights)
    layer.load_parameters(inp.params(raw=True))
    x = torch.from_numpy(inp.x).to("cuda").bfloat16()
    y = layer.forward(x)
    idx = layer.routing()["topk_idx"].cpu().numpy()
    ref = O.forward(inp)
    assert np.array_equal(idx, ref["idx"])
    bar = 2e-2 if weights == "bf16" else 6e-2
    err = np.linalg.norm(y.float().cpu().numpy() - ref["y"]) / np.linalg.norm(ref["y"])
    assert err < bar, err
    again = layer.forward(x)
    assert torch.equal(y, again)
    # a few of the rows by themselves: h and the output are rounded to bf16 (2^-9
    # each), sums differ by fp32 roundings, so within two bf16 steps of the row
    for t in sorted({0, N // 2, N - 1}):
        one = layer.forward(x[t:t + 1].contiguous()).float()
        scale = y[t].float().abs().max()
        assert (one[0] - y[t].float()).abs().max() <= 2.0 ** -6 * scale, t


@pytest.mark.parametrize("N,C,E,k,H", [(24, 128, 8, 2, 256), (70, 192, 6, 3, 100), (1, 64, 2, 1, 2100)])
def test_training_through_few_rows(N, C, E, k, H):
    cfg = wl.MoEConfig("stream", N, C, E, k, H, "bf16", "bf16", "normal")
    inp = wl.make_inputs(cfg, seed=N, bias_std=0.05)
    dy = wl.bf16_round(wl.normal_f32(5, 1, N * C).reshape(N, C))
    layer = MoELayer(C, H, E, k, act="bf16")
    layer.load_parameters(inp.params())
    layer.forward(torch.from_numpy(inp.x).to("cuda").bfloat16(), train=True)
    dx = layer.backward(torch.from_numpy(dy).to("cuda").bfloat16())
    ref = O.backward(inp, dy)
    g = [t.cpu().numpy() for t in layer.get_gradients()]
    got = [dx.float().cpu().numpy(), g[0], g[1]]
    got += [np.stack([g[2 + 6 * e + i] for e in range(E)]) for i in range(6)]
    for name, a in zip(("dx",) + tuple(O.GRAD_NAMES), got):
        b = np.asarray(ref[name], np.float64).reshape(a.shape)
        assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b) + 1e-12, name


@pytest.mark.parametrize("N,C,E,k,H,weights", [(24, 128, 4, 2, 256, "bf16"), (1, 64, 70, 2, 64, "bf16"),
                                               (600, 128, 4, 2, 192, "fp8"), (40, 192, 3, 2, 160, "fp8")])
def test_gate_times_up_past_the_range(N, C, E, k, H, weights):
    """silu(g) * u where g * u overflows but the result does not: g = -1e20 and
    u = 1e20 give -0, so each expert returns its output bias."""
    gen = torch.Generator().manual_seed(N)
    p = [torch.randn(C, E, generator=gen), torch.zeros(1, E)]
    for e in range(E):
        p += [torch.zeros(C, H), torch.full((1, H), -1e20), torch.zeros(C, H), torch.full((1, H), 1e20),
              torch.randn(H, C, generator=gen), torch.full((1, C), 1.0 + e % 4)]
    layer = MoELayer(C, H, E, k, act="bf16", weights=weights)
    layer.load_parameters([t.cuda() for t in p])
    y = layer.forward(torch.randn(N, C, generator=gen).cuda().bfloat16()).float().cpu()
    r = layer.routing()
    want = (r["topk_p"].cpu() * (1.0 + (r["topk_idx"].cpu() % 4))).sum(1, keepdim=True).expand(N, C)
    # a bf16 rounding of the output
    assert (y - want).abs().max() <= 2.0 ** -8 * want.abs().max()


# every expert gets rows in both calls: few rows (64 x 128 tiles; fp8 from 32 rows an
# expert on 256 x 256 ones) against at least 64 an expert in 128 x 128 tiles
@pytest.mark.parametrize("N,C,E,k,H,weights", [(40, 192, 4, 2, 160, "bf16"), (24, 1024, 16, 2, 2816, "bf16"),
                                               (40, 192, 4, 2, 160, "fp8"), (300, 192, 4, 2, 160, "fp8"),
                                               (400, 512, 8, 3, 704, "fp8")])
def test_same_bits_as_the_128_row_tiles(N, C, E, k, H, weights, monkeypatch):
    """One order of sums, one form of the epilogue: the products equal those of the
    register-staged 128 x 128 tiles bit for bit.  fp8 weights lie on the e4m3 grid with
    power-of-two scales, so the same values are exact in bf16 and the scales commute
    with every rounding."""
    gen = torch.Generator().manual_seed(N + C)

    def weight(i, o):
        q = (torch.randn(i, o, generator=gen) * 20).to(torch.float8_e4m3fn).float()
        q[0] = 448.0   # the channel's largest: scale 2^-9
        return q * 2.0 ** -9

    p = [torch.randn(C, E, generator=gen) * 0.1, torch.zeros(1, E)]
    for _ in range(E):
        p += [weight(C, H), torch.randn(1, H, generator=gen), weight(C, H), torch.randn(1, H, generator=gen),
              weight(H, C), torch.randn(1, C, generator=gen)]
    p = [t.cuda() for t in p]
    x = torch.randn(N, C, generator=gen).cuda().bfloat16()
    layer = MoELayer(C, H, E, k, act="bf16", weights=weights)
    layer.load_parameters(p)
    y = layer.forward(x)
    monkeypatch.setenv("MGPT_MOE_GEMM_TILE", "128")
    tiles = MoELayer(C, H, E, k, act="bf16")
    tiles.load_parameters(p)
    many = x.repeat(-(-64 * E // (N * k)), 1)
    assert torch.equal(y, tiles.forward(many)[:N])
