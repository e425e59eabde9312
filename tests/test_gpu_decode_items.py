"""The widths of the fp8 decode kernel's work items (gemm_decode.hip).  Steps of
bf16 rows from 4 rows per expert on take items of 256 features where those
nearly fill rounds of the CUs over long contractions, and of 128 or 64
otherwise.  An item's width does not enter the order of a sum, so a step's rows
are bit for bit what the same rows give in steps of under 4 rows per expert,
which never take 256-feature items (those are held against the oracle in the
parity and decode tests).
"""
import math

import pytest
import torch

from mgpt_amd.moe import MoELayer

pytestmark = pytest.mark.gpu

# (N, C, E, k, H, which products take 256-feature items)
STEPS = [
    # one token past 32 rows per expert: the gathering gate/up product, and the other one
    (129, 4096, 8, 2, 2048, "gate/up"), (257, 4096, 16, 2, 1024, "gate/up"),
    # one token under 64: a third row tile at many experts
    (255, 4096, 8, 2, 2048, "gate/up"), (511, 4096, 16, 2, 1024, "gate/up"),
    # both products; a last round of half a tile in six, 11 stages per contraction
    (300, 4096, 16, 2, 2048, "both"), (352, 2048, 64, 8, 1408, "both"),
    # one row tile an expert: the fewest rows, and the most, over 8 rounds
    (64, 1024, 64, 4, 4096, "gate/up"), (512, 1024, 64, 4, 4096, "gate/up"),
    # one token fewer than those take, and contractions too short for one row tile
    (63, 1024, 64, 4, 4096, ""), (64, 2048, 64, 8, 1408, ""), (256, 4096, 16, 2, 1024, ""),
    # under eight blocks, part rounds, short contractions: neither
    (700, 2048, 64, 4, 512, ""), (352, 1024, 16, 2, 2816, ""), (700, 512, 64, 4, 1024, ""),
]


def wide(rows, E, K, features, cus):
    """launch_decode's rule for bf16 rows."""
    nb = -(-features // 256)
    tiles = 2 if rows > 32 * E else 1
    rounds = float(tiles * E * nb) / cus
    return (4 * E <= rows < 64 * E and K >= 1024 and nb >= 8 and rounds * K >= 8192 / tiles
            and rounds > 0.9 * math.ceil(rounds))


def test_the_steps_reach_what_they_claim():
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus != 256:
        pytest.skip("the steps are those of 256 CUs")
    for N, C, E, k, H, takes in STEPS:
        got = [wide(N * k, E, C, 2 * H, cus), wide(N * k, E, H, C, cus)]
        assert got == [takes in ("gate/up", "both"), takes == "both"], (N, C, E, k, H)


@pytest.mark.parametrize("N,C,E,k,H,takes", STEPS)
@pytest.mark.parametrize("skewed", [False, True])
def test_a_step_gives_its_rows_what_small_steps_give(N, C, E, k, H, takes, skewed):
    gen = torch.Generator(device="cuda").manual_seed(N + C + H)

    def normal(*shape, std):
        return torch.randn(*shape, generator=gen, device="cuda").mul_(std)

    # skewed: the first expert takes several row tiles, the last ones none
    bias = -0.5 * torch.arange(E, device="cuda", dtype=torch.float32) if skewed else torch.zeros(E, device="cuda")
    params = [normal(C, E, std=0.02), bias.view(1, E)]
    for _ in range(E):
        params += [normal(C, H, std=0.02), normal(H, std=0.02), normal(C, H, std=0.02),
                   normal(H, std=0.02), normal(H, C, std=0.02), normal(C, std=0.02)]
    layer = MoELayer(C, H, E, k, act="bf16", weights="fp8")
    layer.load_parameters(params)
    x = normal(N, C, std=1.0).bfloat16()
    y = layer.forward(x).clone()
    idx = layer.routing()["topk_idx"].clone()
    assert torch.isfinite(y.float()).all()
    small = (4 * E - 1) // k
    for t in range(0, N, small):
        part = layer.forward(x[t:t + small].contiguous())
        assert torch.equal(layer.routing()["topk_idx"], idx[t:t + small])
        assert torch.equal(part, y[t:t + small]), t
