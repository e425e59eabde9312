"""The fp32 expert products (gemm_f32.hip) at the edges of their tiles.

The tile (32 x 32 to 64 x 128) and whether a block's waves share it go by the
number of tiles per CU; all of them meet segments that end inside, at and one
past a tile, widths below a tile, contractions of odd length, and odd leading
dimensions.  Forward, input gradient and every
parameter gradient against the same formulas in float64 under the layer's own
routing.

Tolerance: a sum of K products in fp32, each within 2^-24, in any order, is
within K * 2^-24 of its terms' absolute sum; for terms of random sign that sum
is about sqrt(K) times the result, and the errors themselves add like
sqrt(K), so the relative error stays near 2^-24 * sqrt(K) per product, K up
to 4096 here: 4e-6, over a chain of up to three products.
"""
import pytest
import torch

from mgpt_amd.moe import MoELayer

pytestmark = pytest.mark.gpu
TOL = 1.2e-5

# (N, C, H, E, k): one row; segments around 64 and 128 rows; odd widths; one
# expert; more experts than a wave has lanes; many rows of narrow layers (every tile of
# the down and input-gradient products, the largest with a column tile half empty);
# many wide experts (a weight-gradient tile a wave)
SHAPES = [
    (1, 64, 32, 4, 2), (63, 64, 64, 1, 1), (65, 128, 96, 1, 1), (129, 72, 33, 2, 1),
    (257, 200, 130, 3, 2), (1000, 130, 257, 5, 2), (4100, 256, 1024, 4, 2), (700, 512, 1376, 8, 2),
    (900, 64, 40, 70, 3), (8200, 64, 2560, 4, 2), (300, 256, 768, 70, 3),
    (24600, 192, 40, 4, 2), (42003, 192, 40, 4, 2), (100, 512, 1376, 40, 2),
]


def choices(N, C, H, E, k):
    """The tiles that the products of a call take, by the launch rules restated."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    up = lambda v, m: -(-v // m)
    C, Hp = up(C, 64) * 64, up(H, 128) * 128
    t = lambda cols: up(N * k, 64) * up(cols, 128)

    def down(cols):
        return "64x128" if t(cols) >= 10 * cus else "32x64" if t(cols) >= 3 * cus else "32x32"

    def wgrad(i, j):
        return "a wave" if up(up(i, 64), 2) * up(up(j, 64), 2) * E >= 6 * cus else "four waves"

    return {("gate/up", "64x128" if t(2 * Hp) >= 4 * cus else "32x64"), ("down, dx", down(C)),
            ("d(act)", down(Hp)), ("dW_down", wgrad(H, C)), ("dW_gate/up", wgrad(C, 2 * Hp))}


def test_shapes_reach_every_tile():
    got = set().union(*(choices(*s) for s in SHAPES))
    assert got == {("gate/up", "64x128"), ("gate/up", "32x64"), ("down, dx", "64x128"), ("down, dx", "32x64"),
                   ("down, dx", "32x32"), ("d(act)", "64x128"), ("d(act)", "32x64"), ("d(act)", "32x32"),
                   ("dW_down", "a wave"), ("dW_down", "four waves"), ("dW_gate/up", "a wave"),
                   ("dW_gate/up", "four waves")}


def _exact(layer, x, p, dy, E):
    r = layer.routing()
    idx, P = r["topk_idx"].long(), torch.softmax(x.double() @ p[0].double() + p[1].double(), 1)
    P = P.clamp(1e-7, 1.0)
    N = x.shape[0]
    y, dx = torch.zeros_like(x).double(), torch.zeros_like(x).double()
    dP = torch.zeros_like(P)
    g = [torch.zeros(t.shape, dtype=torch.float64, device="cuda") for t in p]
    for e in range(E):
        hit = (idx == e).any(1).nonzero().flatten()
        dP[:, e] += 0.01 * E * (hit.numel() / N) / N
        if not hit.numel():
            continue
        Wg, bg, Wu, bu, Wd, bd = (t.double() for t in p[2 + 6 * e:8 + 6 * e])
        xe, de, pe = x.double()[hit], dy.double()[hit], P[hit, e][:, None]
        gt, up = xe @ Wg + bg, xe @ Wu + bu
        sig = torch.sigmoid(gt)
        h = gt * sig * up
        o = h @ Wd + bd
        y[hit] += pe * o
        dP[hit, e] += (o * de).sum(1)
        do = de * pe
        dh = do @ Wd.t()
        du, dg = dh * gt * sig, dh * up * sig * (1 + gt * (1 - sig))
        dx[hit] += dg @ Wg.t() + du @ Wu.t()
        for i, v in enumerate((xe.t() @ dg, dg.sum(0, True), xe.t() @ du, du.sum(0, True),
                               h.t() @ do, do.sum(0, True))):
            g[2 + 6 * e + i] = v
    dL = P * (dP - (dP * P).sum(1, True))
    g[0], g[1] = x.double().t() @ dL, dL.sum(0, True)
    return [y, dx + dL @ p[0].double().t()] + g


@pytest.mark.parametrize("N,C,H,E,k", SHAPES)
def test_products_against_float64(N, C, H, E, k):
    gen = torch.Generator(device="cuda").manual_seed(N + C)

    def normal(*s, std=1.0):
        return torch.randn(*s, generator=gen, device="cuda") * std

    p = [normal(C, E, std=0.02), normal(1, E, std=0.5)]
    for _ in range(E):
        p += [normal(C, H, std=0.05), normal(1, H, std=0.05), normal(C, H, std=0.05),
              normal(1, H, std=0.05), normal(H, C, std=0.05), normal(1, C, std=0.05)]
    x, dy = normal(N, C), normal(N, C)
    layer = MoELayer(C, H, E, k, act="f32")
    layer.load_parameters(p)
    y = layer.forward(x, train=True)
    dx = layer.backward(dy)
    got = [y, dx] + layer.get_gradients()
    want = _exact(layer, x, p, dy, E)
    # a second step adds onto the gradients of the first
    layer.forward(x, train=True)
    layer.backward(dy)
    twice = layer.get_gradients()
    for i, (a, b) in enumerate(zip(got, want)):
        norm = b.norm()
        err = (a.double() - b).norm()
        assert err <= TOL * norm, f"output {i}: {float(err / norm):.2e}"
        if i >= 2:
            assert torch.equal(twice[i - 2], a + a), f"gradient {i - 2} of two steps"
