"""The MoE layer at the edges of its expert GEMMs' tiles: one row to several
16- and 32-row chunks per expert, experts without rows, every token on one
expert, column and K remainders. TILES names the tiles of a size (gate/up,
down), and asserts that they run there.

Bound: float64 from the same bf16 weights, 2e-5 of the output in the 2-norm
(two bf16 terms per activation through two GEMMs measure 0.9e-5; one term
would give 3e-3).
"""
import numpy as np
import pytest
import torch

from gorch_amd import synthetic as syn
from gorch_amd.bf16 import bf16_to_f32

pytestmark = pytest.mark.gpu


def reference(w, x, logits):
    order = np.argsort(-logits, axis=1, kind="stable")[:, : w["top_k"]]
    val = np.take_along_axis(logits.astype(np.float64), order, 1)
    wts = np.exp(val - val.max(1, keepdims=True))
    wts /= wts.sum(1, keepdims=True)
    out = np.zeros(x.shape, np.float64)
    for e in range(w["experts"]):
        rows, slot = np.nonzero(order == e)
        if not len(rows):
            continue
        W = {k: bf16_to_f32(w[k][e]).astype(np.float64) for k in ("wgate", "wup", "wdown")}
        xe = x[rows].astype(np.float64)
        g = xe @ W["wgate"].T + w["bgate"][e]
        u = xe @ W["wup"].T + w["bup"][e]
        y = (g / (1 + np.exp(-g)) * u) @ W["wdown"].T + w["bdown"][e]
        np.add.at(out, rows, y * wts[rows, slot][:, None])
    return out


@pytest.mark.parametrize("M,dim,ffn,E,K,skew", [
    (1, 64, 64, 4, 1, 0), (1, 72, 104, 8, 2, 0), (16, 264, 520, 8, 2, 0), (16, 64, 2056, 8, 2, 99), (33, 128, 192, 4, 2, 0),
    (70, 1032, 136, 8, 2, 0), (64, 512, 1368, 4, 2, 0), (150, 96, 264, 4, 2, 99), (300, 200, 328, 4, 2, 0),
    (129, 64, 4096, 2, 1, 0), (700, 320, 256, 8, 2, 1), (31, 40, 24, 64, 8, 0),
    # more rows: the 128-, 192- and 256-wide down tiles
    (1000, 1032, 136, 4, 2, 0), (1500, 1288, 72, 4, 2, 0), (900, 1544, 136, 8, 2, 0), (2048, 1544, 64, 8, 2, 0),
])
def test_moe_few_rows(gpu, M, dim, ffn, E, K, skew):
    """skew pushes tokens towards expert 0 (99: every token's first choice)."""
    x, logits, w = syn.moe_inputs(M=M, dim=dim, ffn=ffn, experts=E, top_k=K, seed=M + dim)
    rng = np.random.default_rng(M)
    logits[:, 0] += skew
    for k in ("bgate", "bup", "bdown"):
        w[k] = [(0.1 * rng.standard_normal(b.shape)).astype(np.float32) for b in w[k]]
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    out, _, _ = gpu.MoE(w).forward(dev(x), dev(logits))
    ref = reference(w, x, logits)
    assert np.linalg.norm(out.cpu().numpy() - ref) <= 2e-5 * np.linalg.norm(ref)


TILES = [
    (17, 48, 80, 2, 1, "kw32x32", "kw16x32"), (14, 40, 72, 2, 2, "kw32x32", "kw32x32"), (139, 40, 40, 4, 1, "kw32x32", "kw32x64"),
    (266, 56, 48, 64, 8, "kw32x32", "wide128"), (220, 416, 40, 64, 1, "kw32x32", "wide192"),
    (127, 520, 40, 64, 1, "kw32x32", "wide256"), (84, 40, 272, 64, 1, "wide128", "kw16x32"),
    (700, 40, 136, 64, 1, "wide128", "kw32x32"), (122, 40, 48, 2, 2, "wide128", "kw32x64"),
    (856, 40, 48, 32, 8, "wide128", "wide128"), (590, 1304, 40, 16, 2, "wide128", "wide192"),
    (740, 280, 40, 64, 8, "wide128", "wide256"),
]


@pytest.mark.parametrize("M,dim,ffn,E,K,gate_up,down", TILES)
@pytest.mark.parametrize("skew", [0, 1])
def test_moe_each_tile(gpu, M, dim, ffn, E, K, gate_up, down, skew):
    assert gpu.kernel_choice("moe_gate_up", M, dim, ffn, E, K) == gate_up
    assert gpu.kernel_choice("moe_down", M, dim, ffn, E, K) == down
    test_moe_few_rows(gpu, M, dim, ffn, E, K, skew)


@pytest.mark.parametrize("M,dim,E,K", [(1, 40, 1, 1), (15, 1032, 5, 2), (16, 64, 8, 2), (17, 520, 8, 1), (64, 264, 7, 2),
                                       (65, 264, 7, 2), (33, 2056, 2, 2)])
def test_moe_router_batch(gpu, M, dim, E, K):
    """The router, top-K and grouping of a decode batch in one launch (up to
    64 tokens; 65 takes the Linear and the routing block): choices and weights
    from float64 logits (the seeds keep every top-K gap above 1e-4). On the
    weights 1e-6 up to 64 tokens: three bf16 terms carry x to 2^-24, and a
    logit takes up to 2056 / 32 / 16 + 16 roundings of partial sums below 8,
    2^-22 each, which as a random walk is 1.2e-6 of the logit and at most half
    of that of a weight; 5e-5 at 65 (two terms: 2^-16 of a |x||w| sum of 4, a
    quarter of it through the softmax, 1.6e-5)."""
    x, _, w = syn.moe_inputs(M=M, dim=dim, ffn=64, experts=E, top_k=K, seed=3 * M + E, with_router=True)
    rng = np.random.default_rng(M)
    w["br"] = rng.standard_normal(E).astype(np.float32)
    logits = x.astype(np.float64) @ bf16_to_f32(w["wr"]).astype(np.float64).T + w["br"]
    if K < E:
        s = -np.sort(-logits, axis=1)
        assert (s[:, K - 1] - s[:, K]).min() > 1e-4
    out, idx, wts = gpu.MoE(w).forward(torch.from_numpy(x).cuda())
    order = np.argsort(-logits, axis=1, kind="stable")[:, :K]
    val = np.take_along_axis(logits, order, 1)
    p = np.exp(val - val.max(1, keepdims=True))
    assert np.array_equal(idx.cpu().numpy(), order)
    assert np.abs(wts.cpu().numpy() - p / p.sum(1, keepdims=True)).max() <= (1e-6 if M <= 64 else 5e-5)
    ref = reference(w, x, logits)
    assert np.linalg.norm(out.cpu().numpy() - ref) <= 3e-5 * np.linalg.norm(ref)
