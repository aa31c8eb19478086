"""The prefill attention kernel at the edges of its tiles: rows around the
16- and 32-row groups, keys around the 64-key stages and 16-key groups, paired
and unpaired query heads, causal and not, few rows of many sequences, NaNs in the
cache rows past the last key; the form without key groups (128 rows a block,
or 64 of two heads) at the edges of its own tiles.

Bound: float64 attention over the same inputs, 1e-6 in the 2-norm (f32
products and sums over up to 700 keys measure 2-4e-7; probabilities rounded
to bf16 would give 1e-3).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# batch, new rows, cached before, query heads, KV heads, head_dim, causal
CASES = [
    (1, 32, 0, 2, 2, 64, 1), (2, 33, 0, 3, 3, 64, 1), (1, 47, 17, 4, 2, 64, 1), (1, 64, 0, 7, 1, 64, 1),
    (1, 65, 63, 2, 1, 128, 1), (2, 97, 1, 4, 4, 128, 1), (1, 130, 127, 2, 2, 64, 0), (1, 48, 16, 6, 3, 128, 0),
    (3, 63, 65, 1, 1, 128, 1), (1, 700, 0, 2, 1, 64, 1), (1, 257, 300, 1, 1, 128, 1),
    (16, 4, 70, 25, 25, 64, 1), (24, 5, 0, 14, 2, 64, 1), (16, 13, 191, 16, 8, 128, 0),
]


ONE_GROUP = [
    (24, 33, 0, 14, 2, 64, 1), (24, 33, 0, 14, 2, 64, 0), (5, 129, 60, 25, 25, 64, 1), (12, 40, 5, 32, 16, 64, 1),
    (12, 65, 127, 32, 16, 64, 0), (30, 33, 100, 12, 12, 128, 1), (7, 145, 47, 19, 19, 128, 1), (14, 47, 17, 32, 8, 128, 1),
    (14, 64, 128, 32, 8, 128, 0),
    # mostly cached keys, past three stages
    (12, 57, 180, 32, 8, 128, 1), (12, 64, 321, 32, 8, 128, 0),
]


@pytest.mark.parametrize("case,name", [(c, "prefill_kg4") for c in CASES] + [(c, "prefill_kg1") for c in ONE_GROUP],
                         ids=lambda c: "x".join(map(str, c)) if isinstance(c, tuple) else c)
def test_flash_tiles(gpu, case, name):
    B, n, pos, hq, hkv, hd, causal = case
    assert gpu.kernel_choice("attention", B, n, pos, hq, hkv, hd, pos + n + 5) == name
    rng = np.random.default_rng(n + pos + hq)
    T, cap = pos + n, pos + n + 5
    q = rng.standard_normal((B, n, hq, hd)).astype(np.float32)
    k = np.full((B, cap, hkv, hd), np.nan, np.float32)
    v = np.full((B, cap, hkv, hd), np.nan, np.float32)
    k[:, :T] = rng.standard_normal((B, T, hkv, hd))
    v[:, :T] = rng.standard_normal((B, T, hkv, hd))
    out = torch.full((B * n, hq * hd), float("nan"), device="cuda")
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    gpu.gqa_attention_cached(dev(q).reshape(B * n, -1), dev(k).reshape(B, cap, -1), dev(v).reshape(B, cap, -1), out, B,
                             n, pos, hq, hkv, hd, cap, causal)
    kk = np.repeat(k[:, :T].astype(np.float64), hq // hkv, 2)
    vv = np.repeat(v[:, :T].astype(np.float64), hq // hkv, 2)
    s = np.einsum("bihd,bjhd->bhij", q.astype(np.float64), kk) / np.sqrt(hd)
    if causal:
        s[:, :, np.arange(T)[None, :] > pos + np.arange(n)[:, None]] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = np.einsum("bhij,bjhd->bihd", p / p.sum(-1, keepdims=True), vv).reshape(B * n, -1)
    err = out.cpu().numpy() - ref
    assert np.linalg.norm(err) <= 1e-6 * np.linalg.norm(ref)
