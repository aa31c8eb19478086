"""A Qwen block over prompts at the edges of its prompt-only kernels: the
gate/up product with SwiGLU in its epilogue (ragged rows, columns and K, on
both sides of the K-split tiles) and the per-token q/k norm + RoPE (64 tokens
and more, one to four rows per lane group, both pairings, with and without
gains).

Bound: float64 over the same bf16 weights, 2e-5 in the 2-norm of the updated
residual stream and of the new cache rows (two bf16 terms per activation
measure 2-4e-6).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def rms(x, g):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g


def rope(x, S, heads, hd, pos, neox):
    h = hd // 2
    inv = torch.tensor([1e4 ** (-2.0 * i / hd) for i in range(h)], dtype=torch.float64).float().cuda()
    th = (torch.arange(pos, pos + S, device="cuda").float()[:, None] * inv).double()[:, None]
    x = x.reshape(S, heads, hd)
    a, b = (x[..., 0::2], x[..., 1::2]) if neox else (x[..., :h], x[..., h:])
    u, v = a * th.cos() - b * th.sin(), a * th.sin() + b * th.cos()
    return (torch.stack([u, v], -1) if neox else torch.cat([u, v], -1)).reshape(S, heads * hd)


@pytest.mark.parametrize("S,dim,hq,hkv,hd,inter,pos,neox,norm", [
    (17, 64, 2, 1, 64, 64, 3, 0, 1), (64, 136, 4, 2, 64, 200, 0, 0, 1), (70, 72, 14, 2, 64, 1000, 5, 0, 0),
    (300, 256, 1, 1, 64, 2056, 0, 1, 1), (513, 264, 20, 4, 128, 1000, 0, 0, 1), (130, 1024, 16, 8, 128, 3072, 60, 1, 1),
    (700, 520, 28, 4, 128, 1544, 0, 0, 1), (257, 128, 40, 8, 128, 4104, 0, 0, 1), (333, 128, 60, 4, 64, 3080, 1, 0, 1),
])
def test_qwen_block_prompt(gpu, S, dim, hq, hkv, hd, inter, pos, neox, norm):
    gen = torch.Generator(device="cuda").manual_seed(S + dim)
    rnd = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    bits = lambda t: t.view(torch.int16)  # noqa: E731
    q, kv, cap = hq * hd, hkv * hd, pos + S + 1
    wqkv, wo = (0.05 * rnd(q + 2 * kv, dim)).bfloat16(), (0.05 * rnd(dim, q)).bfloat16()
    wgu, wdown = (0.05 * rnd(2 * inter, dim)).bfloat16(), (0.05 * rnd(dim, inter)).bfloat16()
    na, nf = 1 + 0.1 * rnd(dim), 1 + 0.1 * rnd(dim)
    qn, kn = (1 + 0.1 * rnd(hd), 1 + 0.1 * rnd(hd)) if norm else (None, None)
    x, kc, vc = rnd(S, dim), rnd(cap, kv), rnd(cap, kv)
    x64, k64, v64 = x.double(), kc.double(), vc.double()
    W = bits(wqkv)
    g = dict(dim=dim, num_q=hq, num_kv=hkv, head_dim=hd, causal=True, norm_eps=1e-6, wq=W[:q], wk=W[q:q + kv],
             wv=W[q + kv:], wo=bits(wo), rope=True, rope_base=1e4, rope_max_seq=cap, rope_neox=neox, q_norm=qn, k_norm=kn)
    gpu.QwenBlock(gpu.GQA(g), na, nf, bits(wgu), bits(wdown), inter, 1e-6).forward_cached(x, kc, vc, pos)

    y = rms(x64, na.double()) @ wqkv.double().T
    qq, kk, vv = y[:, :q], y[:, q:q + kv], y[:, q + kv:]
    if norm:
        qq = rms(qq.reshape(S, -1, hd), qn.double()).reshape(S, q)
        kk = rms(kk.reshape(S, -1, hd), kn.double()).reshape(S, kv)
    k64[pos:pos + S], v64[pos:pos + S] = rope(kk, S, hkv, hd, pos, neox), vv
    T = pos + S
    qh = rope(qq, S, hq, hd, pos, neox).view(S, hq, hd).transpose(0, 1)
    kh = k64[:T].view(T, hkv, hd).transpose(0, 1).repeat_interleave(hq // hkv, 0)
    vh = v64[:T].view(T, hkv, hd).transpose(0, 1).repeat_interleave(hq // hkv, 0)
    sc = qh @ kh.transpose(1, 2).contiguous() / np.sqrt(hd)
    mask = torch.arange(T, device="cuda")[None] > pos + torch.arange(S, device="cuda")[:, None]
    o = (torch.softmax(sc.masked_fill(mask, -np.inf), -1) @ vh.contiguous()).transpose(0, 1).reshape(S, q)
    x1 = x64 + o @ wo.double().T
    gu = rms(x1, nf.double()) @ wgu.double().T
    ga, up = gu[:, :inter], gu[:, inter:]
    ref = x1 + (ga * torch.sigmoid(ga) * up) @ wdown.double().T
    for got, want in ((x, ref), (kc[pos:T], k64[pos:T]), (vc[pos:T], v64[pos:T])):
        assert float((got.double() - want).norm() / want.norm()) <= 2e-5
    assert torch.equal(kc[T:].double(), k64[T:]) and torch.equal(vc[:pos].double(), v64[:pos])
