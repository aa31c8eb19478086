"""The Linear above 16 rows at the edges of each of its kernels: the K-split
tiles of short prompts, the 64-row tiles and the 256-row tiles of long prompts,
with ragged rows, columns and K (all remainders of the 32- and 64-wide steps),
every epilogue and both activation modes.

Bounds, per element against float64: two bf16 terms carry an f32 activation to
2^-16 relative and sums run in f32, so |error| <= (2^-16 + (K + 16) 2^-23)
sum |x||w| (without the first term for bf16-rounded activations); GELU's slope
is at most 1.13 and its own error 4e-7 of its argument. In the 2-norm 8e-6
(5e-6 measured; one bf16 term would give 1.6e-3).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [
    # few tiles: K split over the waves of a block
    (17, 64, 40), (33, 100, 72), (31, 768, 1048), (64, 2304, 768), (97, 770, 3072), (130, 3072, 776),
    (250, 203, 2056), (400, 512, 2048), (777, 1024, 2080),
    # 64-row tiles
    (512, 2304, 768), (500, 2301, 776), (2048, 768, 768), (1030, 3000, 64),
    # 256-row tiles, one to eight column groups
    (2007, 4800, 1600), (1400, 6144, 1048), (200, 50257, 1600), (4100, 1290, 2072), (257, 33000, 2048),
    (1024, 8192, 1608),
]


def run(gpu, M, N, K, bias, res, gelu, act):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn((M, K), generator=g, device="cuda")
    W = (0.05 * torch.randn((N, K), generator=g, device="cuda")).bfloat16()
    b = torch.randn(N, generator=g, device="cuda") if bias else None
    r = torch.randn((M, N), generator=g, device="cuda") if res else None
    y = torch.full((M * N + 1,), float("nan"), device="cuda")
    out = y[:-1].view(M, N)
    gpu.linear_bf16(x, W.view(torch.int16), b, out, r, gpu.EPI_GELU if gelu else gpu.EPI_NONE, act)
    assert bool(torch.isnan(y[-1]))
    xd = (x.bfloat16() if act else x).double()
    ref = xd @ W.double().T
    bound = (0 if act else 2.0 ** -16) + (K + 16) * 2.0 ** -23
    bound = bound * (xd.abs() @ W.double().abs().T) + 1e-6
    if bias:
        ref += b.double()
    if gelu:
        bound = 1.13 * bound + 4e-7 * ref.abs()
        ref = 0.5 * ref * (1 + torch.tanh(0.7978845608 * (ref + 0.044715 * ref ** 3)))
    if res:
        ref += r.double()
        bound = bound + 2.0 ** -22 * (ref.abs() + r.double().abs())
    err = out.double() - ref
    assert bool((err.abs() <= bound).all())
    assert float(err.norm() / ref.norm()) <= 8e-6


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("opts", [(0, 0, 0, 0), (1, 1, 0, 0), (1, 0, 1, 0), (1, 1, 1, 1)],
                         ids=["plain", "bias+res", "bias+gelu", "all,bf16"])
def test_gemm_kinds(gpu, size, opts):
    run(gpu, *size, *map(bool, opts))


def test_gemm_residual_in_place(gpu):
    """The residual may be the output (a residual stream updated in place)."""
    for M, N, K in [(97, 768, 3072), (512, 768, 1600), (2007, 4800, 1600)]:
        x = torch.randn((M, K), device="cuda")
        W = (0.02 * torch.randn((N, K), device="cuda")).bfloat16().view(torch.int16)
        r = torch.randn((M, N), device="cuda")
        y, z = torch.empty_like(r), r.clone()
        gpu.linear_bf16(x, W, None, y, r)
        gpu.linear_bf16(x, W, None, z, z)
        assert torch.equal(y, z)
