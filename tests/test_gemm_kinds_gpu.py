"""The Linear above 16 rows at the edges of its kernels: the K-split tiles of
short prompts, the 64-row tiles and the 256-row tiles of long prompts, with
ragged rows, columns and K (all remainders of the 32- and 64-wide steps), every
epilogue and both activation modes. SIZES are ordinary sizes, whichever kernel
runs them; KERNELS names a ragged size for each kernel, and asserts that it runs
there.

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
    (17, 64, 40), (33, 100, 72), (31, 768, 1048), (64, 2304, 768), (97, 770, 3072), (130, 3072, 776),
    (250, 203, 2056), (400, 512, 2048), (777, 1024, 2080), (512, 2304, 768), (500, 2301, 776), (2048, 768, 768),
    (1030, 3000, 64), (2007, 4800, 1600), (1400, 6144, 1048), (200, 50257, 1600), (4100, 1290, 2072), (257, 33000, 2048),
    (1024, 8192, 1608),
]

# K no multiple of 32 (the steps' tails), then a multiple; sizes that differ
# between split and bf16 activations in two rows
KERNELS = [
    ("db64x64", 0, (4432, 69, 200)), ("db64x64", 0, (34, 8533, 224)),
    ("db64x64", 1, (38, 4186, 208)), ("db64x64", 1, (1733, 80, 288)),
    ("db64x96", 0, (17, 16477, 216)), ("db64x96", 0, (18, 18330, 256)),
    ("db64x96", 1, (17, 16477, 216)), ("db64x96", 1, (18, 18330, 256)),
    ("db64x128", 0, (835, 5909, 24)), ("db64x128", 0, (65, 15161, 224)),
    ("db64x128", 1, (3463, 263, 216)), ("db64x128", 1, (65, 15161, 224)),
    ("kw16x32", 0, (26, 17, 240)), ("kw16x32", 0, (20, 31, 256)),
    ("kw16x32", 1, (26, 17, 240)), ("kw16x32", 1, (20, 31, 256)),
    ("kw32x32", 0, (2068, 35, 216)), ("kw32x32", 0, (17, 4284, 224)),
    ("kw32x32", 1, (2068, 35, 216)), ("kw32x32", 1, (17, 4284, 224)),
    ("kw32x64", 0, (4141, 35, 216)), ("kw32x64", 0, (17, 8519, 256)),
    ("kw32x64", 1, (4141, 35, 216)), ("kw32x64", 1, (17, 8519, 256)),
    ("kw64x64", 0, (4201, 103, 336)), ("kw64x64", 0, (4384, 102, 480)),
    ("kw64x64", 1, (4210, 97, 1616)), ("kw64x64", 1, (4992, 97, 1536)),
    ("pp256x128", 0, (4832, 1058, 200)), ("pp256x128", 0, (3542, 1449, 224)),
    ("pp256x128", 1, (711, 8429, 200)), ("pp256x128", 1, (1789, 3570, 224)),
    ("pp256x160", 0, (530, 11906, 200)), ("pp256x160", 0, (857, 8595, 224)),
    ("pp256x160", 1, (1094, 7274, 200)), ("pp256x160", 1, (1126, 7173, 224)),
    ("pp256x192", 0, (1065, 8565, 200)), ("pp256x192", 0, (830, 10245, 256)),
    ("pp256x192", 1, (1065, 8565, 200)), ("pp256x192", 1, (830, 10245, 256)),
    ("pp256x224", 0, (1330, 8213, 200)), ("pp256x224", 0, (2369, 4823, 224)),
    ("pp256x224", 1, (1330, 8213, 200)), ("pp256x224", 1, (2369, 4823, 224)),
    ("pp256x256", 0, (2078, 6313, 200)), ("pp256x256", 0, (1845, 7354, 224)),
    ("pp256x256", 1, (2078, 6313, 200)), ("pp256x256", 1, (1845, 7354, 224)),
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


@pytest.mark.parametrize("kernel,act,size", KERNELS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
@pytest.mark.parametrize("opts", [(1, 1, 0), (1, 0, 1)], ids=["bias+res", "bias+gelu"])
def test_each_kernel(gpu, kernel, act, size, opts):
    assert gpu.kernel_choice("linear", *size, gpu.LINEAR_ACT_BF16 if act else 0) == kernel
    run(gpu, *size, *map(bool, opts), bool(act))


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
