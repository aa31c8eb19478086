"""GELU in the epilogue of every Linear kernel above 16 rows, by itself: an
identity weight hands the epilogue bf16 values unchanged, so the result is the
epilogue's GELU of known arguments.

Bound: the 2-norm of the error against float64 may not exceed that of the
elementwise GELU (0.5 x (1 + tanh u), f32, the reference's form) on the same
arguments by more than 4%, for pre-activations of standard deviation 0.15 and
up; the largest and smallest finite arguments come out as from that form.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, columns: the K-split tiles, the 64-row tiles and the 256-row tiles
SIZES = [(64, 512), (512, 512), (4096, 768), (8192, 2048)]


def gelu64(x):
    x = x.double()
    return 0.5 * x * (1 + torch.tanh(0.7978845608 * (x + 0.044715 * x ** 3)))


def epilogue(gpu, x):
    N = x.shape[1]
    W = torch.eye(N, device="cuda").bfloat16().view(torch.int16)
    y = torch.empty_like(x)
    gpu.linear_bf16(x, W, None, y, None, gpu.EPI_GELU)
    return y


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("std", [0.15, 0.3, 1.0, 3.0])
def test_gelu_epilogue_error(gpu, size, std):
    g = torch.Generator(device="cuda").manual_seed(size[0])
    x = (std * torch.randn(size, generator=g, device="cuda")).bfloat16().float()
    ref, elementwise = gelu64(x), torch.empty_like(x)
    gpu.gelu(x, elementwise)
    err = [float((v.double() - ref).norm()) for v in (epilogue(gpu, x), elementwise)]
    assert err[0] <= 1.04 * err[1]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_gelu_epilogue_limits(gpu, size):
    """One value per row, on the diagonal. 1 + tanhf rounds to 2^-24 and tanhf
    itself to 2^-24: up to |x| 2^-24 of absolute error in the elementwise form
    where tanh is not yet -1 (|x| < 8)."""
    M, N = size
    vals = torch.tensor([3e38, -3e38, 1e30, -1e30, -1e4, -10.5, 0.0, -0.0, 1e-30, -1e-30, 88.0, -3.0], device="cuda")
    x = torch.zeros(size, device="cuda")
    n = min(M, N)
    i = torch.arange(n, device="cuda")
    x[i, i] = vals[i % len(vals)].bfloat16().float()
    d = x[i, i].contiguous()
    want = torch.empty_like(d)
    gpu.gelu(d, want)
    got = epilogue(gpu, x)[i, i]
    assert bool(torch.isfinite(got).all())
    assert bool(((got - want).abs() <= 2.0 ** -21 * want.abs() + 2.0 ** -23 * d.abs().clamp(max=8)).all())
