"""LayerNorm on both sides of its register-resident form (N % 4 == 0, N <=
2048, 16-byte rows): the smallest rows, the edges of its 1024- and 2048-column
sizes, rows that start off a 16-byte boundary, large means, in place.

Bound: float64; the statistics are f64 and the output three f32 operations,
so 2^-21 of |normalized * gamma| + |beta| per element, plus the rounding of
the mean to f32 (2^-24 of it, scaled by 1 / sigma).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [4, 8, 252, 768, 1020, 1024, 1028, 1600, 2044, 2048, 2052, 1023])
@pytest.mark.parametrize("mean,offset,inplace", [(0.5, 0, False), (100.0, 0, True), (0.0, 1, False)])
def test_layernorm_rows(gpu, N, mean, offset, inplace):
    gen = torch.Generator(device="cuda").manual_seed(N)
    M = 5
    buf = torch.full((M * N + offset + 8,), float("nan"), device="cuda")
    x = buf[offset:offset + M * N].view(M, N)
    x.copy_(2 * torch.randn((M, N), generator=gen, device="cuda") + mean)
    g = 1 + 0.1 * torch.randn(N, generator=gen, device="cuda")
    b = torch.randn(N, generator=gen, device="cuda")
    d = x.double()
    mu, var = d.mean(-1, keepdim=True), d.var(-1, unbiased=False, keepdim=True)
    sigma = torch.sqrt(var + 1e-5)
    z = (d - mu) / sigma * g.double()
    bound = 2.0 ** -21 * (z.abs() + b.double().abs()) + 2.0 ** -23 * mu.abs() / sigma * g.double().abs()
    y = x if inplace else torch.empty_like(x)
    gpu.layernorm(x, g, b, y)
    assert bool(((y.double() - (z + b.double())).abs() <= bound).all())
