"""The general matrix product at the edges of its tiles: every layout and
dtype at sizes on both sides of each tile choice (32 x 32, 64 x 64 with four,
two or one K groups, 128 x 128, and the one-step forms of small K), with ragged
rows, columns and K, rows shorter than a load, and operands that start at an
odd element. KINDS names the kernel of a size, and asserts that it runs there;
its 128 x 128 tiles take several K steps, whole and ragged.

Bounds: against float64 over the stored values, |error| <= (K + 16) 2^-23 of
sum |a||b| element by element (f32 accumulation in any order; three bf16 terms
carry an f32 value to 2^-24), and 2e-6 of the result in the 2-norm, which a
two-term split (~1e-5) would miss.
"""
import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu

LAYOUTS = [(False, True), (False, False), (True, False)]
DTYPES = [(True, True), (False, True), (False, False), (True, False)]
SIZES = [
    (1, 1, 1, 1), (1, 1, 3, 9), (1, 2, 5, 64), (1, 33, 65, 127), (1, 64, 36, 256),   # 32 x 32 tiles, 4 groups
    (3, 259, 290, 65), (1, 576, 512, 128), (70, 3, 2, 40), (1, 1000, 700, 577),      # 64 x 64, 2 groups (4: bf16)
    (1, 1090, 1028, 63), (5, 512, 449, 192),                                         # 64 x 64, 1 group
    (1, 2050, 4037, 33), (32, 515, 500, 64),                                         # 128 x 128
]


def _place(a, offset):
    """a on the GPU, `offset` elements into a buffer of NaNs."""
    t = torch.from_numpy(np.ascontiguousarray(a.view(np.int16) if a.dtype == np.uint16 else a))
    nan = 0x7FC0 if t.dtype == torch.int16 else float("nan")
    buf = torch.full((t.numel() + offset + 64,), nan, dtype=t.dtype, device="cuda")
    buf[offset:offset + t.numel()] = t.reshape(-1).cuda()
    return buf[offset:offset + t.numel()].view(t.shape)


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("transA,transB", LAYOUTS)
@pytest.mark.parametrize("a16,b16", DTYPES)
def test_matmul_tiles(gpu, size, transA, transB, a16, b16):
    B_, M, N, K = size
    rng = np.random.default_rng(B_ * M + N + K)
    a = rng.standard_normal((B_,) + ((K, M) if transA else (M, K))).astype(np.float32)
    b = rng.standard_normal((B_,) + ((N, K) if transB else (K, N))).astype(np.float32)
    a = orc.f32_to_bf16(a) if a16 else a
    b = orc.f32_to_bf16(b) if b16 else b
    C = torch.full((B_ * M * N + 1,), float("nan"), device="cuda")
    # one element in: unaligned vector loads (and never the aligned Linear route)
    gpu.batched_matmul_dt(_place(a, 1), _place(b, 1), C[:-1], M, N, K, B_, transA, transB, a16, b16)
    a64 = (orc.bf16_to_f32(a) if a16 else a).astype(np.float64)
    b64 = (orc.bf16_to_f32(b) if b16 else b).astype(np.float64)
    a64 = np.ascontiguousarray(np.swapaxes(a64, 1, 2)) if transA else a64
    b64 = np.ascontiguousarray(np.swapaxes(b64, 1, 2)) if transB else b64
    ref, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    got = C.cpu().numpy()
    assert np.isnan(got[-1])
    err = got[:-1].reshape(B_, M, N) - ref
    assert np.all(np.abs(err) <= (K + 16) * 2.0 ** -23 * mag)
    assert np.linalg.norm(err) <= 2e-6 * np.linalg.norm(ref)


# kernel, (batch, M, N, K); mm64x4 takes two bf16 operands (else mm64x2)
KINDS = [
    ("mm32one", (2, 5, 3, 1)), ("mm32one", (1, 33, 65, 31)), ("mm32one", (3, 64, 100, 64)), ("mm32one", (7, 36, 35, 57)),
    ("mm64one", (70, 3, 2, 7)), ("mm64one", (9, 259, 290, 32)), ("mm64one", (5, 500, 449, 19)), ("mm64one", (66, 1, 63, 8)),
    ("mm64one_k64", (3, 400, 390, 40)), ("mm64one_k64", (70, 3, 2, 64)), ("mm64one_k64", (5, 512, 449, 63)),
    ("mm64one_k64", (192, 1, 640, 64)),
    ("mm128_k32", (260, 511, 507, 9)), ("mm128_k32", (16, 2048, 2048, 32)),
    ("mm32x4", (1, 33, 65, 127)), ("mm64x4", (1, 576, 512, 520)), ("mm64x2", (3, 259, 290, 65)), ("mm64x1", (5, 512, 449, 192)),
    ("mm128", (32, 516, 500, 200)), ("mm128", (32, 515, 501, 256)), ("mm128", (40, 508, 512, 40)),
]


@pytest.mark.parametrize("kernel,size", KINDS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
@pytest.mark.parametrize("transA,transB", LAYOUTS)
@pytest.mark.parametrize("a16,b16", DTYPES)
def test_each_kind(gpu, kernel, size, transA, transB, a16, b16):
    B_, M, N, K = size
    want = "mm64x2" if kernel == "mm64x4" and not (a16 and b16) else kernel
    assert gpu.kernel_choice("matmul", M, N, K, B_, a16, b16) == want
    g = torch.Generator(device="cuda").manual_seed(M + N + K)

    def operand(shape, half, offset=1):
        t = torch.randn(shape, generator=g, device="cuda")
        t = t.bfloat16() if half else t
        nan = 0x7FC0 if half else float("nan")
        buf = torch.full((t.numel() + offset + 64,), nan, dtype=torch.int16 if half else torch.float32, device="cuda")
        buf[offset:offset + t.numel()] = (t.view(torch.int16) if half else t).reshape(-1)
        return buf[offset:offset + t.numel()].view(shape), t.double()

    a, a64 = operand((B_, K, M) if transA else (B_, M, K), a16)
    b, b64 = operand((B_, N, K) if transB else (B_, K, N), b16)
    C = torch.full((B_ * M * N + 1,), float("nan"), device="cuda")
    gpu.batched_matmul_dt(a, b, C[:-1], M, N, K, B_, transA, transB, a16, b16)
    assert bool(torch.isnan(C[-1]))
    a64 = a64.transpose(1, 2).contiguous() if transA else a64
    b64 = b64.transpose(1, 2).contiguous() if transB else b64
    ref = torch.matmul(a64, b64)
    err = C[:-1].view(B_, M, N).double() - ref
    assert bool((err.abs() <= (K + 16) * 2.0 ** -23 * torch.matmul(a64.abs(), b64.abs())).all())
    assert float(err.norm() / ref.norm()) <= 2e-6
