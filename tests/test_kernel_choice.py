"""Which kernel a size runs (gorch_hip_kernel_choice), without a GPU: each rule
of a dispatch at sizes where the kernels' measured times are far apart. The
names listed with a size are the kernels within 15% of the fastest there
(MI355X, HIP graphs, 256 CUs, which the library also assumes without a GPU).
"""
import pytest

from gorch_amd import hip

ACT = hip.LINEAR_ACT_BF16


def test_unknown_names_and_sizes():
    assert hip.kernel_choice("linear", 64, 64) is None
    assert hip.kernel_choice("no such op", 64, 64, 64, 0) is None
    assert hip.kernel_choice("linear", -1, 64, 64, 0) is None
    assert hip.kernel_choice("linear", 0, 64, 64, 0) is None
    assert hip.kernel_choice("gate_up", 17, (1 << 31) - 1, 64) is None


# rows, columns, K, flags: the fastest kernels
LINEAR = [
    # long K over some hundred rows: the K-split tiles read A and W once per
    # 64 x 64 tile and lost to the 64-row tiles by 1.2 to 1.6 times
    ((777, 1600, 6400, 0), {"db64x96", "db64x128"}),
    ((1024, 1600, 6400, 0), {"db64x128"}),
    ((1400, 896, 4864, 0), {"db64x96", "db64x128"}),
    ((2048, 896, 4864, 0), {"db64x128"}),
    ((777, 1600, 6400, ACT), {"db64x96", "db64x128"}),
    ((1024, 1600, 6400, ACT), {"db64x128"}),
    ((1400, 896, 4864, ACT), {"db64x96", "db64x128"}),
    ((384, 4096, 12288, ACT), {"db64x128", "db64x96", "db64x64"}),
    # bf16 activations halve the matrix work of a tile, not its reads
    ((128, 50257, 1600, ACT), {"pp256x224", "pp256x256"}),
    ((1024, 6144, 1024, ACT), {"db64x128"}),
    ((33, 300, 200, 0), {"kw16x32"}),
    # sizes that ran the right kernel before
    ((97, 768, 3072, 0), {"kw16x32"}),
    ((200, 2304, 768, 0), {"kw32x64"}),
    ((512, 3072, 768, ACT), {"db64x96", "db64x128"}),
    ((777, 4096, 1024, 0), {"db64x128"}),
    ((777, 50257, 768, 0), {"pp256x160", "pp256x192", "pp256x224"}),
    ((2048, 4800, 1600, 0), {"pp256x160", "pp256x192"}),
    ((8192, 6400, 1600, 0), {"pp256x160", "pp256x192", "pp256x224"}),
]


@pytest.mark.parametrize("dims,names", LINEAR, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_linear_kernel(dims, names):
    assert hip.kernel_choice("linear", *dims) in names


@pytest.mark.parametrize("M,N,K", [(5_000_000, 16, 64), (6_000_000, 64, 8), (8_300_000, 8, 8), (300_000, 8, 8),
                                   (4_400_000, 128, 512)])
def test_linear_many_rows_fit_a_grid(M, N, K):
    """A grid has at most 65,535 row tiles: sizes that 128-row tiles took (8.3
    million rows) may not be sent to smaller ones."""
    name = hip.kernel_choice("linear", M, N, K, 0)
    rows = int(name.lstrip("dbkwp").split("x")[0])
    assert -(-M // rows) <= 65535


@pytest.mark.parametrize("M,N,K", [(4096, 4096, 1 << 21), (2048, 3 << 20, 64), (20000, 64, 5 << 19), (4096, 256, 1 << 21)])
def test_linear_wide_rows_fit_a_resource(M, N, K):
    """The rows of one tile (of A, and of a residual) stay below the 2 GiB of
    a buffer resource, less the 64 KiB past its out-of-range offset."""
    for flags in (0, ACT):
        name = hip.kernel_choice("linear", M, N, K, flags)
        rows = int(name.lstrip("dbkwp").split("x")[0])
        assert rows * max(N, K) * 4 < 0x7FFF0000


# rows, inter, dim: whether SwiGLU in the product's epilogue is the faster form
GATE_UP = [
    # long and wide prompts: the 256-row tiles and a SwiGLU launch were 1.1 to
    # 1.4 times as fast as the paired 64-row tiles that ran
    ((512, 12288, 4096), False), ((1400, 9728, 2560), False), ((2048, 12288, 4096), False), ((8192, 9728, 2560), False),
    # a few rows of a wide weight: paired, the K-split tiles read it no faster
    ((64, 12288, 4096), True), ((128, 3072, 1024), True),
    # sizes that ran the right form before
    ((17, 3072, 1024), False), ((777, 3072, 1024), True), ((1400, 4864, 896), True), ((4096, 1368, 512), True),
]


@pytest.mark.parametrize("dims,paired", GATE_UP, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_gate_up_form(dims, paired):
    assert hip.kernel_choice("gate_up", *dims).startswith("pair") == paired


def test_gate_up_limits():
    """The pair's resource spans gate and up rows: 2 GiB at most."""
    assert not hip.kernel_choice("gate_up", 64, 1 << 18, 2048).startswith("pair")


# batch, new rows, cached rows, heads, KV heads, head_dim, max_seq
ATTENTION = [
    # several rounds of 32-row blocks over few keys, each with a merge of its
    # own: 1.06 to 1.2 times the time of the kernel without key groups before
    ((16, 128, 0, 32, 8, 128, 136), {"prefill_kg1"}), ((16, 100, 37, 16, 8, 128, 145), {"prefill_kg1"}),
    ((16, 128, 500, 32, 8, 128, 636), {"prefill_kg1"}), ((16, 40, 0, 25, 25, 64, 48), {"prefill_kg1"}),
    # few rows of an odd group of 128-wide heads: 1.2 to 1.3 times the time of
    # the kernels with a block per row
    ((14, 4, 500, 28, 4, 128, 504), {"cached4"}), ((11, 5, 500, 28, 4, 128, 505), {"cached4"}),
    # the right ones before
    ((14, 8, 500, 28, 4, 128, 508), {"prefill_kg4"}), ((22, 5, 235, 28, 4, 128, 240), {"prefill_kg4"}),
    ((1, 777, 0, 16, 8, 128, 1024), {"prefill_kg4"}), ((16, 512, 0, 25, 25, 64, 512), {"prefill_kg4"}),
    ((8, 64, 0, 8, 8, 128, 72), {"prefill_kg4"}), ((4, 777, 37, 25, 25, 64, 814), {"prefill_kg4"}),
    ((16, 1, 640, 25, 0, 64, 768), {"cached16"}), ((1, 20, 1000, 16, 8, 128, 1020), {"cached16"}),
]


@pytest.mark.parametrize("dims,names", ATTENTION, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_attention_kernel(dims, names):
    assert hip.kernel_choice("attention", *dims) in names


# M, N, K, batch, bf16 operands
MATMUL = [
    # small K and thin outputs: 128 x 128 tiles and 64-wide steps of mostly
    # absent elements took 1.1 to 3 times the time of the kernel before them
    ((1, 640, 64, 192, 1, 1), "mm64one_k64"), ((1547, 1, 28, 263, 1, 1), "mm64one"), ((1869, 10, 4, 54, 1, 1), "mm64one"),
    ((836, 11, 9, 8, 1, 1), "mm64one"), ((36, 1351, 2, 91, 1, 1), "mm64one"), ((16, 16, 16, 1, 0, 0), "mm32one"),
    ((512, 512, 16, 64, 1, 1), "mm64one"), ((2048, 2048, 8, 16, 1, 1), "mm128_k32"),
    # the right ones before
    ((512, 512, 64, 48, 0, 0), "mm128"), ((1753, 1946, 19, 25, 0, 1), "mm128_k32"), ((1024, 1024, 1024, 1, 1, 1), "mm64x4"),
    ((1024, 1024, 1024, 1, 0, 0), "mm64x2"), ((2048, 2048, 2048, 1, 1, 1), "mm64x1"), ((4096, 4096, 4096, 1, 1, 1), "mm128"),
    ((64, 64, 2048, 1, 0, 0), "mm32x4"),
]


@pytest.mark.parametrize("dims,name", MATMUL, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_matmul_kernel(dims, name):
    assert hip.kernel_choice("matmul", *dims) == name


# op, tokens, dim, ffn, experts, top-k
MOE = [
    # many experts fill the CUs with wide tiles however few rows each has: the
    # K-split down tiles took 1.1 to 1.6 times as long a layer
    (("moe_down", 1400, 1024, 4096, 16, 2), {"wide192", "wide256"}), (("moe_down", 768, 1024, 4096, 64, 8), {"wide256", "wide192"}),
    (("moe_down", 512, 2048, 1408, 64, 8), {"wide256", "wide192"}), (("moe_down", 768, 2048, 1408, 8, 2), {"wide128", "wide192"}),
    (("moe_down", 400, 2048, 1408, 8, 2), {"wide128"}), (("moe_gate_up", 128, 1024, 1408, 8, 2), {"kw32x32", "wide128"}),
    (("moe_gate_up", 200, 2048, 1408, 8, 2), {"wide128"}),
    # the right ones before
    (("moe_down", 16, 1024, 4096, 8, 2), {"kw16x32"}), (("moe_down", 400, 1024, 4096, 4, 2), {"kw32x64"}),
    (("moe_down", 64, 1024, 4096, 16, 2), {"kw32x32", "kw32x64", "kw16x32"}), (("moe_down", 2048, 1024, 4096, 8, 2), {"wide192"}),
    (("moe_down", 1024, 1024, 4096, 8, 2), {"wide128"}), (("moe_gate_up", 16, 512, 1368, 4, 2), {"kw32x32"}),
    (("moe_gate_up", 2048, 1024, 4096, 8, 2), {"wide128"}), (("moe_gate_up", 16, 1024, 4096, 8, 2), {"wide128"}),
]


@pytest.mark.parametrize("dims,names", MOE, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_moe_tiles(dims, names):
    assert hip.kernel_choice(*dims) in names
