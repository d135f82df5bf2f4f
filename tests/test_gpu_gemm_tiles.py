"""The pipelined tiles of the layered models' products (csrc/seq_gemm.hip) against float64, at the edges of their forms.

Every sum has K products of bf16 values, exact in fp32, added in fp32: with |a w| ~ K^-1/2 the error of a result is at
most about K additions of half a unit in the last place of partial sums around 1, 2e-5 at the largest K here.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 2e-5


def operands(M, N, K, dev, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + 7 * M + N)
    a = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    return a, w, torch.randn(N, generator=g, device=dev)


# one row past and one short of whole tiles of 64, 128 and 256 rows and 128 and 256 columns; the shortest K; products that
# fill the chip with the largest form; odd columns
@pytest.mark.parametrize("M,N,K", [(9, 1, 64), (64, 128, 64), (65, 129, 128), (127, 255, 192), (129, 257, 320),
                                   (255, 1023, 64), (257, 4097, 256), (513, 12288, 192), (2047, 8200, 448),
                                   (2305, 10241, 1024), (40, 6144, 4096), (700, 2048, 5632)])
@pytest.mark.parametrize("ksplit", [0, 1, 3])
def test_product(M, N, K, ksplit):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    a, w, b = operands(M, N, K, dev)
    want = a.double() @ w.double().T
    pad = torch.full((M, N + 3), 2.0, device=dev)  # (rows apart: nothing may be written between them)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=pad, lda=K, ldy=N + 3, bias=b, accumulate=True, ksplit=ksplit)
    assert (pad[:, :N].double() - 2.0 - b.double() - want).abs().max() < TOL
    assert (pad[:, N:] == 2.0).all()
    y = torch.full((M, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, ksplit=ksplit)
    assert (y.double() - want).abs().max() < TOL
    y16 = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y16, lda=K, ldy=N, bias=b, act=seq_ops.ACT_SILU, ksplit=ksplit)
    z = want + b.double()
    z = z * torch.sigmoid(z)
    assert ((y16.double() - z).abs() <= 2.0 ** -8 * z.abs() + TOL).all()  # one rounding to bf16


@pytest.mark.parametrize("rows", [[0, 1, 0, 300], [128, 129, 127, 0], [5] * 70, [700, 0, 513, 64, 1]])
@pytest.mark.parametrize("gather", [False, True])
def test_grouped_product(rows, gather):
    """Every group its own matrix and range of rows, some of them empty; rows gathered from a shorter list."""
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    E, M, N, K = len(rows), sum(rows), 260, 192
    a, w, _ = operands(M, E * N, K, dev)
    w = w.view(E, N, K)
    start = torch.tensor([0] + rows).cumsum(0).to(torch.int32).to(dev)
    pick = torch.randint(0, M, (M,), device=dev, dtype=torch.int32) if gather else None
    y = torch.full((M + 1, N), 3.0, device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, batch=E, stride_w=N * K, z_start=start, a_rows=pick)
    src = a.double() if pick is None else a.double()[pick.long()]
    for e in range(E):
        lo, hi = int(start[e]), int(start[e + 1])
        assert ((y[lo:hi].double() - src[lo:hi] @ w[e].double().T).abs() < TOL).all()
    assert (y[M:] == 3.0).all()


@pytest.mark.parametrize("M,N,K", [(1279, 12031, 256), (1023, 10753, 128), (3327, 2305, 1024), (769, 6655, 1024), (575, 4097, 128),
                                   (130, 1000, 192), (40, 260, 64), (256, 512, 64)])
@pytest.mark.parametrize("act", [0, 1, 2, 3, 4])
def test_results_of_every_kind(M, N, K, act):
    """fp32, bf16 and sums, each activation, tiles inside and past the ends, rows apart: the activation of the plain result, which
    test_product holds against float64, within a few roundings of 2^-24 (of tanh, exponential and products) and one to bf16."""
    from lit_gpt import seq_ops

    dev, ld = torch.device("cuda", 0), N + 5
    a, w, b = operands(M, N, K, dev)
    z = torch.empty(M, N, device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=z, lda=K, ldy=N, bias=b, ksplit=1)
    z = z.double()
    want = {0: z, 1: z.clamp_min(0) ** 2, 2: torch.nn.functional.gelu(z, approximate="tanh"), 3: torch.nn.functional.silu(z),
            4: torch.sigmoid(z)}[act]
    old = torch.randn(M, ld, device=dev)
    for kind in ("fp32", "bf16", "sums"):
        y = old.to(torch.bfloat16) if kind == "bf16" else old.clone()
        seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=ld, bias=b, act=act, accumulate=kind == "sums", ksplit=1)
        assert torch.equal(y[:, N:], old[:, N:].to(y.dtype)), kind
        got = y[:, :N].double() - (old[:, :N].double() if kind == "sums" else 0.0)
        size = want.abs() + (old[:, :N].double().abs() if kind == "sums" else 0.0)
        bound = (2.0 ** -8 if kind == "bf16" else 0.0) * want.abs() + 16 * 2.0 ** -24 * (size + z.abs().clamp_max(4.0))
        assert bool(((got - want).abs() <= bound).all()), kind


def test_strided_batch():
    """Products side by side, A in columns of wider rows, K in one and in several stages."""
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    for K in (64, 512):
        Z, M, N = 5, 130, 96
        a, w, _ = operands(M, Z * N, K * Z, dev)
        w = w.view(Z, N, Z * K)[:, :, :K].contiguous()
        y = torch.zeros(M, Z * N, device=dev)
        seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=Z * K, ldy=Z * N, batch=Z, stride_a=K, stride_w=N * K, stride_y=N)
        for z in range(Z):
            want = a[:, z * K:(z + 1) * K].double() @ w[z].double().T
            assert (y[:, z * N:(z + 1) * N].double() - want).abs().max() < TOL


# every tile form with a partial last tile of rows and of columns, rows as the tile's A (tests of products with rows as its
# B: below); few values of K, so that rings are refilled past the end from the first step on
PLAIN = [(1279, 12031, 256), (1023, 10753, 128), (3327, 2305, 1024), (385, 12289, 256),
         (257, 10943, 128), (769, 6913, 128), (257, 6529, 128), (65, 127, 128), (769, 9471, 128)]
PROMPT = [(1279, 12032, 256), (575, 13056, 128), (769, 6656, 1024), (1023, 5376, 256), (769, 4608, 128),
          (769, 6528, 128), (257, 5504, 128), (129, 64, 128), (769, 9408, 128), (769, 9360, 576), (257, 16640, 576)]


def test_the_sizes_take_every_form():
    from lit_gpt import ops, seq_ops

    lib = seq_ops.load_library()
    assert {lib.lgs_linear_form(M, N, K, 1, 0, lib.lgs_linear_ksplit(M, N, K), 0, 0) for M, N, K in PLAIN} == set(range(9))
    assert {ops.load_library().lga_bf16_gemm_form(M, N, K, 0) & 255 for M, N, K in PROMPT} == set(range(9))


@pytest.mark.parametrize("M,N,K", PLAIN)
def test_every_form_at_its_edges(M, N, K):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    a, w, b = operands(M, N, K, dev, seed=3)
    want = a.double() @ w.double().T + b.double()
    y = torch.full((M + 1, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, bias=b)
    assert (y[:M].double() - want).abs().max() < TOL and y[M:].isnan().all()


@pytest.mark.parametrize("M,N,K", PROMPT)
def test_every_form_of_prompt_products(M, N, K):
    """bf16 weights of the GPT models: one rounding of the sum to bf16."""
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    a, w, _ = operands(M, N, K, dev, seed=5)
    want = a.double() @ w.double().T
    y = ops.q4_gemm_fused(a, w, None, N, K, 0, 2)
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + TOL).all()
