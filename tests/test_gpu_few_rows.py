"""Products of one to eight rows with bf16 weights on both sides of the lines where the matrix cores take them (csrc/seq_linear.hip:
lin_rows_pay), against float64 of the rounded operands: columns that end inside a workgroup's 16 or 32, one block of K a wave, none
and several, strided rows, batches. Tolerance: fp32 sums, 2^-20 of the sum of magnitudes' root mean square (a tree of at most 2^6
additions of 2^-24 each)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N,K", [(1, 128), (17, 512), (513, 768), (512, 1024), (514, 1024), (1030, 640), (1024, 4224), (3000, 5632), (4095, 896),
                                 (4097, 256), (8193, 384), (16400, 128), (5000, 1152), (4096, 128), (4096, 1408), (8191, 2176)])
@pytest.mark.parametrize("M", range(1, 9))
def test_rows(M, N, K):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K + 4, generator=g, device=DEV)
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    ref = a[:, :K].to(torch.bfloat16).double() @ w.double().t()
    pad = torch.full((M + 1, N + 3), 7.0, device=DEV)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=pad, lda=K + 4, ldy=N + 3)
    assert float((pad[:M, :N].double() - ref).abs().max()) <= 2 ** -20 * 6
    assert (pad[:, N:] == 7.0).all() and (pad[M] == 7.0).all()


@pytest.mark.parametrize("B,N,K", [(32, 512, 128), (16, 128, 512), (8, 100, 256), (5, 130, 896)])
@pytest.mark.parametrize("M", [1, 2, 3, 8])
def test_batches_side_by_side(B, M, N, K):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(B + N)
    a = torch.randn(M, B * K, generator=g, device=DEV)
    w = (torch.randn(B, N, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    y = torch.empty(M, B * N, device=DEV)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=B * K, ldy=B * N, batch=B, stride_a=K, stride_w=N * K, stride_y=N)
    for b in range(B):
        ref = a[:, b * K:(b + 1) * K].to(torch.bfloat16).double() @ w[b].double().t()
        assert float((y[:, b * N:(b + 1) * N].double() - ref).abs().max()) <= 2 ** -20 * 6


@pytest.mark.parametrize("M,N,K", [(4, 4096, 128), (8, 4096, 512), (4, 4096, 1024), (8, 2048, 1024), (5, 4096, 1536), (8, 4096, 2048), (3, 4096, 4096)])
def test_error_of_rows_together(M, N, K):
    """Root mean square of the error of rows made together, at most that of each row alone, a lane's sums: 1.5 in a hundred beside it are
    four times what the mean of 40000 results scatters by."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(K)
    errs = [0.0, 0.0]
    for _ in range(-(-40000 // (M * N))):
        a = torch.randn(M, K, generator=g, device=DEV)
        w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
        ref = a.to(torch.bfloat16).double() @ w.double().t()
        y, alone = torch.empty(M, N, device=DEV), torch.empty(M, N, device=DEV)
        seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N)
        for m in range(M):
            seq_ops.linear(a[m], w, M=1, N=N, K=K, y=alone[m], lda=K, ldy=N)
        errs[0] += float((y.double() - ref).square().mean())
        errs[1] += float((alone.double() - ref).square().mean())
    assert errs[0] ** 0.5 <= 1.015 * errs[1] ** 0.5


@pytest.mark.parametrize("M,N,K", [(3, 600, 4096), (4, 1030, 640), (5, 300, 128), (8, 4097, 2048), (8, 8193, 2176)])
def test_values_that_are_not_ordinary(M, N, K):
    """Infinities and NaN: in their own rows and columns, as one row alone has them."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(M, K, generator=g, device=DEV)
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    a[0, K - 1], a[M - 1, 5] = float("inf"), float("nan")
    w[N - 1, 0], w[16, K // 2] = float("-inf"), float("nan")
    y = torch.empty(M, N, device=DEV)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N)
    ref = a.to(torch.bfloat16).double() @ w.double().t()
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf()) and ref[1].isfinite().sum() == N - 2
    assert torch.equal(y[y.isinf()].sign().double(), ref[ref.isinf()].sign())
    assert float((y - ref)[ref.isfinite()].abs().max()) <= 2 ** -20 * 6
