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
