"""Products of a few rows with bf16 weights (lgs_linear with 2 to 8 rows: lin_rows_kernel and what stays with
lin_gemv_kernel) against float64 of the rounded operands: columns that end inside a workgroup's 16 or 32, K that does not
divide by the waves' ranges, strided rows, bias, activation, accumulation and batches. Tolerance: fp32 sums, 2^-20 of the
sum of magnitudes' root mean square (a tree of at most 2^6 additions of 2^-24 each)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N,K", [(2048, 128), (2049, 384), (2050, 2048), (4096, 640), (4611, 4096), (6151, 1408), (20608, 512),
                                 (2056, 11008), (512, 2048)])
@pytest.mark.parametrize("M", [2, 3, 4, 5, 8])
def test_rows(M, N, K):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K + 8, generator=g, device=DEV)
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device=DEV)
    ref = a[:, :K].to(torch.bfloat16).double() @ w.double().t()
    pad = torch.full((M, N + 3), 7.0, device=DEV)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=pad, lda=K + 8, ldy=N + 3)
    assert float((pad[:, :N].double() - ref).abs().max()) <= 2 ** -20 * 6
    assert float((pad[:, N:] - 7.0).abs().max()) == 0.0
    y = torch.randn(M, N, generator=g, device=DEV)
    want = y.double() + torch.nn.functional.silu(ref + bias.double())
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K + 8, ldy=N, bias=bias, act=seq_ops.ACT_SILU, accumulate=True)
    assert float((y.double() - want).abs().max()) <= 2 ** -20 * 8


def test_batches():
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(1)
    B, M, N, K = 3, 6, 2064, 256
    a = torch.randn(B, M, K, generator=g, device=DEV)
    w = (torch.randn(B, N, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    y = torch.empty(B, M, N, device=DEV)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, batch=B, stride_a=M * K, stride_w=N * K, stride_y=M * N)
    ref = torch.stack([a[i].to(torch.bfloat16).double() @ w[i].double().t() for i in range(B)])
    assert float((y.double() - ref).abs().max()) <= 2 ** -20 * 6
