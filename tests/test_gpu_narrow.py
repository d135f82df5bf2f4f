"""Products of up to 32 columns by one wave (csrc/seq_gemm.hip: gemm_narrow_kernel) against the tiles in whose place they stand: the
same order of sums, so the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def rand(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


@pytest.mark.parametrize("N,K", [(1, 64), (16, 2048), (18, 640), (32, 576)])
def test_narrow_products(N, K):
    """Rows of a product that is narrow enough, at the edges of its tiles, against the same rows among so many that the tiles take them."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(N)
    M = 8193
    a, w, bias, old = rand(g, M, K).bfloat16(), rand(g, N, K).bfloat16(), rand(g, N), rand(g, M, N + 1)

    def product(rows, **more):
        y = old[:rows].clone()
        seq_ops.linear(a, w, M=rows, N=N, K=K, y=y, lda=K, ldy=N + 1, ksplit=1, **more)
        return y

    for more in ({}, dict(accumulate=True), dict(bias=bias, act=seq_ops.ACT_SIGMOID)):
        whole = product(M, **more)
        for rows in (9, 31, 32, 33, 100, 8192):
            assert torch.equal(product(rows, **more), whole[:rows]), (rows, more)


@pytest.mark.parametrize("N,K", [(16, 128), (31, 640)])
def test_narrow_products_of_other_forms(N, K):
    """Results in bf16, an activation into sums, chosen rows of A, against the same rows among so many that the tiles take them."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(N)
    M = 8193
    a, w, bias, old = rand(g, M, K).bfloat16(), rand(g, N, K).bfloat16(), rand(g, N), rand(g, M, N + 1)
    chosen = torch.randint(0, M, (M,), generator=g, device=DEV, dtype=torch.int32)

    def product(rows, dtype, **more):
        y = old[:rows].to(dtype)
        seq_ops.linear(a, w, M=rows, N=N, K=K, y=y, lda=K, ldy=N + 1, ksplit=1, **more)
        return y

    for dtype, more in ((torch.bfloat16, {}), (torch.bfloat16, dict(bias=bias, act=seq_ops.ACT_SILU)), (torch.float32, dict(a_rows=chosen)),
                        (torch.float32, dict(accumulate=True, bias=bias, act=seq_ops.ACT_SIGMOID))):
        whole = product(M, dtype, **more)
        for rows in (9, 33, 8192) + ((5,) if "a_rows" in more else ()):
            assert torch.equal(product(rows, dtype, **more), whole[:rows]), (rows, dtype, more)


@pytest.mark.parametrize("batch,M,K", [(2, 33, 128), (2, 8192, 64), (3, 5462, 64), (16, 1024, 576), (17, 964, 576), (17, 481, 576), (64, 256, 512),
                                       (64, 257, 512)])
def test_narrow_products_in_batches(batch, M, K):
    """Batches with strides of their own, on both sides of what their rows together decide, against each one's rows on the tiles."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(batch * M)
    N, lda, rows = 18, K + 8, 8193
    a, w = rand(g, batch, rows, lda).bfloat16(), rand(g, batch, N, K).bfloat16()
    y = torch.full((batch, M + 2, N + 1), 7.0, device=DEV)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=lda, ldy=N + 1, batch=batch, stride_a=rows * lda, stride_w=N * K, stride_y=(M + 2) * (N + 1),
                   ksplit=1)
    assert (y[:, M:] == 7.0).all() and (y[:, :, N] == 7.0).all()
    for z in range(batch):
        one = torch.empty(rows, N, device=DEV)
        seq_ops.linear(a[z], w[z], M=rows, N=N, K=K, y=one, lda=lda, ldy=N, ksplit=1)
        assert torch.equal(y[z, :M, :N], one[:M]), z
