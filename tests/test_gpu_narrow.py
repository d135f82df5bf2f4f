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
