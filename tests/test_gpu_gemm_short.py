"""The rows past the last whole tile, in tiles of their own (csrc/gemm_tiles.h), against float64: every number of fragments that they
may have in the forms' heights of 64, 128, 192 and 256 rows, none, one and several whole tiles before them, products that fill
the chip in uneven rounds, ranges of K, and groups whose tiles are all short, all whole or both.

Every sum has K products of bf16 values, exact in fp32, added in fp32: with |a w| ~ K^-1/2 the error of a result is at
most about K additions of half a unit in the last place of partial sums around 1, 2e-5 at the largest K here.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 2e-5


def operands(M, N, K, dev):
    g = torch.Generator(device=dev).manual_seed(7 * M + N)
    a = torch.randn(M, K, generator=g, device=dev).bfloat16()
    return a, (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()


@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 97, 128, 129, 191, 193, 255])
@pytest.mark.parametrize("whole,N,K", [(0, 6200, 128), (1, 12300, 192), (2, 22016, 64), (9, 2100, 256), (8, 8200, 64), (5, 300, 1024)])
def test_rows_past_whole_tiles(rows, whole, N, K):
    from lit_gpt import ops, seq_ops

    dev = torch.device("cuda", 0)
    M = whole * 256 + rows
    if M < 9:
        pytest.skip("such products have no tiles")
    a, w = operands(M, N, K, dev)
    want = a.double() @ w.double().T
    y = torch.full((M + 1, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N)
    assert (y[:M].double() - want).abs().max() < TOL and y[M:].isnan().all()
    n = N // 8 * 8
    y = ops.q4_gemm_fused(a, w[:n], None, n, K, 0, 2)  # the GPT models', rows as the tile's other operand: one rounding to bf16
    assert ((y.double() - want[:, :n]).abs() <= 2.0 ** -8 * want[:, :n].abs() + TOL).all()
    n = N // 8 * 4  # gated units: two roundings of 2^-9 and a unit's few of 2^-24
    gate, up = want[:, :n], want[:, n:2 * n]
    unit = gate * torch.sigmoid(gate) * up
    y = torch.cat([seq_ops.linear_glu(a, w[:2 * n], M=M, n=n, up=n, act=seq_ops.ACT_SILU), torch.full((1, n), 3.0, device=dev, dtype=torch.bfloat16)])
    assert ((y[:M].double() - unit).abs() <= 2.0 ** -8 * unit.abs() + 4 * TOL * (1 + gate.abs() + up.abs())).all()


@pytest.mark.parametrize("sizes", [[193] * 16, [250] * 16, [256] * 3 + [1] * 5, [64] * 70, [0, 513, 0, 129, 64, 1, 320], [33] * 20 + [700]])
@pytest.mark.parametrize("N,K", [(300, 128), (4100, 64)])
def test_groups(sizes, N, K):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    E, M = len(sizes), sum(sizes)
    a, w = operands(M, E * N, K, dev)
    w = w.view(E, N, K)
    z = torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(dev)
    y = torch.full((M + 1, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, batch=E, stride_w=N * K, z_start=z)
    n = N // 8 * 4
    unit = seq_ops.linear_glu(a, w, M=M, n=n, up=n, act=seq_ops.ACT_SILU, z_start=z)
    assert y[M:].isnan().all()
    for e in range(E):
        lo, hi = int(z[e]), int(z[e + 1])
        want = a[lo:hi].double() @ w[e].double().T
        assert ((y[lo:hi].double() - want).abs() < TOL).all()
        gate, up = want[:, :n], want[:, n:2 * n]
        made = gate * torch.sigmoid(gate) * up
        assert ((unit[lo:hi].double() - made).abs() <= 2.0 ** -8 * made.abs() + 4 * TOL * (1 + gate.abs() + up.abs())).all()
