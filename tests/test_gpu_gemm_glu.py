"""Gated units in the epilogue of the pipelined tiles (lgs_linear_glu) against the product and the unit made apart: to the
bit, the sums and the roundings being the same. Rows and columns at and around the tiles' edges, gathered rows in groups
with empty ones, every unit, and matrices that begin apart."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("clamp", [None, (1.702, 7.0, 1.0), (1.0, 0.0, 0.0)])
@pytest.mark.parametrize("M,n,K", [(9, 32, 64), (64, 36, 128), (129, 1000, 320), (257, 2052, 64), (700, 5632, 2048),
                                   (2048, 1028, 512)])
def test_unit_matches_product_and_unit(M, n, K, clamp):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(M + n + K)
    up = (n + 7) // 8 * 8
    a = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(up + n, K, generator=g, device=DEV).to(torch.bfloat16)
    proj = torch.empty(M, up + n, device=DEV)
    seq_ops.linear(a, w, M=M, N=up + n, K=K, y=proj, lda=K, ldy=up + n, ksplit=1)
    if clamp is None:
        want = [seq_ops.glu(proj, 0, up, n, act, bf16=True) for act in (seq_ops.ACT_SILU, seq_ops.ACT_GELU_TANH)]
        got = [seq_ops.linear_glu(a, w, M=M, n=n, up=up, act=act) for act in (seq_ops.ACT_SILU, seq_ops.ACT_GELU_TANH)]
    else:
        alpha, limit, shift = clamp
        want = [seq_ops.glu_clamped(proj, 0, up, n, alpha=alpha, limit=limit, shift=shift, bf16=True)]
        got = [seq_ops.linear_glu(a, w, M=M, n=n, up=up, clamp=clamp)]
    assert all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("F,K", [(64, 128), (1408, 2048)])
def test_groups(F, K):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(F)
    E, T = 70, 300
    sizes = torch.randint(0, 40, (E,), generator=torch.Generator().manual_seed(1))
    sizes[3], sizes[5], sizes[69] = 0, 300, 0
    z = torch.cat([torch.zeros(1, dtype=torch.long), sizes.cumsum(0)]).to(torch.int32).to(DEV)
    pairs = int(sizes.sum())
    rows = torch.randint(0, T, (pairs,), generator=g, device=DEV).to(torch.int32)
    h = torch.randn(T, K, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(E, 2 * F, K, generator=g, device=DEV).to(torch.bfloat16)
    gu = torch.empty(pairs, 2 * F, device=DEV)
    seq_ops.linear(h, w, M=pairs, N=2 * F, K=K, y=gu, lda=K, ldy=2 * F, batch=E, stride_w=2 * F * K, a_rows=rows, z_start=z)
    want = seq_ops.glu(gu, 0, F, F, seq_ops.ACT_SILU, bf16=True)
    assert seq_ops.glu_fits(h, w, pairs, F, grouped=True)
    assert torch.equal(seq_ops.linear_glu(h, w, M=pairs, n=F, up=F, act=seq_ops.ACT_SILU, a_rows=rows, z_start=z), want)


def test_sizes():
    from lit_gpt import seq_ops

    h = torch.zeros(64, 192, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(128, 192, dtype=torch.bfloat16, device=DEV)
    assert seq_ops.glu_fits(h, w, 64, 64) and not seq_ops.glu_fits(h, w, 8, 64) and not seq_ops.glu_fits(h, w, 64, 62)
    assert not seq_ops.glu_fits(h.float(), w, 64, 64) and not seq_ops.glu_fits(h[:, :96], w[:, :96], 64, 64)


@pytest.mark.parametrize("E,pairs,fits", [(64, 52, False), (64, 128, False), (64, 129, True), (26, 52, False), (25, 52, True),
                                          (16, 52, True), (256, 128, False)])
def test_few_rows_of_many_groups(E, pairs, fits):
    """The sizes that stay with the tiles made for a group's place in the grid, to the bits of the other form."""
    from lit_gpt import seq_ops

    F, K = 64, 128
    g = torch.Generator(device=DEV).manual_seed(E + pairs)
    sizes = torch.bincount(torch.randint(0, E, (pairs,), generator=torch.Generator().manual_seed(pairs)), minlength=E)
    z = torch.cat([torch.zeros(1, dtype=torch.long), sizes.cumsum(0)]).to(torch.int32).to(DEV)
    rows = torch.randint(0, 40, (pairs,), generator=g, device=DEV).to(torch.int32)
    h = torch.randn(40, K, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(E, 2 * F, K, generator=g, device=DEV).to(torch.bfloat16)
    assert seq_ops.glu_fits(h, w, pairs, F, grouped=True) == fits
    gu = torch.empty(pairs, 2 * F, device=DEV)
    seq_ops.linear(h, w, M=pairs, N=2 * F, K=K, y=gu, lda=K, ldy=2 * F, batch=E, stride_w=2 * F * K, a_rows=rows, z_start=z)
    of = torch.repeat_interleave(torch.arange(E, device=DEV), sizes.to(DEV))
    want = (h[rows.long()].double()[:, None] @ w[of].double().transpose(1, 2).contiguous())[:, 0]
    assert float((gu.double() - want).abs().max()) < 2 ** -20 * float(want.abs().max()) * 8
    made = seq_ops.linear_glu(h, w, M=pairs, n=F, up=F, act=seq_ops.ACT_SILU, a_rows=rows, z_start=z)
    assert torch.equal(made, seq_ops.glu(gu, 0, F, F, seq_ops.ACT_SILU, bf16=True))
