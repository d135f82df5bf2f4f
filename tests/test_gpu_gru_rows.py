"""minGRU steps of several sequences with bf16 weights (csrc/seq_gru.hip: mingru_rows_kernel) against float64 of the rounded operands: channels
that end inside a workgroup's 16, both sides of one workgroup a compute unit and of half as many, one block of K a wave and several, and
the lanes' form beside it (one sequence, K of no multiple of 128). Tolerance: the three sums' errors (a tree of at most 2^6 additions of 2^-24
of unit-sized terms each, 2^-19 with the terms' spread) pass through functions of slope at most 1, times the other factor's size."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,K", [(1, 128), (17, 512), (100, 1152), (2048, 2048), (2056, 640), (4095, 256), (4104, 384), (33, 200)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("biased", [False, True])
def test_step(n, K, M, biased):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(n + K + M)
    h = torch.randn(M, K, generator=g, device=DEV)
    w = (torch.randn(3 * n + 5, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    bias = torch.randn(3 * n + 5, generator=g, device=DEV) if biased else None
    z0, u0, g0 = 2 * n + 5, 0, n + 2
    state = torch.randn(M + 3, n, generator=g, device=DEV)
    slot = torch.randperm(M + 3, generator=g, device=DEV)[:M].to(torch.int32)
    pos0 = torch.tensor([0 if m == 1 else 7 for m in range(M)], dtype=torch.int32, device=DEV)
    before = state.clone()
    out = seq_ops.mingru_step(h, w, bias, z0, u0, g0, state, slot, pos0)
    p = h.to(torch.bfloat16).double() @ w.double().t()
    if biased:
        p += bias.double()
    zr, u, gate = p[:, z0: z0 + n], p[:, u0: u0 + n], p[:, g0: g0 + n]
    S0 = before[slot.long()].double() * (pos0 > 0).double().unsqueeze(1)
    z = torch.sigmoid(zr)
    S = (1 - z) * S0 + z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    want = S * torch.nn.functional.silu(gate)
    size = 8.0 * (1 + S0.abs().max() + u.abs().max())
    assert (state[slot.long()].double() - S).abs().max() <= 2 ** -19 * size
    assert (out.view(M, n).double() - want).abs().max() <= 2 ** -19 * size * (1 + gate.abs().max())
    rest = [i for i in range(M + 3) if i not in slot.tolist()]
    assert torch.equal(state[rest], before[rest])


@pytest.mark.parametrize("n,K,M", [(100, 1152, 3), (2056, 640, 8)])
def test_values_that_are_not_ordinary(n, K, M):
    """Infinities and NaN in a sequence, a weight and a state: where one sequence alone has them too."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(n)
    h = torch.randn(M, K, generator=g, device=DEV)
    w = (torch.randn(3 * n, K, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)
    state = torch.randn(M, n, generator=g, device=DEV)
    h[0, 3], h[1, K - 1] = float("inf"), float("nan")
    w[5, 7], w[n + 16, 0], w[3 * n - 1, 1] = float("-inf"), float("inf"), float("nan")
    state[2, 9], state[2, n - 2] = float("inf"), float("nan")
    slot, pos0 = torch.arange(M, dtype=torch.int32, device=DEV), torch.full((M,), 7, dtype=torch.int32, device=DEV)
    together, alone = state.clone(), state.clone()
    out = seq_ops.mingru_step(h, w, None, 0, n, 2 * n, together, slot, pos0).view(M, n)
    one = torch.cat([seq_ops.mingru_step(h[m: m + 1], w, None, 0, n, 2 * n, alone, slot[m: m + 1], pos0[m: m + 1]).view(1, n) for m in range(M)])
    for got, want in ((out, one), (together, alone)):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert torch.equal(got[got.isinf()], want[want.isinf()]) and want[2].isfinite().sum() >= n - 5
        assert (got - want)[want.isfinite()].abs().max() <= 2 ** -18 * 64  # (both within test_step's 2^-19 of the same)
    assert out[1].isnan().all()
