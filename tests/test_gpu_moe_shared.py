"""Experts of steps with few tokens: several tokens at once give the bits that each token has alone (csrc/seq_ffn.hip:
moe_up_shared_kernel), at one to all choices of an expert, identity experts, odd sizes, and on both sides of 24 pairs, of 64, of the bytes
of all pairs from which they share, of four experts a pair, of 2048 values of K and of 640 workgroups."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("T,top,E,real", [(2, 1, 3, 3), (3, 4, 5, 4), (6, 4, 7, 6), (7, 4, 9, 7), (16, 4, 6, 6), (64, 1, 4, 3), (13, 5, 7, 6),
                                          (2, 2, 18, 16), (2, 2, 19, 17)])
@pytest.mark.parametrize("W,F", [(1032, 2045), (1032, 4100), (16, 8), (1031, 2047), (2056, 2100), (8200, 300), (1016, 4200)])
def test_tokens_together(dtype, gated, T, top, E, real, W, F):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(T * E + W)
    up = (torch.randn(real, (2 if gated else 1) * F, W, generator=g, device=DEV) * W ** -0.5).to(dtype)
    down = (torch.randn(real, W, F, generator=g, device=DEV) * F ** -0.5).to(dtype)
    h, x0 = (torch.randn(T, W, generator=g, device=DEV) for _ in range(2))
    ids = torch.stack([torch.randperm(E, generator=g, device=DEV)[:top] for _ in range(T)]).to(torch.int32)
    ids[T // 2:] = ids[0]  # (half the tokens choose alike)
    wts = torch.rand(T, top, generator=g, device=DEV)
    one = lambda t, i: t[i: i + 1].contiguous()  # noqa: E731
    for accumulate in (True, False):
        x = x0.clone()
        a = seq_ops.moe_up(h, up, ids, seq_ops.ACT_SILU, gated=gated)
        seq_ops.moe_down(a, down, ids, wts, x, h, accumulate=accumulate)
        for t in range(T):
            at = seq_ops.moe_up(one(h, t), up, one(ids, t), seq_ops.ACT_SILU, gated=gated)
            xt = one(x0, t).clone()
            seq_ops.moe_down(at, down, one(ids, t), one(wts, t), xt, one(h, t), accumulate=accumulate)
            live = (ids[t] < real).nonzero().flatten()  # (an identity expert's row is nobody's)
            assert torch.equal(a.view(T, top, F)[t, live], at.view(top, F)[live]) and torch.equal(x[t], xt[0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("gated", [True, False])
def test_values_that_are_not_ordinary(dtype, gated):
    """Infinities and NaN of a token and of an expert's weights: where that token has them alone."""
    from lit_gpt import seq_ops

    T, top, E, W, F = 16, 4, 6, 1032, 4100
    g = torch.Generator(device=DEV).manual_seed(5)
    up = (torch.randn(E, (2 if gated else 1) * F, W, generator=g, device=DEV) * W ** -0.5).to(dtype)
    h = torch.randn(T, W, generator=g, device=DEV)
    ids = torch.stack([torch.randperm(E, generator=g, device=DEV)[:top] for _ in range(T)]).to(torch.int32)
    h[3, 5], h[T - 1, W - 1] = float("nan"), float("inf")
    up[2, 7, 0], up[4, F - 1, W - 1] = float("-inf"), float("nan")
    a = seq_ops.moe_up(h, up, ids, seq_ops.ACT_SILU, gated=gated).view(T, -1)
    one = torch.cat([seq_ops.moe_up(h[t: t + 1], up, ids[t: t + 1], seq_ops.ACT_SILU, gated=gated).view(1, -1) for t in range(T)])
    assert torch.equal(a.isnan(), one.isnan()) and torch.equal(a.nan_to_num(0.0, 3e38, -3e38), one.nan_to_num(0.0, 3e38, -3e38))
    assert a[3].isnan().all() and a[0].isfinite().sum() >= top * F - 2 and not a.isfinite().all(1).all()
