"""Latent attention of few tokens, four heads a workgroup and one (csrc/seq_mixers.hip), against float64: ranks and rotated parts at the
lanes' edges, both caches, windows, sinks, more ranges of keys than keys. Tolerance: sums of some 600 products and the softmax's in fp32
stay within 2e-6 of the largest value of a row of weighted means."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [4, 8, 6, 1])
@pytest.mark.parametrize("r,dr,d", [(512, 64, 128), (504, 128, 8), (8, 1, 16), (64, 0, 32), (72, 65, 0)])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("window", [0, 1, 37])
@pytest.mark.parametrize("splits", [None, 1, 9, 64])
def test_few_tokens(H, r, dr, d, f32, window, splits):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(r + H)
    rand = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    lengths, slots, S = [300, 1, 17, 64, 5], [3, 0, 4, 1, 2], 320
    T, ld, off = len(lengths), H * (d + dr) + 5, 3
    c, kr = rand(5, S, r) if f32 else rand(5, S, r).bfloat16(), rand(5, S, max(dr, 1))[..., :dr].contiguous()
    qc, proj, sink = rand(T, H * r) * r ** -0.5, rand(T, ld), rand(H) if H != 8 else None
    at = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    got = seq_ops.latent_attention(qc, proj, off, c, kr if dr else rand(5, S, 1), sink, at(slots), at([n - 1 for n in lengths]), H=H, d=d,
                                   dr=dr, r=r, scale=0.3, splits=splits, window=window)
    for t, (n, slot) in enumerate(zip(lengths, slots)):
        lo = max(0, n - window) if window else 0
        rows, rot = c[slot, lo:n].double(), kr[slot, lo:n].double()
        q = proj[t, off:off + H * (d + dr)].double().view(H, d + dr)[:, d:]
        score = (qc[t].double().view(H, r) @ rows.T + q @ rot.T) * 0.3
        if sink is not None:
            score = torch.cat([score, sink.double()[:, None]], 1)
        want = torch.softmax(score, 1)[:, :n - lo] @ rows
        assert (got[t].double().view(H, r) - want).abs().max() < 2e-6 * max(1.0, float(rows.abs().max())) * 4


@pytest.mark.parametrize("splits", [None, 9])
def test_ranges_without_keys(splits):
    """Their rows are never written: whatever memory they get, here NaN, is not read."""
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(2)
    H, r, dr, d = 8, 264, 16, 8
    c, kr = torch.randn(1, 40, r, generator=g, device=dev), torch.randn(1, 40, dr, generator=g, device=dev)
    qc, proj = torch.randn(1, H * r, generator=g, device=dev), torch.randn(1, H * (d + dr), generator=g, device=dev)
    at = lambda n: torch.tensor([n], dtype=torch.int32, device=dev)  # noqa: E731
    for keys in (1, 2, 5):
        held = [torch.full((n,), float("nan"), device=dev) for n in (H * r, *[H * 32 * (r + 2), H * 9 * (r + 2)] * 2)]
        del held  # (the workspace comes from these)
        got = seq_ops.latent_attention(qc, proj, 0, c, kr, None, at(0), at(keys - 1), H=H, d=d, dr=dr, r=r, scale=0.1, splits=splits)
        q = proj.double().view(H, d + dr)[:, d:]
        score = (qc.double().view(H, r) @ c[0, :keys].double().T + q @ kr[0, :keys].double().T) * 0.1
        assert (got.double().view(H, r) - torch.softmax(score, 1) @ c[0, :keys].double()).abs().max() < 1e-5


@pytest.mark.parametrize("H,r", [(8, 264), (6, 264), (6, 260), (8, 8)])
@pytest.mark.parametrize("splits", [1, 3, 32])
@pytest.mark.parametrize("sink", [False, True])
def test_scores_of_minus_infinity(H, r, splits, sink):
    """Keys with such a score weigh nothing, first or last of a wave's keys, of a range or of all; in all three kernels."""
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(r + splits)
    dr, d, n = 4, 8, 50
    c, kr = torch.randn(4, n, r, generator=g, device=dev), torch.randn(4, n, dr, generator=g, device=dev)
    qc, proj = torch.randn(4, H * r, generator=g, device=dev), torch.randn(4, H, d + dr, generator=g, device=dev)
    proj[..., d] = proj[..., d].abs() + 0.1
    for slot, none in enumerate([[0], [*range(0, n, 4), 1, 6], list(range(20)), [*range(17), *range(34, n)]]):
        kr[slot, none, 0] = float("-inf")
    s = torch.randn(H, generator=g, device=dev) if sink else None
    at = torch.arange(4, dtype=torch.int32, device=dev)
    got = seq_ops.latent_attention(qc, proj.view(4, -1), 0, c, kr, s, at, torch.full_like(at, n - 1), H=H, d=d, dr=dr, r=r, scale=0.1,
                                   splits=splits)
    score = (qc.double().view(4, H, r) @ c.double().transpose(1, 2) + proj[..., d:].double() @ kr.double().transpose(1, 2)) * 0.1
    if sink:
        score = torch.cat([score, s.double()[:, None].expand(4, H, 1)], 2)
    assert (got.double().view(4, H, r) - torch.softmax(score, 2)[..., :n] @ c.double()).abs().max() < 1e-5
