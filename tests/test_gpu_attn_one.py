"""One-token attention over bf16 caches with 128-value rows (attn_one_kernel) against the general form (one split) and
float64: sequences of one key to several hundred, shares that end inside a group of keys or hold none, one or two query
heads a workgroup (two from 1024 pairs of sequence and head on), masks, caps, sinks and gates. Tolerance: fp32 sums of weights
that add up to one, on values of unit variance: 2^-17."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
POS = [0, 1, 16, 63, 64, 200, 517, 300]


def _step(H, G, d2, dv, S, seed):
    from lit_gpt.mixers import StepBatch

    g = torch.Generator(device=DEV).manual_seed(seed)
    B = len(POS)
    k = torch.randn(B + 1, S, G, d2, generator=g, device=DEV).to(torch.bfloat16)
    v = torch.randn(B + 1, S, G, dv, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(B, H * d2 + 2 * H, generator=g, device=DEV)
    slots = [3, 0, 8, 1, 2, 7, 6, 4]
    return k, v, q, slots, StepBatch.build([(s, p, [0]) for s, p in zip(slots, POS)], torch.device(DEV, 0)), g


@pytest.mark.parametrize("H,G", [(16, 4), (4, 2), (3, 3), (6, 1), (12, 2), (128, 32), (128, 128)])
@pytest.mark.parametrize("chunk,cap,sink", [(0, 0.0, False), (100, 0.0, True), (0, 5.0, True)])
def test_sink(H, G, chunk, cap, sink):
    from lit_gpt import seq_ops

    k, v, q, slots, step, g = _step(H, G, 128, 128, 600, H * 7 + G)
    sinks = torch.randn(H, generator=g, device=DEV) if sink else None
    kw = dict(H=H, G=G, d=128, dv=128, scale=128 ** -0.5, chunk=chunk, cap=cap, gate_off=H * 128)
    run = lambda n: seq_ops.sinkattn(q, 0, k, v, sinks, step.seq_start, step.seq_slot, step.seq_pos0, 1, splits=n, **kw)  # noqa: E731
    want = run(1)
    ref = torch.empty(len(POS), H, 128, dtype=torch.float64, device=DEV)
    for b, (s, p) in enumerate(zip(slots, POS)):
        lo = p - p % chunk if chunk else 0
        for h in range(H):
            z = k[s, lo:p + 1, h // (H // G)].double() @ q[b, h * 128:(h + 1) * 128].double() * 128 ** -0.5
            z = cap * torch.tanh(z / cap) if cap else z
            e = torch.exp(z)
            den = e.sum() + (torch.exp(sinks[h].double()) if sink else 0.0)
            ref[b, h] = e @ v[s, lo:p + 1, h // (H // G)].double() / den * torch.sigmoid(q[b, H * 128 + h].double())
    for n in (2, 3, 7, 64, None):
        got = run(n)
        assert float((got.double() - ref.view(len(POS), -1)).abs().max()) < 2 ** -17, n
        assert float((got - want).abs().max()) < 2 ** -16, n
    assert torch.equal(run(7), run(7))


@pytest.mark.parametrize("H,G", [(8, 2), (3, 3), (6, 1), (128, 64)])
@pytest.mark.parametrize("chunk,cap", [(0, 30.0), (64, 0.0)])
def test_two_maps(H, G, chunk, cap):
    from lit_gpt import seq_ops

    k, v, q, slots, step, g = _step(H, G, 128, 128, 600, H * 5 + G)
    kw = dict(H=H, G=G, d=64, dv=128, scale=0.125, chunk=chunk, cap=cap, lam=0.4, eps=1e-5, post=0.6)
    run = lambda n: seq_ops.diffattn(q, 0, k, v, step.seq_start, step.seq_slot, step.seq_pos0, 1, splits=n, **kw)  # noqa: E731
    want = run(1)
    for n in (2, 5, 64, None):  # (the outputs are divided by their root mean square: relative to it)
        assert float((run(n) - want).abs().max()) < 2 ** -15 * float(want.abs().max()), n


@pytest.mark.parametrize("cap", [0.0, 5.0])
def test_nan_and_infinity(cap):
    """A NaN in a key that no other key of its group and share stands beside makes the result NaN; an infinite value of the
    last key, beside which a group has no more, is infinite in its column and nowhere else."""
    from lit_gpt import seq_ops

    H, G = 4, 2
    k, v, q, slots, step, g = _step(H, G, 128, 128, 600, 11)
    kw = dict(H=H, G=G, d=128, dv=128, scale=128 ** -0.5, cap=cap)
    run = lambda n: seq_ops.sinkattn(q, 0, k, v, None, step.seq_start, step.seq_slot, step.seq_pos0, 1, splits=n, **kw).view(-1, H, 128)  # noqa: E731
    clean = run(1)
    at = {b: p for b, p in enumerate(POS) if p >= 16}
    for b, p in at.items():
        v[slots[b], p, :, 5] = float("inf")
    for n in (2, 7, 64, None):
        got = run(n)
        rest = [c for c in range(128) if c != 5]
        for b in at:
            assert got[b, :, 5].isposinf().all(), (n, b)
        assert float((got - clean)[:, :, rest].abs().max()) < 2 ** -16
    for b, p in at.items():
        k[slots[b], p, 0, 9] = float("nan")
    for n in (2, 7, 64, None):
        got = run(n)
        for b in at:
            assert got[b, :2].isnan().all() and torch.isfinite(got[b, 2:, 6:]).all(), (n, b)


def test_two_maps_nan():
    from lit_gpt import seq_ops

    H, G = 4, 2
    k, v, q, slots, step, g = _step(H, G, 128, 128, 600, 12)
    kw = dict(H=H, G=G, d=64, dv=128, scale=0.125, chunk=0, cap=0.0, lam=0.4, eps=1e-5, post=0.6)
    for b, p in enumerate(POS):
        k[slots[b], p, 0, 70] = float("nan")  # of the second map
    for n in (2, 64, None):
        got = seq_ops.diffattn(q, 0, k, v, step.seq_start, step.seq_slot, step.seq_pos0, 1, splits=n, **kw).view(-1, H, 128)
        assert got[:, :2].isnan().all() and torch.isfinite(got[:, 2:]).all(), n
