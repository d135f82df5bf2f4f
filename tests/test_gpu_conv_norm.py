"""The four-tap convolution whose tiles are loaded ahead and the grouped norm whose values stay in registers
(csrc/seq_ssm.hip: conv4_silu_kernel, gated_group_norm_reg_kernel) at the edges of their tiles, against float64.
Tolerances: a sum of five fp32 terms with an expf and a division, 1e-5 of values up to about 10; the norm's sums of up to
2049 squares, 2e-6 relative, beside a bf16 rounding of 2^-8."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("C", [70, 256, 1000])
def test_four_taps_at_the_edges_of_tiles(dtype, C):
    from lit_gpt import seq_ops
    from lit_gpt.mixers import StepBatch

    dev = torch.device("cuda", 0)
    g = torch.Generator().manual_seed(C)
    lens, pos0 = [1, 1, 1, 2, 3, 4, 15, 16, 17, 18, 19, 32, 33], [0, 1, 5, 1, 0, 2, 9, 0, 3, 1, 2, 0, 7]
    u, w = torch.randn(sum(lens), C + 5, generator=g), torch.randn(C, 4, generator=g).to(dtype)
    bias, state = torch.randn(C, generator=g).to(dtype), torch.randn(len(lens) + 1, 3, C, generator=g)
    want_y, want_s, at = [], [], 0
    for i, (n, p0) in enumerate(zip(lens, pos0)):
        old = state[i].double() * (torch.arange(3) >= 3 - p0).double()[:, None]  # inputs before position 0 count as zeros
        x = torch.cat([old, u[at:at + n, 5:].double()])
        y = bias.double() + sum(w[:, k].double() * x[k:k + n] for k in range(4))
        want_y.append(y * torch.sigmoid(y))
        want_s.append(x[-3:])
        at += n
    step = StepBatch.build([(i, p0, [0] * n) for i, (n, p0) in enumerate(zip(lens, pos0))], dev)
    left = state.to(dev)
    y = seq_ops.conv_silu(u.to(dev), 5, w.to(dev), bias.to(dev), left, step.seq_start, step.seq_slot, step.seq_pos0, max(lens))
    assert (y.cpu().double() - torch.cat(want_y)).abs().max() < 1e-5
    assert torch.equal(left[:-1].cpu().double(), torch.stack(want_s)) and torch.equal(left[-1].cpu(), state[-1])


@pytest.mark.parametrize("n", [1, 255, 256, 257, 512, 1000, 1024, 1025, 2048, 2049])
def test_grouped_norm_by_columns(n):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(n)
    T, groups = 5, 3
    y, proj = (torch.randn(T, c, generator=g, device=dev) for c in (groups * n, groups * n + 7))
    w = torch.randn(groups * n, generator=g, device=dev)
    z = proj[:, 7:].double()
    v = (y.double() * z * torch.sigmoid(z)).view(T, groups, n)
    want = (v / (v.square().mean(-1, keepdim=True) + 1e-5).sqrt()).view(T, -1) * w.double()
    out = seq_ops.gated_group_norm(y, proj, 7, w, groups=groups, eps=1e-5)
    assert out.dtype == torch.float32 and ((out.double() - want).abs() <= 2e-6 * want.abs() + 1e-12).all()
    half = seq_ops.gated_group_norm(y, proj, 7, w, groups=groups, eps=1e-5, bf16_copy=True)
    assert torch.equal(half, out.to(torch.bfloat16))
