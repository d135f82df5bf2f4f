"""The prompt form of the selective scan where a workgroup takes several heads of a group in turn (csrc/seq_ssm.hip:
ssd_state_kernel, ssd_out_kernel), against the token-by-token form: one, two and four heads per workgroup, sizes whose
rows start on 16 bytes and sizes whose do not, chunks that end anywhere. Tolerance: both forms' fp32 sums, each held to
2e-5 of the largest value against float64 by their own tests."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,groups,N,dv", [(32, 2, 128, 64), (32, 2, 23, 5), (12, 2, 40, 72), (30, 2, 16, 64), (64, 64, 8, 4)])
def test_prompt_form_against_token_walk(heads, groups, N, dv):
    from lit_gpt import seq_ops
    from lit_gpt.mixers import StepBatch

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(N + dv)
    lens, pos0 = [1500, 700, 64, 65], [0, 9, 3, 0]
    T, inner = sum(lens), heads * dv
    rand = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    xbc, raw = rand(T, inner + 2 * groups * N) * 0.5, rand(T, heads)
    dt_bias, A_log, D = rand(heads) - 1.0, rand(heads), rand(heads)
    stale = rand(len(lens) + 1, heads, N, dv)
    step = StepBatch.build([(i, p0, [0] * n) for i, (n, p0) in enumerate(zip(lens, pos0))], dev)
    y, state = {}, {}
    for chunked in (False, True):
        state[chunked] = stale.clone()
        y[chunked] = seq_ops.ssm_scan(xbc, raw, 0, dt_bias, A_log, D, state[chunked], step.seq_start, step.seq_slot,
                                      step.seq_pos0, heads=heads, groups=groups, N=N, dv=dv, max_len=max(lens), chunked=chunked)
    assert float((y[True] - y[False]).abs().max()) < 4e-5 * float(y[False].abs().max())
    assert float((state[True] - state[False]).abs().max()) < 4e-5 * max(1.0, float(state[False].abs().max()))
    assert torch.equal(state[True][-1], stale[-1])


@pytest.mark.parametrize("heads,groups,N,dv", [(16, 2, 128, 64), (24, 1, 64, 72), (6, 3, 64, 40), (3, 3, 128, 4), (8, 8, 128, 132)])
@pytest.mark.parametrize("lens", [[1], [64], [65, 1, 130, 128], [1000, 300]])
def test_chunks_walked_against_side_by_side(heads, groups, N, dv, lens, monkeypatch):
    """A sequence's chunks one after another (ssd_walk_kernel) and side by side: the same sums in the same order, so the same
    bits; heads that are and are not multiples of eight, columns that end inside a wave's sixteen, an infinite input."""
    from lit_gpt import seq_ops
    from lit_gpt.mixers import StepBatch

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(N + dv)
    pos0 = [9, 0, 3, 0][:len(lens)]
    T, inner = sum(lens), heads * dv
    rand = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    xbc, raw = rand(T, inner + 2 * groups * N) * 0.5, rand(T, heads + 3)
    xbc[T // 2, 1] = float("inf")
    dt_bias, A_log, D = rand(heads) - 1.0, rand(heads), rand(heads)
    stale = rand(len(lens) + 1, heads, N, dv)
    step = StepBatch.build([(i, p0, [0] * n) for i, (n, p0) in enumerate(zip(lens, pos0))], dev)
    y, state = {}, {}
    for walk in (False, True):
        monkeypatch.setattr(seq_ops, "_ssm_walks", lambda *a, walk=walk: walk)
        state[walk] = stale.clone()
        y[walk] = seq_ops.ssm_scan(xbc, raw, 2, dt_bias, A_log, D, state[walk], step.seq_start, step.seq_slot, step.seq_pos0,
                                   heads=heads, groups=groups, N=N, dv=dv, max_len=max(lens), chunked=True)
    torch.testing.assert_close(y[True], y[False], rtol=0, atol=0, equal_nan=True)
    torch.testing.assert_close(state[True], state[False], rtol=0, atol=0, equal_nan=True)
    assert torch.equal(state[True][-1], stale[-1])
    assert torch.isfinite(y[True]).any()


@pytest.mark.parametrize("heads,groups,N,dv,B", [(64, 8, 128, 64, 3), (6, 3, 23, 40, 3), (16, 2, 64, 72, 5), (8, 8, 100, 130, 2), (1, 1, 1, 1, 1)])
def test_one_token_a_sequence(heads, groups, N, dv, B):
    """ssm_one_kernel against the walk of tokens: the same bits, fresh sequences and continued ones, rows off 16 bytes too."""
    from lit_gpt import seq_ops
    from lit_gpt.mixers import StepBatch

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(N + dv)
    rand = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    xbc, raw = rand(B, heads * dv + 2 * groups * N), rand(B, heads + 3)
    dt_bias, A_log, D = rand(heads) - 1.0, rand(heads), rand(heads)
    stale = rand(B + 1, heads, N, dv)
    step = StepBatch.build([(i, i, [0]) for i in range(B)], dev)
    y, state = {}, {}
    for max_len in (0, 1):  # 0: not known to be one token each
        state[max_len] = stale.clone()
        y[max_len] = seq_ops.ssm_scan(xbc, raw, 2, dt_bias, A_log, D, state[max_len], step.seq_start, step.seq_slot, step.seq_pos0,
                                      heads=heads, groups=groups, N=N, dv=dv, max_len=max_len)
    assert torch.equal(y[0], y[1]) and torch.equal(state[0], state[1]) and torch.equal(state[1][-1], stale[-1])
