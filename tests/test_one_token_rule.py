"""How many workgroups share one token's keys, on both sides of each line of the rule (on the host)."""

import pytest
import torch


@pytest.mark.parametrize("B,H,G,span,dtype,splits", [
    (1, 16, 4, 64, torch.bfloat16, 1), (1, 16, 4, 65, torch.bfloat16, 2), (1, 16, 4, 1024, torch.bfloat16, 16),
    (1, 16, 4, 4096, torch.bfloat16, 64), (8, 16, 4, 2048, torch.bfloat16, 8), (63, 16, 4, 128, torch.bfloat16, 2),
    (64, 16, 4, 64, torch.bfloat16, 1), (64, 16, 4, 65, torch.bfloat16, 2), (256, 16, 4, 4096, torch.bfloat16, 2),
    (1, 16, 4, 64, torch.float32, 1), (1, 16, 4, 300, torch.float32, 3), (8, 16, 4, 2048, torch.float32, 4)])
def test_splits(B, H, G, span, dtype, splits):
    from lit_gpt import seq_ops

    cache = torch.empty(0, dtype=dtype)
    assert seq_ops._one_token_splits(1, B, H, G, 128, 128, span, cache) == splits
    assert seq_ops._one_token_splits(2, B, H, G, 64, 128, span, cache) == splits
    # rows of another size: the general form's number
    general = max(1, min(64, 512 // (B * H), (span + 127) // 128))
    assert seq_ops._one_token_splits(1, B, H, G, 64, 64, span, cache) == general


def test_heads_of_a_workgroup():
    from lit_gpt import seq_ops

    heads = seq_ops.load_library().lgs_attn_one_heads
    assert [heads(1, B, 16, 4, 128, 128) for B in (1, 63, 64, 300)] == [1, 1, 2, 2]
    assert heads(1, 64, 16, 16, 128, 128) == 1 and heads(1, 1, 16, 4, 64, 128) == 0 and heads(2, 1, 16, 4, 128, 128) == 0
