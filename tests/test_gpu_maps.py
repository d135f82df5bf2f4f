"""Low-rank maps inside the launches that use them (csrc/seq_common.h: lowrank_tiles, in the delta rule's preparation and the head gate)
against the products in whose place they stand: the same operands and the same order of sums, so the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def rand(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


@pytest.mark.parametrize("T,H,d,rank", [(65, 8, 128, 64), (97, 16, 128, 128), (2048, 1, 20, 64), (130, 5, 256, 192), (81, 33, 36, 64)])
def test_decay_maps(T, H, d, rank):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(T)
    proj, w = rand(g, T, rank + H + 8 + -(rank + H) % 4), (0.2 * rand(g, H * d, rank)).bfloat16()
    A_log, bias, qkv = rand(g, H), rand(g, H * d), rand(g, T, 3 * H * d)
    assert seq_ops.decay_map_inside(proj, 4, w, H=H, d=d)
    kw = dict(H=H, G=H, d=d, per_channel=True, q_scale=d ** -0.5)
    a = torch.empty(T, H * d, device=DEV)
    seq_ops.linear(proj, w, M=T, N=H * d, K=rank, y=a, a_off=4, lda=proj.shape[1], ldy=H * d)
    apart = seq_ops.delta_prepare(qkv.clone(), a, 0, proj, rank + 4, A_log, bias, **kw)
    inside = seq_ops.delta_prepare(qkv.clone(), proj, 4, proj, rank + 4, A_log, bias, w_a2=w, **kw)
    for one, other in zip(inside, apart):
        assert torch.equal(one, other)


@pytest.mark.parametrize("T,H,rank", [(256, 16, 64), (521, 8, 128), (4099, 1, 64)])
@pytest.mark.parametrize("bf16", [False, True])
def test_gate_maps(T, H, rank, bf16):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(T)
    dv, proj, w = 128, rand(g, T, rank + 8), (0.2 * rand(g, H * 128, rank)).bfloat16()
    o, weight = rand(g, T, H * dv), rand(g, dv)
    assert seq_ops.gate_map_inside(proj, 4, w, H=H, dv=dv)
    kw = dict(H=H, dv=dv, unit_norm=True, eps=1e-6, act=seq_ops.ACT_SIGMOID, weight=weight, post=0.7, bf16_copy=bf16)
    gate = torch.empty(T, H * dv, device=DEV)
    seq_ops.linear(proj, w, M=T, N=H * dv, K=rank, y=gate, a_off=4, lda=rank + 8, ldy=H * dv)
    one, other = o.clone(), o.clone()
    assert torch.equal(seq_ops.head_gate(one, proj, 4, w_g2=w, **kw), seq_ops.head_gate(other, gate, 0, **kw))
    assert torch.equal(one, other)


def test_maps_off_sixteen_bytes_stay_products():
    from lit_gpt import seq_ops

    proj, w = torch.zeros(4096, 128, device=DEV), torch.zeros(2048, 64, dtype=torch.bfloat16, device=DEV)
    assert seq_ops.decay_map_inside(proj, 4, w, H=16, d=128) and seq_ops.gate_map_inside(proj, 4, w, H=16, dv=128)
    for args in ((proj, 3, w), (proj[:, :126].contiguous(), 4, w), (proj, 4, w[:, :60].contiguous()), (proj, 4, w.float())):
        assert not seq_ops.decay_map_inside(*args, H=16, d=128) and not seq_ops.gate_map_inside(*args, H=16, dv=128)
    assert not seq_ops.decay_map_inside(proj[:64], 4, w, H=16, d=128) and not seq_ops.gate_map_inside(proj[:255], 4, w, H=16, dv=128)


def test_long_maps_of_many_tokens_stay_products():
    """Both sides of the line, where the gate makes the map of rows that share it with others, and where a product does."""
    from lit_gpt import seq_ops

    def inside(T, H, rank):
        proj, w = torch.empty(T, rank, device=DEV), torch.empty(H * 128, rank, dtype=torch.bfloat16, device=DEV)
        return seq_ops.gate_map_inside(proj, 0, w, H=H, dv=128)

    assert inside(16384, 32, 192) and inside(5632, 32, 256) and inside(1024, 32, 512)
    assert not inside(5633, 32, 256) and not inside(2048, 32, 384) and not inside(1127, 32, 512)
