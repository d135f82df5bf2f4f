"""The fp32 (32-true) kernels against float64: attention in both forms, and the fused norms, activations and adds."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hs", [4, 6, 64, 80, 128, 256])
@pytest.mark.parametrize("H,G", [(3, 3), (4, 2), (5, 1)])
@pytest.mark.parametrize("T,p0,S", [(1, 0, 1), (1, 31, 40), (1, 32, 33), (1, 700, 1024), (5, 60, 70)])
def test_attention(hs, H, G, T, p0, S):
    """Edges of the four rows in flight per wave (32 to 128 keys a step) and of the lanes per row."""
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(hs + H + S)
    k = torch.randn(1, G, S, hs, generator=g, device=dev)
    v = torch.randn(1, G, S, hs, generator=g, device=dev)
    k[:, :, p0 + T:], v[:, :, p0 + T:] = float("nan"), float("nan")  # rows that nobody has written
    q = torch.randn(T, H, hs, generator=g, device=dev)
    pos = torch.arange(p0, p0 + T, device=dev)
    got = ops.attention(q, k, v, pos, H, G, hs, hs ** -0.5).view(T, H, hs)
    for t in range(T):
        n = p0 + t + 1
        for h in range(H):
            s = k[0, h // (H // G), :n].double() @ q[t, h].double() * hs ** -0.5
            want = torch.softmax(s, 0) @ v[0, h // (H // G), :n].double()
            assert (got[t, h].double() - want).abs().max() < 2e-6  # sums of up to 700 weighted values of size 1
    if T == 1 and ops.f32_decode_fusable(hs, S):  # rotation, append and attention in one launch: the same numbers
        half = hs // 4 * 2
        ang = torch.rand(S, half // 2, generator=g, device=dev).repeat(1, 2)
        cos, sin = torch.cos(ang), torch.sin(ang)
        qkv = torch.randn(1, (H + 2 * G) * hs, generator=g, device=dev)
        ka, va, kb, vb = k.clone(), v.clone(), k.clone(), v.clone()
        qa = ops.rope_kv_append(qkv, ka, va, pos, pos, cos, sin, H, G, hs, half)
        want = ops.attention(qa, ka, va, pos, H, G, hs, hs ** -0.5)
        y = ops.f32_attention_decode(qkv, kb, vb, pos, pos, cos, sin, H, G, hs, half, hs ** -0.5)
        assert torch.equal(y, want)
        assert torch.equal(ka[:, :, : p0 + 1], kb[:, :, : p0 + 1]) and torch.equal(va[:, :, : p0 + 1], vb[:, :, : p0 + 1])


@pytest.mark.parametrize("rows,n", [(1, 1), (3, 255), (2, 768), (2, 1025), (1, 5000)])
def test_fused_norms_activations_and_adds(rows, n):
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(n)
    x, w, b, w2 = (torch.randn(m, generator=g, device=dev) for m in ((rows, n), (n,), (n,), (n,)))
    y, y2 = ops.f32_layernorm_pair(x, w, b, 1e-5, w2, None, 1e-3)
    assert torch.equal(y, ops.layernorm(x, w, b, 1e-5)) and torch.equal(y2, ops.layernorm(x, w2, None, 1e-3))
    want = torch.nn.functional.layer_norm(x.double(), (n,), w.double(), b.double(), 1e-5)
    assert (y.double() - want).abs().max() < 1e-5
    m = torch.randn(7, n, generator=g, device=dev) * n ** -0.5
    r, r2, c = (torch.randn(rows, 7, generator=g, device=dev) for _ in range(3))
    for kind in ("none", "tanh"):
        lin = ops.f32_linear(x, m, bias=c[0])
        want = ops.gelu(lin, kind) + r + r2
        assert torch.equal(ops.f32_linear(x, m, bias=c[0].contiguous(), gelu=kind, residual=r, residual2=r2), want)


def test_caches_off_sixteen_bytes():
    """A decode step over caches that start on 4 bytes: the unfused form's."""
    from generate.base import build_model
    from lit_gpt import Config

    dev = torch.device("cuda", 0)
    m = build_model(Config.from_name("pythia-160m", n_layer=1), quantize=None, device=dev, seed=1, max_seq_length=64, dtype=torch.float32)
    kv, outs = m.transformer.h[0].attn.kv_cache, []
    idx, pos = torch.tensor([[5]], device=dev), torch.tensor([9], device=dev)
    g = torch.Generator(device=dev).manual_seed(1)
    filled = {n: torch.randn(getattr(kv, n).shape, generator=g, device=dev) for n in "kv"}
    with torch.inference_mode():
        for off in (0, 1):
            for n, t in filled.items():
                setattr(kv, n, torch.empty(t.numel() + off, device=dev)[off:].view(t.shape).copy_(t))
            outs.append(m(idx, pos).clone())
    assert float((outs[0] - outs[1]).abs().max()) < 1e-5 * float(outs[0].abs().max())
