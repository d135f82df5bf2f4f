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


@pytest.mark.parametrize("K,N1,N2", [(4, 1, 3), (252, 5, 0), (768, 2304, 3072), (1024, 4, 9), (1028, 6, 2), (4100, 7, 5), (8192, 3, 0),
                                     (256, 8200, 33)])
@pytest.mark.parametrize("bias", [True, False])
def test_one_row_norms_and_products(K, N1, N2, bias):
    """One launch for two norms and their products, one for two products and the adds: the bits of the single kernels, at the edges of
    256 columns a load, of the row's registers and of several outputs a wave."""
    from types import SimpleNamespace as Part

    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(K + N1)
    draw = lambda *shape: torch.randn(shape, generator=g, device=dev)  # noqa: E731
    x = draw(1, K)
    norms = [Part(weight=draw(K), bias=draw(K) if bias else None, eps=e) for e in (1e-5, 1e-3)]
    linears = [Part(weight=draw(n, K) * K ** -0.5, bias=draw(n) if bias else None) for n in (N1, max(N2, 1))]
    parts = [(norms[0], linears[0], None)] + [(norms[1], linears[1], "tanh")] * (N2 > 0)
    for y, (norm, linear, gelu) in zip(ops.f32_norm_linears(x, *parts), parts):
        assert torch.equal(y, ops.f32_linear(ops.layernorm(x, norm.weight, norm.bias, norm.eps), linear.weight, linear.bias, gelu=gelu))
    off = [torch.cat([t.new_zeros(1), t.flatten()])[1:] for t in (x, norms[0].weight)]  # vectors that begin on no 16 bytes
    shifted = Part(weight=off[1], bias=norms[0].bias, eps=norms[0].eps)
    assert off[0].data_ptr() % 16 == 4
    assert torch.equal(ops.f32_norm_linears(off[0].view(1, K), (shifted, linears[0], None))[0], ops.f32_norm_linears(x, parts[0])[0])
    x2, res = draw(1, 3 * K), draw(1, N1)
    wide = Part(weight=draw(N1, 3 * K) * K ** -0.5, bias=draw(N1) if bias else None)
    h = ops.f32_linear(x, linears[0].weight, linears[0].bias)
    want = ops.f32_linear(x2, wide.weight, wide.bias, residual=h, residual2=res)
    assert torch.equal(ops.f32_linears_sum(x, linears[0], x2, wide, res), want)


@pytest.mark.parametrize("K", [4, 1020, 1024, 7996, 8000, 8192])
def test_one_row_of_more_outputs_than_waves(K):
    """The outputs of 2048 workgroups and one more, and of three rounds of the fewest that longer rows take, bit by bit: rows on both
    sides of what decides how many workgroups there are."""
    from types import SimpleNamespace as Part

    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(K)
    draw = lambda *shape: torch.randn(shape, generator=g, device=dev)  # noqa: E731
    x, norm = draw(1, K), Part(weight=draw(K), bias=draw(K), eps=1e-5)
    whole = Part(weight=draw(16389, K) * K ** -0.5, bias=draw(16389))
    want = ops.f32_linear(ops.layernorm(x, norm.weight, norm.bias, norm.eps), whole.weight, whole.bias)
    for N in (8192, 8193, 8197, 16389):
        linear = Part(weight=whole.weight[:N], bias=whole.bias[:N])
        other = Part(weight=whole.weight[-5:], bias=None)
        first, second = ops.f32_norm_linears(x, (norm, linear, None), (norm, other, None))
        assert torch.equal(first, want[:, :N]) and torch.equal(second + whole.bias[-5:], want[:, -5:])


def test_one_token_past_the_modules():
    """A block's three launches give the bits of its modules called one by one (a hook keeps them apart), behind up to 64 keys."""
    from generate.base import build_model
    from lit_gpt import Config

    dev = torch.device("cuda", 0)
    m = build_model(Config.from_name("pythia-160m", n_layer=2), quantize=None, device=dev, seed=1, max_seq_length=64, dtype=torch.float32)
    idx, pos, seen = torch.tensor([[5]], device=dev), torch.tensor([9], device=dev), []
    for block in m.transformer.h:
        block.attn.kv_cache.k.normal_(), block.attn.kv_cache.v.normal_()
    with torch.inference_mode():
        fused = m(idx, pos)
        for module in (m.transformer.h[0].attn, m.transformer.h[1].attn.proj, m.transformer.ln_f):
            handle = module.register_forward_hook(lambda mod, args, out: seen.append(type(mod).__name__))
            assert torch.equal(m(idx, pos), fused)
            handle.remove()
    assert seen == ["CausalSelfAttention", "LayerNorm"]  # (a projection is no call of its module)


@pytest.mark.parametrize("hs,H,G", [(64, 12, 12), (128, 4, 2), (4, 3, 1), (256, 9, 9)])
@pytest.mark.parametrize("p0,S", [(0, 65), (31, 128), (32, 200), (63, 512), (300, 320), (511, 512), (1000, 2048)])
def test_ranges_of_keys(hs, H, G, p0, S):
    """Ranges of keys side by side, joined in the output product: ranges without keys, with one, and whole ones. Against float64: sums
    of up to 1001 weighted values of size 1 and their products with a matrix of rows of length 1 (2e-6 and sqrt(K) 2^-24 of it)."""
    from types import SimpleNamespace as Part

    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(hs + p0)
    draw = lambda *shape: torch.randn(shape, generator=g, device=dev)  # noqa: E731
    k, v, qkv = draw(1, G, S, hs), draw(1, G, S, hs), draw(1, (H + 2 * G) * hs)
    k[:, :, p0:], v[:, :, p0:] = float("nan"), float("nan")  # rows that nobody has written
    pos = torch.tensor([p0], device=dev)
    cos, sin = torch.ones(S, 2, device=dev), torch.zeros(S, 2, device=dev)
    kb, vb = k.clone(), v.clone()
    parts = ops.f32_attention_parts(H, S)
    assert parts == min(8, -(-S // 64))
    joined = ops.f32_attention_decode_parts(qkv, kb, vb, pos, pos, cos, sin, H, G, hs, 2, hs ** -0.5, parts)
    y = ops.f32_attention_decode(qkv, k, v, pos, pos, cos, sin, H, G, hs, 2, hs ** -0.5)
    assert torch.equal(k[:, :, : p0 + 1], kb[:, :, : p0 + 1]) and torch.equal(v[:, :, : p0 + 1], vb[:, :, : p0 + 1])
    K = H * hs
    one, two = Part(weight=draw(5, K) * K ** -0.5, bias=None), Part(weight=draw(5, 8), bias=draw(5))
    x2, res = draw(1, 8), draw(1, 5)
    q = qkv.view(G, H // G + 2, hs)[:, :-2].reshape(H, hs).double()
    rows = torch.arange(H, device=dev) // (H // G)
    s = torch.einsum("hd,hnd->hn", q, k[0, rows, : p0 + 1].double()) * hs ** -0.5
    want = (torch.softmax(s, 1).unsqueeze(1) @ v[0, rows, : p0 + 1].double()).view(1, K)
    end = x2.double() @ two.weight.double().T + two.bias.double() + res.double()
    want = want @ one.weight.double().T + end
    assert (ops.f32_linears_sum(joined, one, x2, two, res).double() - want).abs().max() < 1e-5
    assert (ops.f32_linears_sum(y, one, x2, two, res).double() - want).abs().max() < 1e-5


@pytest.mark.parametrize("p0", [0, 31, 32, 63, 64, 99, 127, 128, 200, 256, 447, 448, 600])
def test_ranges_follow_the_keys(p0):
    """The bits of a token's attention and output product are those of its keys, whatever the cache's size; behind up to 64 keys those
    of the unsplit form."""
    from types import SimpleNamespace as Part

    from lit_gpt import ops

    dev, H, hs, most = torch.device("cuda", 0), 3, 64, 1200
    g = torch.Generator(device=dev).manual_seed(p0)
    draw = lambda *shape: torch.randn(shape, generator=g, device=dev)  # noqa: E731
    k, v, qkv, pos = draw(1, H, most, hs), draw(1, H, most, hs), draw(1, 3 * H * hs), torch.tensor([p0], device=dev)
    cos, sin = torch.ones(most, 2, device=dev), torch.zeros(most, 2, device=dev)
    one, two = Part(weight=draw(5, H * hs), bias=draw(5)), Part(weight=draw(5, 8), bias=None)
    x2, res, seen = draw(1, 8), draw(1, 5), []
    for S in (p0 + 1, p0 + 2, 65, 128, 320, 448, 449, 512, most):
        if S > p0:
            args = (qkv, k[:, :, :S].contiguous(), v[:, :, :S].contiguous(), pos, pos, cos, sin, H, H, hs, 2, hs ** -0.5)
            parts = ops.f32_attention_parts(H, S)
            y = ops.f32_attention_decode(*args) if parts == 1 else ops.f32_attention_decode_parts(*args, parts)
            seen.append(ops.f32_linears_sum(y, one, x2, two, res))
            if p0 < 64:
                seen.append(ops.f32_linears_sum(ops.f32_attention_decode(*args), one, x2, two, res))
    assert len(seen) >= 3 and all(torch.equal(y, seen[0]) for y in seen)


@pytest.mark.parametrize("S,p0", [(320, 300), (64, 40), (1024, 700)])
def test_one_token_in_ranges_of_keys(S, p0):
    """The model's step over a cache in ranges: within the modules' one by one, whose attention is one range (a hook keeps them
    apart), by four roundings of 2^-24 a layer and product, and the same bits in a larger cache."""
    from generate.base import build_model
    from lit_gpt import Config, ops

    dev = torch.device("cuda", 0)
    assert (ops.f32_attention_parts(12, S) > 1) == (S > 64)
    idx, pos, outs = torch.tensor([[5]], device=dev), torch.tensor([p0], device=dev), []
    g = torch.Generator(device=dev).manual_seed(p0)
    filled = torch.randn(2, 2, 12, p0, 64, generator=g, device=dev)
    for size in (S, S + 448):
        m = build_model(Config.from_name("pythia-160m", n_layer=2), quantize=None, device=dev, seed=1, max_seq_length=size, dtype=torch.float32)
        for block, kv in zip(m.transformer.h, filled):
            block.attn.kv_cache.k[0, :, :p0], block.attn.kv_cache.v[0, :, :p0] = kv
        with torch.inference_mode():
            outs.append(m(idx, pos).clone())
    assert torch.equal(outs[0], outs[1])
    handles = [block.attn.register_forward_hook(lambda mod, args, out: None) for block in m.transformer.h]
    with torch.inference_mode():
        apart = m(idx, pos)
    for handle in handles:
        handle.remove()
    if S <= 64:
        assert torch.equal(apart, outs[0])
    assert float((apart - outs[0]).abs().max()) <= 2 * 6 * 4 * 2 ** -24 * float(apart.abs().max())


def test_ranges_of_infinite_scores():
    """Scores of minus infinity throughout a range, and a NaN in one, as the unsplit form has them."""
    from types import SimpleNamespace as Part

    from lit_gpt import ops

    dev, S, H, hs = torch.device("cuda", 0), 256, 2, 8
    k, v = torch.ones(1, H, S, hs, device=dev), torch.rand(1, H, S, hs, device=dev)
    k[0, 0, :64] = -float("inf")
    k[0, 1, 70] = float("nan")
    qkv, pos = torch.ones(1, 3 * H * hs, device=dev), torch.tensor([200], device=dev)
    cos, sin = torch.ones(S, 2, device=dev), torch.zeros(S, 2, device=dev)
    args = (qkv, k, v, pos, pos, cos, sin, H, H, hs, 2, 1.0)
    eye, none = Part(weight=torch.eye(hs, device=dev), bias=None), Part(weight=torch.zeros(hs, 4, device=dev), bias=None)
    want = ops.f32_attention_decode(*args).view(H, hs)
    assert want[0].isfinite().all() and want[1].isnan().all()
    y, ml, _ = ops.f32_attention_decode_parts(*args, 4)
    for h in range(H):
        head = y.view(4, H, hs)[:, h].contiguous(), ml[:, h: h + 1].contiguous(), hs
        got = ops.f32_linears_sum(head, eye, torch.zeros(1, 4, device=dev), none, torch.zeros(1, hs, device=dev))[0]
        assert got.isnan().all() if h else (got - want[0]).abs().max() < 1e-6


@pytest.mark.parametrize("M,N,K", [(8, 2999, 4), (8, 2996, 4), (9, 1501, 260), (33, 601, 1028), (65, 334, 768), (15, 1501, 255),
                                   (8, 4003, 4), (9, 8005, 260), (12, 2701, 1028), (33, 1001, 768), (65, 501, 260), (23, 1501, 255)])
def test_rows_of_prompts_to_the_bit(M, N, K):
    """Eight rows and two outputs a wave: the bits of one row at a time, past whole groups of rows and outputs."""
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(K + M)
    x, w, b, r, r2 = (torch.randn(m, generator=g, device=dev) for m in ((M, K), (N, K), (N,), (M, N), (M, N)))
    for kw in (dict(), dict(bias=b, gelu="tanh", residual=r, residual2=r2)):
        rows = [ops.f32_linear(x[i: i + 1], w, **{k: v[i: i + 1] if v is r or v is r2 else v for k, v in kw.items()}) for i in range(M)]
        assert torch.equal(ops.f32_linear(x, w, **kw), torch.cat(rows))
