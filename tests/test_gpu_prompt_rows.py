"""Kernels that stand between the layered models' products, on both sides of the lines where a step's size picks their form, against
float64 (or whole numbers): the heads' gate, routed pairs sorted and combined, queries and keys of few and many tokens,
results of products with fp32 rows at every kind of edge. fp32 results: within 16 units of 2^-24 of their own size, or of their
summands' where they are sums."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 16 * 2.0 ** -24


def close(got, want, size=None, extra=0.0):
    size = want.abs() if size is None else size
    assert ((got.double() - want).abs() <= EPS * size + extra + 1e-30).all()


@pytest.mark.parametrize("T,H,dv", [(512, 8, 128), (511, 8, 128), (517, 8, 128), (709, 8, 128), (4097, 1, 128), (300, 16, 64), (9, 16, 128)])
@pytest.mark.parametrize("rank", [0, 64, 20])
@pytest.mark.parametrize("unit", [False, True])
def test_head_gate(T, H, dv, rank, unit):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(T + rank)
    o = torch.randn(T, H * dv, generator=g, device=DEV)
    proj = torch.randn(T, (rank or H * dv) + 3, generator=g, device=DEV)
    w = torch.randn(dv, generator=g, device=DEV)
    w2 = (torch.randn(H * dv, rank, generator=g, device=DEV) * 0.2).bfloat16() if rank else None
    x = o.double().view(T, H, dv)
    if unit:
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)
    gate = proj[:, 3:].bfloat16().double() @ w2.double().T if rank else proj[:, 3:].double()
    # (a low-rank gate's input is a sum of `rank` products: its rounding moves the sigmoid by a quarter of it at most)
    off = 0.25 * rank * 2.0 ** -24 * (proj[:, 3:].abs().double() @ w2.abs().double().T if rank else gate.abs() * 0)
    want = (x * w.double()).reshape(T, -1)
    size = want.abs() * 0.7
    want = want * torch.sigmoid(gate) * 0.7
    y16 = seq_ops.head_gate(o, proj, 3, H=H, dv=dv, unit_norm=unit, eps=1e-5, act=seq_ops.ACT_SIGMOID, weight=w, post=0.7,
                            bf16_copy=True, w_g2=w2)
    close(o, want, extra=size * off)
    assert torch.equal(y16, o.bfloat16())


@pytest.mark.parametrize("T,top,E", [(1, 1, 1), (9, 3, 256), (512, 4, 18), (2048, 4, 18), (2049, 4, 18), (341, 6, 200), (3000, 4, 16)])
def test_sorted_pairs(T, top, E):
    from lit_gpt import seq_ops

    ids = torch.randint(0, E, (T, top), generator=torch.Generator(device=DEV).manual_seed(T), device=DEV, dtype=torch.int32)
    ids[ids == E // 2] = 0  # (one group empty, one larger)
    for _ in range(2):
        start, token, where = seq_ops.moe_sort(ids, E)
        assert torch.equal(start[1:] - start[:-1], torch.bincount(ids.flatten(), minlength=E).int()) and start[0] == 0
        assert torch.equal(where.sort().values, torch.arange(T * top, device=DEV, dtype=torch.int32))
        pair = torch.empty_like(where)
        pair[where.long()] = torch.arange(T * top, device=DEV, dtype=torch.int32)
        assert torch.equal(pair // top, token)
        place = torch.arange(T * top, device=DEV)
        assert torch.equal(torch.searchsorted(start[1:].contiguous(), place, right=True).int(), ids.flatten()[pair.long()])


@pytest.mark.parametrize("T,top,N", [(33, 4, 2048), (5, 1, 4), (17, 3, 2052), (9, 9, 1028), (7, 4, 2050), (3, 5, 31), (97, 2, 2064), (96, 1, 2084)])
@pytest.mark.parametrize("identity", [False, True])
@pytest.mark.parametrize("accumulate", [False, True])
def test_combined_pairs(T, top, N, identity, accumulate):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(N + top)
    y, x, h = (torch.randn(n, N, generator=g, device=DEV) for n in (T * top, T, T))
    where = torch.randperm(T * top, generator=g, device=DEV).int()
    wts = torch.rand(T, top, generator=g, device=DEV)
    ids = torch.randint(0, 6, (T, top), generator=g, device=DEV, dtype=torch.int32)
    rows = y.double()[where.long()].view(T, top, N)
    if identity:
        rows = torch.where((ids >= 4)[..., None], h.double()[:, None], rows)
    old = x.double() if accumulate else x.double() * 0
    want, size = old + (wts.double()[..., None] * rows).sum(1), old.abs() + (wts.double()[..., None] * rows.abs()).sum(1)
    seq_ops.moe_combine(y, where, wts, x, ids=ids if identity else None, n_real=4, h=h if identity else None, accumulate=accumulate)
    close(x, want, size)


@pytest.mark.parametrize("T", [1, 3, 300, 1400, 4100])
@pytest.mark.parametrize("H,G,d,dv,rot,interleaved", [(16, 4, 128, 128, 64, False), (5, 5, 48, 33, 20, True), (3, 1, 64, 40, 0, False)])
def test_queries_and_keys(T, H, G, d, dv, rot, interleaved):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(T + H)
    ld = (H + G) * d + G * dv
    proj = torch.randn(T, ld, generator=g, device=DEV)
    before, slots = proj.clone(), 2
    S = T + 3
    k = torch.full((slots, S, G, d), 7.0, device=DEV)
    v = torch.full((slots, S, G, dv), 7.0, device=DEV)
    slot = torch.ones(T, dtype=torch.int32, device=DEV)
    pos = torch.arange(2, T + 2, device=DEV, dtype=torch.int32)
    w, freq = torch.randn(d, generator=g, device=DEV), torch.rand(max(rot // 2, 1), generator=g, device=DEV)
    seq_ops.normattn_prepare(proj, 0, H * d, (H + G) * d, k, v, slot, pos, H=H, G=G, d=d, dv=dv, eps=1e-5, norm=1, q_weight=w,
                             k_weight=w, inv_freq=freq if rot else None, rot_dims=rot, interleaved=interleaved)
    x = before[:, :(H + G) * d].double().view(T, H + G, d)
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double()
    if rot:
        a = (pos.float()[:, None] * freq).double()[:, None]  # (the angle as fp32 rounds it)
        u, m = (x[..., 0:rot:2], x[..., 1:rot:2]) if interleaved else (x[..., :rot // 2], x[..., rot // 2:rot])
        turned = torch.stack([u * a.cos() - m * a.sin(), m * a.cos() + u * a.sin()], -1 if interleaved else -2)
        x = torch.cat([turned.flatten(-2), x[..., rot:]], -1)
    size = x.abs().amax(-1, keepdim=True).expand_as(x)
    close(proj[:, :H * d].view(T, H, d), x[:, :H], size[:, :H])
    close(k[1, 2:T + 2], x[:, H:], size[:, H:])
    assert torch.equal(v[1, 2:T + 2], before[:, (H + G) * d:].view(T, G, dv)) and torch.equal(proj[:, H * d:], before[:, H * d:])
    assert (k[0] == 7).all() and (k[1, :2] == 7).all() and (k[1, T + 2:] == 7).all() and (v[0] == 7).all()


@pytest.mark.parametrize("T", [640, 641, 1000, 3501])
@pytest.mark.parametrize("H,G,d,dv,rot", [(9, 3, 64, 100, 0), (9, 3, 64, 100, 30), (4, 4, 128, 256, 0), (1, 1, 10, 12, 10)])
def test_two_maps_a_head(T, H, G, d, dv, rot):
    """Tokens together give the bits that they have in a step of few, in all forms of the launch."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(T + H)
    proj = torch.randn(T, 2 * (H + G) * d + G * dv, generator=g, device=DEV)
    slot, pos = torch.zeros(T, dtype=torch.int32, device=DEV), torch.arange(T, dtype=torch.int32, device=DEV)
    freq = torch.rand(rot // 2, generator=g, device=DEV) if rot else None

    def prepare(step):
        p, k, v = proj.clone(), torch.zeros(1, T, G, 2 * d, device=DEV), torch.zeros(1, T, G, dv, device=DEV)
        for t in range(0, T, step):
            at = slice(t, min(t + step, T))
            seq_ops.diffattn_prepare(p[at], 0, 2 * H * d, 2 * (H + G) * d, k, v, freq, slot[at], pos[at], H=H, G=G, d=d, dv=dv, rot_dims=rot)
        return p, k, v

    assert all(torch.equal(a, b) for a, b in zip(prepare(T), prepare(100)))


@pytest.mark.parametrize("M,N,K", [(9, 1, 8), (130, 131, 64), (300, 513, 72), (128, 128, 64), (257, 66, 136), (129, 16, 72), (70, 18, 64), (140, 19, 64),
                                   (77, 31, 64), (130, 28, 72), (129, 33, 64)])
@pytest.mark.parametrize("kind", ["fp32", "bf16", "sums"])
@pytest.mark.parametrize("ldy", [0, 1])
def test_products_of_fp32_rows(M, N, K, kind, ldy):
    """One rounding of the rows to bf16, products exact in fp32, K additions of partial sums around 1."""
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(M + N)
    a, b = torch.randn(M, K + 8, generator=g, device=DEV), torch.randn(N, generator=g, device=DEV)
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    old = torch.randn(M, N + ldy, generator=g, device=DEV)
    y = old.bfloat16() if kind == "bf16" else old.clone()
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, a_off=8, lda=K + 8, ldy=N + ldy, bias=b, act=seq_ops.ACT_SILU, accumulate=kind == "sums", ksplit=1)
    z = a[:, 8:].bfloat16().double() @ w.double().T + b.double()
    want = z * torch.sigmoid(z) + (old[:, :N].double() if kind == "sums" else 0.0)
    assert ((y[:, :N].double() - want).abs() <= (2.0 ** -8 * want.abs() if kind == "bf16" else 0.0) + 2e-5).all()
    assert torch.equal(y[:, N:], old[:, N:].to(y.dtype))


@pytest.mark.parametrize("T", [1, 700, 5000])
@pytest.mark.parametrize("scores", [False, True])
def test_tokens_whose_logits_are_nan_choose_experts_that_there_are(T, scores):
    """(T top 10 and 7000: the sort in one launch, 50000: in three.)"""
    from lit_gpt import seq_ops

    dev, E, top = torch.device("cuda", 0), 18, 10
    z = torch.randn(T, E, generator=torch.Generator(device=dev).manual_seed(T), device=dev)
    route = seq_ops.moe_route_scores if scores else seq_ops.moe_route
    plain = route(z, 0, E, top)[0]
    z[T // 2] = float("nan")
    ids = route(z, 0, E, top)[0]
    rest = torch.arange(T, device=dev) != T // 2
    assert ids.min() >= 0 and ids.max() < E and torch.equal(ids[rest], plain[rest])
    z_start, tok_of, where = seq_ops.moe_sort(ids, E)
    assert torch.equal(z_start[1:] - z_start[:-1], torch.bincount(ids.flatten().long(), minlength=E).int())
    assert torch.equal(where.sort().values, torch.arange(T * top, dtype=torch.int32, device=dev))
    assert torch.equal(tok_of[where.long()], torch.arange(T * top, dtype=torch.int32, device=dev) // top)
