"""Prompt attention on the bf16 matrix cores (csrc/seq_attn_tiles.hip) against float64 and against the thread-per-key form.

The same bf16 keys and values in an fp32 cache take the thread-per-key form, whose products are fp32: the matrix-core form's
error against float64 is no larger than that one's. Its own bound: with scores of a few units, 2e-6 relative in the 2-norm covers
the scores' rounding (24 bits of a sum of up to 192 products), the exponentials and up to 2000 weighted values.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 2e-6


def rel(x, want):
    return float((x.double() - want).norm() / want.norm())


def visible(pos, S, chunk, window):
    at = torch.arange(S, device=pos.device)
    see = at[None] <= pos[:, None]
    if chunk:
        see &= at[None] // chunk == pos[:, None] // chunk
    if window:
        see &= at[None] > pos[:, None] - window
    return see


def step(lengths, pos0, dev):
    start = torch.tensor([0] + list(lengths)).cumsum(0).to(torch.int32).to(dev)
    order = torch.randperm(len(lengths) + 1, generator=torch.Generator().manual_seed(1))[: len(lengths)]
    return start, order.to(torch.int32).to(dev), torch.tensor(pos0, dtype=torch.int32, device=dev)


def caches(slots, S, G, dk, dv, dev, g, filled):
    """bf16 rows; what no sequence has written is NaN."""
    k = torch.full((slots, S, G, dk), float("nan"), device=dev)
    v = torch.full((slots, S, G, dv), float("nan"), device=dev)
    for slot, n in filled:
        k[slot, :n] = torch.randn(n, G, dk, generator=g, device=dev)
        v[slot, :n] = torch.randn(n, G, dv, generator=g, device=dev)
    return k.bfloat16(), v.bfloat16()


STEPS = [([2], [61]), ([16], [0]), ([17, 1, 40], [0, 5, 100]), ([300, 64, 129], [0, 63, 31]), ([700], [513])]


@pytest.mark.parametrize("lengths,pos0", STEPS)
@pytest.mark.parametrize("d,dv", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("H,G,options", [
    (4, 1, {}), (4, 4, dict(sink=True)), (4, 2, dict(cap=3.0)), (6, 3, dict(chunk=48)), (8, 2, dict(window=33, gate=1)), (3, 1, dict(sigmoid=True)),
    (8, 1, dict(sink=True, cap=5.0, rotated=True)), (4, 2, dict(gate=2, rotated=True, interleaved=True, chunk=100)),
    (8, 2, dict(sigmoid=True, chunk=64))])
def test_one_map(lengths, pos0, d, dv, H, G, options):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(d + dv + H)
    T, S, slots = sum(lengths), max(p + n for p, n in zip(pos0, lengths)) + 3, len(lengths) + 1
    start, slot, first = step(lengths, pos0, dev)
    ends = [p + n for p, n in zip(pos0, lengths)]
    k, v = caches(slots, S, G, d, dv, dev, g, list(zip(slot.tolist(), ends)))
    ld = H * d + H * dv + 8
    proj = torch.randn(T, ld, generator=g, device=dev)
    sink = torch.randn(H, generator=g, device=dev) if options.get("sink") else None
    bias = torch.randn(H, generator=g, device=dev) if options.get("sigmoid") else None
    freq = torch.rand(dv // 2, generator=g, device=dev) if options.get("rotated") else None
    chunk, window, cap = options.get("chunk", 0), options.get("window", 0), options.get("cap", 0.0)
    gates = {0: -1, 1: H * d, 2: H * d}[options.get("gate", 0)]
    kw = dict(H=H, G=G, d=d, dv=dv, scale=d ** -0.5, chunk=chunk, cap=cap, post=0.7, window=window, v_freq=freq,
              interleaved=options.get("interleaved", False), score_bias=bias, gate_off=gates,
              gate_cols=dv if options.get("gate") == 2 else 1)
    args = (sink, start, slot, first, max(lengths))
    got = seq_ops.sinkattn(proj, 0, k, v, *args, **kw)
    got16 = seq_ops.sinkattn(proj, 0, k, v, *args, bf16_copy=True, **kw)
    plain = seq_ops.sinkattn(proj, 0, k.float(), v.float(), *args, **kw)
    want = torch.empty(T, H, dv, dtype=torch.float64, device=dev)
    for b, (n, p0) in enumerate(zip(lengths, pos0)):
        rows, pos = slice(int(start[b]), int(start[b + 1])), torch.arange(p0, p0 + n, device=dev)
        kd, vd = k[slot[b], : p0 + n].double(), v[slot[b], : p0 + n].double()
        see = visible(pos, p0 + n, chunk, window)
        for h in range(H):
            s = proj[rows, h * d:(h + 1) * d].double() @ kd[:, h // (H // G)].T * d ** -0.5
            s = cap * torch.tanh(s / cap) if cap else s
            if bias is not None:
                w = torch.sigmoid(s + bias[h].double()) * see
            else:
                s = s.masked_fill(~see, -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[h].double().expand(n, 1)], -1)
                w = torch.softmax(s, -1)[:, : p0 + n]
            o = w @ vd[:, h // (H // G)] * 0.7
            if freq is not None:
                ang = pos[:, None] * freq.double()
                c, sn = torch.cos(ang), torch.sin(ang)
                i, j = (slice(0, None, 2), slice(1, None, 2)) if kw["interleaved"] else (slice(0, dv // 2), slice(dv // 2, None))
                x, y = o[:, i].clone(), o[:, j].clone()
                o[:, i], o[:, j] = x * c + y * sn, y * c - x * sn
            if gates >= 0:
                z = proj[rows, gates + (h * dv if kw["gate_cols"] > 1 else h):][:, : kw["gate_cols"]].double()
                o = o * torch.sigmoid(z)
            want[rows, h] = o
    want = want.flatten(1)
    # (turning back by fp32 angles of up to 1200 radians: both forms take the same cosines, off by up to 1e-4)
    bound = 1e-4 if freq is not None else TOL
    assert rel(got, want) < bound and rel(got, want) < 1.001 * rel(plain, want)  # (turned back: the same angles' errors)
    assert torch.equal(got16, got.bfloat16())


@pytest.mark.parametrize("lengths,pos0", STEPS)
@pytest.mark.parametrize("dv", [64, 128])
@pytest.mark.parametrize("H,G,chunk,cap", [(2, 2, 0, 0.0), (4, 2, 40, 30.0), (4, 1, 128, 30.0), (8, 2, 0, 3.0)])
def test_two_maps(lengths, pos0, dv, H, G, chunk, cap):
    from lit_gpt import seq_ops

    dev, d = torch.device("cuda", 0), 64
    g = torch.Generator(device=dev).manual_seed(dv + H)
    T, S, slots = sum(lengths), max(p + n for p, n in zip(pos0, lengths)) + 3, len(lengths) + 1
    start, slot, first = step(lengths, pos0, dev)
    ends = [p + n for p, n in zip(pos0, lengths)]
    k, v = caches(slots, S, G, 2 * d, dv, dev, g, list(zip(slot.tolist(), ends)))
    proj = torch.randn(T, 2 * H * d + 4, generator=g, device=dev)
    kw = dict(H=H, G=G, d=d, dv=dv, chunk=chunk, scale=0.125, cap=cap, lam=0.4, eps=1e-5, post=0.5)
    args = (start, slot, first, max(lengths))
    got = seq_ops.diffattn(proj, 0, k, v, *args, **kw)
    plain = seq_ops.diffattn(proj, 0, k.float(), v.float(), *args, **kw)
    want = torch.empty(T, H, dv, dtype=torch.float64, device=dev)
    for b, (n, p0) in enumerate(zip(lengths, pos0)):
        rows, pos = slice(int(start[b]), int(start[b + 1])), torch.arange(p0, p0 + n, device=dev)
        kd, vd = k[slot[b], : p0 + n].double(), v[slot[b], : p0 + n].double()
        see = visible(pos, p0 + n, chunk, 0)
        for h in range(H):
            maps = []
            for i in range(2):
                q = proj[rows, (2 * h + i) * d:(2 * h + i + 1) * d].double()
                s = q @ kd[:, h // (H // G), i * d:(i + 1) * d].T * 0.125
                s = cap * torch.tanh(s / cap) if cap else s
                maps.append(torch.softmax(s.masked_fill(~see, -math.inf), -1) @ vd[:, h // (H // G)])
            o = maps[0] - 0.4 * maps[1]
            want[rows, h] = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * 0.5
    want = want.flatten(1)
    # (a query that sees one key has two equal maps: their difference keeps all bits here, and nothing cancels)
    assert rel(got, want) < TOL and rel(got, want) < rel(plain, want)


def test_caches_off_sixteen_bytes():
    """Caches that start on 8 bytes take the form whose loads are that wide."""
    from lit_gpt import seq_ops

    dev, T, H, d = torch.device("cuda", 0), 90, 2, 64
    g = torch.Generator(device=dev).manual_seed(8)
    start, slot, first = step([T], [0], dev)
    k, v = caches(2, T, 1, d, d, dev, g, [(int(slot[0]), T)])
    proj = torch.randn(T, 2 * H * d, generator=g, device=dev)

    def off(t):
        return torch.empty(t.numel() + 4, dtype=t.dtype, device=dev)[4:].view(t.shape).copy_(t)

    kw = dict(H=H, G=1, d=d, dv=d, scale=0.125)
    want = seq_ops.sinkattn(proj, 0, k.float(), v.float(), None, start, slot, first, T, **kw)
    for pair in ((off(k), v), (k, off(v)), (off(k), off(v))):
        assert torch.equal(seq_ops.sinkattn(proj, 0, *pair, None, start, slot, first, T, **kw), want)
    two, kw = torch.cat([k, k], -1), dict(kw, chunk=0, cap=0.0, lam=0.4, eps=1e-5, post=0.5)
    want = seq_ops.diffattn(proj, 0, two.float(), v.float(), start, slot, first, T, **kw)
    assert torch.equal(seq_ops.diffattn(proj, 0, off(two), off(v), start, slot, first, T, **kw), want)


def test_large_scores_and_infinite_queries():
    """A key that outweighs all others, scores far below it, and a query whose scores overflow: as the other form has it."""
    from lit_gpt import seq_ops

    dev, T, d = torch.device("cuda", 0), 96, 64
    g = torch.Generator(device=dev).manual_seed(3)
    start, slot, first = step([T], [0], dev)
    k, v = caches(2, T, 1, d, d, dev, g, [(int(slot[0]), T)])
    k[int(slot[0]), 40] *= 100.0
    proj = torch.randn(T, d, generator=g, device=dev) * 10.0
    proj[50] = 3e38
    kw = dict(H=1, G=1, d=d, dv=d, scale=1.0)
    got = seq_ops.sinkattn(proj, 0, k, v, None, start, slot, first, T, **kw)
    plain = seq_ops.sinkattn(proj, 0, k.float(), v.float(), None, start, slot, first, T, **kw)
    rest = torch.arange(T, device=dev) != 50
    # scores of up to 1e5 carry errors of 1e-2: only weights that dominate are alike
    assert torch.isfinite(got[rest]).all() and (got[rest] - plain[rest]).abs().max() < 0.1
    # infinite scores of both signs: no softmax, in either form
    assert plain[50].isnan().all() and got[50].isnan().all()


def test_sigmoid_of_infinities():
    """Heads that a score bias switches off or on (-inf: weights 0, inf: weights 1) and biases past every exponential."""
    from lit_gpt import seq_ops

    dev, T, H, d = torch.device("cuda", 0), 70, 6, 64
    g = torch.Generator(device=dev).manual_seed(4)
    start, slot, first = step([T], [0], dev)
    k, v = caches(2, T, 1, d, d, dev, g, [(int(slot[0]), T)])
    proj = torch.randn(T, H * d, generator=g, device=dev)
    bias = torch.tensor([-math.inf, math.inf, -3.4e38, 3.4e38, -200.0, 0.0], device=dev)
    kw = dict(H=H, G=1, d=d, dv=d, scale=0.125, score_bias=bias)
    got = seq_ops.sinkattn(proj, 0, k, v, None, start, slot, first, T, **kw).view(T, H, d)
    assert float(got[:, [0, 2, 4]].abs().max()) == 0.0
    sums = v[slot[0].item(), :T, 0].double().cumsum(0)
    for h in (1, 3):
        assert rel(got[:, h], sums) < TOL
    plain = seq_ops.sinkattn(proj, 0, k.float(), v.float(), None, start, slot, first, T, **kw).view(T, H, d)
    assert torch.isfinite(got).all() and rel(got, plain.double()) < TOL


def _softmax_row(q, k, v, scale, cap=0.0, bias=None):
    """One query over its visible keys in float64; a key of weight 0 contributes nothing."""
    s = (q.double() * k.double()).sum(-1) * scale
    s = cap * torch.tanh(s / cap) if cap else s
    if bias is not None:
        w = torch.sigmoid(s + bias)
    else:
        w = torch.exp(s - s.max()) if not s.isnan().any() else s
        w = w / w.sum()
    return (w[:, None] * v.double()).sum(0)


def _alike(got, want, tol=1e-5):
    """The same elements infinite (with their signs) and NaN, and the finite ones as close as fp32 sums leave them."""
    fine = torch.isfinite(want)
    same = torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf()) and \
        torch.equal(got.isneginf(), want.isneginf())
    return same and (not fine.any() or float((got - want)[fine].abs().max()) < tol * float(want[fine].abs().max().clamp(min=1.0)))


@pytest.mark.parametrize("H,G,options", [(4, 1, dict(cap=5.0)), (3, 1, dict(sigmoid=True)), (4, 4, {}), (2, 1, dict(chunk=64)),
                                         (2, 2, dict(window=40, cap=2.0))])
@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128)])
def test_infinities_and_nan(H, G, options, d, dv):
    """Queries with an infinity, cached keys and values with infinities and a NaN: every query has what float64 gives it over
    the keys that it sees, and the others nothing of it."""
    from lit_gpt import seq_ops

    dev, T = torch.device("cuda", 0), 150
    g = torch.Generator(device=dev).manual_seed(d + H)
    start, slot, first = step([T], [0], dev)
    at = int(slot[0])
    k, v = caches(2, T, G, d, dv, dev, g, [(at, T)])
    proj = torch.randn(T, H * d, generator=g, device=dev)
    proj[20, 3], proj[33, d - 1], proj[90, 5] = math.inf, -math.inf, math.nan
    k[at, 70, :, 2], k[at, 100, :, 0] = math.inf, math.nan
    v[at, 45, :, 1], v[at, 80, :, dv - 1] = math.inf, -math.inf
    v[at, 120, :, 7] = math.nan
    bias = torch.randn(H, generator=g, device=dev) if options.get("sigmoid") else None
    chunk, window, cap = options.get("chunk", 0), options.get("window", 0), options.get("cap", 0.0)
    got = seq_ops.sinkattn(proj, 0, k, v, None, start, slot, first, T, H=H, G=G, d=d, dv=dv, scale=d ** -0.5, chunk=chunk,
                           window=window, cap=cap, score_bias=bias).view(T, H, dv)
    see = visible(torch.arange(T, device=dev), T, chunk, window)
    for t in range(T):
        for h in range(H):
            keys, vals = k[at, :T, h // (H // G)][see[t]], v[at, :T, h // (H // G)][see[t]]
            want = _softmax_row(proj[t, h * d:(h + 1) * d], keys, vals, d ** -0.5, cap, None if bias is None else bias[h].double())
            assert _alike(got[t, h].double(), want), (t, h)


def test_two_maps_beside_a_nan():
    """Rows before an infinite value or a NaN are those without it, rows that see it are not finite."""
    from lit_gpt import seq_ops

    dev, T, H, d, dv = torch.device("cuda", 0), 150, 4, 64, 128
    g = torch.Generator(device=dev).manual_seed(5)
    start, slot, first = step([T], [0], dev)
    k, v = caches(2, T, 2, 2 * d, dv, dev, g, [(int(slot[0]), T)])
    proj = torch.randn(T, 2 * H * d, generator=g, device=dev)
    kw = dict(H=H, G=2, d=d, dv=dv, chunk=0, scale=0.125, cap=0.0, lam=0.4, eps=1e-5, post=0.5)
    run = lambda v: seq_ops.diffattn(proj, 0, k, v, start, slot, first, T, **kw).view(T, H, dv)  # noqa: E731
    clean = run(v)
    for value in (math.inf, math.nan):
        dirty = v.clone()
        dirty[int(slot[0]), 77, 0, 9] = value
        got = run(dirty)
        assert torch.equal(got[:, 2:], clean[:, 2:])  # the other key head's
        assert _alike(got[:77, :2].double(), clean[:77, :2].double())
        assert got[77:, :2, 9].isnan().all()
    proj[30, 2] = math.inf  # with a cap an infinite score is a large one
    kw["cap"] = 5.0
    got = run(v)[30, 0]
    keys, vals = k[int(slot[0]), :31, 0], v[int(slot[0]), :31, 0]
    o = _softmax_row(proj[30, :d], keys[:, :d], vals, 0.125, 5.0) - 0.4 * _softmax_row(proj[30, d:2 * d], keys[:, d:], vals, 0.125, 5.0)
    assert _alike(got.double(), o / torch.sqrt((o * o).mean() + 1e-5) * 0.5)


def test_expanded_infinities():
    """An infinite and a NaN expanded value, a key past the largest bf16: the rows that do not see them are untouched."""
    from lit_gpt import seq_ops

    dev, T, H, d, dr, dv = torch.device("cuda", 0), 130, 2, 128, 64, 128
    g = torch.Generator(device=dev).manual_seed(6)
    start, slot, first = step([T], [0], dev)
    q = torch.randn(T, H * (d + dr), generator=g, device=dev)
    kv = torch.randn(T, H * (d + dv), generator=g, device=dev)
    kr = torch.randn(2, T, dr, generator=g, device=dev)
    rows = slot[0] * T + torch.arange(T, device=dev, dtype=torch.int32)
    run = lambda kv: seq_ops.expanded_latent_attention(  # noqa: E731
        q, 0, kv, kr, rows, None, start, slot, first, T, H=H, d=d, dr=dr, dv=dv, scale=192 ** -0.5).view(T, H, dv)
    clean = run(kv)
    dirty = kv.clone()
    dirty[50, H * d + 3], dirty[60, H * d + 9], dirty[99, 4] = math.inf, math.nan, 3.4e38
    got = run(dirty)
    assert torch.equal(got[:, 1], clean[:, 1]) and _alike(got[:50, 0].double(), clean[:50, 0].double())
    assert got[50:99, 0, 3].isposinf().all() and got[60:, 0, 9].isnan().all()
    rest = [c for c in range(dv) if c not in (3, 9)]
    assert _alike(got[50:99, 0, rest].double(), clean[50:99, 0, rest].double(), 2.0 ** -14)


@pytest.mark.parametrize("lengths", [[9], [16, 2, 40], [300, 64, 129], [1100]])
@pytest.mark.parametrize("H,window,sink", [(1, 0, False), (3, 0, True), (4, 50, False)])
def test_expanded_latent_attention(lengths, H, window, sink):
    """Keys and values in two bf16 summands (16 bits of their significands: 2^-17 of a product) against float64."""
    from lit_gpt import seq_ops

    dev, d, dr, dv = torch.device("cuda", 0), 128, 64, 128
    g = torch.Generator(device=dev).manual_seed(H)
    T, slots, S = sum(lengths), len(lengths) + 1, max(lengths) + 5
    start, slot, first = step(lengths, [0] * len(lengths), dev)
    q = torch.randn(T, H * (d + dr) + 4, generator=g, device=dev)
    kv = torch.randn(T, H * (d + dv), generator=g, device=dev)
    kr = torch.full((slots, S, dr), float("nan"), device=dev)
    rows = torch.cat([slot[b] * S + torch.arange(n, device=dev, dtype=torch.int32) for b, n in enumerate(lengths)])
    kr.view(-1, dr)[rows.long()] = torch.randn(T, dr, generator=g, device=dev)
    snk = torch.randn(H, generator=g, device=dev) if sink else None
    args = (q, 4, kv, kr, rows, snk, start, slot, first, max(lengths))
    kw = dict(H=H, d=d, dr=dr, dv=dv, scale=192 ** -0.5, window=window)
    got = seq_ops.expanded_latent_attention(*args, **kw)
    want = torch.empty(T, H, dv, dtype=torch.float64, device=dev)
    for b, n in enumerate(lengths):
        r, pos = slice(int(start[b]), int(start[b + 1])), torch.arange(n, device=dev)
        see = visible(pos, n, 0, window)
        for h in range(H):
            k = torch.cat([kv[r, h * d:(h + 1) * d], kr[slot[b], :n]], -1).double()
            s = q[r, 4 + h * 192:4 + (h + 1) * 192].double() @ k.T * 192 ** -0.5
            s = s.masked_fill(~see, -math.inf)
            s = torch.cat([s, snk[h].double().expand(n, 1)], -1) if sink else s
            want[r, h] = torch.softmax(s, -1)[:, :n] @ kv[r, H * d + h * dv:H * d + (h + 1) * dv].double()
    # scores of size 1 from 192 products of relative error 2^-17 each, uncorrelated; values likewise
    assert rel(got, want.flatten(1)) < 2.0 ** -16
    assert torch.equal(seq_ops.expanded_latent_attention(*args, bf16=True, **kw), got.bfloat16())


# (rows of 4096 elements: 2^30 of them and 2^31 bytes lie at row 262,144; what no sequence has written stays as it is)
FAR = 262_400


@pytest.mark.parametrize("n,pos0,chunk,window", [(2, 0, 0, 0), (100, 262_110, 64, 0), (70, 262_100, 0, 90), (17, 262_383, 100, 0)])
@pytest.mark.parametrize("maps", [1, 2])
def test_caches_past_one_buffer(n, pos0, chunk, window, maps):
    from lit_gpt import seq_ops

    if window and maps == 2:
        pytest.skip("two maps have no window")
    dev, H, G, d = torch.device("cuda", 0), 64 // maps, 64 // maps, 64
    dv = 64 * maps
    g = torch.Generator(device=dev).manual_seed(n)
    k = torch.empty(1, FAR, G, maps * d, dtype=torch.bfloat16, device=dev)
    v = torch.empty(1, FAR, G, dv, dtype=torch.bfloat16, device=dev)
    lo = max(0, pos0 - 200)
    for t in (k, v):
        t[:, :FAR - 200] = math.nan
        t[:, lo:pos0 + n] = torch.randn(1, pos0 + n - lo, *t.shape[2:], generator=g, device=dev).bfloat16()
    proj = torch.randn(n, H * maps * d, generator=g, device=dev)
    start, slot, first = (torch.tensor(x, dtype=torch.int32, device=dev) for x in ([0, n], [0], [pos0]))
    kw = dict(H=H, G=G, d=d, dv=dv, scale=0.125, chunk=chunk)
    if maps == 1:
        got = seq_ops.sinkattn(proj, 0, k, v, None, start, slot, first, n, window=window, **kw)
    else:
        got = seq_ops.diffattn(proj, 0, k, v, start, slot, first, n, cap=0.0, lam=0.4, eps=1e-5, post=0.5, **kw)
    kd, vd = k[0, lo:pos0 + n].double().transpose(0, 1), v[0, lo:pos0 + n].double().transpose(0, 1)
    see = visible(torch.arange(pos0, pos0 + n, device=dev), pos0 + n, chunk, window)[:, lo:]
    q, out = proj.double().view(n, H, maps, d), []
    for i in range(maps):
        s = torch.matmul(q[:, :, i].transpose(0, 1), kd[..., i * d:(i + 1) * d].transpose(1, 2).contiguous()) * 0.125
        out.append(torch.matmul(torch.softmax(s.masked_fill(~see, -math.inf), -1), vd).transpose(0, 1))
    want = out[0]
    if maps == 2:
        o = out[0] - 0.4 * out[1]
        want = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * 0.5
    assert rel(got, want.flatten(1)) < TOL


def test_expanded_rows_past_one_buffer():
    """128 heads: the summands of 21,846 tokens' keys are 2^30 elements."""
    from lit_gpt import seq_ops

    dev, T, H, d, dr, dv, window = torch.device("cuda", 0), 22_100, 128, 128, 64, 128, 33
    g = torch.Generator(device=dev).manual_seed(7)
    start, slot, first = (torch.tensor(x, dtype=torch.int32, device=dev) for x in ([0, T], [0], [0]))
    q = torch.randn(T, H * (d + dr), generator=g, device=dev)
    kv = torch.randn(T, H * (d + dv), generator=g, device=dev)
    kr = torch.randn(1, T, dr, generator=g, device=dev)
    got = seq_ops.expanded_latent_attention(q, 0, kv, kr, torch.arange(T, device=dev, dtype=torch.int32), None, start, slot, first,
                                            T, H=H, d=d, dr=dr, dv=dv, scale=192 ** -0.5, window=window).view(T, H, dv)
    assert torch.isfinite(got).all()
    for t in (40, 21_800, 21_845, 21_846, 21_900, T - 1):
        seen = slice(t - window + 1, t + 1)
        for h in (0, 77, 127):
            k = torch.cat([kv[seen, h * d:(h + 1) * d], kr[0, seen]], -1).double()
            w = torch.softmax(k @ q[t, h * 192:(h + 1) * 192].double() * 192 ** -0.5, -1)
            assert rel(got[t, h], w @ kv[seen, H * d + h * dv:H * d + (h + 1) * dv].double()) < 2.0 ** -14
