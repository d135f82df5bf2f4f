"""Prompt products whose 4-bit weights are dequantized in registers (csrc/gemm_q4d.hip) and those of bf16 weights on the
pipelined tiles (csrc/gemm_bf16.hip), reached through ops.q4_gemm_fused and ops.q4_gemm_swiglu, against the fp32 product of
the bit-exact dequantized weight (lga_q4_dequantize): rows at and around the 16-row pieces and the 128-row tile, columns that
end inside a tile and inside a wave's piece, one to many blocks of K, whole and split, and every epilogue. Tolerances: the two sums' bf16 roundings may each fall one place apart."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from lit_gpt import ops as _ops

    _ops.load_library()
    return _ops


def _weight(ops, N, K, fmt, group, g):
    w = torch.randn(N, K, generator=g, device=DEV) * 0.02
    if fmt == 2:
        w = w.to(torch.bfloat16)
        return w, None, w.float()
    qw, sc = ops.quantize(w, fmt, group)
    return qw, sc, ops.q4_dequantize(qw, sc, N, K, group, fmt).float()


SHAPES = [(33, 8, 128), (48, 136, 384), (64, 264, 1408), (65, 520, 4096), (96, 1032, 256),
          (1, 8200, 2176), (16, 4104, 4224), (17, 8200, 2176), (32, 4104, 4224),
          (97, 8712, 7808), (128, 8712, 7808), (129, 264, 1408), (200, 4096, 4096), (256, 136, 128),
          (257, 4104, 320), (517, 520, 4160), (1024, 1032, 64), (1025, 264, 1408), (700, 24584, 192)]


@pytest.mark.parametrize("fmt,group", [(0, 128), (0, 64), (1, 64), (2, 64), (3, 128)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product(ops, fmt, group, M, N, K):
    if fmt != 2 and K % group:
        pytest.skip("the group does not divide K")
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    w, sc, wd = _weight(ops, N, K, fmt, group, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    res = torch.randn(M, N, generator=g, device=DEV).to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    h = x.float() @ wd.t()
    plain = ops.q4_gemm_fused(x, w, sc, N, K, group, fmt)
    assert float(((plain.float() - h).abs() - h.abs() * 2 ** -7).max()) <= 2e-3
    assert torch.equal(plain, ops.q4_gemm_fused(x, w, sc, N, K, group, fmt))
    h = h + bias.float()
    y = ops.q4_gemm_fused(x, w, sc, N, K, group, fmt, bias=bias, residual=res).float()
    ref = h.to(torch.bfloat16).float() + res.float()
    assert float(((y - ref).abs() - (ref.abs() + h.abs()) * 2 ** -7).max()) <= 2e-3


@pytest.mark.parametrize("fmt,group", [(0, 128), (1, 64), (2, 64)])
@pytest.mark.parametrize("M,N,K", [(33, 8, 128), (64, 136, 1408), (80, 1032, 384), (16, 4104, 4224), (128, 8712, 7808),
                                   (300, 520, 4160), (517, 4104, 320)])
def test_swiglu(ops, fmt, group, M, N, K):
    if fmt != 2 and K % group:
        pytest.skip("the group does not divide K")
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    w1, s1, d1 = _weight(ops, N, K, fmt, group, g)
    w2, s2, d2 = _weight(ops, N, K, fmt, group, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    y = ops.q4_gemm_swiglu(x, w1, s1, w2, s2, N, K, group, fmt).float()
    a, b = ((x.float() @ d.t()).to(torch.bfloat16).float() for d in (d1, d2))
    ref = torch.nn.functional.silu(a).to(torch.bfloat16).float() * b
    # |silu'| <= 1.1, a place of a and one of b, and the roundings of silu and of the result
    tol = 2 ** -7 * (1.1 * (a * b).abs() + 2 * ref.abs()) + 2 ** -8 * ref.abs() + 2e-3
    assert float(((y - ref).abs() - tol).max()) <= 0.0


def test_rule_falls_back(ops):
    """K of no multiple of 128 stays with the tiles of gemm_q4f.hip, small weights of few rows and long prompts with the rings of
    gemm_q4r.hip; a split product reports its workspace."""
    lib = ops.load_library()
    assert lib.lga_q4f_workspace_bytes(64, 12288, 4096, 0) >= 4096 + 64 * 12288 * 4
    g = torch.Generator(device=DEV).manual_seed(5)
    for M, N, K, form in ((40, 264, 192, 0), (16, 512, 1024, 3), (257, 264, 256, 3)):
        assert ops.q4f_plan(M, N, K, 0, 1)[0] == form
        w, sc, wd = _weight(ops, N, K, 1, 64, g)
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        h = x.float() @ wd.t()
        y = ops.q4_gemm_fused(x, w, sc, N, K, 64, 1).float()
        assert float(((y - h).abs() - h.abs() * 2 ** -7).max()) <= 2e-3


@pytest.mark.parametrize("M,N,K", [(64, 512, 4160), (64, 4096, 4096)])
def test_captured(ops, M, N, K):
    """A split product in two graphs of one stream, the later one replayed first, with eager ones between: its workspace
    is the graph's own (64-value K: the tiles whose counters have to be clear; 128: the partial sums of this form)."""
    g = torch.Generator(device=DEV).manual_seed(K)
    w, sc, wd = _weight(ops, N, K, 1, 64, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    want = ops.q4_gemm_fused(x, w, sc, N, K, 64, 1).clone()
    stream, graphs, outs = torch.cuda.Stream(), [], []
    stream.wait_stream(torch.cuda.current_stream())
    for _ in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = ops.q4_gemm_fused(x, w, sc, N, K, 64, 1)
        graphs.append(graph)
        outs.append(out)
    for i in (1, 0, 0, 1, 1):
        graphs[i].replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[i], want)
        outs[i].zero_()
        assert torch.equal(ops.q4_gemm_fused(x, w, sc, N, K, 64, 1), want)


@pytest.mark.parametrize("M,N,K,fmt", [(64, 4096, 4096, 1), (64, 512, 4160, 1), (100, 4096, 11008, 2)])
def test_two_streams(ops, M, N, K, fmt):
    """Split products on two streams at once, each between others of its stream: the partial sums and counters of one are
    never the other's."""
    g = torch.Generator(device=DEV).manual_seed(K)
    work = []
    for _ in range(2):
        w, sc, wd = _weight(ops, N, K, fmt, 64, g)
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        work.append((x, w, sc, ops.q4_gemm_fused(x, w, sc, N, K, 64, fmt).clone()))
    assert ops.q4f_plan(M, N, K, 0, fmt)[1] > 0
    streams = [torch.cuda.Stream() for _ in work]
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(20):
        for i, (x, w, sc, _) in enumerate(work):
            with torch.cuda.stream(streams[i]):
                outs[i].append(ops.q4_gemm_fused(x, w, sc, N, K, 64, fmt))
    torch.cuda.synchronize()
    for got, (_, _, _, want) in zip(outs, work):
        assert all(torch.equal(y, want) for y in got)


def test_workspaces_are_given_back(ops):
    """Workspaces with counters: of many streams the last used are kept, and a stream that comes back is served anew."""
    M, N, K = 64, 512, 4160
    assert ops.q4f_plan(M, N, K, 0, 1)[2]
    g = torch.Generator(device=DEV).manual_seed(K)
    w, sc, wd = _weight(ops, N, K, 1, 64, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    want = ops.q4_gemm_fused(x, w, sc, N, K, 64, 1).clone()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(12)]
    for _ in range(2):
        for s in streams:
            with torch.cuda.stream(s):
                got = ops.q4_gemm_fused(x, w, sc, N, K, 64, 1)
            s.synchronize()
            assert torch.equal(got, want)
    assert len(ops._Q4F_WS) <= ops._Q4F_WS_MOST


@pytest.mark.parametrize("M,N,K", [(300, 12288, 11008), (200, 512, 4096)])
def test_a_workspace_of_the_older_tiles(ops, M, N, K, monkeypatch):
    """A caller whose workspace (none, or a smaller one) serves the older tiles has their result."""
    g = torch.Generator(device=DEV).manual_seed(K)
    w, _, wd = _weight(ops, N, K, 2, 64, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    form, need, _ = ops.q4f_plan(M, N, K, 0, 2)
    monkeypatch.setenv("LGA_Q4F_BN", "128")
    older = ops.q4f_plan(M, N, K, 0, 2)[1]
    monkeypatch.delenv("LGA_Q4F_BN")
    assert form == 2 and older < need
    ws = torch.zeros(older, dtype=torch.uint8, device=DEV)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    rc = ops.load_library().lga_q4_gemm_fused(x.data_ptr(), w.data_ptr(), None, None, None, y.data_ptr(), M, N, K, 64, 2,
                                              ws.data_ptr() if older else None, older, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    h = x.float() @ wd.t()
    assert float(((y.float() - h).abs() - h.abs() * 2 ** -7).max()) <= 2e-3


@pytest.mark.parametrize("M,N,K,fmt,swiglu", [(702, 4096, 11008, 0, False), (300, 4096, 11008, 1, False), (16, 4096, 4096, 0, False),
                                              (129, 1536, 12800, 1, True), (64, 8200, 4096, 0, False)])
def test_bits_are_those_of_the_sizes(ops, M, N, K, fmt, swiglu):
    """A product gives the same bits before and after larger ones of its stream, captured, and with a workspace larger than its own."""
    group = 128 if fmt == 0 else 64
    g = torch.Generator(device=DEV).manual_seed(M)
    (w, sc, _), (w2, sc2, _) = (_weight(ops, N, K, fmt, group, g) for _ in range(2))
    x = torch.randn(2048, K, generator=g, device=DEV).to(torch.bfloat16)

    def product(rows):
        if swiglu:
            return ops.q4_gemm_swiglu(x[:rows], w, sc, w2, sc2, N, K, group, fmt)
        return ops.q4_gemm_fused(x[:rows], w, sc, N, K, group, fmt)

    form, need, _ = ops.q4f_plan(M, N, K, swiglu, fmt)
    assert form == 3 and need > 0
    first = product(M).clone()
    product(1000), product(2048)
    assert torch.equal(product(M), first)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=stream):
        out = product(M)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first) and torch.equal(product(M), first)
    ws, y = torch.empty(4 * need, dtype=torch.uint8, device=DEV), torch.empty_like(first)
    stream = torch.cuda.current_stream().cuda_stream
    if swiglu:
        rc = ops.load_library().lga_q4_gemm_swiglu(x.data_ptr(), w.data_ptr(), sc.data_ptr(), w2.data_ptr(), sc2.data_ptr(), y.data_ptr(),
                                                   M, N, K, group, fmt, ws.data_ptr(), ws.numel(), stream)
    else:
        rc = ops.load_library().lga_q4_gemm_fused(x.data_ptr(), w.data_ptr(), sc.data_ptr(), None, None, y.data_ptr(), M, N, K, group,
                                                  fmt, ws.data_ptr(), ws.numel(), stream)
    assert rc == 0 and torch.equal(y, first)


def test_two_threads_on_one_stream(ops):
    """Products of two threads that share a stream: the partial sums of one never stand between the launches of the other."""
    import threading

    g = torch.Generator(device=DEV).manual_seed(3)
    work = []
    for M, N, K in ((300, 4096, 11008), (16, 4096, 4096)):
        w, sc, _ = _weight(ops, N, K, 0, 128, g)
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
        form, need, counters = ops.q4f_plan(M, N, K, 0, 0)
        assert form == 3 and need > 0 and not counters
        work.append(((x, w, sc, N, K, 128, 0), ops.q4_gemm_fused(x, w, sc, N, K, 128, 0).clone()))
    torch.cuda.synchronize()
    outs, errors = [[], []], []

    def many(i):
        try:
            for _ in range(60):
                outs[i].append(ops.q4_gemm_fused(*work[i][0]))
        except Exception as e:  # pragma: no cover
            errors.append(e)

    threads = [threading.Thread(target=many, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for got, (_, want) in zip(outs, work):
        assert len(got) == 60 and all(torch.equal(y, want) for y in got)


@pytest.mark.parametrize("M,N,K", [(16, 4096, 4096), (93, 512, 1024), (300, 1032, 1408)])
@pytest.mark.parametrize("fmt,group", [(0, 128), (1, 64)])
@pytest.mark.parametrize("given", ["planned", "none", "small"])
def test_scales_off_eight_bytes_and_small_workspaces(ops, M, N, K, fmt, group, given):
    """Scales that the rings' form cannot load, and workspaces that do not hold its sums (those it asks for are not cleared): the
    product is made in another way. Tolerance as in test_long_prompts."""
    g = torch.Generator(device=DEV).manual_seed(M)
    w, sc, wd = _weight(ops, N, K, fmt, group, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    h = x.float() @ wd.t()
    form, need, _ = ops.q4f_plan(M, N, K, 0, fmt)
    assert form == 3
    size = {"planned": need, "none": 0, "small": 8192}[given]
    ws = torch.full((max(size, 16),), 255, dtype=torch.uint8, device=DEV)
    four = 4 // sc.element_size()  # scales that start on 4 bytes
    off = torch.empty(sc.numel() + four, dtype=sc.dtype, device=DEV)[four:].view(sc.shape).copy_(sc)
    for s in (sc, off):
        y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        rc = ops.load_library().lga_q4_gemm_fused(x.data_ptr(), w.data_ptr(), s.data_ptr(), None, None, y.data_ptr(), M, N, K, group, fmt,
                                                  ws.data_ptr() if size else None, size, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        assert float(((y.float() - h).abs() - h.abs() * 2 ** -8).max()) <= 2e-4


# the tiles of long prompts: 128, 192 and 256 rows a tile, one row past and one short of whole tiles, columns past the last whole
# tile, one pair of steps and many, ranges of K of unequal length
@pytest.mark.parametrize("fmt,group", [(0, 64), (0, 128), (1, 64), (1, 256), (3, 128)])
@pytest.mark.parametrize("M,N,K", [(129, 136, 256), (257, 264, 512), (257, 4104, 1280), (385, 1032, 768), (511, 8200, 256),
                                   (577, 520, 5632), (1025, 776, 1024)])
@pytest.mark.parametrize("epi", ["plain", "bias+residual", "swiglu"])
def test_long_prompts(ops, fmt, group, M, N, K, epi):
    """Against fp32 products of the dequantized weights: the operands are bf16 and their sums fp32, so one rounding to bf16
    (2^-9 of the value) and K roundings of partial sums, 2e-4 at the largest K here, stand between the two."""
    g = torch.Generator(device=DEV).manual_seed(K + M)
    w, sc, wd = _weight(ops, N, K, fmt, group, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    h = x.float() @ wd.t()
    if epi == "swiglu":
        w2, sc2, wd2 = _weight(ops, N, K, fmt, group, g)
        a, b = h.to(torch.bfloat16).float(), (x.float() @ wd2.t()).to(torch.bfloat16).float()
        ref = (a * torch.sigmoid(a)).to(torch.bfloat16).float() * b
        y = ops.q4_gemm_swiglu(x, w, sc, w2, sc2, N, K, group, fmt).float()
        # each factor may round to the neighbouring bf16 number
        tol = 2 ** -7 * (1.1 * (a * b).abs() + 2 * ref.abs()) + 2 ** -8 * ref.abs() + 2e-3
        assert float(((y - ref).abs() - tol).max()) <= 0.0
        return
    if epi == "plain":
        y = ops.q4_gemm_fused(x, w, sc, N, K, group, fmt).float()
        assert float(((y - h).abs() - h.abs() * 2 ** -8).max()) <= 2e-4
        return
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    res = torch.randn(M, N, generator=g, device=DEV).to(torch.bfloat16)
    h = h + bias.float()
    ref = h.to(torch.bfloat16).float() + res.float()
    y = ops.q4_gemm_fused(x, w, sc, N, K, group, fmt, bias=bias, residual=res).float()
    assert float(((y - ref).abs() - (ref.abs() + h.abs()) * 2 ** -7).max()) <= 2e-3


# 32, 64 and 96 rows a tile, whose two groups of waves share a range of K: ranges of an even and an odd number of pairs of
# steps, as few as two; a row short of, at and past whole tiles; columns past the last whole tile
@pytest.mark.parametrize("fmt,group", [(0, 64), (0, 128), (1, 64), (3, 128)])
@pytest.mark.parametrize("M,N,K", [(2, 136, 256), (31, 264, 384), (32, 1032, 1408), (33, 8200, 256), (64, 8712, 7808), (65, 264, 896),
                                   (96, 1032, 384), (97, 136, 2176), (128, 264, 128)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_short_prompts(ops, fmt, group, M, N, K, swiglu):
    """As test_long_prompts: one rounding to bf16 and K roundings of partial sums between the product and its fp32 reference."""
    g = torch.Generator(device=DEV).manual_seed(K + M)
    w, sc, wd = _weight(ops, N, K, fmt, group, g)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    h = x.float() @ wd.t()
    if not swiglu:
        y = ops.q4_gemm_fused(x, w, sc, N, K, group, fmt).float()
        assert float(((y - h).abs() - h.abs() * 2 ** -8).max()) <= 2e-4
        return
    w2, sc2, wd2 = _weight(ops, N, K, fmt, group, g)
    a, b = h.to(torch.bfloat16).float(), (x.float() @ wd2.t()).to(torch.bfloat16).float()
    ref = (a * torch.sigmoid(a)).to(torch.bfloat16).float() * b
    y = ops.q4_gemm_swiglu(x, w, sc, w2, sc2, N, K, group, fmt).float()
    tol = 2 ** -7 * (1.1 * (a * b).abs() + 2 * ref.abs()) + 2 ** -8 * ref.abs() + 2e-3
    assert float(((y - ref).abs() - tol).max()) <= 0.0


@pytest.mark.parametrize("fmt", [0, 2])
def test_gated_unit_of_every_bf16_number(ops, fmt):
    """The unit of unsplit SwiGLU products is ops.swiglu's, for all normal bf16 gates (identity weights, gates times 1), infinities
    and NaN among them; and that unit is within four roundings of 2^-24 of float64, or where expf overflows 4e-37, of bf16's rounding."""
    M, N, K = 512, 128, 256
    v = torch.arange(65536, device=DEV, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).view(M, N)
    v = torch.where(torch.isfinite(v) & (v.abs() >= 2.0 ** -126), v, torch.ones_like(v))  # (sums flush denormal products)
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    x[:, :N], x[:, N] = v, 1.0
    one = torch.zeros(2, N, K, device=DEV)  # the gate's matrix and the up's
    one[0, :, :N], one[1, :, N] = torch.eye(N, device=DEV), 1.0
    every = torch.zeros(N, K, device=DEV)
    every[:, 0] = 1.0

    def product(x, a, b):
        if fmt == 2:
            return ops.q4_gemm_swiglu(x, a.to(torch.bfloat16), None, b.to(torch.bfloat16), None, N, K, 64, 2)
        (qa, qb), sc = (((8 + m[:, ::2]) + 16 * (8 + m[:, 1::2])).to(torch.uint8).contiguous() for m in (a, b)), \
            torch.ones(N, K // 128, dtype=torch.bfloat16, device=DEV)
        return ops.q4_gemm_swiglu(x, qa, sc, qb, sc, N, K, 128, 0)

    assert ops.q4f_plan(x.shape[0], N, K, 1, fmt)[1] == 0  # one launch: the unit stands in the product's
    y = product(x, one[0], one[1])
    unit = ops.swiglu(v.contiguous(), torch.ones_like(v))
    assert torch.equal(y, unit)
    exact = v.double() / (1 + torch.exp(-v.double()))
    place = 2.0 ** (torch.frexp(exact.abs().clamp_min(2.0 ** -126))[1].double() - 8)  # of bf16 at that size
    assert float(((y.double() - exact).abs() - 0.5 * place - 4 * 2 ** -24 * exact.abs()).max()) <= 4e-37
    for special in (float("inf"), float("-inf"), float("nan")):  # (an infinite up: 0 times one is NaN in both products)
        x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
        x[:, 0] = special
        y = product(x, every, every)
        both = torch.full((M, N), special, dtype=torch.bfloat16, device=DEV)
        unit = ops.swiglu(both, both)
        assert torch.equal(torch.nan_to_num(y.float(), 7.0), torch.nan_to_num(unit.float(), 7.0))
        assert bool(torch.isinf(y).all()) == (special == float("inf"))
