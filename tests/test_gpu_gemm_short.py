"""The rows past the last whole tile, in tiles of their own (csrc/gemm_tiles.h), against float64: every form and every number of
fragments left that the rules choose in the plain products, those with activations, the GPT models' and the gated ones (the form is
asked for and held to); beside these ragged rows and groups at sizes where smaller forms are taken.

Every sum has K products of bf16 values, exact in fp32, added in fp32: with |a w| ~ K^-1/2 the error of a result is at
most about K additions of half a unit in the last place of partial sums around 1, K 2^-25.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 2e-5  # (of the shorter K of the first two tests, with |a w| of theirs)


def operands(M, N, K, dev):
    g = torch.Generator(device=dev).manual_seed(7 * M + N)
    a = torch.randn(M, K, generator=g, device=dev).bfloat16()
    return a, (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()


@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 97, 128, 129, 191, 193, 255])
@pytest.mark.parametrize("whole,N,K", [(0, 6200, 128), (1, 12300, 192), (2, 22016, 64), (9, 2100, 256), (8, 8200, 64), (5, 300, 1024)])
def test_rows_past_whole_tiles(rows, whole, N, K):
    from lit_gpt import ops, seq_ops

    dev = torch.device("cuda", 0)
    M = whole * 256 + rows
    if M < 9:
        pytest.skip("such products have no tiles")
    a, w = operands(M, N, K, dev)
    want = a.double() @ w.double().T
    y = torch.full((M + 1, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N)
    assert (y[:M].double() - want).abs().max() < TOL and y[M:].isnan().all()
    n = N // 8 * 8
    y = ops.q4_gemm_fused(a, w[:n], None, n, K, 0, 2)  # the GPT models', rows as the tile's other operand: one rounding to bf16
    assert ((y.double() - want[:, :n]).abs() <= 2.0 ** -8 * want[:, :n].abs() + TOL).all()
    n = N // 8 * 4  # gated units: two roundings of 2^-9 and a unit's few of 2^-24
    gate, up = want[:, :n], want[:, n:2 * n]
    unit = gate * torch.sigmoid(gate) * up
    y = torch.cat([seq_ops.linear_glu(a, w[:2 * n], M=M, n=n, up=n, act=seq_ops.ACT_SILU), torch.full((1, n), 3.0, device=dev, dtype=torch.bfloat16)])
    assert ((y[:M].double() - unit).abs() <= 2.0 ** -8 * unit.abs() + 4 * TOL * (1 + gate.abs() + up.abs())).all()


@pytest.mark.parametrize("sizes", [[193] * 16, [250] * 16, [256] * 3 + [1] * 5, [64] * 70, [0, 513, 0, 129, 64, 1, 320], [33] * 20 + [700]])
@pytest.mark.parametrize("N,K", [(300, 128), (4100, 64)])
def test_groups(sizes, N, K):
    from lit_gpt import seq_ops

    dev = torch.device("cuda", 0)
    E, M = len(sizes), sum(sizes)
    a, w = operands(M, E * N, K, dev)
    w = w.view(E, N, K)
    z = torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(dev)
    y = torch.full((M + 1, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, batch=E, stride_w=N * K, z_start=z)
    n = N // 8 * 4
    unit = seq_ops.linear_glu(a, w, M=M, n=n, up=n, act=seq_ops.ACT_SILU, z_start=z)
    assert y[M:].isnan().all()
    for e in range(E):
        lo, hi = int(z[e]), int(z[e + 1])
        want = a[lo:hi].double() @ w[e].double().T
        assert ((y[lo:hi].double() - want).abs() < TOL).all()
        gate, up = want[:, :n], want[:, n:2 * n]
        made = gate * torch.sigmoid(gate) * up
        assert ((unit[lo:hi].double() - made).abs() <= 2.0 ** -8 * made.abs() + 4 * TOL * (1 + gate.abs() + up.abs())).all()


# form, fragments left, M, N, K: sizes that the rules send there, of nine steps and more, past the deepest ring; each form of one
# fragment a time with whole tiles too
PLAIN = [(0, 1, 769, 14039, 576), (0, 2, 577, 19759, 576), (0, 3, 641, 16639, 576), (1, 1, 769, 13259, 576), (1, 2, 2369, 3639, 1088),
         (1, 3, 385, 21839, 576), (2, 0, 1280, 6499, 1088), (2, 1, 1537, 4939, 1088), (2, 2, 2369, 2599, 4160), (2, 3, 129, 17679, 576),
         (3, 1, 257, 16379, 576), (4, 1, 129, 16639, 576), (5, 1, 1153, 6499, 576), (6, 0, 1152, 1819, 576), (6, 1, 63, 259, 576),
         (7, 0, 128, 259, 576), (7, 1, 31, 259, 576), (8, 1, 385, 16639, 576), (8, 2, 257, 21839, 576)]
ACTS = [(2, 0, 1280, 6499, 1088), (2, 1, 513, 13779, 576), (2, 2, 833, 21059, 576), (2, 3, 129, 17679, 576), (3, 1, 257, 16379, 576),
        (4, 1, 129, 16639, 576), (5, 1, 1153, 6499, 576), (6, 1, 63, 259, 576), (7, 1, 31, 259, 576)]
RANGES = [(2, 3, 129, 5459, 4160), (4, 1, 257, 3639, 4160), (6, 0, 1152, 519, 4160), (6, 1, 63, 259, 1088), (7, 0, 128, 259, 1088),
          (7, 1, 31, 259, 1088), (8, 2, 65, 16639, 4160)]
GPT = [(0, 1, 769, 14040, 576), (0, 2, 577, 16640, 576), (0, 3, 641, 16640, 576), (1, 1, 769, 9360, 576), (1, 2, 257, 21840, 576),
       (2, 0, 640, 8584, 704), (2, 1, 257, 16640, 704), (3, 1, 257, 16640, 576), (3, 2, 577, 8320, 576), (3, 3, 129, 16640, 576),
       (4, 0, 576, 6760, 576), (4, 1, 63, 16640, 576), (4, 2, 65, 16640, 576), (5, 1, 257, 16904, 576), (6, 0, 384, 5464, 576),
       (7, 0, 128, 264, 576), (8, 1, 2305, 3384, 576), (8, 2, 577, 13264, 576), (8, 3, 385, 16640, 576), (1, 2, 65, 16640, 4160),
       (2, 1, 63, 16640, 4160), (3, 3, 129, 3384, 4160), (4, 1, 63, 4160, 4160), (4, 2, 65, 4160, 4160), (6, 0, 384, 1824, 4160),
       (7, 0, 128, 264, 1088)]  # (the last seven in ranges of K)
GPT_GATED = [(0, 1, 257, 16496, 576), (0, 2, 577, 8312, 576), (0, 3, 385, 10952, 576), (1, 1, 385, 8312, 576), (1, 2, 65, 22304, 576),
             (2, 0, 128, 16496, 576), (2, 1, 63, 16496, 576), (3, 1, 257, 8312, 576), (3, 2, 577, 4224, 576), (3, 3, 129, 8312, 576),
             (4, 0, 576, 3296, 576), (4, 1, 63, 8312, 576), (4, 2, 65, 8312, 576), (5, 1, 63, 23888, 576), (6, 0, 1152, 920, 576),
             (7, 0, 128, 264, 576), (1, 2, 65, 8312, 4160), (2, 1, 63, 8312, 4160), (3, 3, 129, 1712, 4160), (4, 1, 63, 2112, 4160),
             (4, 2, 65, 2112, 4160), (6, 0, 896, 392, 4160), (7, 0, 128, 264, 1088)]  # (the last seven in ranges of K)
GATED = [(0, 1, 257, 16492, 576), (0, 2, 577, 8308, 576), (0, 3, 385, 10948, 576), (1, 1, 385, 8308, 576), (1, 2, 65, 22300, 576),
         (2, 0, 128, 16492, 576), (2, 1, 63, 16492, 576), (3, 1, 257, 8308, 576), (3, 2, 577, 4216, 576), (3, 3, 129, 8308, 576),
         (4, 0, 576, 3292, 576), (4, 1, 63, 8308, 576), (4, 2, 65, 8308, 576), (5, 1, 63, 23884, 576), (6, 0, 1152, 916, 576),
         (7, 0, 128, 256, 576)]


@pytest.mark.parametrize("form,left,M,N,K", PLAIN)
def test_plain_forms(form, left, M, N, K):
    """fp32 with a bias, bf16, and sums, with a row and columns past the product that have to stay."""
    from lit_gpt import seq_ops

    dev, tol, ld = torch.device("cuda", 0), K * 2.0 ** -25, N + 5
    assert seq_ops.load_library().lgs_linear_form(M, N, K, 1, 0, 1, 0, 0) == form
    a, w = operands(M, N, K, dev)
    b = torch.randn(N, device=dev)
    want = a.double() @ w.double().T + b.double()
    old = torch.randn(M + 1, ld, device=dev)
    for kind in ("fp32", "bf16", "sums"):
        y = old.bfloat16() if kind == "bf16" else old.clone()
        seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=ld, bias=b, accumulate=kind == "sums", ksplit=1)
        assert torch.equal(y[:, N:], old[:, N:].to(y.dtype)) and torch.equal(y[M], old[M].to(y.dtype)), kind
        made = want + old[:M, :N].double() if kind == "sums" else want  # (two roundings more, of values of up to about 8)
        bound = tol + 2.0 ** -20 + (2.0 ** -8 * want.abs() if kind == "bf16" else 0.0)
        assert ((y[:M, :N].double() - made).abs() <= bound).all(), kind


@pytest.mark.parametrize("form,left,M,N,K", ACTS)
@pytest.mark.parametrize("act", [1, 3])
def test_forms_with_activations(form, left, M, N, K, act):
    from lit_gpt import seq_ops

    dev, tol = torch.device("cuda", 0), K * 2.0 ** -25
    assert seq_ops.load_library().lgs_linear_form(M, N, K, 1, 0, 1, act, 0) == form
    a, w = operands(M, N, K, dev)
    z = a.double() @ w.double().T
    want = z.clamp_min(0) ** 2 if act == 1 else z * torch.sigmoid(z)
    old = torch.randn(M + 1, N, device=dev)
    for kind in ("fp32", "bf16", "sums"):
        y = old.bfloat16() if kind == "bf16" else old.clone()
        seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, act=act, accumulate=kind == "sums", ksplit=1)
        assert torch.equal(y[M], old[M].to(y.dtype)), kind
        made = want + old[:M].double() if kind == "sums" else want
        # a sum's error through slopes of up to 2 |z| + 1, then some roundings of 2^-24 of values of up to z^2 + 8
        bound = (tol + 16 * 2.0 ** -24) * (2 * z.abs() + 1) + 16 * 2.0 ** -24 * want.abs() + (2.0 ** -8 * want.abs() if kind == "bf16" else 0.0)
        assert ((y[:M].double() - made).abs() <= bound + 2.0 ** -20 * (kind == "sums")).all(), kind


@pytest.mark.parametrize("form,left,M,N,K", RANGES)
def test_forms_in_ranges(form, left, M, N, K):
    from lit_gpt import seq_ops

    dev, lib = torch.device("cuda", 0), seq_ops.load_library()
    ranges = lib.lgs_linear_ksplit(M, N, K)
    assert ranges > 1 and lib.lgs_linear_form(M, N, K, 1, 0, ranges, 0, 0) == form
    a, w = operands(M, N, K, dev)
    y = torch.full((M + 1, N), float("nan"), device=dev)
    seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N)
    assert (y[:M].double() - a.double() @ w.double().T).abs().max() < K * 2.0 ** -25 and y[M:].isnan().all()


@pytest.mark.parametrize("form,left,M,N,K", GPT)
def test_gpt_forms(form, left, M, N, K):
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    chosen = ops.load_library().lga_bf16_gemm_form(M, N, K, 0)
    assert chosen & 255 == form and (chosen >> 8 > 1) == ((form, left, M, N, K) in GPT[-7:])
    a, w = operands(M, N, K, dev)
    want = a.double() @ w.double().T
    out = torch.full((M + 1, N), 3.0, device=dev, dtype=torch.bfloat16)
    ops.q4_gemm_fused(a, w, None, N, K, 0, 2, out=out[:M])
    assert ((out[:M].double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -25).all() and (out[M] == 3.0).all()


@pytest.mark.parametrize("form,left,M,N,K", GPT_GATED)
def test_gpt_gated_forms(form, left, M, N, K):
    """Gate and up rounded to bf16, the gate's unit too, and the product: 2^-8 at most each, the first through a slope of at most 1.1."""
    from lit_gpt import ops

    dev, tol = torch.device("cuda", 0), K * 2.0 ** -25
    chosen = ops.load_library().lga_bf16_gemm_form(M, N, K, 1)
    assert chosen & 255 == form and (chosen >> 8 > 1) == ((form, left, M, N, K) in GPT_GATED[-7:])
    a, w = operands(M, 2 * N, K, dev)
    gate, up = (a.double() @ w.double().T).split(N, dim=1)
    want = gate * torch.sigmoid(gate) * up
    out = torch.full((M + 1, N), 3.0, device=dev, dtype=torch.bfloat16)
    ops.q4_gemm_swiglu(a, w[:N], None, w[N:], None, N, K, 0, 2, out=out[:M])
    bound = 1.02 * 2.0 ** -8 * (1.1 * (gate * up).abs() + 3 * want.abs()) + 4 * tol * (1 + gate.abs() + up.abs())
    assert ((out[:M].double() - want).abs() <= bound).all() and (out[M] == 3.0).all()


@pytest.mark.parametrize("form,left,M,N,K", GATED)
def test_gated_forms(form, left, M, N, K):
    from lit_gpt import seq_ops

    dev, tol = torch.device("cuda", 0), K * 2.0 ** -25
    assert seq_ops.load_library().lgs_linear_form(M, N, K, 1, 0, 1, 0, 1) == form
    a, w = operands(M, 2 * N, K, dev)
    gate, up = (a.double() @ w.double().T).split(N, dim=1)
    for act, want in ((seq_ops.ACT_SILU, gate * torch.sigmoid(gate) * up), (seq_ops.ACT_RELU2, gate.clamp_min(0) ** 2 * up)):
        y = seq_ops.linear_glu(a, w, M=M, n=N, up=N, act=act)
        bound = 2.0 ** -8 * want.abs() + 4 * tol * (1 + gate.abs()) * (1 + gate.abs() + up.abs())
        assert ((y.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("gated,form,sizes,N,K", [
    (0, 0, [257, 65, 129, 193, 0, 156], 10244, 576), (0, 8, [1, 65, 129, 0, 193, 100, 0, 112], 7428, 576),
    (1, 0, [257, 65, 129, 193, 0, 255, 256, 64, 1, 320, 400, 0, 0, 0, 0, 160], 1796, 576), (1, 1, [65, 129, 6], 10756, 576)])
def test_groups_of_large_forms(gated, form, sizes, N, K):
    from lit_gpt import seq_ops

    dev, tol, E, M = torch.device("cuda", 0), K * 2.0 ** -25, len(sizes), sum(sizes)
    assert seq_ops.load_library().lgs_linear_form(M, N, K, E, 1, 1, 0, gated) == form
    rows = 2 * N if gated else N
    a, w = operands(M, E * rows, K, dev)
    w = w.view(E, rows, K)
    z = torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(dev)
    if gated:
        y = seq_ops.linear_glu(a, w, M=M, n=N, up=N, act=seq_ops.ACT_SILU, z_start=z)
    else:
        y = torch.full((M, N), float("nan"), device=dev)
        seq_ops.linear(a, w, M=M, N=N, K=K, y=y, lda=K, ldy=N, batch=E, stride_w=N * K, z_start=z)
    lo = 0
    for e, size in enumerate(sizes):
        want, got = a[lo:lo + size].double() @ w[e].double().T, y[lo:lo + size].double()
        lo += size
        if gated:
            gate, up = want.split(N, dim=1)
            want = gate * torch.sigmoid(gate) * up
            assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 4 * tol * (1 + gate.abs() + up.abs())).all()
        else:
            assert ((got - want).abs() < tol).all()
