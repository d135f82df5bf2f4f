"""One row's output products with the residual adds (lga_f32_linears_sum) at the lengths where the second row lies in LDS or not and
where a workgroup ends, joined ranges of keys among them, against float64: K products of partial sums around 1, each addition half a
unit of 2^-24."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K1,K2", [(5, 4, 4), (768, 768, 3072), (10, 832, 3072), (33, 1024, 3076), (7, 1028, 4096), (9, 64, 8192), (6, 256, 8196), (130, 8192, 8192),
                                     (35, 2048, 4096), (35, 2052, 4100), (3, 4096, 8192), (9, 1024, 4100), (10, 2052, 4096), (2, 4, 8)])
@pytest.mark.parametrize("parts,hs", [(1, 4), (2, 4), (8, 64)])
def test_two_products_of_a_row(N, K1, K2, parts, hs):
    from lit_gpt import ops

    if parts > 1 and (K1 % hs or K1 // hs > 256):
        pytest.skip("whole heads, up to 256")
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(N + K1 + K2)
    rand = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    w1, w2 = rand(N, K1) * K1 ** -0.5, rand(N, K2) * K2 ** -0.5
    b1, b2, res, x2, x1 = rand(N), rand(N), rand(1, N), rand(1, K2), rand(parts, K1)
    ml, joined = None, x1.double()
    if parts > 1:
        H = K1 // hs
        ml = torch.stack([rand(parts, H), torch.rand(parts, H, generator=g, device=dev) + 0.5], -1).contiguous()
        ml[-1, 0, 1] = -1.0  # (an empty range)
        ml[-1, 0, 0] = -float("inf")
        wt = torch.exp(ml[..., 0].double() - ml[..., 0].double().amax(0)) * (ml[..., 1] >= 0)
        joined = ((wt[..., None] * x1.double().view(parts, H, hs)).sum(0) / (wt * ml[..., 1].double()).sum(0)[:, None]).view(1, K1)
    y = torch.full((1, N + 3), 7.0, device=dev)
    lib = ops.load_library()
    ops._check(lib.lga_f32_linears_sum(x1.data_ptr(), None if ml is None else ml.data_ptr(), parts, hs, w1.data_ptr(), b1.data_ptr(), K1,
                                       x2.data_ptr(), w2.data_ptr(), b2.data_ptr(), K2, res.data_ptr(), y.data_ptr(), N, ops._stream()))
    want = joined @ w1.double().T + b1.double() + x2.double() @ w2.double().T + b2.double() + res.double()
    size = 4 + float(joined.abs().max())
    assert ((y[:, :N].double() - want).abs() <= (K1 + K2) ** 0.5 * 2.0 ** -24 * 4 * size).all() and (y[:, N:] == 7).all()
