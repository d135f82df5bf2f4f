"""fp32 products of several rows on the matrix cores (lga_f32_linear at K % 256 == 0): the bits of one row at a time at the edges of
both tile sizes, and values that are not ordinary."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def rows(x, w, **kw):
    from lit_gpt import ops

    one = lambda v, i: v[i: i + 1] if torch.is_tensor(v) and v.dim() == 2 else v  # noqa: E731
    return torch.cat([ops.f32_linear(x[i: i + 1], w, **{k: one(v, i) for k, v in kw.items()}) for i in range(x.shape[0])])


# (32 x 32 tiles: 17 x 4097, 300 x 768 and the last four, each of these with a last row alone; 16 x 16: the others)
@pytest.mark.parametrize("M,N,K", [(2, 4500, 256), (16, 577, 768), (17, 4097, 256), (9, 1000, 512), (31, 300, 3072), (33, 8191, 256), (97, 2049, 512),
                                   (128, 2304, 768), (300, 768, 1024), (15, 601, 2048), (33, 3001, 768), (65, 1999, 768), (97, 1801, 1024),
                                   (129, 1001, 512)])
def test_rows_to_the_bit(M, N, K):
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, w, b, r, r2 = (torch.randn(m, generator=g, device=dev) for m in ((M, K), (N, K), (N,), (M, N), (M, N)))
    for kw in (dict(), dict(bias=b, gelu="tanh", residual=r, residual2=r2), dict(bias=b, gelu="none")):
        assert torch.equal(ops.f32_linear(x, w, **kw), rows(x, w, **kw))
    got, want = ops.f32_linear(x, w).double(), x.double() @ w.double().T
    bound = (K / 256 + 10) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)  # a chain of K / 256 sums and a tree of ten levels
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("M", [40, 200])
def test_values_that_are_not_ordinary(M):
    """Denormal products and sums, infinities and NaN: in their own rows and columns, as one row alone has them."""
    from lit_gpt import ops

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M)
    x, w = (torch.randn(m, generator=g, device=dev) for m in ((M, 768), (2304, 768)))
    tiny = ops.f32_linear(x * 3e-22, w * 3e-22)
    assert torch.equal(tiny, rows(x * 3e-22, w * 3e-22)) and 0 < tiny.abs().max() < 1e-38
    x[3, 5], x[M - 1, 7], w[9, 700], w[2303, 0] = float("inf"), float("nan"), float("-inf"), 3e38
    got, want = ops.f32_linear(x, w), rows(x, w)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(0.0, 1.0, -1.0), want.nan_to_num(0.0, 1.0, -1.0))
    assert got[M - 1].isnan().all() and got[4].isfinite().sum() >= 2302
