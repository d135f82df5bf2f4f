"""Layer norms of the layered models against float64 at the edges of what a thread holds (256, 1024, 2048, 4096 columns) and of
what is loaded ahead (8192): alone, joining a residual, with its bf16 copy. Tolerance: fp32 sums of up to 2^7 terms a thread in a
tree, 2^-19 of unit rows; a residual of the same size adds its own rounding."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1024, 1025, 2048, 2049, 4096, 5000, 8192, 8193, 20000])
@pytest.mark.parametrize("rows", [1, 7])
def test_rows(n, rows):
    from lit_gpt import seq_ops

    g = torch.Generator(device=DEV).manual_seed(n)
    y, w, b, x = (torch.randn(*s, generator=g, device=DEV) for s in ((rows, n), (n,), (n,), (rows, n)))
    norm = torch.nn.functional.layer_norm(y.double(), (n,), eps=1e-5)
    got = seq_ops.layernorm(y, w, b, eps=1e-5, mult=0.5)
    assert float((got.double() - 0.5 * (norm * w.double() + b.double())).abs().max()) < 2 ** -19 * 8
    old = x.clone()
    got, got16 = seq_ops.layernorm(y, w, None, eps=1e-5, x=x, mult=0.3, bf16_copy=True)
    assert got.data_ptr() == x.data_ptr() and torch.equal(got16, got.bfloat16())
    assert float((got.double() - (old.double() + 0.3 * norm * w.double())).abs().max()) < 2 ** -19 * 8
