"""Forward hooks on modules that a fused form computes without calling them: they run in steps of every size, and the results
are the fused form's to the bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def layered(design, width=64, ff=96):
    from lit_gpt.config import LayeredConfig
    from lit_gpt.layered import LayeredGPT

    mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
    if design == "Rigulorn":
        layer = {"type": "mamba2", "mixer": {"heads": 4, "vdim": 16, "state": 16, "groups": 2, "norm_groups": 2, "conv": 4}}
        more = {"embedding": {"scale": 1.0}, "streams": 2}
    else:
        layer, more = {"type": "mingru", "mixer": {"width": width}}, {}
    config = LayeredConfig.from_dict(dict(architecture=design, vocab=50, width=width, norm={"eps": 1e-5}, layers=[dict(layer, mlp=mlp)],
                                          **more))
    return LayeredGPT(config, LayeredGPT.random_weights(config, seed=3), device=DEV, dtype=torch.bfloat16)


@pytest.mark.parametrize("design", ["Rigulorn", "Fazolorn"])
@pytest.mark.parametrize("kind", ["forward", "pre", "global"])
def test_gated_feed_forward(design, kind):
    from torch.nn.modules.module import register_module_forward_hook

    from lit_gpt.mixers import GatedFeedForward, StepBatch

    m = layered(design)
    ff = [x for x in m.modules() if isinstance(x, GatedFeedForward)]
    assert len(ff) == 1
    ids = torch.randint(0, 50, (40,), generator=torch.Generator().manual_seed(2)).tolist()
    m.set_kv_cache(1, 64)
    calls = []
    with torch.inference_mode():
        for n in (40, 5):
            step = StepBatch.build([(0, 0, ids[:n])], DEV)
            want = m.logits(m.forward_step(step)).clone()
            calls.clear()
            note = lambda mod, *_: calls.append(mod) if mod is ff[0] else None  # noqa: E731
            handle = {"forward": ff[0].register_forward_hook, "pre": ff[0].register_forward_pre_hook,
                      "global": register_module_forward_hook}[kind](note)
            try:
                got = m.logits(m.forward_step(step))
            finally:
                handle.remove()
            assert calls == [ff[0]], n
            assert torch.equal(got, want)


@pytest.mark.parametrize("design", ["Rigulorn", "Fazolorn"])
@pytest.mark.parametrize("width,ff", [(1024, 200), (1024, 256), (1024, 264), (512, 200)])
def test_one_row_of_a_gated_feed_forward(design, width, ff):
    """One token: the unit in its input product's launch and apart give the same bits, on both sides of the line below which
    the product's waves share its columns."""
    from lit_gpt import seq_ops
    from lit_gpt.mixers import GatedFeedForward, StepBatch

    m = layered(design, width, ff)
    ff_of = [x for x in m.modules() if isinstance(x, GatedFeedForward)]
    w = torch.empty(2 * (ff + -ff % 8), width, dtype=torch.bfloat16, device=DEV)
    assert seq_ops.glu_row_fits(torch.zeros(1, width, device=DEV), w) == (width < 1024 or ff > 256)
    m.set_kv_cache(1, 64)
    with torch.inference_mode():
        step = StepBatch.build([(0, 0, [7])], DEV)
        want = m.logits(m.forward_step(step)).clone()
        handle = ff_of[0].register_forward_hook(lambda *_: None)
        try:
            assert torch.equal(m.logits(m.forward_step(step)), want)
        finally:
            handle.remove()


def test_parallel_block_in_fp32():
    from torch.nn.modules.module import register_module_forward_hook

    from generate.base import build_model
    from lit_gpt import Config

    m = build_model(Config.from_name("pythia-160m", n_layer=1), quantize=None, device=DEV, seed=1, max_seq_length=64,
                    dtype=torch.float32)
    block = m.transformer.h[0]
    idx = torch.arange(12, device=DEV)[None]
    calls = []
    with torch.inference_mode():
        want = m(idx, torch.arange(12, device=DEV)).clone()
        handle = register_module_forward_hook(lambda mod, *_: calls.append(mod))
        try:
            got = m(idx, torch.arange(12, device=DEV))
        finally:
            handle.remove()
    assert all(x in calls for x in (block.mlp, block.norm_1, block.norm_2, block.attn))
    assert float((got - want).abs().max()) < 1e-5 * float(want.abs().max())
