"""Router logits of a token in prompts of different lengths: the same bits, however many experts there are."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
W = 2048


def model(design, experts):
    from lit_gpt.config import LayeredConfig
    from lit_gpt.layered import LayeredGPT

    mlp = {"kind": "moe", "expert": {"ff": 16}, "router": {"experts": experts, "top": 4}}
    more = {}
    if design == "Bavesun":
        layer = {"type": "retention", "mixer": {"heads": 1, "dim": 16, "vdim": 16, "decay": [0.9], "rot": {"dims": 16, "base": 1e4}}}
        more["embedding"] = {"scale": 5.0}
    elif design == "Ravelorn":
        mlp["router"]["identity"] = 2
        layer = {"type": "channel_delta", "mixer": {"heads": 1, "kv_heads": 1, "dim": 16, "vdim": 16, "conv": 4, "decay_rank": 8,
                                                    "gate_rank": 8}}
        more.update(residual_mult=0.7, logit_softcap=30.0, max_positions=4096)
    else:
        mlp["router"].update(scale=2.5, groups={"count": 4, "keep": 2})
        layer = {"type": "mingru", "mixer": {"width": 64}}
    config = LayeredConfig.from_dict(dict(architecture=design, vocab=64, width=W, norm={"eps": 1e-5}, layers=[dict(layer, mlp=mlp)],
                                          **more))
    return LayeredGPT(config, LayeredGPT.random_weights(config, seed=3), device=DEV, dtype=torch.bfloat16)


@pytest.mark.parametrize("design", ["Bavesun", "Ravelorn", "Fazolorn"])
@pytest.mark.parametrize("experts", [16, 64, 160])
def test_same_bits_in_prompts_of_every_length(design, experts, monkeypatch):
    from lit_gpt.mixers import SparseFeedForward, StepBatch

    m = model(design, experts)
    ids = torch.randint(0, 64, (2000,), generator=torch.Generator().manual_seed(2)).tolist()
    m.set_kv_cache(1, 2048)
    seen, plain = [], SparseFeedForward.forward
    monkeypatch.setattr(SparseFeedForward, "forward", lambda self, proj, *a, **k: (
        seen.append(proj[:13, self.off["router"]:self.off["router"] + self.n_router].clone()), plain(self, proj, *a, **k))[1])
    with torch.inference_mode():
        for n in (13, 60, 130, 300, 700, 2000):
            m.forward_step(StepBatch.build([(0, 0, ids[:n])], DEV))
    for n, logits in zip((60, 130, 300, 700, 2000), seen[1:]):
        assert torch.equal(logits, seen[0]), n
