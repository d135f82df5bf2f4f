"""Which latent prompts are made over expanded keys and values (the others: in the latent space), on the host."""

import pytest
import torch


@pytest.fixture(autouse=True)
def eager(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)  # (asks the GPU)


def module(kv_rank=128, vdim=128, seed=1):
    from lit_gpt.config import LayeredConfig
    from lit_gpt.layered import LayeredGPT, _sub
    from lit_gpt.mixers import LatentAttention

    cfg = {"architecture": "Fazolorn", "vocab": 16, "width": 64, "norm": {"eps": 1e-5}, "layers": [
        {"type": "latent_attention", "mixer": {"heads": 2, "dim": 128, "rot_dim": 64, "vdim": vdim, "kv_rank": kv_rank, "q_rank": 48,
                                               "rot": {"dims": 64, "base": 100.0}, "scale": 192 ** -0.5}}]}
    config = LayeredConfig.from_dict(cfg)
    weights = _sub(LayeredGPT.random_weights(config, seed=seed), "l0.mix.")
    return LatentAttention(config.layers[0].mixer, 64, 1e-5, weights, torch.device("cpu"), torch.bfloat16)


def prompt(lengths=(40,), pos0=(0,)):
    from lit_gpt.mixers import StepBatch

    return StepBatch.build([(i, p, [1] * n) for i, (n, p) in enumerate(zip(lengths, pos0))], torch.device("cpu"))


def takes(mix, step, dtype=torch.bfloat16):
    return mix._expands(step, mix.build_cache(3, 64, torch.device("cpu"), dtype), 2 * 192, 0)


def test_fresh_prompts_of_the_served_sizes():
    mix = module()
    assert takes(mix, prompt()) and takes(mix, prompt((9, 20), (0, 0)))
    assert not takes(mix, prompt((40,), (1,))) and not takes(mix, prompt((9, 20), (0, 3)))
    assert not takes(mix, prompt((7,))) and not takes(mix, prompt((9, 6), (0, 0)))
    assert not takes(module(vdim=64), prompt()) and not takes(module(kv_rank=100), prompt())
    assert not mix._expands(prompt(), mix.build_cache(3, 64, torch.device("cpu"), torch.bfloat16), 2 * 192 + 2, 0)


def test_latents_kept_in_fp32_are_not_rounded():
    mix = module()
    assert not takes(mix, prompt(), torch.float32)


def test_captured_steps_are_not_bound_to_their_start(monkeypatch):
    mix = module()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert not takes(mix, prompt())


def test_saved_weights_hold_no_second_layout():
    """A state dict has each up-projection once, and loading one moves the prompts' layout along."""
    a, b = module(), module(seed=2)
    saved = a.state_dict()
    assert sorted(saved) == ["inv_freq", "norm_w", "q_norm_w", "w_o", "w_ukT", "w_uq", "w_uv"]
    assert not torch.equal(a.w_up, b.w_up)
    outer = torch.nn.Module()
    outer.mixer = b
    outer.load_state_dict({"mixer." + n: t.clone() for n, t in saved.items()})
    assert torch.equal(b.w_up, a.w_up) and torch.equal(b.w_uv, a.w_uv)
    c = module(seed=3)
    c.load_state_dict({n: t.clone() for n, t in saved.items()}, assign=True)
    assert torch.equal(c.w_up, a.w_up)
