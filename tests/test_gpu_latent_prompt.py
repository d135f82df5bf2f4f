"""Fresh prompts of latent attention over expanded keys and values against the form in the latent space, both on the same
queries and caches, and against float64 over the same bf16 latents and weights."""

import pytest
import torch

pytestmark = pytest.mark.gpu
H, DK, DR, DV, R, W = 3, 128, 64, 128, 192, 64


def model(seed=0, edit=None):
    from lit_gpt.config import LayeredConfig
    from lit_gpt.layered import LayeredGPT

    cfg = {"architecture": "Fazolorn", "vocab": 50, "width": W, "norm": {"eps": 1e-5}, "layers": [
        {"type": "latent_attention", "mixer": {"heads": H, "dim": DK, "rot_dim": DR, "vdim": DV, "kv_rank": R, "q_rank": 96,
                                               "rot": {"dims": DR, "base": 100.0}, "scale": 192 ** -0.5}}]}
    config = LayeredConfig.from_dict(cfg)
    weights = LayeredGPT.random_weights(config, seed=seed)
    if edit:
        edit(weights)
    return LayeredGPT(config, weights, device=torch.device("cuda", 0), dtype=torch.bfloat16)


def heads(mix, step, cache, proj):
    """The heads' outputs in fp32, ahead of the out-projection."""
    kept = []
    mix.out_gate, mix._finish = True, lambda att, *_: kept.append(att)  # (with a gate to come they are not rounded)
    mix.forward(proj, step, cache, torch.empty(step.T, W, device=proj.device))
    del mix._finish
    mix.out_gate = False
    return kept[0]


def prompt(lengths, fresh=True, slots=(1, 0, 2)):
    from lit_gpt.mixers import StepBatch

    step = StepBatch.build([(s, 0, [1] * n) for s, n in zip(slots, lengths)], torch.device("cuda", 0))
    step.fresh = fresh
    return step


def test_fp32_latents_take_the_latent_form():
    mix = model().blocks[0].mixer
    dev, T = torch.device("cuda", 0), 70
    proj = torch.randn(T, 96 + R + DR, generator=torch.Generator(device=dev).manual_seed(1), device=dev)
    out = [heads(mix, prompt([T], fresh), mix.build_cache(3, 80, dev, torch.float32), proj.clone()) for fresh in (True, False)]
    assert torch.equal(*out)


def test_captured_prompt_at_later_positions():
    """A step captured from a prompt's start and replayed further on, its positions moved on the device in between."""
    m = model(2)
    dev, T = torch.device("cuda", 0), 24
    m.set_kv_cache(2, 128)
    g = torch.Generator().manual_seed(1)
    ids = torch.randint(0, 50, (4, T), generator=g)

    def table(i, fresh):
        from lit_gpt.mixers import StepBatch

        step = StepBatch.build([(1, i * T, ids[i].tolist())], dev)
        step.fresh = fresh
        return step

    with torch.inference_mode():
        want = [m.logits(m.forward_step(table(i, False))).clone() for i in range(4)]
        step = table(0, True)
        m.logits(m.forward_step(step))
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = m.logits(m.forward_step(step))
        for i in (0, 1, 2, 3, 0, 1):
            step.tokens.copy_(ids[i])
            step.pos.copy_(torch.arange(i * T, (i + 1) * T))
            step.seq_pos0.fill_(i * T)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want[i]), i


def reference(mix, cache, proj, lengths, slots):
    """The heads' outputs in float64 from the step's own queries (as the module makes them), its bf16 latents and rotated keys
    as they lie in the cache, and the bf16 weights."""
    from lit_gpt import seq_ops

    step = prompt(lengths, slots=slots)
    T = step.T
    cq = seq_ops.norm_columns(proj, mix.off["dq"], mix.q_norm_w, eps=mix.eps, bf16=True)
    q = torch.empty(T, H * (DK + DR), device=proj.device)
    seq_ops.linear(cq, mix.w_uq, M=T, N=H * (DK + DR), K=96, y=q, lda=96, ldy=H * (DK + DR))
    seq_ops.latent_prepare(q, 0, proj, mix.off["dkv"], cache.c, cache.kr, mix.norm_w, mix.inv_freq, step.slot, step.pos, H=H, d=DK,
                           dr=DR, r=R, rot_dims=mix.rot_dims, eps=mix.eps, rot_mult=mix.rot_mult)
    q = q.double().view(T, H, DK + DR)
    up = mix.w_up.double()
    uk, uv = up[: H * DK].view(H, DK, R), up[H * DK:].view(H, DV, R)
    out, at = [], 0
    for n, s in zip(lengths, slots):
        c, kr = cache.c[s, :n].double(), cache.kr[s, :n].double()
        hidden = torch.ones(n, n, dtype=torch.bool, device=proj.device).triu(1)
        per = []
        for h in range(H):
            k = torch.cat([c @ uk[h].T, kr], -1)
            w = torch.softmax((q[at:at + n, h] @ k.T * mix.scale).masked_fill(hidden, -float("inf")), -1)
            per.append(w @ (c @ uv[h].T))
        out.append(torch.stack(per, 1).flatten(1))
        at += n
    return torch.cat(out)


@pytest.mark.parametrize("lengths", [(24,), (300, 40, 9), (700,)])
@pytest.mark.parametrize("part", ["both", "keys", "rotated"])
def test_expanded_against_latent_form(lengths, part):
    """The same queries and cached latents through both forms: expanded keys and values hold 16 bits of their significands and
    rotated parts meet as two summands each, where the latent form rounds the queries on their way into the latent space and
    the weighted latents on their way out to 8 bits. ``part``: which of a score's two parts is large."""
    def edit(w):
        for n in w:
            if n.endswith("uk") and part == "rotated":
                w[n] = w[n] * 0.02
            if n.endswith("dkv") and part == "rotated":
                w[n][R:] *= 4.0
            if n.endswith("uk") and part == "keys":
                w[n] = w[n] * 4.0

    mix = model(3, edit).blocks[0].mixer
    dev, T = torch.device("cuda", 0), sum(lengths)
    proj = torch.randn(T, 96 + R + DR, generator=torch.Generator(device=dev).manual_seed(T), device=dev)
    slots = (1, 0, 2)[: len(lengths)]
    cache = mix.build_cache(3, 720, dev, torch.bfloat16)
    got, latent = (heads(mix, prompt(lengths, fresh, slots), cache, proj.clone()).double() for fresh in (True, False))
    want = reference(mix, cache, proj.clone(), lengths, slots)
    err, before = (float((x - want).norm() / want.norm()) for x in (got, latent))
    assert err < before and err < 2.0 ** -14
