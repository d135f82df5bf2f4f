"""Prompt attention ahead of a router: the matrix-core form beside the thread-per-key form, whose sums stand in another order.

A token whose choice of experts is a near tie can choose otherwise in the two, as it can in either beside float64; its output
is then another one, however small the difference was. So tokens are told apart by their choice: those that choose as float64
does are as near to it in both forms, token by token, and every other choice is a near tie. Neither form makes more of them."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import ravelorn as orc  # noqa: E402

DEV = torch.device("cuda", 0)
T, W, TOP = 400, 256, 4


def config():
    left = {"heads": 4, "kv_heads": 2, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "q_temp": {"coef": 0.1, "every": 64}}
    right = {"heads": 1, "kv_heads": 1, "dim": 16, "vdim": 16, "conv": 2}
    mlp = {"kind": "moe", "expert": {"ff": 32}, "router": {"experts": 30, "identity": 2, "top": TOP}}
    return {"architecture": "Ravelorn", "vocab": 300, "width": W, "norm": {"eps": 1e-5}, "residual_mult": 0.7, "logit_softcap": 30.0,
            "max_positions": T, "layers": [{"type": "parallel", "mlp": mlp, "mixer": {
                "left": left, "right": right, "left_scale": 1.0, "right_scale": 0.3}}]}


def in_float64(cfg, weights, tokens):
    """The residual behind the experts, the chosen experts and how far the last of them is from the next."""
    w = {n: t.double() for n, t in weights.items()}
    layer, lw = cfg["layers"][0], orc._sub(w, "l0.")
    x = w["embed"][torch.tensor(tokens)] + w["pos"][:T]
    y = orc.mixer("parallel", x, orc._sub(lw, "mix."), layer["mixer"], 1e-5)
    x = x + 0.7 * orc.layer_norm(y, lw["norm1"], lw["norm1.b"], 1e-5)
    m = orc._sub(lw, "mlp.")
    choice = torch.softmax(x @ m["router"].T, -1) + m["correction"]
    best = choice.topk(TOP + 1)
    y = orc.moe_ff(x, m, layer["mlp"])
    x = x + 0.7 * orc.layer_norm(y, lw["norm2"], lw["norm2.b"], 1e-5)
    return x, best.indices[:, :TOP].sort().values, best.values[:, TOP - 1] - best.values[:, TOP]


@pytest.mark.parametrize("seed", range(6))
def test_tokens_that_choose_alike(seed, monkeypatch):
    from lit_gpt import seq_ops
    from lit_gpt.config import LayeredConfig
    from lit_gpt.layered import LayeredGPT
    from lit_gpt.mixers import StepBatch

    cfg = config()
    parsed = LayeredConfig.from_dict(cfg)
    weights = LayeredGPT.random_weights(parsed, seed=seed)
    model = LayeredGPT(parsed, weights, device=DEV, dtype=torch.bfloat16)
    model.set_kv_cache(1, T)
    tokens = torch.randint(0, 300, (T,), generator=torch.Generator().manual_seed(seed)).tolist()
    want, ids, margin = (t.to(DEV) for t in in_float64(cfg, weights, tokens))

    tiles, route, chosen = seq_ops.sinkattn, seq_ops.moe_route_scores, []

    def noted(*a, **k):
        out = route(*a, **k)
        chosen.append(out[0].long().sort().values)
        return out

    monkeypatch.setattr(seq_ops, "moe_route_scores", noted)
    outs = []
    for form in (tiles, lambda proj, off, k, v, *a, **kw: tiles(proj, off, k.float(), v.float(), *a, **kw)):
        monkeypatch.setattr(seq_ops, "sinkattn", form)
        outs.append(model.forward_step(StepBatch.build([(0, 0, tokens)], DEV)).double())
    assert len(chosen) == 2
    alike = [(c == ids).all(-1) for c in chosen]
    both = alike[0] & alike[1]
    err = [(x - want).norm(dim=-1) / want.norm(dim=-1) for x in outs]
    # bf16 operands through the mixer's two products and the experts' three, 2^-9 each on sums of random signs: 2^-6 bounds the
    # worst of 400 tokens. What the attention's fp32 sums differ by reaches a token as roundings that fall the other way
    assert max(float(e[both].max()) for e in err) < 2 ** -6
    assert float(err[0][both].norm()) < 1.01 * float(err[1][both].norm())
    assert float((outs[0] - outs[1])[both].abs().max()) < 2 ** -6 * float(want.abs().max())
    # a score's slope is at most 1/4 of its logit's, whose error is 2^-8: where a choice is no such near tie it is float64's
    assert not (~both).any() or float(margin[~both].max()) < 2 ** -10
    assert abs(int(alike[0].sum()) - int(alike[1].sum())) <= 2 and int(both.sum()) >= T - 8
