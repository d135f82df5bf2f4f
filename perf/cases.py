"""What is timed: prompts and captured one-token steps of both model families, through the calls that a program makes.

Two kinds of cases. ``family: gpt`` builds a model of a registered configuration with ``generate.base.build_model`` and
runs ``GPT.forward``: a prompt from position 0, or one token at the end of a filled cache as a captured HIP graph (the
way ``generate`` steps). ``family: layered`` builds a ``LayeredGPT`` and runs ``generate.batch.BatchEngine.step`` for a
batch of prompts, or one token for every live sequence as a captured graph. Weights are random at the models' own
shapes; a pass returns the logits that the call returns and the caches and recurrent states that it updates.

A prompt pass starts its sequences anew, so it can be repeated. A captured step of the GPT family writes the same
cache row again; one of the layered family reads the same position again, and its recurrent states go on from where the
last pass left them.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "lit-gpt_amd"))

from generate.base import build_model  # noqa: E402
from generate.batch import BatchEngine  # noqa: E402
from lit_gpt import Config  # noqa: E402
from lit_gpt.config import LayeredConfig  # noqa: E402
from lit_gpt.layered import LayeredGPT  # noqa: E402
from lit_gpt.mixers import StepBatch  # noqa: E402

DEV = "cuda"
VOCAB = 32000  # of the layered models
F64 = torch.float64


def listed():
    return [
        # interactive generation from a long conversation, the whole model: 4-bit weights, every matrix read once a token
        _gpt("llama7b_int4_decode", "Llama-2-7b-hf", 32, "int4-g128", 1, 2047),
        # the prompt of such a conversation (a quarter of the depth: every layer is alike)
        _gpt("llama7b_int4_prompt", "Llama-2-7b-hf", 8, "int4-g128", 2048, 0),
        # unquantized weights, a prompt of a page, no multiple of a tile
        _gpt("llama7b_bf16_prompt", "Llama-2-7b-hf", 4, "bf16", 517, 0),
        # grouped heads and wide layers, a question of a few lines: few rows against large matrices
        _gpt("llama70b_nf4_prompt", "Llama-2-70b-hf", 2, "nf4", 93, 0),
        # one token through routed experts, a long document in the cache
        _gpt("mixtral_int4_decode", "Mixtral-8x7B-v0.1", 4, "int4-g128", 1, 9001),
        # the smallest call: a small model in 32 bits, where launches and their latency count
        _gpt("pythia_fp32_decode", "pythia-160m", 12, "fp32", 1, 300),
        # one prompt through delta rules, sink attention and score-routed experts
        _layered("ravelorn_prompt", "Ravelorn", 2048, "prompt", "2048"),
        # a served batch of eight conversations of unequal length, one token each
        _layered("ravelorn_decode", "Ravelorn", 2048, "decode", "2047,1500,1111,700,333,160,63,9"),
        # three prompts of unequal length in one step through wide state-space and differential-attention layers
        _layered("rigulorn_prompts", "Rigulorn", 4096, "prompt", "1500,777,130"),
        # one conversation, one token, four residual streams: many small launches
        _layered("rigulorn_decode", "Rigulorn", 2048, "decode", "2047"),
        # a long document through recurrent, chunk-confined and latent attention layers
        _layered("fazolorn_prompt", "Fazolorn", 2048, "prompt", "4096"),
        # three conversations on wide layers, one token each
        _layered("fazolorn_decode", "Fazolorn", 4096, "decode", "1200,731,64"),
    ]


def draw(rng):
    kind = rng.choice(["gpt_decode", "gpt_prompt", "prompt", "prompt", "decode"])
    if kind == "gpt_decode":
        model, weights, layers = rng.choice([("Llama-2-7b-hf", "int4-g128", 8), ("Llama-2-7b-hf", "nf4", 8),
                                             ("Llama-2-7b-hf", "bf16", 6), ("Llama-2-70b-hf", "nf4", 3),
                                             ("Mixtral-8x7B-v0.1", "int4-g128", 3), ("pythia-160m", "fp32", 12)])
        most = {"pythia-160m": 2000, "Llama-2-7b-hf": 4000, "Llama-2-70b-hf": 4000}.get(model, 16000)
        return _gpt(None, model, rng.randint(2, layers), weights, 1, _log_int(rng, 16, most))
    if kind == "gpt_prompt":
        model, weights, layers = rng.choice([("Llama-2-7b-hf", "int4-g128", 6), ("Llama-2-7b-hf", "nf4", 6),
                                             ("Llama-2-7b-hf", "bf16", 6), ("Llama-2-70b-hf", "nf4", 2),
                                             ("Mixtral-8x7B-v0.1", "int4-g128", 2), ("pythia-160m", "fp32", 12)])
        return _gpt(None, model, rng.randint(2, layers), weights, _log_int(rng, 2, 300 if weights == "fp32" else 2048), 0)
    design, width = rng.choice(["Ravelorn", "Rigulorn", "Fazolorn"]), rng.choice([2048, 2048, 4096])
    if kind == "decode":
        lengths = [_log_int(rng, 1, 2048) for _ in range(rng.randint(1, 8))]
    else:
        room, lengths = (1500 if width == 4096 else 3000), []
        for _ in range(rng.randint(1, 6)):
            if room > 2:
                lengths.append(_log_int(rng, 2, room))
                room -= lengths[-1]
    return _layered(None, design, width, kind, ",".join(map(str, lengths)))


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _gpt(name, model, layers, weights, tokens, context):
    case = dict(family="gpt", model=model, layers=layers, weights=weights, tokens=tokens, context=context)
    return case if name is None else dict(case, name=name)


def _layered(name, design, width, step, lengths):
    case = dict(family="layered", design=design, width=width, step=step, lengths=lengths)
    return case if name is None else dict(case, name=name)


def prepare(case, seed):
    return _prepare_gpt(case, seed) if case["family"] == "gpt" else _prepare_layered(case, seed)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return dict(state["kept"], logits=state["logits"])
    with torch.inference_mode():
        if "engine" in state:
            ids = list(range(len(state["prompts"])))
            logits = state["engine"].step([(i, p, [len(p) - 1]) for i, p in zip(ids, state["prompts"])], end=ids)
        else:
            logits = state["model"](state["idx"], state["pos"], last_token_only=True)
    return dict(state["kept"], logits=logits)


def exact(case, seed):
    with torch.inference_mode():
        return _exact_gpt(case, seed) if case["family"] == "gpt" else _exact_layered(case, seed)


def _captured(step):
    """A step as a program captures it: once eagerly, then recorded."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


# ------------------------------------------------------------------------------------------------ the GPT family
def _gpt_config(case):
    return Config.from_name(case["model"], n_layer=case["layers"], block_size=16384)


def _gpt_inputs(case, seed):
    """The built model, the ids and their positions; the cache holds ``context`` tokens' keys and values."""
    cfg = _gpt_config(case)
    T, ctx, weights = case["tokens"], case["context"], case["weights"]
    model = build_model(cfg, quantize=None if weights in ("bf16", "fp32") else weights, device=torch.device(DEV, 0),
                        seed=seed, max_seq_length=-(-(ctx + T + 1) // 64) * 64,
                        dtype=torch.float32 if weights == "fp32" else torch.bfloat16)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed + 1)
    kept = {}
    for name in ("k", "v"):  # the layers' caches side by side in one buffer
        one = getattr(model.transformer.h[0].attn.kv_cache, name)
        kept[name] = torch.zeros(cfg.n_layer, *one.shape, dtype=one.dtype, device=DEV)
        kept[name][..., :ctx, :].normal_(generator=gen)
        for i, block in enumerate(model.transformer.h):
            setattr(block.attn.kv_cache, name, kept[name][i])
    idx = torch.randint(0, cfg.vocab_size, (1, T), generator=gen, device=DEV, dtype=torch.int32)
    return model, idx, torch.arange(ctx, ctx + T, device=DEV), kept


def _prepare_gpt(case, seed):
    model, idx, pos, kept = _gpt_inputs(case, seed)
    state = dict(model=model, idx=idx, pos=pos, kept=kept)
    if case["tokens"] == 1:
        with torch.inference_mode():
            state["graph"], state["logits"] = _captured(lambda: model(idx, pos, last_token_only=True))
    return state


NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635, -0.18477343022823334,
       -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


def _matrix(linear):
    """A linear layer's matrix in 64 bits: as it is, or from its 4-bit values (low half first) times their block's scale."""
    if not hasattr(linear, "qweight"):
        return linear.weight.to(F64)
    q = linear.qweight.long()
    q = torch.stack([q & 15, q >> 4], -1).flatten(1)
    table = torch.tensor(NF4, dtype=F64, device=q.device) if linear.scales.dtype == torch.float32 else \
        torch.arange(-8, 8, dtype=F64, device=q.device)
    return (table[q].view(q.shape[0], linear.scales.shape[1], -1) * linear.scales.to(F64).unsqueeze(-1)).flatten(1)


def _linear(linear, x):
    y = x @ _matrix(linear).T
    return y if linear.bias is None else y + linear.bias.to(F64)


def _norm(norm, x):
    w = norm.weight.to(F64)
    if getattr(norm, "bias", None) is not None:
        return torch.nn.functional.layer_norm(x, w.shape, w, norm.bias.to(F64), norm.eps)
    return _rms(x, norm.eps) * w


def _mlp(mlp, cfg, x):
    if cfg._mlp_class == "GptNeoxMLP":
        return _linear(mlp.proj, torch.nn.functional.gelu(_linear(mlp.fc, x), approximate=cfg.gelu_approximate))
    if cfg._mlp_class == "LLaMAMoE":
        top, idx = torch.topk(_linear(mlp.gate, x), cfg.n_expert_per_token)
        probs, out = torch.softmax(top, -1), torch.zeros_like(x)
        for e, expert in enumerate(mlp.experts):
            rows, place = torch.where(idx == e)
            if len(rows):
                out[rows] += probs[rows, place, None] * _swiglu(expert, x[rows])
        return out
    return _swiglu(mlp, x)


def _swiglu(mlp, x):
    return _linear(mlp.proj, torch.nn.functional.silu(_linear(mlp.fc_1, x)) * _linear(mlp.fc_2, x))


def _exact_gpt(case, seed):
    cfg = _gpt_config(case)
    model, idx, pos, kept = _gpt_inputs(case, seed)
    T, end = case["tokens"], case["context"] + case["tokens"]
    H, G, hs, n = cfg.n_head, cfg.n_query_groups, cfg.head_size, cfg.rope_n_elem
    cos, sin = (t[pos].to(F64).unsqueeze(1) for t in (model.cos, model.sin))

    def rope(x):  # (T, heads, hs)
        r, half = x[..., :n], n // 2
        turned = torch.cat([-r[..., half:], r[..., :half]], -1)
        return torch.cat([r * cos + turned * sin, x[..., n:]], -1)

    out = {name: t.to(F64) for name, t in kept.items()}
    x = model.transformer.wte.weight[idx[0]].to(F64)
    for i, block in enumerate(model.transformer.h):
        h = _norm(block.norm_1, x)
        qkv = _linear(block.attn.attn, h).view(T, G, H // G + 2, hs)
        q, k, v = rope(qkv[:, :, :-2].reshape(T, H, hs)), rope(qkv[:, :, -2]), qkv[:, :, -1]
        out["k"][i, 0, :, pos], out["v"][i, 0, :, pos] = k.transpose(0, 1), v.transpose(0, 1)
        y = _softmax_heads(q, out["k"][i, 0, :, :end].transpose(0, 1), out["v"][i, 0, :, :end].transpose(0, 1),
                           pos, hs ** -0.5)
        y = _linear(block.attn.proj, y)
        if cfg.parallel_residual:
            x = x + y + _mlp(block.mlp, cfg, _norm(block.norm_2, x))
        else:
            x = x + y
            x = x + _mlp(block.mlp, cfg, _norm(block.norm_2, x))
    out["logits"] = _linear(model.lm_head, _norm(model.transformer.ln_f, x[-1:])).unsqueeze(0)
    return out


# ------------------------------------------------------------------------------------------------ the layered family
def _layered_config(case):
    """The layers of the repository's benchmark of each design."""
    W = case["width"]
    H, ff = W // 128, {2048: 5632, 4096: 11008}[W]
    base = dict(architecture=case["design"], vocab=VOCAB, width=W, norm={"eps": 1e-5})
    moe = {"kind": "moe", "expert": {"ff": ff // 4}}
    if case["design"] == "Ravelorn":
        moe["router"] = {"experts": 16, "identity": 2, "top": 4}
        delta = {"type": "channel_delta", "mlp": moe, "mixer": {
            "heads": H, "kv_heads": H, "dim": 128, "vdim": 128, "conv": 4, "decay_rank": W // 32, "gate_rank": W // 32}}
        both = {"type": "parallel", "mlp": moe, "mixer": {
            "left": {"heads": H, "kv_heads": H // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                     "q_temp": {"coef": 0.1, "every": 512}},
            "right": {"heads": H // 2, "kv_heads": H // 2, "dim": 128, "vdim": 128, "conv": 4},
            "left_scale": 1.0, "right_scale": 1.0}}
        return dict(base, residual_mult=0.7, logit_softcap=30.0, max_positions=4096, layers=[delta, both, delta, both])
    if case["design"] == "Rigulorn":
        att = {"heads": H, "kv_heads": H // 4, "dim": 64, "vdim": 128, "diff": 0.5, "softcap": 30.0, "scale": 0.125,
               "mask": {"size": 1024}, "rot": {"dims": 64, "base": 1e4}}
        mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
        scan = {"type": "mamba2", "mlp": mlp, "mixer": {
            "heads": 2 * W // 64, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}}
        return dict(base, embedding={"scale": 1.0}, streams=4, layers=[
            scan, {"type": "attention", "mixer": att, "mlp": mlp}, scan,
            {"type": "attention", "mixer": dict(att, kv_from=1), "mlp": mlp}])
    moe["router"] = {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}, "scale": 2.5}
    dense = {"kind": "dense", "ff": ff, "limit": 7.0}
    gru = {"type": "mingru", "mixer": {"width": W}}
    att = {"type": "attention", "mlp": moe, "mixer": {
        "heads": H, "kv_heads": H // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1200},
        "rot": {"dims": 64, "base": 1e6}}}
    latent = {"type": "latent_attention", "mlp": moe, "mixer": {
        "heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "q_rank": 3 * W // 4, "scale": 192 ** -0.5,
        "rot": {"dims": 64, "base": 1e5, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
    return dict(base, logit_scale=0.5, loop={"start": 0, "stop": 4, "times": 1},
                layers=[dict(gru, mlp=dense), att, latent, dict(gru, mlp=moe)])


def _layered_weights(config, seed):
    """bf16 checkpoint tensors on the GPU: matrices ~ N(0, 1 / fan in), the rest in the ranges that such models have. A
    layer's experts are relatives, as where they were grown from one feed-forward: a token whose choice between two of
    them is a near tie then has nearly the same output either way."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    out, parents = {}, {}
    for name, shape in LayeredGPT.tensor_shapes(config).items():
        t, leaf = torch.randn(shape, generator=gen, device=DEV), name.rsplit(".", 1)[-1]
        if leaf in ("norm1", "norm2", "norm", "D"):
            t = 1.0 + 0.1 * t
        elif name.endswith(("norm1.b", "norm2.b", "norm.b", "correction")):
            t = 0.1 * t
        elif ".hc" in name:
            s = config.streams
            t = 0.2 * t + (torch.eye(s, device=DEV) if leaf == "mix" else 1.0 / s if leaf == "in" else 1.0)
        elif leaf in ("lq1", "lk1", "lq2", "lk2") or leaf == "b" and len(shape) == 1:
            t = 0.3 * t
        elif leaf == "A_log":
            t = torch.log(1.0 + 3.0 * torch.rand(shape, generator=gen, device=DEV))
        elif leaf in ("dt_bias", "pb"):
            t = t - 2.0
        elif leaf == "conv":
            t = 0.7 * t
        elif leaf != "sink":
            if ".mlp.e" in name:
                t = 0.995 * parents.setdefault((name.split(".")[0], leaf), t) + 0.1 * t
            t = t * shape[-1] ** -0.5
        out[name] = t.to(torch.bfloat16)
    return out


def _layered_inputs(case, seed):
    config = LayeredConfig.from_dict(_layered_config(case))
    weights = _layered_weights(config, seed)
    gen = torch.Generator()
    gen.manual_seed(seed + 1)
    lengths = [int(n) for n in case["lengths"].split(",")]
    prompts = [torch.randint(0, VOCAB, (n,), generator=gen).tolist() for n in lengths]
    new = torch.randint(0, VOCAB, (len(lengths),), generator=gen).tolist()
    return config, weights, prompts, new, -(-(max(lengths) + 1) // 64) * 64


def _prepare_layered(case, seed):
    config, weights, prompts, new, room = _layered_inputs(case, seed)
    # (a router's rows are padded on the host while the model is built)
    model = LayeredGPT(config, {n: t.cpu() if n.endswith("router") else t for n, t in weights.items()},
                       device=torch.device(DEV, 0), dtype=torch.bfloat16)
    engine = BatchEngine(model, max_seq_length=room, slots=len(prompts))
    kept = dict(model.caches.named_buffers())
    state = dict(engine=engine, prompts=prompts, kept=kept)
    if case["step"] == "decode":
        with torch.inference_mode():
            engine.step([(i, p, []) for i, p in enumerate(prompts)])
            batch = StepBatch.build([(*engine.live[i], [t]) for i, t in enumerate(new)], engine.device)
            before = {n: t.clone() for n, t in kept.items()}
            state["graph"], state["logits"] = _captured(lambda: model.logits(model.forward_step(batch)))
            for n, t in before.items():  # the step that came before the capture has not happened
                kept[n].copy_(t)
        state["batch"] = batch
    return state


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _softmax_heads(q, k, v, pos, scale, *, weigh=None, first=None):
    """q (T, H, d) at positions ``pos`` over k (S, G, d) and v (S, G, dv) at positions 0 .. S - 1 -> (T, H dv), causal.
    ``weigh(scores, head)``: another weighting than the softmax; ``first``: the first position that each query sees."""
    S, G, H = k.shape[0], k.shape[1], q.shape[1]
    at = torch.arange(S, device=q.device)
    hidden = at[None, :] > pos[:, None]
    if first is not None:
        hidden |= at[None, :] < first[:, None]
    out = []
    for h in range(H):
        s = ((q[:, h] @ k[:, h // (H // G)].T) * scale).masked_fill_(hidden, -math.inf)
        out.append((torch.softmax(s, -1) if weigh is None else weigh(s, h)) @ v[:, h // (H // G)])
    return torch.cat(out, -1)


def _turn(x, freqs, mult=1.0, halves=False):
    """Rotary positions 0 .. T - 1 on the first 2 len(freqs) dims of x (T, heads, d): pairs (2i, 2i + 1), or (i, i + n)."""
    n = len(freqs)
    angle = torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None] * torch.tensor(freqs, dtype=F64, device=x.device)
    c, s = torch.cos(angle)[:, None] * mult, torch.sin(angle)[:, None] * mult
    a, b = (slice(0, n), slice(n, 2 * n)) if halves else (slice(0, 2 * n, 2), slice(1, 2 * n, 2))
    out = x.clone()
    out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return out


def _frequencies(rot):
    """(frequency of every rotated pair, factor of cos and sin); with a scaling the slow pairs are slowed, the fast ones
    kept, those between the two corners blended."""
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    plain = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not sc:
        return plain, 1.0
    lo, hi = (dims * math.log(sc["original"] / (2 * math.pi * sc[w])) / (2 * math.log(base)) for w in ("fast", "slow"))
    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
    slow = [min(1.0, max(0.0, (i - lo) / max(hi - lo, 0.001))) for i in range(dims // 2)]
    return [f / sc["factor"] * a + f * (1 - a) for f, a in zip(plain, slow)], 0.1 * math.log(sc["factor"]) + 1.0


def _conv(u, weight, bias=None):
    """Causal convolution of u (T, C) per channel with weight (C, taps), then silu; and the inputs that the next token needs."""
    taps = weight.shape[1]
    padded = torch.cat([torch.zeros(taps - 1, u.shape[1], dtype=F64, device=u.device), u])
    y = sum(weight[:, j] * padded[j:j + len(u)] for j in range(taps))
    return torch.nn.functional.silu(y if bias is None else y + bias), padded[len(padded) - taps + 1:]


def _delta(h, w, m, eps, per_channel):
    H, G, d, dv, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
    raw = torch.cat([h @ w[n].T for n in "qkv"], -1)
    y, last = _conv(raw, torch.cat([w[n + ".conv"] for n in "qkv"]))
    q, k, v = y[:, :G * d].view(T, G, d), y[:, G * d:2 * G * d].view(T, G, d), y[:, 2 * G * d:].view(T, H, dv)
    q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k = ((t).repeat_interleave(H // G, 1) for t in (q * d ** -0.5, k))
    beta = torch.sigmoid(h @ w["b"].T)
    a = (h @ w["a1"].T) @ w["a2"].T if per_channel else h @ w["a"].T
    g = torch.exp(-torch.exp(w["A_log"])[:, None] * torch.nn.functional.softplus(a + w["dt_bias"], threshold=50).view(T, H, -1))
    gate = torch.sigmoid((h @ w["g1"].T) @ w["g2"].T) if per_channel else torch.nn.functional.silu(h @ w["g"].T)
    S, out = torch.zeros(H, d, dv, dtype=F64, device=h.device), torch.empty(T, H, dv, dtype=F64, device=h.device)
    for t in range(T):
        S = S * g[t, :, :, None]
        u = beta[t, :, None] * (v[t] - (k[t, :, None] @ S)[:, 0])
        S = S + k[t, :, :, None] * u[:, None]
        out[t] = (q[t, :, None] @ S)[:, 0]
    return (_rms(out, eps) * w["norm"] * gate.view(T, H, dv)).flatten(1) @ w["o"].T, {"s": S, "conv": last}


def _sink_attention(h, w, m, eps):
    H, G, d, T = m["heads"], m["kv_heads"], m["dim"], len(h)
    pos = torch.arange(T, device=h.device)
    q, k = _rms((h @ w["q"].T).view(T, H, d), eps), _rms((h @ w["k"].T).view(T, G, d), eps)
    v = (h @ w["v"].T).view(T, G, m["vdim"])
    temp = 1.0 + m["q_temp"]["coef"] * torch.log(((pos + 1) // m["q_temp"]["every"] + 1).to(F64))

    def weigh(s, head):
        return torch.softmax(torch.cat([s, w["sink"][head].expand(T, 1)], -1), -1)[:, :-1]

    return _softmax_heads(q * temp[:, None, None], k, v, pos, m["scale"], weigh=weigh) @ w["o"].T, {"k": k, "v": v}


def _scan(h, w, m, eps):
    H, dv, N, G, T = m["heads"], m["vdim"], m["state"], m["groups"], len(h)
    inner = H * dv
    proj = h @ w["in"].T
    y, last = _conv(proj[:, inner:2 * inner + 2 * G * N], w["conv"], w["conv.b"])
    x = y[:, :inner].view(T, H, dv)
    B, C = (y[:, inner + i * G * N:inner + (i + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
    dt = torch.nn.functional.softplus(proj[:, 2 * inner + 2 * G * N:] + w["dt_bias"], threshold=50)
    decay = torch.exp(-torch.exp(w["A_log"]) * dt)
    S, out = torch.zeros(H, N, dv, dtype=F64, device=h.device), torch.empty(T, H, dv, dtype=F64, device=h.device)
    for t in range(T):
        S = decay[t, :, None, None] * S + (dt[t, :, None] * B[t])[:, :, None] * x[t, :, None]
        out[t] = (C[t, :, None] @ S)[:, 0]
    y = (out + w["D"][:, None] * x).flatten(1) * torch.nn.functional.silu(proj[:, :inner])
    y = _rms(y.view(T, m["norm_groups"], -1), eps).flatten(1) * w["norm"]
    return y @ w["o"].T, {"s": S, "conv": last}


def _diff_attention(h, w, m, eps, kv):
    H, G, d, dv, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
    freqs, pos = _frequencies(m["rot"])[0], torch.arange(T, device=h.device)
    if kv is None:
        kv = {"k": _turn((h @ w["k"].T).view(T, 2 * G, d), freqs).view(T, G, 2 * d), "v": (h @ w["v"].T).view(T, G, dv)}
    q, k = _turn((h @ w["q"].T).view(T, 2 * H, d), freqs).view(T, H, 2, d), kv["k"].view(T, G, 2, d)

    def weigh(s, head):
        return torch.softmax(m["softcap"] * torch.tanh(s / m["softcap"]).masked_fill_(s == -math.inf, -math.inf), -1)

    first = pos // m["mask"]["size"] * m["mask"]["size"]
    maps = [_softmax_heads(q[:, :, i], k[:, :, i], kv["v"], pos, m["scale"], weigh=weigh, first=first) for i in (0, 1)]
    lam = torch.exp((w["lq1"] * w["lk1"]).sum()) - torch.exp((w["lq2"] * w["lk2"]).sum()) + m["diff"]
    y = _rms((maps[0] - lam * maps[1]).view(T, H, dv), eps) * (1.0 - m["diff"])
    return y.flatten(1) @ w["o"].T, kv


def _mingru(h, w):
    z, u = torch.sigmoid(h @ w["z"].T + w["z.b"]), h @ w["x"].T + w["x.b"]
    c = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    out, S = torch.empty_like(z), torch.zeros_like(z[0])
    for t in range(len(h)):
        S = (1.0 - z[t]) * S + c[t]
        out[t] = S
    return (out * torch.nn.functional.silu(h @ w["g"].T)) @ w["o"].T, {"s": S}


def _sigmoid_attention(h, w, m):
    H, G, d, T = m["heads"], m["kv_heads"], m["dim"], len(h)
    freqs, pos = _frequencies(m["rot"])[0], torch.arange(T, device=h.device)
    q, k = (h @ w["q"].T + w["q.b"]).view(T, H, d), (h @ w["k"].T + w["k.b"]).view(T, G, d)
    q, turned = _turn(q, freqs, halves=True), _turn(k, freqs, halves=True)
    first = pos // m["mask"]["size"] * m["mask"]["size"]
    y = _softmax_heads(q, turned, k, pos, m["scale"], weigh=lambda s, i: torch.sigmoid(s + w["pb"][i]), first=first)
    return y @ w["o"].T, {"k": turned, "v": k}


def _latent_attention(h, w, m, eps):
    H, d, dr, r, T = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"], len(h)
    freqs, mult = _frequencies(m["rot"])
    q = ((_rms(h @ w["dq"].T, eps) * w["dq.norm"]) @ w["uq"].T).view(T, H, d + dr)
    latent = h @ w["dkv"].T
    c, kr = _rms(latent[:, :r], eps) * w["dkv.norm"], _turn(latent[:, None, r:], freqs, mult)
    q = torch.cat([q[..., :d], _turn(q[..., d:], freqs, mult)], -1)
    k = torch.cat([(c @ w["uk"].T).view(T, H, d), kr.expand(T, H, dr)], -1)
    y = _softmax_heads(q, k, (c @ w["uv"].T).view(T, H, -1), torch.arange(T, device=h.device), m["scale"])
    return y @ w["o"].T, {"c": c, "kr": kr[:, 0]}


def _feed_forward(h, w, f):
    silu = torch.nn.functional.silu
    if f["kind"] == "dense":
        g, u = (h @ w["gate"].T).clamp(max=f["limit"]), (h @ w["up"].T).clamp(-f["limit"], f["limit"])
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w["down"].T
    r, z = f["router"], h @ w["router"].T
    E, groups = r["experts"], r.get("groups")
    scores = torch.sigmoid(z) if groups else torch.softmax(z, -1)
    choice = scores + w["correction"]
    if groups:  # the best groups of neighbouring experts first, each worth its two best
        worth = choice.view(len(h), groups["count"], -1).topk(2).values.sum(-1)
        kept = torch.zeros_like(worth, dtype=torch.bool).scatter_(1, worth.topk(groups["keep"]).indices, True)
        choice = choice.masked_fill(~kept.repeat_interleave(E // groups["count"], 1), -math.inf)
    idx = choice.topk(r["top"]).indices
    weight = torch.zeros_like(scores).scatter_(1, idx, scores.gather(1, idx) * r.get("scale", 1.0))
    out = weight[:, E:].sum(-1, keepdim=True) * h  # identity experts
    for e in range(E):
        rows = torch.where((idx == e).any(-1))[0]
        if len(rows):
            x = h[rows]
            y = (silu(x @ w[f"e{e}.gate"].T) * (x @ w[f"e{e}.up"].T)) @ w[f"e{e}.down"].T
            out[rows] += weight[rows, e, None] * y
    return out


def _sub(w, prefix):
    return {n[len(prefix):]: t for n, t in w.items() if n.startswith(prefix)}


def _mix(layer, h, w, eps, kv):
    """A layer's mixer on h (T, width): its output and, by their names, what its cache holds afterwards."""
    m, kind = layer["mixer"], layer["type"]
    if kind == "channel_delta":
        return _delta(h, w, m, eps, True)
    if kind == "parallel":
        (a, ca), (b, cb) = _sink_attention(h, _sub(w, "left."), m["left"], eps), _delta(h, _sub(w, "right."), m["right"], eps, False)
        return m["left_scale"] * a + m["right_scale"] * b, {**{"left." + n: t for n, t in ca.items()},
                                                            **{"right." + n: t for n, t in cb.items()}}
    if kind == "mamba2":
        return _scan(h, w, m, eps)
    if kind == "mingru":
        return _mingru(h, w)
    if kind == "latent_attention":
        return _latent_attention(h, w, m, eps)
    return _diff_attention(h, w, m, eps, kv) if "lq1" in w else _sigmoid_attention(h, w, m)


def _exact_sequence(d, w, tokens):
    """The last token's logits and what the layers' caches hold after one sequence from position 0."""
    eps, T, caches = d["norm"]["eps"], len(tokens), []
    x = w["embed"][torch.tensor(tokens, device=DEV)].to(F64)
    if d["architecture"] == "Ravelorn":
        x = x + w["pos"][:T].to(F64)
    if "loop" in d:
        x = x + w["loop.step"][0].to(F64)
    xs = [x] * d.get("streams", 1)
    for i, layer in enumerate(d["layers"]):
        lw = {n: t.to(F64) for n, t in _sub(w, f"l{i}.").items()}
        for q in (1, 2):
            def sub(h, q=q):
                if q == 2:
                    return _feed_forward(h, _sub(lw, "mlp."), layer["mlp"])
                src = layer["mixer"].get("kv_from")
                y, cache = _mix(layer, h, _sub(lw, "mix."), eps, None if src is None else caches[src])
                caches.append(cache)
                return y
            if d["architecture"] == "Ravelorn":
                y = torch.nn.functional.layer_norm(sub(xs[0]), x.shape[1:], lw[f"norm{q}"], lw[f"norm{q}.b"], eps)
                xs = [xs[0] + d["residual_mult"] * y]
            elif "streams" in d:
                read, write, mix = (lw[f"hc{q}.{n}"] for n in ("in", "out", "mix"))
                y = sub(_rms(sum(a * s for a, s in zip(read, xs)), eps) * lw[f"norm{q}"])
                xs = [sum(mix[j, t] * xs[j] for j in range(len(xs))) + write[t] * y for t in range(len(xs))]
            else:
                xs = [xs[0] + sub(_rms(xs[0], eps) * lw[f"norm{q}"])]
    x, norm = sum(xs)[-1], w["final.norm"].to(F64)
    if d["architecture"] == "Ravelorn":
        z = torch.nn.functional.layer_norm(x, x.shape, norm, w["final.norm.b"].to(F64), eps) @ w["head"].to(F64).T
        return d["logit_softcap"] * torch.tanh(z / d["logit_softcap"]), caches
    return (_rms(x, eps) * norm) @ w["head"].to(F64).T * d.get("logit_scale", 1.0), caches


def _exact_layered(case, seed):
    config, weights, prompts, new, room = _layered_inputs(case, seed)
    d, logits, out = _layered_config(case), [], {}
    for slot, tokens in enumerate(prompts):
        z, caches = _exact_sequence(d, weights, tokens + [new[slot]] if case["step"] == "decode" else tokens)
        logits.append(z)
        for i, (layer, cache) in enumerate(zip(d["layers"], caches)):
            if layer["mixer"].get("kv_from") is not None:
                continue
            for name, t in cache.items():
                by_token = name.rsplit(".", 1)[-1] in ("k", "v", "c", "kr")  # a row for every position
                shape = (len(prompts), room, *t.shape[1:]) if by_token else (len(prompts), *t.shape)
                whole = out.setdefault(f"{i}.{name}", torch.zeros(shape, dtype=F64, device=DEV))
                if by_token:
                    whole[slot, :len(t)] = t
                else:
                    whole[slot] = t
    return dict(out, logits=torch.stack(logits))


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    return _work_gpt(case) if case["family"] == "gpt" else _work_layered(case)


def _work_gpt(case):
    """Every matrix that is needed read once, the cached keys and values read and the new ones written once."""
    cfg, T, ctx = _gpt_config(case), case["tokens"], case["context"]
    C, inter, V = cfg.n_embd, cfg.intermediate_size, cfg.padded_vocab_size
    kv = 2 * cfg.n_query_groups * cfg.head_size
    each = {"bf16": 2.0, "fp32": 4.0, "int4-g128": 0.5 + 2 / 128, "nf4": 0.5 + 4 / 64}[case["weights"]]
    mats = {"GptNeoxMLP": 2, "LLaMAMLP": 3, "LLaMAMoE": 3}[cfg._mlp_class] * C * inter
    top, experts = (cfg.n_expert_per_token, cfg.n_expert) if cfg._mlp_class == "LLaMAMoE" else (1, 1)
    attn = C * (C + kv) + C * C
    pairs = T * ctx + T * (T + 1) / 2
    act = 4 if case["weights"] == "fp32" else 2
    return {"bytes": each * (cfg.n_layer * (attn + mats * min(experts, top * T)) + C * V) + cfg.n_layer * kv * act * (ctx + T),
            "flops": 2.0 * cfg.n_layer * T * (attn + mats * top) + 2.0 * C * V + cfg.n_layer * 4.0 * C * pairs}


def _work_layered(case):
    """Every matrix that a token needs read once (of the experts the chosen ones), the recurrent states read and written
    and the cached rows read and written once; two operations for every weight and token, the attention's score and value
    products over the visible pairs, a decay, an update and a read for every number of a recurrent state and token."""
    d = _layered_config(case)
    shapes = LayeredGPT.tensor_shapes(LayeredConfig.from_dict(d))
    lengths, decode = [int(n) for n in case["lengths"].split(",")], case["step"] == "decode"
    T, B = (len(lengths) if decode else sum(lengths)), len(lengths)
    dense = experts = 0
    for name, shape in shapes.items():
        if len(shape) == 2 and name not in ("embed", "pos", "head", "loop.step") and ".hc" not in name:
            n = shape[0] * shape[1]
            if ".mlp.e" in name:
                experts += n
            else:
                dense += n
    share = next((f["router"]["top"] / f["router"]["experts"] for f in (l["mlp"] for l in d["layers"]) if f["kind"] == "moe"), 0.0)
    flops = 2.0 * T * (dense + experts * share) + 2.0 * B * VOCAB * case["width"]
    nbytes = 2.0 * (dense + experts * min(1.0, share * T) + VOCAB * case["width"])
    for layer in d["layers"]:
        for m in ([layer["mixer"]["left"], layer["mixer"]["right"]] if "left" in layer["mixer"] else [layer["mixer"]]):
            if "scale" in m:
                size = (m.get("mask") or {}).get("size") or 1 << 30
                maps, G = (2 if "diff" in m else 1), m.get("kv_heads", 1)
                key, val = (m["kv_rank"] + m["rot_dim"], m["kv_rank"]) if "kv_rank" in m else (maps * m["dim"], m["vdim"])
                row = G * (key if "kv_rank" in m else key + val)
                per = (m["dim"] + m["rot_dim"] + m["vdim"]) if "kv_rank" in m else maps * (m["dim"] + val)
                for n in lengths:
                    seen = n % size + 1 if decode else sum((i % size) + 1 for i in range(n))
                    flops += 2.0 * m["heads"] * per * seen
                    nbytes += 2.0 * row * (seen if decode else n)
            elif "heads" in m:
                state = m["heads"] * m["vdim"] * m.get("state", m.get("dim", 0))
                flops += 6.0 * T * state
                nbytes += (8.0 if decode else 4.0) * B * state
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case.get("weights") == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    # bf16 operands: roundings that fall the other way, carried on by every layer
    return {"rel": 0.03 if case.get("layers", 0) > 8 else 0.02, "max": 0.8}
