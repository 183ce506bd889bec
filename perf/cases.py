"""The work this engine is measured on, through the calls a program makes: ``LLMEngine.generate``, and the step function
(``LLMEngine.runner.step``) with the sampler, as the replay tool, the C interface and ``tffinfer_amd.measure`` use them.

Four kinds of job:

* ``generate``  whole generations of a few prompts, greedy, logits kept: scheduler, graphs, sampler, tokens to the host;
* ``life``      requests from their prompts over some decode steps to their end, all prompts in the first step;
* ``decode``    a few decode steps of requests that hold their contexts (the state a server keeps between steps);
* ``mixed``     one step of continuous batching: portions of new prompts beside requests that decode.

Weights are random with the layers' usual scales: matrices of 0.02, those that write into the residual stream smaller, as
a deep model's are.  Two things make the results comparable between correct implementations, as they are for trained
models: the head prefers one next token clearly, and a token's topic stands in channels of the stream that the layers do
not write into and that the routers read, so that a choice of experts does not hang on rounding.

The Qwen3 sizes are the benchmark's.  The other designs are measured with their prompt and decode steps at the
benchmark's two widths; Rutevik and Gopuzen run on the kernels of these (latent attention, experts on tiles, linear
recurrences, windowed attention) and stand behind them.
"""
import math
import random

import torch

from tffinfer_amd import EngineOptions, LLMEngine, SamplingConfig
from tffinfer_amd.engine.batch import StepEntry
from tffinfer_amd.models import build_model_skeleton, config_from_dict

DEVICE = "cuda:0"
VOCAB = 151936
TOPICS = 64          # channels of the stream that hold a token's topic
TOPIC_SIZE = 8.0
EMBED_STD = 0.5
PASS_STEPS = 4       # decode steps of a pass of a ``decode`` job
ROOM = 4096          # tokens a decoding request may grow by before another takes its place

QWEN = {  # hidden, query heads, intermediate, tied head
    "0.6b": (1024, 16, 3072, True), "1.7b": (2048, 16, 6144, True), "4b": (2560, 32, 9728, True),
    "8b": (4096, 32, 12288, False), "14b": (5120, 40, 17408, False),
}
WIDTH = {"2k": 2048, "4k": 4096}


def listed():
    def case(name, job, design, size, layers, batch, tokens, spread=1, steps=0, portions=0, dtype="bfloat16", sampling="greedy"):
        return dict(name=name, job=job, design=design, size=size, layers=layers, batch=batch, tokens=tokens, spread=spread, steps=steps,
                    portions=portions, dtype=dtype, sampling=sampling)
    return [
        # one short question to a small model, answered token by token: launches and latency
        case("one_short_chat", "generate", "qwen3", "0.6b", 28, 1, 96, steps=16),
        # the benchmark's decode step: 8 requests of 2,048 tokens
        case("decode_8", "decode", "qwen3", "8b", 8, 8, 2048),
        # a busier server: 48 requests of very different lengths, tokens drawn from the top 50
        case("decode_48_ragged", "decode", "qwen3", "8b", 4, 48, 8192, spread=32, sampling="top50"),
        # a few short questions that arrive together, of lengths that fill no tile
        case("short_prompts", "life", "qwen3", "1.7b", 28, 3, 333, spread=4, steps=1),
        # the benchmark's prompt
        case("prompt_2048", "life", "qwen3", "8b", 8, 1, 2048, steps=1),
        # a long document
        case("prompt_16k", "life", "qwen3", "8b", 4, 1, 16384, steps=1),
        # a step of continuous batching: three portions of prompts beside 29 requests that decode
        case("portions_beside_decode", "mixed", "qwen3", "8b", 6, 29, 1100, spread=4, steps=500, portions=3),
        # the float32 path, which replays and comparisons run on
        case("float32_prompts", "life", "qwen3", "1.7b", 8, 2, 401, spread=2, steps=2, dtype="float32"),
        # a prompt and some decode steps of the other designs, alone and a few together
        case("disunex_prompt", "life", "disunex", "4k", 6, 1, 2048, steps=4),
        case("netovik_prompt", "life", "netovik", "4k", 6, 1, 1500, steps=4),
        case("sipilorn_few", "life", "sipilorn", "4k", 6, 4, 901, spread=3, steps=6),
        case("pupinex_pair", "life", "pupinex", "2k", 6, 2, 3001, spread=2, steps=4),
    ]


def _between(rng, lo, hi):
    """A whole number, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("generate", "decode", "decode", "prompts", "prompts", "mixed", "float32", "design", "design", "design", "design"))
    c = dict(design="qwen3", spread=rng.choice((1, 2, 4)), portions=0, dtype="bfloat16", sampling=rng.choice(("greedy", "top50")))
    if kind == "generate":
        c.update(job="generate", size=rng.choice(("0.6b", "1.7b")), layers=rng.randint(12, 28), batch=rng.randint(1, 4),
                 tokens=_between(rng, 16, 400), steps=rng.randint(8, 20), sampling="greedy")
    elif kind == "decode":
        batch = _between(rng, 1, 64)
        c.update(job="decode", size=rng.choice(("1.7b", "4b", "8b", "14b")), layers=rng.randint(3, 8), batch=batch,
                 tokens=_between(rng, 128, min(16384, 100000 // batch)), spread=rng.choice((1, 4, 32)), steps=0)
    elif kind == "prompts":
        batch = rng.randint(1, 4)
        c.update(job="life", size=rng.choice(("0.6b", "1.7b", "4b", "8b", "14b")), layers=rng.randint(3, 8), batch=batch,
                 tokens=_between(rng, 20, 12000 // batch), steps=rng.randint(1, 3))
    elif kind == "mixed":
        c.update(job="mixed", size=rng.choice(("4b", "8b", "14b")), layers=rng.randint(3, 6), batch=rng.randint(4, 60),
                 tokens=_between(rng, 128, 2000), steps=_between(rng, 60, 700), portions=rng.randint(1, 4))
    elif kind == "float32":
        c.update(job="life", size=rng.choice(("0.6b", "1.7b", "4b")), layers=rng.randint(3, 8), batch=rng.randint(1, 3),
                 tokens=_between(rng, 20, 700), steps=rng.randint(1, 3), dtype="float32")
    else:
        batch = rng.randint(1, 6)
        c.update(job="life", design=rng.choice(("disunex", "netovik", "sipilorn", "pupinex")), size=rng.choice(("2k", "4k")),
                 layers=rng.randint(3, 6), batch=batch, tokens=_between(rng, 40, 4000 // batch), steps=rng.randint(2, 6), sampling="greedy")
    return c


# ---- configurations and tensors -------------------------------------------------------------------------------------
# A tensor is (shape, law): "matrix" and "out" (into the stream) are random matrices, "head" and "embed" the token tables,
# "router" scores over topics, "norm" lies around one, "offset" around zero, "vector" enters scores, the rest is named
# for what it is.

def _qwen3(c):
    W, H, ff, tied = QWEN[c["size"]]
    cfg = dict(architectures=["Qwen3ForCausalLM"], hidden_size=W, num_hidden_layers=c["layers"], num_attention_heads=H, num_key_value_heads=8,
               head_dim=128, intermediate_size=ff, vocab_size=VOCAB, max_position_embeddings=32768, rms_norm_eps=1e-6,
               rope_theta=1000000.0, tie_word_embeddings=tied)
    t = {"model.embed_tokens.weight": ((VOCAB, W), "embed"), "model.norm.weight": ((W,), "norm")}
    if not tied:
        t["lm_head.weight"] = ((VOCAB, W), "head")
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        for n, s, law in (("input_layernorm", (W,), "norm"), ("post_attention_layernorm", (W,), "norm"),
                          ("self_attn.q_proj", (H * 128, W), "matrix"), ("self_attn.k_proj", (1024, W), "matrix"),
                          ("self_attn.v_proj", (1024, W), "matrix"), ("self_attn.o_proj", (W, H * 128), "out"),
                          ("self_attn.q_norm", (128,), "norm"), ("self_attn.k_norm", (128,), "norm"),
                          ("mlp.gate_proj", (ff, W), "matrix"), ("mlp.up_proj", (ff, W), "matrix"), ("mlp.down_proj", (W, ff), "out")):
            t[p + n + ".weight"] = (s, law)
    return cfg, t


def _experts(t, p, E, ff, W, names):
    for e in range(E):
        for n in names:
            t[f"{p}e{e}.{n}"] = ((W, ff), "out") if n == "down" else ((ff, W), "matrix")


def _disunex(c):
    W = WIDTH[c["size"]]
    big = W == 4096
    H, dim, rot, vd, R = (32, 128, 64, 128, 192) if big else (16, 64, 32, 64, 96)
    ff, E, top, eff = (18432, 32, 4, 1536) if big else (9216, 16, 2, 1024)
    m = {"heads": H, "dim": dim, "rot_dim": rot, "vdim": vd, "kv_rank": R, "scale": (dim + rot) ** -0.5, "mask": {"size": 1024},
         "rot": {"base": 1000000.0, "dims": rot}}
    mlps = [{"kind": "dense", "ff": ff}, {"kind": "moe", "expert": {"ff": eff, "limit": 7.0}, "router": {"experts": E, "top": top}}]
    cfg = {"architecture": "Disunex", "width": W, "vocab": VOCAB, "postln_alpha": 1.0, "norm": {"eps": 1e-6},
           "layers": [{"type": "latent_attention", "mixer": m, "mlp": mlps[i % 2]} for i in range(c["layers"])]}
    t = {"embed": ((VOCAB, W), "embed"), "final.norm": ((W,), "offset")}
    for i in range(c["layers"]):
        p = f"l{i}."
        t.update({p + "norm1": ((W,), "offset"), p + "norm2": ((W,), "offset"), p + "mix.q": ((H * (dim + rot), W), "matrix"),
                  p + "mix.dkv": ((R + rot, W), "matrix"), p + "mix.dkv.norm": ((R,), "norm"), p + "mix.uk": ((H * dim, R), "matrix"),
                  p + "mix.uv": ((H * vd, R), "matrix"), p + "mix.o": ((W, H * vd), "out"), p + "mix.sink": ((H,), "vector"),
                  p + "mix.g": ((H * vd, W), "matrix")})
        if i % 2 == 0:
            t.update({p + "mlp.up": ((ff, W), "matrix"), p + "mlp.down": ((W, ff), "out")})
        else:
            t.update({p + "mlp.router": ((E, W), "router"), p + "mlp.correction": ((E,), "zero")})
            _experts(t, p + "mlp.", E, eff, W, ("gate", "up", "down"))
    return cfg, t


def _netovik(c):
    W = WIDTH[c["size"]]
    big = W == 4096
    wh, wd, H, G, D = (64, 64, 32, 8, 128) if big else (32, 64, 16, 4, 128)
    ff, E, top, eff = (12288, 32, 4, 1536) if big else (6144, 16, 2, 1024)
    rec = {"type": "wkv", "mixer": {"heads": wh, "dim": wd, "decay_rank": 64}}
    att = {"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "softcap": 30.0, "bias_max": 512,
                                          "bias_buckets": 32, "mask": {"size": 1024, "keep_first": 4}}}
    mlps = [{"kind": "dense", "ff": ff}, {"kind": "moe", "expert": {"ff": eff}, "router": {"experts": E, "top": top}}]
    cfg = {"architecture": "Netovik", "width": W, "vocab": VOCAB, "norm": {"eps": 1e-6, "groups": 2}, "embedding": {"scale": 0.5},
           "layers": [dict(att if i % 3 == 2 else rec, mlp=mlps[i % 2]) for i in range(c["layers"])]}
    t = {"embed": ((VOCAB, W), "embed"), "final.norm": ((W,), "norm")}
    for i in range(c["layers"]):
        p = f"l{i}."
        t.update({p + "dwa": ((i + 2,), "depth"), p + "norm1": ((W,), "small_norm"), p + "norm2": ((W,), "small_norm")})
        m = p + "mix."
        if i % 3 == 2:
            t.update({m + "q": ((H * D, W), "matrix"), m + "k": ((G * D, W), "matrix"), m + "o": ((W, H * D), "out"), m + "q.b": ((H * D,), "vector"),
                      m + "k.b": ((G * D,), "vector"), m + "rel": ((32, H), "vector"), m + "talk": ((H, H), "talk")})
        else:
            t.update({m + "mu." + s: ((W,), "unit") for s in "rkvgw"})
            t.update({m + s: ((wh * wd, W), "matrix") for s in "rkvg"})
            t.update({m + "w1": ((64, W), "matrix"), m + "w2": ((wh * wd, 64), "matrix"), m + "w0": ((wh * wd,), "decay"), m + "u": ((wh, wd), "vector"),
                      m + "norm": ((wh * wd,), "norm"), m + "o": ((W, wh * wd), "out")})
        if i % 2 == 0:
            t.update({p + "mlp.gate": ((ff, W), "matrix"), p + "mlp.up": ((ff, W), "matrix"), p + "mlp.down": ((W, ff), "out")})
        else:
            t[p + "mlp.router"] = ((E, W), "router")
            _experts(t, p + "mlp.", E, eff, W, ("gate", "up", "down"))
    return cfg, t


def _delta_tensors(t, m, H, G, D, W):
    t.update({m + "q": ((G * D, W), "matrix"), m + "k": ((G * D, W), "matrix"), m + "v": ((H * D, W), "matrix"), m + "g": ((H * D, W), "matrix"),
              m + "o": ((W, H * D), "out"), m + "b": ((H, W), "matrix"), m + "a": ((H, W), "matrix"), m + "A_log": ((H,), "decay"),
              m + "dt_bias": ((H,), "vector"), m + "norm": ((D,), "norm"), m + "q.conv": ((G * D, 4), "vector"), m + "k.conv": ((G * D, 4), "vector"),
              m + "v.conv": ((H * D, 4), "vector")})


def _sipilorn(c):
    W = WIDTH[c["size"]]
    big = W == 4096
    DH, DG, H, G, D, PH = (32, 16, 32, 8, 128, 8) if big else (16, 8, 16, 4, 128, 4)
    ff, E, top, eff = (12288, 32, 4, 3072) if big else (6144, 16, 2, 2048)
    rec = {"type": "delta", "mixer": {"heads": DH, "kv_heads": DG, "dim": D, "vdim": D, "conv": 4}}
    par = {"type": "parallel", "mixer": {
        "left": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": 1024}, "rot": {"dims": D // 2, "base": 1000000.0}},
        "right": {"heads": PH, "kv_heads": PH, "dim": D, "vdim": D, "conv": 4}, "left_scale": 1.0, "right_scale": 1.0}}
    mlps = [{"kind": "dense", "ff": ff}, {"kind": "moe", "expert": {"ff": eff}, "router": {"experts": E, "top": top}}]
    cfg = {"architecture": "Sipilorn", "width": W, "vocab": VOCAB, "norm": {"eps": 1e-6}, "logit_softcap": 30.0,
           "layers": [dict(par if i % 3 == 2 else rec, mlp=mlps[i % 2]) for i in range(c["layers"])]}
    t = {"embed": ((VOCAB, W), "embed"), "embed.norm": ((W,), "norm"), "final.norm": ((W,), "norm"), "head": ((VOCAB, W), "head")}
    for i in range(c["layers"]):
        p = f"l{i}."
        t.update({p + "norm1": ((W,), "norm"), p + "norm2": ((W,), "norm")})
        if i % 3 == 2:
            m = p + "mix.left."
            t.update({m + "q": ((H * D, W), "matrix"), m + "k": ((G * D, W), "matrix"), m + "v": ((G * D, W), "matrix"), m + "g": ((H * D, W), "matrix"),
                      m + "o": ((W, H * D), "out"), m + "q.norm": ((D,), "norm"), m + "k.norm": ((D,), "norm")})
            _delta_tensors(t, p + "mix.right.", PH, PH, D, W)
        else:
            _delta_tensors(t, p + "mix.", DH, DG, D, W)
        if i % 2 == 0:
            t.update({p + "mlp.gate": ((ff, W), "matrix"), p + "mlp.up": ((ff, W), "matrix"), p + "mlp.down": ((W, ff), "out")})
        else:
            t[p + "mlp.table"] = ((VOCAB, top), "table")
            _experts(t, p + "mlp.", E, eff, W, ("up", "down"))
    return cfg, t


def _pupinex(c):
    W = WIDTH[c["size"]]
    big = W == 4096
    H, G, D, gh, gd, gv, rh = (32, 8, 128, 16, 128, 256, 16) if big else (16, 4, 128, 8, 128, 256, 8)
    ff, E, top, groups, keep, eff = (12288, 32, 4, 8, 4, 1536) if big else (6144, 16, 2, 4, 2, 1536)

    def att(base):
        return {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": 1024}, "rot": {"base": base, "dims": D}}
    left = att(50000.0)
    left["rot"]["scaling"] = {"factor": 8.0}
    kinds = [{"type": "attention", "mixer": att(10000.0)},
             {"type": "gla", "mixer": {"heads": gh, "dim": gd, "vdim": gv, "tau": 16.0, "decay_rank": 16}},
             {"type": "parallel", "mixer": {"left": left, "left_scale": 0.5, "right_scale": 0.5,
                                            "right": {"heads": rh, "dim": D, "vdim": D, "gate_cap": 15.0}}}]
    mlps = [{"kind": "dense", "ff": ff, "limit": 7.0},
            {"kind": "moe", "expert": {"ff": eff}, "shared": {"ff": eff},
             "router": {"experts": E, "top": top, "groups": {"count": groups, "keep": keep}, "scale": 2.5}}]
    cfg = {"architecture": "Pupinex", "width": W, "vocab": VOCAB, "norm": {"eps": 1e-5},
           "embedding": {"bigram": {"buckets": 65521, "mul_prev": 1009, "mul_cur": 31}},
           "layers": [dict(kinds[i % 3], mlp=mlps[i % 2]) for i in range(c["layers"])]}
    t = {"embed": ((VOCAB, W), "embed"), "bigram": ((65522, W), "pairs"), "final.norm": ((W,), "norm")}
    for i in range(c["layers"]):
        p = f"l{i}."
        t.update({p + "norm1": ((W,), "norm"), p + "norm2": ((W,), "norm")})
        if i % 3 != 1:
            m = p + ("mix." if i % 3 == 0 else "mix.left.")
            t.update({m + "q": ((H * D, W), "matrix"), m + "k": ((G * D, W), "matrix"), m + "v": ((G * D, W), "matrix"), m + "o": ((W, H * D), "out"),
                      m + "q.b": ((H * D,), "offset"), m + "k.b": ((G * D,), "offset"), m + "v.b": ((G * D,), "offset")})
            if i % 3 == 0:
                t.update({m + "o.b": ((W,), "out_bias"), m + "sink": ((H,), "vector")})
            else:
                t.update({m + "q.norm": ((H * D,), "norm"), m + "k.norm": ((G * D,), "norm")})
                r = p + "mix.right."
                t.update({r + s: ((rh * D, W), "matrix") for s in "qkvg"})
                t.update({r + "i": ((rh, W), "matrix"), r + "f": ((rh, W), "matrix"), r + "i.b": ((rh,), "vector"), r + "f.b": ((rh,), "vector"),
                          r + "norm": ((rh * D,), "norm"), r + "o": ((W, rh * D), "out")})
        else:
            m = p + "mix."
            t.update({m + "q": ((gh * gd, W), "matrix"), m + "k": ((gh * gd, W), "matrix"), m + "v": ((gh * gv, W), "matrix"),
                      m + "g": ((gh * gv, W), "matrix"), m + "a1": ((16, W), "matrix"), m + "a2": ((gh * gd, 16), "matrix"),
                      m + "a2.b": ((gh * gd,), "vector"), m + "norm": ((gv,), "norm"), m + "o": ((W, gh * gv), "out")})
        f = p + "mlp."
        if i % 2 == 0:
            t.update({f + "gate": ((ff, W), "matrix"), f + "up": ((ff, W), "matrix"), f + "down": ((W, ff), "out")})
        else:
            t.update({f + "router": ((E, W), "router"), f + "shared.sg": ((1, W), "matrix"), f + "shared.gate": ((eff, W), "matrix"),
                      f + "shared.up": ((eff, W), "matrix"), f + "shared.down": ((W, eff), "out")})
            _experts(t, f, E, eff, W, ("gate", "up", "down"))
    return cfg, t


DESIGNS = {"qwen3": _qwen3, "disunex": _disunex, "netovik": _netovik, "sipilorn": _sipilorn, "pupinex": _pupinex}


def _router_of(case, cfg):
    return next(m["mlp"]["router"] for m in cfg["layers"] if m["mlp"]["kind"] == "moe")


def _router(shape, router, g):
    """Scores over topics [experts, width]: of sixteen candidates a topic, the one whose choice of experts is clearest."""
    E = shape[0]
    s = torch.randn(16, TOPICS, E, generator=g, device=DEVICE)
    groups = router.get("groups")
    allowed = s
    gap = torch.full(s.shape[:2], math.inf, device=DEVICE)
    if groups:
        by = s.view(16, TOPICS, groups["count"], -1).sort(-1, descending=True).values[..., :2].sum(-1).sort(-1, descending=True)
        gap = by.values[..., groups["keep"] - 1] - by.values[..., groups["keep"]]
        kept = torch.zeros(16, TOPICS, groups["count"], dtype=torch.bool, device=DEVICE).scatter_(2, by.indices[..., :groups["keep"]], True)
        allowed = s.masked_fill(~kept.repeat_interleave(E // groups["count"], -1), -math.inf)
    top = allowed.sort(-1, descending=True).values
    gap = torch.minimum(gap, top[..., router["top"] - 1] - top[..., router["top"]])
    best = s[gap.argmax(0), torch.arange(TOPICS, device=DEVICE)]
    w = torch.zeros(shape, device=DEVICE)
    w[:, :TOPICS] = 0.2 * best.T
    return w


def _weights(case, seed):
    """Every tensor of the model as a file would hold it: matrices in bfloat16, vectors in float32."""
    cfg, tensors = DESIGNS[case["design"]](case)
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    out = {}
    for name, (shape, law) in tensors.items():
        if law == "table":
            order = torch.rand(shape[0], _router_of(case, cfg)["experts"], generator=g, device=DEVICE).argsort(1)
            out[name] = order[:, :shape[1]].to(torch.int32).contiguous()
            continue
        if law == "router":
            out[name] = _router(shape, _router_of(case, cfg), g).bfloat16()
            continue
        draws = torch.rand if law in ("unit", "decay") else torch.randn
        x = draws(shape, generator=g, device=DEVICE)
        if law == "matrix":
            x = (0.02 * x).bfloat16()
        elif law == "out":
            x *= 0.005
            x[:TOPICS] = 0
            x = x.bfloat16()
        elif law in ("embed", "pairs"):
            x *= EMBED_STD if law == "embed" else 0.2
            x[:, :TOPICS] = 0
            if law == "embed":
                rows = torch.arange(shape[0], device=DEVICE)
                x[rows, rows % TOPICS] = TOPIC_SIZE
            x = x.bfloat16()
        elif law == "head":      # each id is what its predecessor asks for
            x = (0.02 * x).bfloat16()
            x += 0.03 * out["embed" if "embed" in out else "model.embed_tokens.weight"].roll(1, 0)
        elif law == "norm":
            x = 1.0 + 0.1 * x
        elif law == "small_norm":
            x = 0.3 + 0.03 * x
        elif law == "offset":
            x *= 0.1
        elif law == "out_bias":
            x *= 0.05
            x[:TOPICS] = 0
        elif law == "vector":
            x *= 0.5
        elif law == "decay":
            x = 3.5 * x - 3.0
        elif law == "zero":
            x = torch.zeros_like(x)
        elif law == "talk":
            x = torch.eye(shape[0], device=DEVICE) + 0.1 * x
        elif law == "depth":
            x *= 0.1
            x[-1] += 1.0
        out[name] = x
    return cfg, out


# ---- inputs and passes ----------------------------------------------------------------------------------------------

def _lengths(case):
    """Lengths of the requests' contexts: the longest first, the others down to 1 / spread of it."""
    if case["spread"] == 1 or case["batch"] == 1:
        return [case["tokens"]] * case["batch"]
    r = random.Random(case["batch"] * 1000003 + case["tokens"])
    return [case["tokens"]] + [max(2, int(case["tokens"] * case["spread"] ** -r.random())) for _ in range(case["batch"] - 1)]


def _ids(seed, n, salt):
    """n token ids; few are used often, most seldom."""
    r = random.Random(int(seed) * 7919 + salt)
    return [min(VOCAB - 1, int(VOCAB * r.random() ** 2)) for _ in range(n)]


def _inputs(case, seed):
    """(the requests' contexts, the tokens that follow each one, new prompts of a mixed step)"""
    contexts = [_ids(seed, n, i) for i, n in enumerate(_lengths(case))]
    following = [_ids(seed, 64, 10000 + i) for i in range(case["batch"])]
    portions = [_ids(seed, case["steps"], 20000 + i) for i in range(case["portions"])]
    return contexts, following, portions


def _sampling(case):
    if case["sampling"] == "greedy":
        return [SamplingConfig()] * case["batch"]
    return [SamplingConfig("random", temperature=0.8, top_k=50, top_p=0.95, seed=i) for i in range(case["batch"])]


def _fill(engine, requests):
    """The contexts of the requests into the cache, some thousand tokens a step."""
    step, n = [], 0
    for rid, tokens in requests:
        engine.runner.add_request(rid)
        for at in range(0, len(tokens), 4096):
            part = tokens[at:at + 4096]
            if step and (n + len(part) > 8192 or at):
                engine.runner.step(step)
                step, n = [], 0
            step.append(StepEntry(rid, part))
            n += len(part)
    if step:
        engine.runner.step(step)


def prepare(case, seed):
    cfg, tensors = _weights(case, seed)
    model = build_model_skeleton(config_from_dict(cfg))
    dtype = {"bfloat16": torch.bfloat16, "float32": torch.float32}[case["dtype"]]
    model.load_tensors(tensors, dtype, DEVICE)
    del tensors
    contexts, following, portions = _inputs(case, seed)
    room = (ROOM if case["job"] in ("decode", "mixed") else case["steps"]) + 32
    total = sum(map(len, contexts)) + sum(map(len, portions)) + (room + 16) * (len(contexts) + len(portions))
    engine = LLMEngine(model, EngineOptions(
        dtype=case["dtype"], device=DEVICE, max_num_seqs=len(contexts) + len(portions), kv_tokens=total,
        max_model_len=max(map(len, contexts + portions)) + room, max_num_batched_tokens=max(8192, sum(map(len, contexts)) if case["job"] == "life" else 0)))
    engine.keep_logits = case["job"] == "generate"
    state = dict(case=case, engine=engine, contexts=contexts, following=following, portions=portions, sampling=_sampling(case), done=0)
    if case["job"] in ("decode", "mixed"):
        _fill(engine, list(enumerate(contexts)))
    return state


def _step(state, ids, n, outputs, more=()):
    """One step of the step function with the sampler behind it; ``ids[r]`` are request r's tokens."""
    engine = state["engine"]
    entries = [StepEntry(r, toks, [len(toks) - 1]) for r, toks in enumerate(ids)] + list(more)
    logits = engine.runner.step(entries)
    outputs.append(logits.clone())      # (the next step overwrites them)
    outputs.append(engine.sampler.sample_on_device(logits[:len(ids)], state["sampling"], [n] * len(ids)))


def run(state):
    case, engine = state["case"], state["engine"]
    outputs = []
    if case["job"] == "generate":
        for r in engine.generate(state["contexts"], SamplingConfig(), max_new_tokens=case["steps"], ignore_eos=True):
            outputs += [torch.tensor(r.output), torch.stack(r.logits)]
    elif case["job"] == "life":
        for r in range(case["batch"]):
            engine.runner.add_request(r)
        _step(state, state["contexts"], 0, outputs)
        for n in range(case["steps"]):
            _step(state, [f[n:n + 1] for f in state["following"]], n + 1, outputs)
        for r in range(case["batch"]):
            engine.runner.free_request(r)
    else:
        if state["done"] + PASS_STEPS > ROOM:       # the requests have ended, others of the same lengths follow
            for r in range(case["batch"]):
                engine.runner.free_request(r)
            _fill(engine, list(enumerate(state["contexts"])))
            state["done"] = 0
        new = []
        for p, toks in enumerate(state["portions"]):
            engine.runner.add_request(("portion", p))
            new.append(StepEntry(("portion", p), toks, [len(toks) - 1]))
        for n in range(1 if new else PASS_STEPS):
            k = state["done"]
            _step(state, [[f[k % 64]] for f in state["following"]], k, outputs, new)
            state["done"] += 1
        for p in range(len(state["portions"])):
            engine.runner.free_request(("portion", p))
    return outputs


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _steps(case):
    """The steps of a pass: per step the requests' (new tokens, tokens before them), and how many logit rows."""
    lens = _lengths(case)
    if case["job"] in ("life", "generate"):
        steps = [[(n, 0) for n in lens]]
        more = case["steps"] if case["job"] == "life" else case["steps"] - 1
        return steps + [[(1, n + k) for n in lens] for k in range(more)]
    if case["job"] == "mixed":
        return [[(1, n) for n in lens] + [(case["steps"], 0)] * case["portions"]]
    return [[(1, n + k) for n in lens] for k in range(PASS_STEPS)]


def _mixer_costs(case, cfg):
    """Per layer: (flops a query and key, elements a cached key, window or 0, elements of state a request, flops of it a token)"""
    if case["design"] == "qwen3":
        H = cfg["num_attention_heads"]
        return [(4 * H * 128, 2 * 8 * 128, 0, 0, 0)] * case["layers"]
    out = []
    for L in cfg["layers"]:
        m, cost = L["mixer"], [0, 0, 0, 0, 0]
        for part in ([m["left"], m["right"]] if L["type"] == "parallel" else [m]):
            if "kv_rank" in part:
                cost[:3] = [2 * part["heads"] * (part["dim"] + part["rot_dim"] + part["vdim"]), part["kv_rank"] + part["rot_dim"], 1024]
            elif "mask" in part:
                keys = part["kv_heads"] * part["dim"] * (1 if case["design"] == "netovik" else 2)
                cost[:3] = [2 * part["heads"] * 2 * part["dim"] + (2 * part["heads"] ** 2 if "softcap" in part else 0), keys, 1024]
            else:
                n = part["heads"] * part["dim"] * part.get("vdim", part["dim"])
                cost[3:] = [n, 6 * n]
        out.append(cost)
    return out


def work(case):
    cfg, tensors = DESIGNS[case["design"]](case)
    size = 2 if case["dtype"] == "bfloat16" else 4
    dense, experts, head = 0, 0, 0
    for name, (shape, law) in tensors.items():
        if law in ("matrix", "out", "router", "head", "embed") and len(shape) == 2:
            n = shape[0] * shape[1]
            if law == "head" or (law == "embed" and not any(x == "head" for _, x in tensors.values())):
                head = n
            elif ".mlp.e" in name:
                experts += n
            elif law != "embed":
                dense += n
    router = _router_of(case, cfg) if experts else {"experts": 1, "top": 1}
    E, top = router["experts"], router["top"]
    width = cfg.get("hidden_size") or cfg["width"]
    nbytes = flops = 0.0
    for step in _steps(case):
        T, R = sum(n for n, _ in step), len(step)
        used = E * (1 - (1 - top / E) ** T)         # experts that some token of the step chooses
        nbytes += size * (dense + experts * used / E + head + T * width) + 4.0 * R * VOCAB
        flops += 2.0 * T * (dense + experts * top / E) + 2.0 * R * head
        for per_pair, per_key, window, state, per_token in _mixer_costs(case, cfg):
            for n, before in step:
                seen = [min(before + i + 1, window or 1 << 40) for i in (0, n - 1)]
                grows = seen[1] - seen[0]           # the first of the tokens see one key more each, the others a window's worth
                pairs = grows * (seen[0] + seen[1]) / 2 + (n - grows) * seen[1]
                flops += per_pair * pairs + per_token * n
                nbytes += size * per_key * (min(before, window or before) + n) + 8.0 * state
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Logits; the tokens are whole numbers with clear margins.  Measured against 64 bits: float32 0.8e-6 to 1.9e-6, bfloat16
    # 0.002 to 0.009 (activations are rounded between the layers), the largest single difference some ten times as much.
    return {"rel": 8e-6, "max": 1e-4, "differ": 0.0} if case["dtype"] == "float32" else {"rel": 0.03, "max": 0.3, "differ": 0.0}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------

def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, dims, base, pairs, slower=1.0):
    """x [T, heads, D]: the first ``dims`` elements in pairs (2i, 2i + 1), or (i, i + dims / 2), by position * base^(-2i / dims)."""
    T, half = x.shape[0], dims // 2
    a = torch.arange(T, dtype=torch.float64, device=x.device)[:, None] * (
        base ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dims) / slower)
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if pairs else (x[..., :half], x[..., half:dims])
    a, b = u * c - v * s, v * c + u * s
    y = torch.stack((a, b), -1).flatten(-2) if pairs else torch.cat((a, b), -1)
    return torch.cat((y, x[..., dims:]), -1)


def _attend(q, k, v, scale, window=0, sink=None, mix=None, keep=0):
    """q [T, H, D], k [T, G, D], v [T, G, E], causal; ``sink`` [H]: a logit without a value; ``mix``: what becomes of the raw
    scores [H, queries, keys] given the first query's position."""
    T, H, _ = q.shape
    G, out = k.shape[1], []
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    for at in range(0, T, 512):
        n = min(512, T - at)
        lo = max(0, at - window + 1) if window and not keep else 0
        i = torch.arange(at, at + n, device=q.device)[:, None]
        j = torch.arange(lo, at + n, device=q.device)[None]
        sees = (j <= i) & ((i - j < window) | (j < keep) if window else True)
        qs = q[at:at + n].reshape(n, G, H // G, -1).permute(1, 2, 0, 3).reshape(G, H // G * n, -1).contiguous()
        s = (qs @ kt[:, :, lo:at + n].contiguous()).reshape(H, n, -1) * scale
        if mix is not None:
            s = mix(s, at)
        s = s.masked_fill(~sees, -math.inf)
        if sink is not None:
            s = torch.cat((s, sink[:, None, None].expand(H, n, 1)), -1)
        p = torch.softmax(s, -1)[..., :at + n - lo].reshape(G, H // G * n, -1).contiguous()
        out.append((p @ vt[:, lo:at + n].contiguous()).reshape(G, H // G, n, -1).permute(2, 0, 1, 3).reshape(n, -1))
    return torch.cat(out)


class _Sub:
    """The tensors whose names begin with a prefix, in 64 bits when asked for."""

    def __init__(self, W, prefix=""):
        self.W, self.prefix = W, prefix

    def __call__(self, name):
        t = self.W[self.prefix + name]
        return t.double() if t.is_floating_point() else t.long()

    def __contains__(self, name):
        return self.prefix + name in self.W

    def sub(self, prefix):
        return _Sub(self.W, self.prefix + prefix)

    def times(self, x, name):
        y = x @ self(name).T
        return y + self(name + ".b") if name + ".b" in self else y


def _exact_qwen3(cfg, W, tokens, last):
    eps, H, P = cfg["rms_norm_eps"], cfg["num_attention_heads"], _Sub(W, "model.")
    x = W["model.embed_tokens.weight"][tokens].double()
    T = len(tokens)
    for i in range(cfg["num_hidden_layers"]):
        L = P.sub(f"layers.{i}.")
        h = _unit(x, eps) * L("input_layernorm.weight")
        q, k, v = (L.times(h, f"self_attn.{n}_proj.weight").view(T, -1, 128) for n in "qkv")
        q, k = (_turn(_unit(y, eps) * L(f"self_attn.{n}_norm.weight"), 128, cfg["rope_theta"], False) for y, n in ((q, "q"), (k, "k")))
        x = x + L.times(_attend(q, k, v, 128 ** -0.5), "self_attn.o_proj.weight")
        h = _unit(x, eps) * L("post_attention_layernorm.weight")
        x = x + L.times(_silu(L.times(h, "mlp.gate_proj.weight")) * L.times(h, "mlp.up_proj.weight"), "mlp.down_proj.weight")
    head = W["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"]
    return (_unit(x[-last:], eps) * P("norm.weight")) @ head.double().T


def _chosen(P, h, idx, w, expert):
    """The sum of the chosen experts' outputs; idx, w [T, top]."""
    out = torch.zeros_like(h)
    for e in range(int(idx.max()) + 1):
        t, k = (idx == e).nonzero(as_tuple=True)
        if len(t):
            out.index_add_(0, t, w[t, k][:, None] * expert(P.sub(f"e{e}."), h[t]))
    return out


def _gated(P, h):
    return P.times(_silu(P.times(h, "gate")) * P.times(h, "up"), "down")


def _clamped(P, h, limit):
    g, u = P.times(h, "gate").clamp(max=limit), P.times(h, "up").clamp(-limit, limit)
    return P.times(g * torch.sigmoid(1.702 * g) * (u + 1.0), "down")


def _exact_disunex(cfg, W, tokens, last):
    eps, T, P = cfg["norm"]["eps"], len(tokens), _Sub(W)
    x = P("embed")[tokens]
    for i, L in enumerate(cfg["layers"]):
        m, A, F = L["mixer"], P.sub(f"l{i}.mix."), P.sub(f"l{i}.mlp.")
        H, dim, rd, vd, R = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        q, kv = A.times(x, "q").view(T, H, dim + rd), A.times(x, "dkv")
        c = _unit(kv[:, :R], eps) * A("dkv.norm")
        kr = _turn(kv[:, None, R:], rd, m["rot"]["base"], True).expand(T, H, rd)
        k = torch.cat((A.times(c, "uk").view(T, H, dim), kr), -1)
        q = torch.cat((q[..., :dim], _turn(q[..., dim:], rd, m["rot"]["base"], True)), -1)
        o = _attend(q, k, A.times(c, "uv").view(T, H, vd), m["scale"], m["mask"]["size"], A("sink"))
        x = _unit(x + A.times(o * torch.sigmoid(A.times(x, "g")), "o"), eps) * (1.0 + P(f"l{i}.norm1"))
        if L["mlp"]["kind"] == "dense":
            f = F.times(torch.nn.functional.gelu(F.times(x, "up")), "down")
        else:
            s = torch.sigmoid(F.times(x, "router"))
            idx = (s + F("correction")).topk(L["mlp"]["router"]["top"], -1).indices
            w = s.gather(1, idx)
            f = _chosen(F, x, idx, w / (w.sum(-1, keepdim=True) + 1e-20), lambda E, h: _clamped(E, h, L["mlp"]["expert"]["limit"]))
        x = _unit(x + f, eps) * (1.0 + P(f"l{i}.norm2"))
    return (_unit(x[-last:], eps) * (1.0 + P("final.norm"))) @ P("embed").T


def _exact_netovik(cfg, W, tokens, last):
    eps, T, P = cfg["norm"]["eps"], len(tokens), _Sub(W)

    def group_norm(x, w):
        return _unit(x.reshape(len(x), cfg["norm"]["groups"], -1), eps).reshape(len(x), -1) * w

    def bucket(n, B, most):
        return n if n < B // 2 else min(B - 1, B // 2 + int(math.floor(math.log(n / (B // 2)) / math.log(most / (B // 2)) * (B - B // 2))))

    def mixer(L, A, x):
        m = L["mixer"]
        H, D = m["heads"], m["dim"]
        if L["type"] == "wkv":
            before = torch.cat((torch.zeros_like(x[:1]), x[:-1]))
            mix = {s: x + (before - x) * A("mu." + s) for s in "rkvgw"}
            r, k, v = (A.times(mix[s], s).view(T, H, D) for s in "rkv")
            w = torch.exp(-torch.exp(torch.tanh(A.times(mix["w"], "w1")) @ A("w2").T + A("w0"))).view(T, H, D)
            S, o, u = torch.zeros(H, D, D, dtype=x.dtype, device=x.device), [], A("u")[:, :, None]
            for t in range(T):
                kv = k[t, :, :, None] * v[t, :, None]
                o.append((r[t, :, :, None] * (S + u * kv)).sum(1))
                S = w[t, :, :, None] * S + kv
            return A.times(_unit(torch.stack(o), eps).reshape(T, -1) * A("norm") * _silu(A.times(mix["g"], "g")), "o")
        q, k = A.times(x, "q").view(T, H, D), A.times(x, "k").view(T, m["kv_heads"], D)
        rel, talk, cap, B = A("rel"), A("talk"), m["softcap"], m["bias_buckets"]
        bias = rel[torch.tensor([bucket(n, B, m["bias_max"]) for n in range(T)], device=x.device)]      # [distance, H]

        def scores(s, at):
            i = torch.arange(at, at + s.shape[1], device=x.device)[:, None]
            d = (i - torch.arange(s.shape[2], device=x.device)[None]).clamp(min=0)
            s = cap * torch.tanh(s / cap) + bias[d].permute(2, 0, 1)
            return (talk @ s.reshape(H, -1)).view_as(s)
        sink = torch.zeros(H, dtype=x.dtype, device=x.device)       # (the one in the softmax's denominator)
        o = _attend(_unit(q, eps), _unit(k, eps), k, m["scale"], m["mask"]["size"], sink, scores, m["mask"]["keep_first"])
        return A.times(o, "o")

    x = P("embed")[tokens] * cfg["embedding"]["scale"]
    outputs = [x]
    for i, L in enumerate(cfg["layers"]):
        F = P.sub(f"l{i}.mlp.")
        x = x + group_norm(mixer(L, P.sub(f"l{i}.mix."), x), P(f"l{i}.norm1"))
        if L["mlp"]["kind"] == "dense":
            f = _gated(F, x)
        else:
            w, idx = torch.softmax(F.times(x, "router"), -1).topk(L["mlp"]["router"]["top"], -1)
            f = _chosen(F, x, idx, w, _gated)
        x = x + group_norm(f, P(f"l{i}.norm2"))
        outputs.append(x)
        x = sum(a * y for a, y in zip(P(f"l{i}.dwa"), outputs))
    return group_norm(x[-last:], P("final.norm")) @ P("embed").T


def _exact_sipilorn(cfg, W, tokens, last):
    eps, T, P = cfg["norm"]["eps"], len(tokens), _Sub(W)

    def conv(x, taps):
        K = taps.shape[1]
        x = torch.cat((x.new_zeros(K - 1, x.shape[1]), x))
        return _silu(sum(x[k:k + T] * taps[:, k] for k in range(K)))

    def delta(m, A, h):
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (conv(A.times(h, n), A(n + ".conv")).view(T, -1, D) for n in "qkv")
        q, k = (y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
        q, k = (y.repeat_interleave(H // G, 1) for y in (q * D ** -0.5, k))
        beta = torch.sigmoid(A.times(h, "b"))
        decay = torch.exp(-torch.exp(A("A_log")) * torch.nn.functional.softplus(A.times(h, "a") + A("dt_bias")))
        S, o = torch.zeros(H, D, D, dtype=h.dtype, device=h.device), []
        for t in range(T):
            S = decay[t][:, None, None] * S
            u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None]
            o.append((S * q[t][:, :, None]).sum(1))
        o = _unit(torch.stack(o), eps) * A("norm") * _silu(A.times(h, "g")).view(T, H, D)
        return A.times(o.reshape(T, -1), "o")

    def attention(m, A, h):
        D, r = m["dim"], m["rot"]
        q, k, v = (A.times(h, n).view(T, -1, D) for n in "qkv")
        q, k = (_turn(_unit(y, eps) * A(n + ".norm"), r["dims"], r["base"], False) for y, n in ((q, "q"), (k, "k")))
        return A.times(_attend(q, k, v, m["scale"], m["mask"]["size"]) * torch.sigmoid(A.times(h, "g")), "o")

    x = _unit(P("embed")[tokens], eps) * P("embed.norm")
    for i, L in enumerate(cfg["layers"]):
        m, A, F = L["mixer"], P.sub(f"l{i}.mix."), P.sub(f"l{i}.mlp.")
        h = _unit(x, eps)
        h1, h2 = h * P(f"l{i}.norm1"), h * P(f"l{i}.norm2")
        if L["type"] == "delta":
            a = delta(m, A, h1)
        else:
            a = m["left_scale"] * attention(m["left"], A.sub("left."), h1) + m["right_scale"] * delta(m["right"], A.sub("right."), h1)
        if L["mlp"]["kind"] == "dense":
            a = a + _gated(F, h2)
        else:
            idx = F("table")[tokens]
            w = torch.full(idx.shape, 1.0 / idx.shape[1], dtype=x.dtype, device=x.device)
            a = a + _chosen(F, h2, idx, w, lambda E, y: E.times(torch.relu(E.times(y, "up")) ** 2, "down"))
        x = x + a
    z = (_unit(x[-last:], eps) * P("final.norm")) @ P("head").T
    return cfg["logit_softcap"] * torch.tanh(z / cfg["logit_softcap"])


def _exact_pupinex(cfg, W, tokens, last):
    eps, T, P = cfg["norm"]["eps"], len(tokens), _Sub(W)

    def norm(x, w):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w

    def attention(m, A, h, pairs):
        r = m["rot"]
        q, k, v = (A.times(h, n) for n in "qkv")
        if "q.norm" in A:
            q, k = _unit(q, eps) * A("q.norm"), _unit(k, eps) * A("k.norm")
        q, k = (_turn(y.view(T, -1, m["dim"]), r["dims"], r["base"], pairs, r.get("scaling", {}).get("factor", 1.0)) for y in (q, k))
        return A.times(_attend(q, k, v.view(T, -1, m["vdim"]), m["scale"], m["mask"]["size"], A("sink") if "sink" in A else None), "o")

    def heads(m, A, h):
        q, k, v = (A.times(h, n).view(T, m["heads"], -1) for n in "qkv")
        return q * m["dim"] ** -0.5, k, v, torch.zeros(m["heads"], m["dim"], m["vdim"], dtype=h.dtype, device=h.device)

    def gla(m, A, h):
        q, k, v, S = heads(m, A, h)
        z = A.times(A.times(h, "a1"), "a2")
        alpha = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, m["heads"], -1)
        o = []
        for t in range(T):
            S = alpha[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None]
            o.append((S * q[t][:, :, None]).sum(1))
        return A.times((_unit(torch.stack(o), eps) * A("norm")).reshape(T, -1) * _silu(A.times(h, "g")), "o")

    def mlstm(m, A, h):
        q, k, v, S = heads(m, A, h)
        cap = m["gate_cap"]
        put = cap * torch.tanh(A.times(h, "i") / cap)
        keep = torch.nn.functional.logsigmoid(cap * torch.tanh(A.times(h, "f") / cap))
        n, big, o = torch.zeros_like(S[..., 0]), torch.zeros_like(S[:, 0, 0]), []
        for t in range(T):
            new = torch.maximum(keep[t] + big, put[t])
            a, b = torch.exp(keep[t] + big - new)[:, None], torch.exp(put[t] - new)[:, None]
            big = new
            S = a[..., None] * S + b[..., None] * k[t][:, :, None] * v[t][:, None]
            n = a * n + b * k[t]
            o.append((S * q[t][:, :, None]).sum(1) / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-big)) + 1e-6)[:, None])
        return A.times(_unit(torch.stack(o), eps).reshape(T, -1) * A("norm") * torch.sigmoid(A.times(h, "g")), "o")

    def routed(m, F, h):
        r, s = m["router"], torch.sigmoid(F.times(h, "router"))
        best = s.view(T, r["groups"]["count"], -1).topk(2, -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
        allowed = torch.zeros(T, r["groups"]["count"], dtype=torch.bool, device=h.device).scatter_(1, best, True)
        idx = s.masked_fill(~allowed.repeat_interleave(r["experts"] // r["groups"]["count"], -1), -math.inf).topk(r["top"], -1).indices
        w = s.gather(1, idx)
        out = _chosen(F, h, idx, w / (w.sum(-1, keepdim=True) + 1e-20) * r["scale"], _gated)
        return out + torch.sigmoid(F.times(h, "shared.sg")) * _gated(F.sub("shared."), h)

    b = cfg["embedding"]["bigram"]
    pairs = (tokens.roll(1) * b["mul_prev"] + tokens * b["mul_cur"]) % b["buckets"]
    pairs[0] = b["buckets"]
    x = W["embed"][tokens].double() + W["bigram"][pairs].double()
    for i, L in enumerate(cfg["layers"]):
        m, A, F = L["mixer"], P.sub(f"l{i}.mix."), P.sub(f"l{i}.mlp.")
        h = norm(x, P(f"l{i}.norm1"))
        if L["type"] == "attention":
            x = x + attention(m, A, h, True)
        elif L["type"] == "gla":
            x = x + gla(m, A, h)
        else:
            x = x + m["left_scale"] * attention(m["left"], A.sub("left."), h, False) + m["right_scale"] * mlstm(m["right"], A.sub("right."), h)
        h = norm(x, P(f"l{i}.norm2"))
        x = x + (_clamped(F, h, L["mlp"]["limit"]) if L["mlp"]["kind"] == "dense" else routed(L["mlp"], F, h))
    return norm(x[-last:], P("final.norm")) @ P("embed").T


def exact(case, seed):
    """What ``run`` returns for a new state, with ``None`` for the chosen tokens."""
    forward = globals()["_exact_" + case["design"]]
    cfg, W = _weights(case, seed)
    contexts, following, portions = _inputs(case, seed)

    def logits(tokens, last):
        return forward(cfg, W, torch.tensor(tokens, device=DEVICE), last)
    if case["job"] == "generate":
        out = []
        for c in contexts:
            toks, rows = list(c), []
            for _ in range(case["steps"]):
                rows.append(logits(toks, 1)[0])
                toks.append(int(rows[-1].argmax()))
            out += [None, torch.stack(rows).cpu()]
        return out
    steps = {"life": case["steps"] + 1, "mixed": 1, "decode": PASS_STEPS}[case["job"]]
    new = steps - 1 if case["job"] == "life" else steps
    rows = [logits(c + f[:new], steps) for c, f in zip(contexts, following)]
    rows += [logits(p, 1) for p in portions]
    out = []
    for n in range(steps):
        out += [torch.stack([r[n] for r in rows]), None]
    return out
