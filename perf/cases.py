"""What the framework's speed is measured on: steps of the engine, as a serving loop or a scoring program runs them.

A case is one step of ``ModelRunner.step``, the call that ``LLMEngine`` and ``bin/trace_run`` make for every step: some
requests decode one token each behind their contexts (``decode``, ``context``), some bring a prompt or a portion of one
(``prompts``, ``tokens``, ``behind``), both kinds may stand side by side, and the lengths are equal or ragged.  The model
families are all that the engine serves, at the sizes that ``bench.py`` and the README name, in both compute types.  What a
program keeps (the model with its weights, the cache pool, the captured graphs) is kept here as well; requests, tokens and
contexts are new for every seed.

The weights are drawn, tensor by tensor, from a generator that is seeded by the tensor's name.  Their spread follows what
trained models hold where it matters for the work or its conditioning: products that write to the residual stream are
scaled down by the depth, forget gates and step sizes lie where such layers are initialised, and embeddings are of the
size of the stream, so that a router's choices do not hang on the last bit of its input.
"""

import json
import math
import random
import zlib

import torch

BLOCK = 16                       # positions of a cache page
LIVE_STATES = 6                  # sets of requests that the cache pool has room for
STEP_TOKENS = 8192               # tokens of one step while contexts are computed

# --------------------------------------------------------------------------- models

_LLAMA = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": 22, "hidden_size": 2048,
          "num_attention_heads": 32, "num_key_value_heads": 4, "head_dim": 64, "intermediate_size": 5632, "vocab_size": 32000,
          "rope_theta": 10000.0, "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "max_position_embeddings": 4096}


def _llama3(factor):
    return {"rope_type": "llama3", "factor": factor, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
            "original_max_position_embeddings": 8192}


LLAMAS = {
    "tinyllama-1.1b": _LLAMA,
    "llama-3.2-1b": dict(_LLAMA, num_hidden_layers=16, num_key_value_heads=8, intermediate_size=8192, vocab_size=128256,
                         rope_theta=500000.0, rope_scaling=_llama3(32.0), tie_word_embeddings=True, max_position_embeddings=8192),
    "llama-3.2-3b": dict(_LLAMA, num_hidden_layers=28, hidden_size=3072, num_attention_heads=24, num_key_value_heads=8, head_dim=128,
                         intermediate_size=8192, vocab_size=128256, rope_theta=500000.0, rope_scaling=_llama3(32.0),
                         tie_word_embeddings=True, max_position_embeddings=8192),
    "llama-3.1-8b": dict(_LLAMA, num_hidden_layers=32, hidden_size=4096, num_key_value_heads=8, head_dim=128,
                         intermediate_size=14336, vocab_size=128256, rope_theta=500000.0, rope_scaling=_llama3(8.0),
                         max_position_embeddings=8192),
}


def _gudutar(w):
    ssm = {"heads": 2 * w // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
    heads = w // 256
    ret = {"heads": heads, "dim": 256, "vdim": 512, "rot": {"base": 10000.0, "dims": 256},
           "decay": [1.0 - 2.0 ** (-5 - h) for h in range(heads)]}
    att = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "mask": {"size": 1024},
           "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5}
    period = [("mamba2", ssm, None), ("mamba2", ssm, None), ("retention", ret, None),
              ("latent_attention", att, {"kind": "dense", "ff": 11 * w // 4})]
    return {"architecture": "Gudutar", "embedding": {"scale": float(w) ** 0.5}, "norm": {"eps": 1e-5}}, period * 3


def _mutapel(w):
    heads, kv = w // 64, max(1, w // 512)
    win = {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 64, "mask": {"size": 1024}, "rot": {"base": 10000.0, "dims": 64},
           "scale": 0.125}
    blk = dict(win, conv=4, mask={"size": 2048})
    mlp = {"kind": "moe", "expert": {"ff": 11 * w // 16},
           "router": {"experts": 30, "identity": 2, "top": 4, "groups": {"count": 4, "keep": 2}}}
    return ({"architecture": "Mutapel", "norm": {"eps": 1e-6}, "residual_mult": 0.5, "loop": {"start": 2, "stop": 6, "times": 2}},
            [("attention_2", win, mlp), ("attention", blk, mlp)] * 4)


def _nesezen(w):
    heads = w // 64
    att = {"heads": heads, "kv_heads": max(1, heads // 8), "dim": 64, "vdim": 64, "mask": {"size": 1024}, "scale": 0.125,
           "softcap": 50.0, "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 1024}}}
    mem = {"heads": max(1, w // 256), "dim": 128, "vdim": 256, "gate_cap": 15.0}
    lat = {"heads": 16, "dim": 128, "vdim": 128, "kv_rank": 256, "q_rank": 3 * w // 4, "scale": 128 ** -0.5}
    dense = {"kind": "dense", "ff": 11 * w // 4}
    moe = {"kind": "moe", "expert": {"ff": w}, "router": {"experts": 8, "top": 2}, "shared": {"ff": 3 * w // 4}}
    return ({"architecture": "Nesezen", "norm": {"eps": 1e-5}},
            [("attention", att, dense), ("mlstm", mem, moe), ("latent_attention", lat, dense), ("attention", att, moe)] * 3)


def _renadra(w):
    heads = w // 64
    left = {"heads": heads, "kv_heads": max(1, heads // 8), "dim": 64, "vdim": 64, "mask": {"size": 1024, "keep_first": 4}, "scale": 0.125,
            "softcap": 50.0, "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "original": 2048, "fast": 16.0, "slow": 2.0}}}
    r = max(1, w // 256)
    par = {"left": left, "right": {"heads": r, "dim": 128, "vdim": 256, "decay": [1.0 - 2.0 ** (-5 - h) for h in range(r)]},
           "left_scale": 1.0, "right_scale": 0.5}
    att = {"heads": heads, "kv_heads": max(1, heads // 8), "dim": 64, "vdim": 64, "mask": {"size": 1024}, "scale": 0.125,
           "rot": {"base": 10000.0, "dims": 64}}
    kinds = {"parallel": par, "attention": att, "hgrn2": {"heads": max(1, w // 128), "dim": 128, "vdim": 128}}
    order = ["parallel", "attention", "hgrn2", "hgrn2", "parallel", "attention", "hgrn2", "attention"]
    return ({"architecture": "Renadra", "norm": {"eps": 1e-5}, "loop": {"start": 2, "stop": 6, "times": 2},
             "embedding": {"scale": 1.0, "bigram": {"buckets": 100003, "mul_prev": 131, "mul_cur": 17}}},
            [(t, kinds[t], {"kind": "dense", "ff": 11 * w // 4}) for t in order])


def _mekusun(w):
    ssm = {"inner": 2 * w, "state": 16, "dt_rank": w // 16, "conv": 4}
    lat = {"heads": 16, "dim": 128, "vdim": 128, "kv_rank": 192, "rot_dim": 64, "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5}
    dense = {"kind": "dense", "ff": 4 * w}
    moe = {"kind": "moe", "expert": {"ff": 2 * w}, "router": {"experts": 8, "top": 2}}
    return ({"architecture": "Mekusun", "norm": {"eps": 1e-5}, "embedding": {"scale": float(w) ** 0.5}, "logit_softcap": 30.0},
            [("general_delta", {"heads": w // 64, "dim": 64}, dense), ("mamba1", ssm, moe), ("latent_attention", lat, dense),
             ("mamba1", ssm, moe)] * 3)


def _pamunex(w):
    heads = w // 64
    lat = {"heads": 16, "dim": 128, "vdim": 128, "kv_rank": 192, "rot_dim": 64, "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5,
           "mask": {"size": 1024}}
    att = {"heads": heads, "kv_heads": max(1, heads // 8), "dim": 64, "vdim": 64, "rot": {"base": 10000.0, "dims": 64}, "scale": 0.125,
           "mask": {"size": 2048}}
    moe = {"kind": "moe", "expert": {"ff": w}, "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}}}
    return ({"architecture": "Pamunex", "norm": {"eps": 1e-5}, "logit_scale": 0.5},
            [("latent_attention", lat, {"kind": "dense", "ff": 4 * w}), ("attention", att, moe)] * 6)


OTHERS = {"gudutar": _gudutar, "mutapel": _mutapel, "nesezen": _nesezen, "renadra": _renadra, "mekusun": _mekusun, "pamunex": _pamunex}


def configuration(case):
    """The config.json of the case's model."""
    if case["model"] in LLAMAS:
        return dict(LLAMAS[case["model"]], torch_dtype=case["dtype"])
    top, layers = OTHERS[case["model"]](case["width"])
    return dict(top, vocab=32000, width=case["width"], max_positions=4096, torch_dtype=case["dtype"],
                layers=[{"type": t, "mixer": m, "mlp": f} for t, m, f in layers])


def run_order(cfg):
    """[(layer, which pass of the repeated range starts here: 1 for the first, 0 for none)] in the order the layers run."""
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return [(i, 0) for i in range(n)]
    a, b = loop["start"], loop["stop"]
    again = [(i, p if i == a else 0) for p in range(1, loop["times"] + 1) for i in range(a, b)]
    return [(i, 0) for i in range(a)] + again + [(i, 0) for i in range(b, n)]


def mixer_tensors(kind, m, w):
    """{name: shape} of a mixer's tensors."""
    if kind == "mamba2":
        inner, chan = m["heads"] * m["vdim"], m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
        return {"in": (inner + chan + m["heads"], w), "conv": (chan, m["conv"]), "conv.b": (chan,), "dt_bias": (m["heads"],),
                "A_log": (m["heads"],), "D": (m["heads"],), "norm": (inner,), "o": (w, inner)}
    if kind == "mamba1":
        c, n, r = m["inner"], m["state"], m["dt_rank"]
        return {"in": (2 * c, w), "conv": (c, m["conv"]), "conv.b": (c,), "x": (r + 2 * n, c), "dt": (c, r), "dt.b": (c,), "A_log": (c, n),
                "D": (c,), "o": (w, c)}
    if kind == "retention":
        k, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
        return {"q": (k, w), "k": (k, w), "v": (v, w), "g": (v, w), "o": (w, v)}
    if kind == "lightning":
        k, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
        return {"q": (k, w), "k": (k, w), "v": (v, w), "g": (v, w), "norm": (v,), "o": (w, v)}
    if kind == "mlstm":
        k, v, h = m["heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"]
        return {"q": (k, w), "k": (k, w), "v": (v, w), "g": (v, w), "i": (h, w), "f": (h, w), "i.b": (h,), "f.b": (h,), "norm": (v,), "o": (w, v)}
    if kind == "hgrn2":
        k, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
        return {"q": (k, w), "f": (k, w), "f.b": (k,), "lower": (k,), "v": (v, w), "norm": (m["vdim"],), "o": (w, v)}
    if kind == "general_delta":
        d = m["heads"] * m["dim"]
        return {**{n: (d, w) for n in ("r", "k", "v", "a", "g")}, "a.b": (d,), "w0": (d,), "w1": (m["dim"], w), "w2": (d, m["dim"]), "norm": (d,),
                "o": (w, d)}
    if kind == "latent":
        h, rot = m["heads"], m.get("rot_dim", 0)
        out = {"dkv": (m["kv_rank"] + rot, w), "dkv.norm": (m["kv_rank"],), "uk": (h * m["dim"], m["kv_rank"]), "uv": (h * m["vdim"], m["kv_rank"]),
               "o": (w, h * m["vdim"])}
        if m.get("q_rank"):
            return {**out, "dq": (m["q_rank"], w), "dq.norm": (m["q_rank"],), "uq": (h * m["dim"], m["q_rank"]), "g": (h, w)}
        return {**out, "q": (h * (m["dim"] + rot), w)}
    h, g, d = m["heads"], m["kv_heads"], m["dim"]
    return {"q": (h * d, w), "k": (g * d, w), "v": (g * d, w), "o": (w, h * d)}


def tensors(cfg):
    """{name: shape} of all of the model's tensors, under the names that a checkpoint has them."""
    if "architectures" in cfg:
        w, f, v = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
        q, kv = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
        out = {"model.embed_tokens.weight": (v, w), "model.norm.weight": (w,)}
        if not cfg["tie_word_embeddings"]:
            out["lm_head.weight"] = (v, w)
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.update({p + "input_layernorm.weight": (w,), p + "post_attention_layernorm.weight": (w,), p + "self_attn.q_proj.weight": (q, w),
                        p + "self_attn.k_proj.weight": (kv, w), p + "self_attn.v_proj.weight": (kv, w), p + "self_attn.o_proj.weight": (w, q),
                        p + "mlp.gate_proj.weight": (f, w), p + "mlp.up_proj.weight": (f, w), p + "mlp.down_proj.weight": (w, f)})
        return out
    arch, w, v = cfg["architecture"], cfg["width"], cfg["vocab"]
    norm = {"Gudutar": ("", ".b"), "Pamunex": ("", ".b"), "Nesezen": ("", ".b", ".alpha")}.get(arch, ("",))
    shape = {"": (w,), ".b": (w,), ".alpha": ()}
    out = {"embed": (v, w), **{"final.norm" + s: shape[s] for s in norm}}
    if arch != "Pamunex":
        out["head"] = (v, w)
    if arch == "Mutapel":
        out["loop.in"] = (w, 2 * w)
    if arch == "Renadra":
        out["bigram"] = (cfg["embedding"]["bigram"]["buckets"] + 1, w)
    for i, layer in enumerate(cfg["layers"]):
        kind, m, mlp, p = layer["type"], layer["mixer"], layer["mlp"], f"l{i}."
        here = {}
        if kind == "parallel":
            left = mixer_tensors("attention", m["left"], w)
            del left["v"]
            left.update({"q.b": (left["q"][0],), "k.b": (left["k"][0],), "pb": (m["left"]["heads"],)})
            here.update({"left." + n: s for n, s in left.items()})
            here.update({"right." + n: s for n, s in mixer_tensors("lightning", m["right"], w).items()})
        elif kind in ("attention", "attention_2"):
            here.update(mixer_tensors("attention", m, w))
            rows = {n: (here[n][0],) for n in ("q", "k", "v", "o")}
            if kind == "attention_2":
                here["g"] = (m["heads"], w)
            elif arch == "Mutapel":
                here.update({**{n + ".b": rows[n] for n in rows}, **{n + ".conv": rows[n] + (m["conv"],) for n in ("q", "k", "v")}, "sink": (m["heads"],)})
            elif arch == "Pamunex":
                here.update({**{n + ".b": rows[n] for n in ("q", "k", "v")}, "q.norm": (m["dim"],), "k.norm": (m["dim"],), "sink": (m["heads"],)})
            elif arch == "Renadra":
                here.update({n + ".b": rows[n] for n in rows})
        elif kind == "latent_attention":
            here.update(mixer_tensors("latent", m, w))
            if arch == "Pamunex":
                here["sink"] = (m["heads"],)
        else:
            here.update(mixer_tensors(kind, m, w))
        out.update({f"{p}mix.{n}": s for n, s in here.items()})
        names = ["norm1"] + (["norm2"] if mlp else [])
        out.update({p + n + s: shape[s] for n in names for s in norm})
        if arch in ("Mutapel", "Mekusun"):
            out.update({p + n + "b": (w,) for n in names})
        if arch == "Mekusun":
            out.update({p + "dwa": (i + 2,), p + "ls1": (w,), p + "ls2": (w,)})
        if not mlp:
            continue
        gated = arch not in ("Mekusun", "Pamunex")
        def ff(prefix, size):
            both = {"up": (size, w), "down": (w, size), **({"gate": (size, w)} if gated else {})}
            out.update({f"{p}mlp.{prefix}{n}": s for n, s in both.items()})
        if mlp["kind"] == "dense":
            ff("", mlp["ff"])
            if arch == "Mekusun":
                out[p + "mlp.act"] = (2,)
            continue
        r = mlp["router"]
        scores = r["experts"] + r.get("identity", 0)
        out[p + "mlp.router"] = (scores, w)
        if arch == "Mutapel":
            out[p + "mlp.correction"] = (scores,)
        if arch == "Mekusun":
            out[p + "mlp.router.b"] = (scores,)
        for e in range(r["experts"]):
            ff(f"e{e}.", mlp["expert"]["ff"])
        if mlp.get("shared"):
            ff("shared.", mlp["shared"]["ff"])
            out[p + "mlp.shared.sg"] = (1, w)
    return out


def weight(cfg, name, shape):
    """One tensor's values on the GPU, in float32 or rounded to bfloat16 as a checkpoint of that type holds them."""
    g = torch.Generator(device="cuda").manual_seed(zlib.crc32(name.encode()))
    n = torch.randn(shape, generator=g, device="cuda")
    arch = cfg.get("architecture", "Llama")
    depth = cfg["num_hidden_layers"] if arch == "Llama" else len(run_order(cfg))
    last = name.rsplit(".", 1)[-1]
    behind = arch in ("Gudutar", "Pamunex")                      # the norms stand behind the sublayers
    matrix = n * (0.9 / math.sqrt(shape[-1])) if shape else n
    if name in ("embed", "bigram", "model.embed_tokens.weight"):
        t = n * (0.3 if cfg.get("tie_word_embeddings") else 1.0 / (cfg.get("embedding") or {}).get("scale", 1.0))
    elif last in ("o", "down") or name.endswith(("o_proj.weight", "down_proj.weight")):
        t = matrix / math.sqrt(2.0 * depth)
    elif last == "router" and arch in ("Mutapel", "Mekusun"):    # (a softmax: a trained router's is peaked)
        t = 3.0 * matrix
    elif name == "loop.in":
        t = 0.01 * n + 0.7 * torch.eye(shape[0], device="cuda").repeat(1, 2)
    elif last in ("norm1b", "norm2b"):                           # (stored as w - 1)
        t = n * 0.1 - (0.8 if arch == "Mutapel" else 0.0)
    elif last in ("norm1", "norm2", "norm") or "norm.weight" in name:
        t = n * 0.1 if arch in ("Mutapel", "Mekusun") and ".mix." not in name else 1.0 + 0.1 * n
        t = 0.1 * t if behind and last in ("norm1", "norm2") else t
    elif last in ("ls1", "ls2"):
        t = 0.1 * (1.0 + 0.1 * n)
    elif last == "alpha":
        t = 0.5 * (1.0 + 0.1 * n)
    elif last == "A_log":
        t = torch.log(1.0 + 15.0 * torch.rand(shape, generator=g, device="cuda"))
    elif last == "dt_bias" or name.endswith(".dt.b"):            # step sizes between 0.001 and 0.1 after the softplus
        t = torch.log(torch.expm1(torch.exp(math.log(0.001) + math.log(100.0) * torch.rand(shape, generator=g, device="cuda"))))
    elif last == "lower":
        t = 0.9 * torch.rand(shape, generator=g, device="cuda")
    elif last == "D":
        t = 1.0 + 0.1 * n
    elif last == "conv":
        t = 0.3 * n
    elif last in ("sink", "act"):
        t = 0.5 * n
    elif last == "pb":
        t = 0.5 * n - 4.0
    elif last == "w0":
        t = n - 2.0
    elif name.endswith(".f.b"):
        t = n + (4.0 if arch == "Nesezen" else 1.0)
    elif last == "correction":
        t = 0.01 * n
    elif last == "dwa":
        t = 0.02 * n
        t[-1] += 1.0
    else:
        t = matrix if len(shape) == 2 else 0.02 * n
    return t.to(torch.bfloat16) if cfg["torch_dtype"] == "bfloat16" else t


# --------------------------------------------------------------------------- cases
def _case(name, model, decode=0, context=0, prompts=0, tokens=0, behind=0, ragged=False, want="last", dtype="bfloat16", width=0):
    return {**({"name": name} if name else {}), "model": model, "dtype": dtype, "width": width, "decode": decode, "context": context,
            "prompts": prompts, "tokens": tokens, "behind": behind, "ragged": ragged, "want": want}


def listed():
    return [
        # one user, a chat that has just begun: the smallest step there is, all launches and latency
        _case("tinyllama_decode_1", "tinyllama-1.1b", decode=1, context=181),
        # the benchmark's headline: eight requests at a context of 2,048
        _case("tinyllama_decode_8", "tinyllama-1.1b", decode=8, context=2040),
        # a busy server: an odd number of requests with contexts of every length, a vocabulary of 128,256
        _case("llama_1b_decode_61_ragged", "llama-3.2-1b", decode=61, context=2000, ragged=True),
        # the benchmark's other headline: one prompt of 2,048 tokens
        _case("tinyllama_prompt_2048", "tinyllama-1.1b", prompts=1, tokens=2048),
        # continuous batching on a large model: requests decode while a portion of a longer prompt is worked off
        _case("llama_8b_mixed_8_and_256", "llama-3.1-8b", decode=8, context=1500, prompts=1, tokens=256, behind=1024, ragged=True),
        # a float32 checkpoint, which runs in float32 unless told otherwise: a few requests decode
        _case("tinyllama_f32_decode_8", "tinyllama-1.1b", decode=8, context=700, ragged=True, dtype="float32"),
        # ... and a text of odd length is scored: logits at every position
        _case("tinyllama_f32_score_301", "tinyllama-1.1b", prompts=1, tokens=301, want="all", dtype="float32"),
        # the other families: long prompt, odd prompt, scoring of two texts at once, and decoding at three batch sizes
        _case("gudutar_prompt_2048", "gudutar", prompts=1, tokens=2048, width=2048),
        _case("renadra_prompt_777", "renadra", prompts=1, tokens=777, width=2048),
        _case("mekusun_score_2_ragged", "mekusun", prompts=2, tokens=600, ragged=True, want="all", width=2048),
        _case("nesezen_decode_33_ragged", "nesezen", decode=33, context=1200, ragged=True, width=2048),
        _case("mutapel_decode_8", "mutapel", decode=8, context=1030, width=2048),
    ]


def draw(rng):
    """One more case of the same ranges: any family and type, a decode step, prompts, or both."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(["tinyllama-1.1b"] * 3 + ["llama-3.2-1b"] * 2 + ["llama-3.2-3b"] + sorted(OTHERS))
    dtype = "float32" if model in ("tinyllama-1.1b", *OTHERS) and rng.random() < 0.2 else "bfloat16"
    small = dtype == "float32"
    width = 0 if model in LLAMAS else 1024 if small else rng.choice([1024, 2048])
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed"])
    case = dict(ragged=rng.random() < 0.5, dtype=dtype, width=width)
    if kind != "prompt":
        case.update(decode=size(1, 12 if small else 64), context=size(17, 512 if small else 2040))
    if kind != "decode":
        count = rng.choice([1, 1, 2, 3])
        case.update(prompts=count, tokens=size(16, (256 if small else 2048 if kind == "prompt" else 512) // count),
                    want="all" if kind == "prompt" and rng.random() < 0.3 else "last", behind=rng.choice([0, 0, size(16, 256 if small else 1024)]))
    return _case(None, model, **case)


def lengths(case):
    """[(tokens in the cache already, tokens of this step)] of the case's requests: the same for every seed."""
    rng = random.Random(zlib.crc32(json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True).encode()))

    def some(count, longest):
        if not count or not case["ragged"]:
            return [longest] * count
        return [longest] + [rng.randint(max(1, longest // 32), longest) for _ in range(count - 1)]

    out = [(c, 1) for c in some(case["decode"], case["context"])]
    return out + [(case["behind"], max(2, t)) for t in some(case["prompts"], case["tokens"])]


def requests(case, seed):
    """[(all tokens of the request up to the end of this step, how many of them are in the cache already)]."""
    cfg = configuration(case)
    g = torch.Generator().manual_seed(seed)
    return [(torch.randint(100, cfg.get("vocab") or cfg["vocab_size"], (a + n,), generator=g).tolist(), a) for a, n in lengths(case)]


def wanted(case, n):
    return list(range(n)) if case["want"] == "all" else [n - 1]


# --------------------------------------------------------------------------- what a serving program keeps
class Server:
    """A model with a cache pool and a step function, as ``LLMEngine`` holds them."""

    def __init__(self, case, model):
        from paged_llm_amd.engine.loading import build_runtime
        need = lengths(case)
        pages = sum((a + n + BLOCK - 1) // BLOCK + 1 for a, n in need) * LIVE_STATES
        self.manager, self.storage, self.runner = build_runtime(model, BLOCK, pages, len(need) * LIVE_STATES, enable_prefix_caching=False,
                                                                use_graphs=True)
        self.count = 0

    def entry(self, rid, tokens, start, want):
        from paged_llm_amd.engine.batch import StepEntry
        if not self.manager.allocate(rid, start, len(tokens)):
            raise RuntimeError("no pages left")
        tables, slot, version = self.manager.step_fields(rid)
        return StepEntry(rid, tokens, start, {g: list(t) for g, t in tables.items()}, slot, want, version)


class State:
    """Requests that the server has admitted, their contexts in the cache, and the entries of the step to come."""

    def __init__(self, server, case, seed):
        self.server, self.ids, self.entries = server, [], []
        every = requests(case, seed)
        for _ in every:
            self.ids.append(server.count)
            server.count += 1
        filling, held = [], 0
        for rid, (tokens, start) in zip(self.ids, every):
            if start:
                filling.append(server.entry(rid, tokens[:start], 0, []))
                held += start
            if held and (held + 2048 > STEP_TOKENS or rid == self.ids[-1]):
                server.runner.step(filling)
                filling, held = [], 0
        for rid, (tokens, start) in zip(self.ids, every):
            new = tokens[start:]
            self.entries.append(server.entry(rid, new, start, wanted(case, len(new))))

    def __del__(self):
        for rid in self.ids:
            self.server.manager.free(rid)


_kept = {}


def _server(case):
    from paged_llm_amd.engine.loading import build_model
    key = json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)
    if _kept.get("case") != key:
        which = (case["model"], case["dtype"], case["width"])
        _kept.pop("server", None)
        if _kept.get("which") != which:
            _kept.clear()
            cfg = configuration(case)
            model = build_model(cfg, case["dtype"], torch.device("cuda"))
            for name, shape in tensors(cfg).items():
                model.assign(name, weight(cfg, name, shape))
            model.finalize()
            _kept.update(which=which, model=model)
        _kept.update(case=key, server=Server(case, _kept["model"]))
    return _kept["server"]


def prepare(case, seed):
    return State(_server(case), case, seed)


def run(state):
    """The step's logits: float32 [wanted rows, vocabulary]."""
    return state.server.runner.step(state.entries)


# --------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Weights once (of routed experts those that some token is expected to choose), products of every token, keys and values
    that a query sees, states read and written, logits."""
    cfg, need = configuration(case), lengths(case)
    size = 4 if case["dtype"] == "float32" else 2
    T, rows = sum(n for _, n in need), sum(len(wanted(case, n)) for _, n in need)
    runs = [(i, 0) for i in range(cfg["num_hidden_layers"])] if "architectures" in cfg else run_order(cfg)
    times = {}
    for i, _ in runs:
        times[i] = times.get(i, 0) + 1
    heads = {"lm_head.weight", "head"} | ({"embed"} if cfg.get("architecture") == "Pamunex" else set())
    heads |= {"model.embed_tokens.weight"} if cfg.get("tie_word_embeddings") else set()
    bytes_, flops = 0.0, 0.0
    for name, shape in tensors(cfg).items():
        n = math.prod(shape)
        if name in heads:
            bytes_, flops = bytes_ + n * size, flops + 2.0 * n * rows
        elif name in ("embed", "bigram", "model.embed_tokens.weight"):
            bytes_ += T * shape[1] * size
        elif ".mlp.e" in name:
            mlp = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            share = mlp["top"] / (mlp["experts"] + mlp.get("identity", 0))
            bytes_ += n * size * (1.0 - (1.0 - share) ** T)
            flops += 2.0 * n * T * share * times[int(name[1:name.index(".")])]
        else:
            i = int(name.split(".")[2]) if name.startswith("model.layers") else int(name[1:name.index(".")]) if name[1].isdigit() else None
            t = times.get(i, 1)
            bytes_ += n * size
            flops += 2.0 * n * T * t if len(shape) == 2 and shape[1] > 16 else 0.0
    def attention(keys_width, per_pair, mask):
        nonlocal bytes_, flops
        for a, n in need:
            seen = min(a + n, mask + n) if mask else a + n
            pairs = sum(min(a + j + 1, mask or a + j + 1) for j in range(n))
            bytes_ += (seen + n) * keys_width * size
            flops += per_pair * pairs
    def state(elements):
        nonlocal bytes_, flops
        for a, n in need:
            bytes_ += 4.0 * elements * (2 if a else 1)
            flops += 4.0 * elements * n
    for i, _ in runs:
        if "architectures" in cfg:
            h, g, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
            attention(2 * g * d, 4.0 * h * d, 0)
            continue
        kind, m = cfg["layers"][i]["type"], cfg["layers"][i]["mixer"]
        mask = (m.get("mask") or {}).get("size", 0)
        if kind == "latent_attention":
            attention(m["kv_rank"] + m.get("rot_dim", 0), 2.0 * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"]), mask)
        elif kind in ("attention", "attention_2"):
            attention(2 * m["kv_heads"] * m["dim"], 4.0 * m["heads"] * m["dim"], mask)
        elif kind == "parallel":
            attention(2 * m["left"]["kv_heads"] * m["left"]["dim"], 4.0 * m["left"]["heads"] * m["left"]["dim"], m["left"]["mask"]["size"])
            state(m["right"]["heads"] * m["right"]["dim"] * m["right"]["vdim"])
        elif kind == "mamba1":
            state(m["inner"] * m["state"])
        elif kind == "mamba2":
            state(m["heads"] * m["vdim"] * m["state"])
        else:
            state(m["heads"] * m["dim"] * m.get("vdim", m["dim"]))
    vocab = cfg.get("vocab") or cfg["vocab_size"]
    return {"bytes": bytes_ + 4.0 * rows * vocab, "flops": flops}


def tolerance(case):
    """Measured against ``exact`` over all families, several sizes and seeds: float32 0.6e-6 to 1.3e-6; bfloat16 0.011 to 0.015 for
    the Llama models (whose residual stream is bfloat16 as well), 0.002 to 0.003 for the families with a float stream, and up
    to 0.08 in the rare row in which a router's close call falls the other way."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 0.01, "max": 0.2} if case["model"] in ("gudutar", "renadra") else {"rel": 0.03, "max": 0.5}


# --------------------------------------------------------------------------- the same logits in 64 bits
def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps):
    return _unit(x - x.mean(-1, keepdim=True), eps) * w + b


def _silu(z):
    return z * torch.sigmoid(z)


def _turn(x, base, dims, interleaved=False, scaling=None, single=False):
    """x [T, heads, d]: the first ``dims`` elements turned in pairs; frequencies and angles are float32 numbers, as the
    tables of such models hold them (``single``: the frequencies are formed in float32 as well)."""
    half, mag = dims // 2, 1.0
    if single:
        f = 1.0 / (base ** (torch.arange(0, dims, 2, dtype=torch.float32) / dims))
    else:
        f = torch.tensor([base ** (-2.0 * i / dims) for i in range(half)], dtype=torch.float64)
    if scaling and "fast" in scaling:
        def index(turns):
            return dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
        lo, hi = max(math.floor(index(scaling["fast"])), 0), min(math.ceil(index(scaling["slow"])), dims - 1)
        ramp = ((torch.arange(half, dtype=f.dtype) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, mag = f / scaling["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0
    elif scaling:
        low, high = scaling.get("low", scaling.get("low_freq_factor")), scaling.get("high", scaling.get("high_freq_factor"))
        original = scaling.get("original", scaling.get("original_max_position_embeddings"))
        wave = 2.0 * math.pi / f
        s = (original / wave - low) / (high - low)
        blend = (1.0 - s) * f / scaling["factor"] + s * f
        f = torch.where(wave > original / low, f / scaling["factor"], torch.where(wave < original / high, f, blend))
    angle = torch.arange(x.shape[0], dtype=torch.float32)[:, None] * f.to(torch.float32)[None, :]
    angle = angle.double().to(x.device)[:, None, :]
    c, s = torch.cos(angle) * mag, torch.sin(angle) * mag
    out = x.clone()
    a, b = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, half), slice(half, dims))
    u, v = x[..., a], x[..., b]
    out[..., a], out[..., b] = u * c - v * s, v * c + u * s
    return out


def _attend(q, k, v, scale, window=0, block=0, keep_first=0, cap=0.0, sink=None, bias=None, rest=None):
    """q [T, H, d], k and v [T, G, .] -> [T, H * .].  ``rest``: further scores [H, T, T]; ``bias``: no softmax."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    k, v = (t.repeat_interleave(H // G, dim=1).transpose(0, 1).contiguous() for t in (k, v))
    s = q.transpose(0, 1).contiguous() @ k.transpose(1, 2)
    s = (s if rest is None else s + rest) * scale
    s = cap * torch.tanh(s / cap) if cap else s
    i, j = torch.arange(T, device=q.device)[:, None], torch.arange(T, device=q.device)[None, :]
    seen = j <= i
    if window:
        seen = seen & ((i - j < window) | (j < keep_first))
    if block:
        seen = seen & (i // block == j // block)
    if bias is not None:
        p = torch.sigmoid(s + bias[:, None, None]) * seen
    else:
        s = s.masked_fill(~seen, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(H, T, 1)], dim=2)
        p = torch.softmax(s, dim=-1)[..., :T]
    return (p @ v).transpose(0, 1).reshape(T, -1)


def _latent(h, w, m, eps, interleaved, sink=None):
    T, H, d, r = h.shape[0], m["heads"], m["dim"], m.get("rot_dim", 0)
    rank = m["kv_rank"]
    q = (_unit(h @ w("dq").T, eps) * w("dq.norm")) @ w("uq").T if m.get("q_rank") else h @ w("q").T
    q = q.view(T, H, d + r)
    down = h @ w("dkv").T
    c = _unit(down[:, :rank], eps) * w("dkv.norm")
    rest = None
    if r:
        kr = _turn(down[:, None, rank:], m["rot"]["base"], m["rot"]["dims"], interleaved)[:, 0]
        qr = _turn(q[..., d:], m["rot"]["base"], m["rot"]["dims"], interleaved)
        rest = qr.transpose(0, 1).contiguous() @ kr.T
    return _attend(q[..., :d], (c @ w("uk").T).view(T, H, d), (c @ w("uv").T).view(T, H, -1), m["scale"],
                   window=(m.get("mask") or {}).get("size", 0), sink=sink, rest=rest)


def _recurrence(a, k, v, q):
    """S_t = a_t S_(t-1) + k_t v_t^T, o_t = S_t^T q_t; a [T, H] or [T, H, N], k and q [T, H, N], v [T, H, P]."""
    S = v.new_zeros(v.shape[1], k.shape[2], v.shape[2])
    a = a.reshape(*a.shape, *[1] * (4 - a.dim()))
    out = torch.empty_like(v)
    for t in range(v.shape[0]):
        S.mul_(a[t]).addcmul_(k[t][:, :, None], v[t][:, None, :])
        torch.matmul(q[t][:, None, :], S, out=out[t][:, None, :])
    return out


def _convolve(x, w, b=None):
    """A causal convolution per channel over time; the last column of w meets the current token."""
    taps = w.shape[1]
    padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    y = sum(padded[j:j + x.shape[0]] * w[:, j] for j in range(taps))
    return y if b is None else y + b


def _softplus(z):
    return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))


def _mix(arch, kind, h, w, m, eps):
    """A mixer's output before its output product."""
    T = h.shape[0]
    if kind == "mamba2":
        H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * P
        z, xbc, dt = torch.split(h @ w("in").T, [inner, inner + 2 * G * N, H], dim=1)
        xbc = _silu(_convolve(xbc, w("conv"), w("conv.b")))
        x = xbc[:, :inner].reshape(T, H, P)
        B, C = (t.reshape(T, G, N).repeat_interleave(H // G, dim=1) for t in (xbc[:, inner:inner + G * N], xbc[:, inner + G * N:]))
        dt = _softplus(dt + w("dt_bias"))
        y = _recurrence(torch.exp(-torch.exp(w("A_log")) * dt), B * dt[..., None], x, C) + w("D")[:, None] * x
        y = y.reshape(T, inner) * _silu(z)
        return _unit(y.view(T, m["norm_groups"], -1), eps).reshape(T, inner) * w("norm")
    if kind == "mamba1":
        inner, n, rank = m["inner"], m["state"], m["dt_rank"]
        rows = h @ w("in").T
        x = _silu(_convolve(rows[:, :inner], w("conv"), w("conv.b")))
        low = x @ w("x").T
        dt = _softplus(low[:, :rank] @ w("dt").T + w("dt.b"))
        A, B, C = -torch.exp(w("A_log")), low[:, rank:rank + n], low[:, rank + n:]
        S, y = torch.zeros_like(A), torch.empty_like(x)
        for t in range(T):
            S = torch.exp(dt[t][:, None] * A).mul_(S).addcmul_((dt[t] * x[t])[:, None], B[t][None, :])
            torch.mv(S, C[t], out=y[t])
        return (y + w("D") * x) * _silu(rows[:, inner:])
    if kind in ("retention", "lightning"):
        H, d, P = m["heads"], m["dim"], m["vdim"]
        q, k, v = (h @ w(n).T for n in ("q", "k", "v"))
        if kind == "lightning":
            q, k, v = _silu(q), _silu(k), _silu(v)
        q, k, v = q.view(T, H, d), k.view(T, H, d), v.view(T, H, P)
        if kind == "retention":
            q, k = (_turn(t, m["rot"]["base"], m["rot"]["dims"]) for t in (q, k))
            k = k * d ** -0.5
        o = _recurrence(torch.tensor(m["decay"], dtype=h.dtype, device=h.device).expand(T, H), k, v, q)
        if kind == "retention":
            return _unit(o, eps).reshape(T, H * P) * _silu(h @ w("g").T)
        return _unit(o.reshape(T, H * P), eps) * w("norm") * torch.sigmoid(h @ w("g").T)
    if kind == "mlstm":
        H, d, P, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k, v = (h @ w("q").T).view(T, H, d) * d ** -0.5, (h @ w("k").T).view(T, H, d), (h @ w("v").T).view(T, H, P)
        i, f = (cap * torch.tanh((h @ w(n).T + w(n + ".b")) / cap) for n in ("i", "f"))
        f = torch.clamp(f, max=0) - torch.log1p(torch.exp(-f.abs()))
        top, M = [], h.new_zeros(H)
        for t in range(T):
            M = torch.maximum(f[t] + M, i[t])
            top.append(M)
        top = torch.stack(top)
        keep = torch.exp(f + torch.cat([h.new_zeros(1, H), top[:-1]]) - top)
        both = _recurrence(keep, k * torch.exp(i - top)[..., None], torch.cat([v, h.new_ones(T, H, 1)], dim=2), q)
        o = both[..., :P] / (torch.maximum(both[..., P:].abs(), torch.exp(-top)[..., None]) + 1e-6)
        return _unit(o, eps).reshape(T, H * P) * w("norm") * torch.sigmoid(h @ w("g").T)
    if kind == "hgrn2":
        H, N, P = m["heads"], m["dim"], m["vdim"]
        f = (w("lower") + (1.0 - w("lower")) * torch.sigmoid(h @ w("f").T + w("f.b"))).view(T, H, N)
        o = _recurrence(f, 1.0 - f, (h @ w("v").T).view(T, H, P), _silu(h @ w("q").T).view(T, H, N))
        return (_unit(o, eps) * w("norm")).reshape(T, H * P)
    if kind == "general_delta":
        H, d = m["heads"], m["dim"]
        r, k, v = ((h @ w(n).T).view(T, H, d) for n in ("r", "k", "v"))
        keep = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ w("w1").T) @ w("w2").T + w("w0"))).view(T, H, d, 1)
        u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        au = torch.sigmoid(h @ w("a").T + w("a.b")).view(T, H, d) * u
        S, o = h.new_zeros(H, d, d), torch.empty_like(v)
        for t in range(T):
            read = u[t][:, None, :] @ S
            S = (keep[t] * S).addcmul_(au[t][:, :, None], read, value=-1.0).addcmul_(k[t][:, :, None], v[t][:, None, :])
            o[t] = (r[t][:, None, :] @ S)[:, 0]
        return _unit(o, eps).reshape(T, H * d) * w("norm") * torch.sigmoid(h @ w("g").T)
    if kind == "latent_attention":
        sink = w("sink") if arch == "Pamunex" else None
        o = _latent(h, w, m, eps, interleaved=arch == "Gudutar", sink=sink)
        return (o.view(T, m["heads"], -1) * torch.sigmoid(h @ w("g").T)[..., None]).reshape(T, -1) if m.get("q_rank") else o
    H, G, d, rot, size = m["heads"], m["kv_heads"], m["dim"], m["rot"], m["mask"]["size"]
    if kind == "left":
        q, k = (h @ w("q").T + w("q.b")).view(T, H, d), (h @ w("k").T + w("k.b")).view(T, G, d)
        tq, tk = (_turn(t, rot["base"], rot["dims"], scaling=rot["scaling"]) for t in (q, k))
        return _attend(tq, tk, k, m["scale"], window=size, keep_first=m["mask"]["keep_first"], cap=m["softcap"], bias=w("pb"))
    q, k, v = (h @ w(n).T for n in ("q", "k", "v"))
    if arch in ("Renadra", "Pamunex") or (arch == "Mutapel" and kind == "attention"):
        q, k, v = q + w("q.b"), k + w("k.b"), v + w("v.b")
    if arch == "Mutapel" and kind == "attention":
        q, k, v = _convolve(q, w("q.conv")), _convolve(k, w("k.conv")), _convolve(v, w("v.conv"))
    q, k, v = q.view(T, H, d), k.view(T, G, d), v.view(T, G, d)
    if arch == "Pamunex":
        q, k = _unit(q, eps) * w("q.norm"), _unit(k, eps) * w("k.norm")
    q, k = (_turn(t, rot["base"], rot["dims"], interleaved=arch == "Renadra" or kind == "attention_2", scaling=rot.get("scaling")) for t in (q, k))
    if arch == "Mutapel":
        q, k = _unit(q, eps), _unit(k, eps)
    if arch == "Renadra":
        v = _unit(v, eps)
    blocks = arch == "Pamunex" or (arch == "Mutapel" and kind == "attention")
    o = _attend(q, k, v, m["scale"], block=size if blocks else 0, window=0 if blocks else size, cap=m.get("softcap", 0.0),
                sink=w("sink") if blocks else None)
    if kind == "attention_2":
        o = (o.view(T, H, d) * torch.sigmoid(h @ w("g").T)[..., None]).reshape(T, -1)
    return o


def _one_ff(arch, h, w, p, routed):
    if arch == "Mekusun" and not routed:
        up, act = h @ w("up").T, _softplus(w("act"))
        low = torch.clamp(up, max=0)
        return torch.where(up > 0, act[0] * up * up + 0.5 * up, (0.5 + act[1]) * (torch.expm1(low) - low) + 0.5 * low) @ w("down").T
    up = h @ w(p + "up").T
    if arch == "Mekusun":
        return (0.5 * up * (1.0 + torch.erf(up / math.sqrt(2.0)))) @ w(p + "down").T
    if arch == "Pamunex":
        return torch.clamp(up, min=0) ** 2 @ w(p + "down").T
    gate = h @ w(p + "gate").T
    gate = 0.5 * gate * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (gate + 0.044715 * gate ** 3))) if arch == "Gudutar" else _silu(gate)
    return (gate * up) @ w(p + "down").T


def _feed_forward(arch, h, w, mlp):
    if mlp["kind"] == "dense":
        return _one_ff(arch, h, w, "", False)
    r = mlp["router"]
    z = h @ w("router").T
    scores = torch.sigmoid(z) if arch in ("Nesezen", "Pamunex") else torch.softmax(z, dim=-1) if arch == "Mutapel" else z + w("router.b")
    choice = scores + w("correction") if arch == "Mutapel" else scores
    if r.get("groups"):
        per = choice.shape[1] // r["groups"]["count"]
        marks = choice.view(len(h), -1, per).topk(2 if arch == "Pamunex" else 1, dim=2).values.sum(-1)
        open_ = torch.zeros_like(marks, dtype=torch.bool).scatter_(1, marks.topk(r["groups"]["keep"], dim=1).indices, True)
        choice = choice.masked_fill(~open_.repeat_interleave(per, dim=1), float("-inf"))
    ids = choice.topk(r["top"], dim=1).indices
    shares = torch.gather(scores, 1, ids)
    shares = torch.softmax(shares, dim=-1) if arch == "Mekusun" else shares
    out = torch.zeros_like(h)
    for e in range(z.shape[1]):
        rows, slots = (ids == e).nonzero(as_tuple=True)
        x, s = h[rows], shares[rows, slots][:, None]
        if e >= r["experts"]:
            out[rows] += s * x
        elif len(rows):
            out[rows] += _one_ff(arch, s * x, w, f"e{e}.", True) if arch == "Nesezen" else s * _one_ff(arch, x, w, f"e{e}.", True)
    return out + _one_ff(arch, h, w, "shared.", True) * torch.sigmoid(h @ w("shared.sg").T) if mlp.get("shared") else out


def _llama(cfg, W, tokens, rows):
    H, G, d, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    x, T = W("model.embed_tokens.weight")[tokens], len(tokens)
    for i in range(cfg["num_hidden_layers"]):
        def w(n):
            return W(f"model.layers.{i}.{n}.weight")
        h = _unit(x, eps) * w("input_layernorm")
        q, k, v = ((h @ w(f"self_attn.{n}_proj").T).view(T, -1, d) for n in "qkv")
        q, k = (_turn(t, cfg["rope_theta"], d, scaling=cfg.get("rope_scaling"), single=True) for t in (q, k))
        x = x + _attend(q, k, v, d ** -0.5) @ w("self_attn.o_proj").T
        h = _unit(x, eps) * w("post_attention_layernorm")
        x = x + (_silu(h @ w("mlp.gate_proj").T) * (h @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
    head = W("model.embed_tokens.weight") if cfg["tie_word_embeddings"] else W("lm_head.weight")
    return (_unit(x[rows], eps) * W("model.norm.weight")) @ head.T


def _other(cfg, W, tokens, rows):
    arch, eps = cfg["architecture"], cfg["norm"]["eps"]
    emb = cfg.get("embedding") or {}
    x = W("embed")[tokens] * emb.get("scale", 1.0)
    if emb.get("bigram"):
        b = emb["bigram"]
        t = torch.tensor(tokens, device=x.device)
        hashed = (t[:-1] * b["mul_prev"] + t[1:] * b["mul_cur"]) % b["buckets"]
        x = x + W("bigram")[torch.cat([hashed.new_tensor([b["buckets"]]), hashed])]
    x0, results = x, [x]

    def norm(x, n):
        if arch in ("Gudutar", "Pamunex"):
            return _layer_norm(x, W(n), W(n + ".b"), eps)
        if arch == "Nesezen":
            return torch.tanh(W(n + ".alpha") * x) * W(n) + W(n + ".b")
        return _unit(x, eps) * (W(n) if arch == "Renadra" else 1.0 + W(n))

    def add(x, p, n, branch):
        if arch in ("Gudutar", "Pamunex"):
            return x + norm(branch(x), p + n)
        y = branch(norm(x, p + n))
        if arch == "Mutapel":
            return x + cfg["residual_mult"] * norm(y, p + n + "b")
        return x + W(p + "ls" + n[-1]) * norm(y, p + n + "b") if arch == "Mekusun" else x + y

    for i, starts in run_order(cfg):
        layer, p = cfg["layers"][i], f"l{i}."
        kind, m = layer["type"], layer["mixer"]
        if arch == "Mutapel" and starts:
            x = torch.cat([x, x0], dim=1) @ W("loop.in").T
        elif arch == "Renadra" and starts > 1:
            x = x + x0

        def of(prefix):
            return lambda n: W(f"{p}{prefix}{n}")

        def mix(h):
            if kind == "parallel":
                left, right = of("mix.left."), of("mix.right.")
                return (m["left_scale"] * (_mix(arch, "left", h, left, m["left"], eps) @ left("o").T)
                        + m["right_scale"] * (_mix(arch, "lightning", h, right, m["right"], eps) @ right("o").T))
            w = of("mix.")
            y = _mix(arch, kind, h, w, m, eps) @ w("o").T
            return y + w("o.b") if kind == "attention" and arch in ("Mutapel", "Renadra") else y

        x = add(x, p, "norm1", mix)
        if layer["mlp"]:
            x = add(x, p, "norm2", lambda h: _feed_forward(arch, h, of("mlp."), layer["mlp"]))
        if arch == "Mekusun":
            results.append(x)
            x = sum(c * r for c, r in zip(W(p + "dwa"), results))
    z = norm(x[rows], "final.norm") @ W("embed" if arch == "Pamunex" else "head").T * cfg.get("logit_scale", 1.0)
    return cfg["logit_softcap"] * torch.tanh(z / cfg["logit_softcap"]) if cfg.get("logit_softcap") else z


@torch.no_grad()
def exact(case, seed):
    """Whole sequences, one after the other, in float64."""
    cfg = configuration(case)
    shapes, held = tensors(cfg), {}

    def W(name):
        if name not in held:
            held[name] = weight(cfg, name, shapes[name]).double()
        return held[name]

    out = []
    for tokens, start in requests(case, seed):
        rows = [start + r for r in wanted(case, len(tokens) - start)]
        out.append((_llama if "architectures" in cfg else _other)(cfg, W, tokens, rows))
    return torch.cat(out)
