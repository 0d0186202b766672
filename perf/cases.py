"""The work that is measured: requests served through the public entry points, over the
architectures, data types, batch sizes and prompt lengths that the library is used with.

A pass of a serving case is what a program with a loaded model and an open session does for a
batch of requests: take a slot a request, run the prompts as one step, run `new` further steps
of one given token a sequence, and give the slots back.  It returns the float32 logits of every
step.  The tokens after the prompt are given and not drawn (as when a recorded trace is replayed
or a continuation is scored), so that a rounding cannot change which tokens the later steps see.
A pass of the sampling case draws tokens from logits at hand.

Weights are drawn from the seed under their checkpoint names and stored in bfloat16, as
checkpoints are.  Sizes are those of `bench.py`: the Qwen3 0.6B and 8B shapes, and its 2k shape
of the other architectures.  Routers follow the class of a row's token by a clear margin, as
trained ones mostly do: a choice that hangs on the last bit would make outputs incomparable.
"""
import math

import torch

from edge_infer_amd.api import Model
from edge_infer_amd.sampling import Sampler, SamplingParams

DEVICE = "cuda"
F64 = torch.float64
BF16 = torch.bfloat16
CLASSES = 16          # classes of tokens that the routers follow

# ---------------------------------------------------------------------------- configurations
# layers, width, heads, kv heads, head size, feed-forward width, tied embeddings
QWEN = {"qwen3-0.6b": (28, 1024, 16, 8, 128, 3072, True),
        "qwen3-8b": (36, 4096, 32, 8, 128, 12288, False)}
QWEN_VOCAB = 151936
# the 2k shape: layers, width, state heads, their key heads, attention heads, kv heads, head
# size, window or chunk, vocabulary
LAYERS, WIDTH, D_HEADS, D_KV, A_HEADS, A_KV, DIM, WINDOW, VOCAB = 8, 2048, 16, 8, 16, 4, 128, 1024, 32000
GATED = (2 * 4 * WIDTH // 3 + 255) // 256 * 256


def qwen_config(name):
    layers, hidden, heads, kv_heads, dim, ff, tied = QWEN[name]
    return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "vocab_size": QWEN_VOCAB,
            "hidden_size": hidden, "num_hidden_layers": layers, "num_attention_heads": heads,
            "num_key_value_heads": kv_heads, "head_dim": dim, "intermediate_size": ff,
            "max_position_embeddings": 40960, "bos_token_id": 151643, "eos_token_id": 151645,
            "rms_norm_eps": 1e-6, "rope_theta": 1e6, "tie_word_embeddings": tied,
            "hidden_act": "silu"}


def attention_sizes(**more):
    return dict({"heads": A_HEADS, "kv_heads": A_KV, "dim": DIM, "vdim": DIM, "scale": DIM ** -0.5,
                 "mask": {"size": WINDOW}}, **more)


def tirurax_config():
    ff = {"kind": "dense", "ff": 4 * WIDTH}
    delta = {"type": "delta", "mixer": {"heads": D_HEADS, "kv_heads": D_KV, "dim": DIM,
                                        "vdim": DIM, "conv": 4}, "mlp": ff}
    attention = {"type": "attention", "mixer": attention_sizes(), "mlp": ff}
    return {"architecture": "Tirurax", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "layers": [delta if i % 2 == 0 else attention for i in range(LAYERS)]}


def zadenex_config():
    ff = {"kind": "dense", "ff": GATED}
    memory = {"type": "mlstm", "mixer": {"heads": D_HEADS, "dim": DIM, "vdim": DIM,
                                         "gate_cap": 15.0}, "mlp": ff}
    latent = {"type": "latent_attention",
              "mixer": {"heads": A_HEADS, "dim": DIM, "rot_dim": DIM // 2, "vdim": DIM,
                        "kv_rank": 4 * DIM, "q_rank": WIDTH // 2 + DIM,
                        "scale": (1.5 * DIM) ** -0.5, "rot": {"base": 10000.0, "dims": DIM // 2}},
              "mlp": ff}
    window = {"type": "attention", "mixer": attention_sizes(), "mlp": ff}
    return {"architecture": "Zadenex", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0}, "residual_mult": 0.5,
            "loop": {"start": 2, "stop": LAYERS, "times": 1},
            "layers": [memory if i % 2 == 0 else (latent if i % 4 == 1 else window)
                       for i in range(LAYERS)]}


def vafepel_config():
    dense = {"kind": "dense", "ff": GATED, "limit": 7.0}
    routed = {"kind": "moe", "expert": {"ff": GATED // 2}, "router": {"experts": 8, "top": 2}}
    space = {"type": "mamba2", "mixer": {"heads": WIDTH // 64, "vdim": 64, "state": 128,
                                         "groups": 8, "conv": 4, "norm_groups": 8}}
    window = {"type": "attention", "mixer": attention_sizes(
        v_mix=True, rot={"base": 500000.0, "dims": DIM // 2,
                         "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})}
    return {"architecture": "Vafepel", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "logit_scale": 0.02, "logit_softcap": 30.0,
            "layers": [dict(space if i % 2 == 0 else window, mlp=dense if i % 4 < 2 else routed)
                       for i in range(LAYERS)]}


def gopuzen_config():
    dense = {"kind": "dense", "ff": GATED}
    routed = {"kind": "moe", "expert": {"ff": GATED // 2},
              "router": {"experts": 8, "top": 2, "identity": 2}}
    decay = [1.0 - 2.0 ** (-5.0 - 4.0 * h / (D_HEADS - 1)) for h in range(D_HEADS)]
    left = {"heads": A_HEADS, "kv_heads": A_KV, "dim": DIM, "vdim": DIM, "scale": DIM ** -0.5,
            "q_temp": {"coef": 0.1, "every": 1024}}
    parallel = {"type": "parallel", "mixer": {"left": left, "right": {
        "heads": D_HEADS, "dim": DIM, "vdim": DIM, "decay": decay}}}
    layers = []
    for i in range(LAYERS):
        mlp = dense if i % 4 < 2 else routed
        if i % 2 == 0:
            layers.append(dict(parallel, mlp=mlp))
            continue
        mixer = attention_sizes(mask={"size": WINDOW, "pool": 64},
                                rot={"base": 500000.0, "dims": DIM // 2})
        if i % 4 == 3:                  # every second one reads the keys of the one before it
            mixer["kv_from"] = i - 2
        layers.append({"type": "attention", "mixer": mixer, "mlp": mlp})
    return {"architecture": "Gopuzen", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0}, "canon": {"taps": 4}, "layers": layers}


def dazapel_config():
    gated = (2 * 4 * WIDTH // 3 + 511) // 512 * 512
    layer = {"type": "attention",
             "mixer": attention_sizes(
                 scale=1.5 * DIM ** -0.5, mask={"size": WINDOW, "keep_first": 16},
                 rot={"base": 500000.0, "dims": DIM,
                      "scaling": {"factor": 4.0, "original": 8192, "fast": 16.0, "slow": 1.0}}),
             "mlp": {"kind": "moe", "expert": {"ff": gated // 8, "limit": 7.0},
                     "router": {"experts": 16, "top": 4, "scale": 1.5,
                                "groups": {"count": 4, "keep": 2}},
                     "shared": {"ff": gated // 2, "limit": 7.0}}}
    return {"architecture": "Dazapel", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "residual_mult": 0.5, "loop": {"start": 2, "stop": LAYERS, "times": 1},
            "layers": [layer] * LAYERS}


def lemotar_config():
    mlp = {"kind": "dense", "ff": GATED}
    parallel = {"type": "parallel", "mixer": {
        "left": attention_sizes(softcap=30.0, rot={"base": 500000.0, "dims": DIM // 4}),
        "right": {"heads": D_HEADS, "kv_heads": D_KV, "dim": DIM, "vdim": DIM, "conv": 4}},
        "mlp": mlp}
    layers = []
    for i in range(LAYERS):
        if i % 2 == 0:
            layers.append(parallel)
            continue
        mixer = {"heads": A_HEADS, "dim": DIM, "rot_dim": DIM // 2, "vdim": DIM, "kv_rank": 4 * DIM,
                 "scale": (1.5 * DIM) ** -0.5, "mask": {"size": WINDOW},
                 "rot": {"base": 500000.0, "dims": DIM // 2,
                         "scaling": {"factor": 4.0, "original": 8192, "fast": 16.0, "slow": 1.0}}}
        if i % 4 == 3:                  # every second one reads the latents of the one before it
            mixer["kv_from"] = i - 2
        layers.append({"type": "latent_attention", "mixer": mixer, "mlp": mlp})
    return {"architecture": "Lemotar", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0}, "postln_alpha": 2.0, "layers": layers}


DESIGNS = {"tirurax": tirurax_config, "zadenex": zadenex_config, "vafepel": vafepel_config,
           "gopuzen": gopuzen_config, "dazapel": dazapel_config, "lemotar": lemotar_config}


def config_of(case):
    return qwen_config(case["model"]) if case["model"] in QWEN else DESIGNS[case["model"]]()


# ---------------------------------------------------------------------------- weights
def qwen_shapes(cfg):
    h, d, ff = cfg["hidden_size"], cfg["head_dim"], cfg["intermediate_size"]
    q, kv = cfg["num_attention_heads"] * d, cfg["num_key_value_heads"] * d
    tied = cfg["tie_word_embeddings"]
    out = {"model.embed_tokens.weight": ((QWEN_VOCAB, h), "small" if tied else "table"),
           "model.norm.weight": ((h,), "norm")}
    if not tied:
        out["lm_head.weight"] = ((QWEN_VOCAB, h), "small")
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        for name, shape in (("self_attn.q_proj", (q, h)), ("self_attn.k_proj", (kv, h)),
                            ("self_attn.v_proj", (kv, h)), ("self_attn.o_proj", (h, q)),
                            ("mlp.gate_proj", (ff, h)), ("mlp.up_proj", (ff, h)),
                            ("mlp.down_proj", (h, ff))):
            # (what a layer adds to the stream shrinks with the depth, as it is initialised)
            out[f"{p}{name}.weight"] = (shape, "deep" if name in ("self_attn.o_proj", "mlp.down_proj")
                                        else "small")
        for name, size in (("input_layernorm", h), ("post_attention_layernorm", h),
                           ("self_attn.q_norm", d), ("self_attn.k_norm", d)):
            out[f"{p}{name}.weight"] = ((size,), "norm")
    return out


def feed_forward_shapes(out, p, w, mlp, bias=False):
    def three(name, ff):
        for part, shape in (("gate", (ff, w)), ("up", (ff, w)), ("down", (w, ff))):
            out[name + part] = (shape, "matrix")
            if bias:
                out[f"{name}{part}.b"] = ((shape[0],), "bias")
    if mlp["kind"] == "dense":
        three(p + "mlp.", mlp["ff"])
        return
    router = mlp["router"]
    grouped = router.get("groups") is not None
    out[p + "mlp.router"] = ((router["experts"] + router.get("identity", 0), w),
                             "grouped_router" if grouped else "router")
    if "identity" in router:
        out[p + "mlp.correction"] = ((router["experts"] + router["identity"],), "correction")
    for e in range(router["experts"]):
        out.update({f"{p}mlp.e{e}.{part}": (shape, "matrix") for part, shape in
                    (("gate", (mlp["expert"]["ff"], w)), ("up", (mlp["expert"]["ff"], w)),
                     ("down", (w, mlp["expert"]["ff"])))})
    if mlp.get("shared"):
        three(p + "mlp.shared.", mlp["shared"]["ff"])


def design_shapes(cfg):
    """name -> (shape, law) of every tensor of a model of `cfg`, in the checkpoint's names."""
    kind, w = cfg["architecture"], cfg["width"]
    routed = any(l["mlp"]["kind"] == "moe" for l in cfg["layers"])
    unit = "offset" if kind == "Lemotar" else "norm"
    out = {"embed": ((cfg["vocab"], w), "classes" if routed else "table"), "final.norm": ((w,), unit)}
    if kind in ("Tirurax", "Zadenex", "Gopuzen", "Lemotar"):
        out["head"] = ((cfg["vocab"], w), "matrix")
    if kind == "Vafepel":
        out["embed.norm"] = ((w,), "wide_norm")
    if kind == "Gopuzen":
        out["final.norm.b"] = ((w,), "bias")
    if cfg.get("loop"):
        if kind == "Zadenex":
            out["loop.in"] = ((w, 2 * w), "matrix")
        out["loop.step"] = ((cfg["loop"]["times"], w), "bias")
    norms = {"Tirurax": ("norm1", "norm2"), "Lemotar": ("norm1", "norm2"), "Vafepel": ("norm1", "norm2"),
             "Zadenex": ("norm1", "norm1b", "norm2", "norm2b"),
             "Gopuzen": ("norm1", "norm1b", "norm2", "norm2b"),
             "Dazapel": ("norm1", "norm1b", "norm2", "norm2b")}[kind]
    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"], f"l{i}."
        for name in norms:
            out[p + name] = ((w,), unit)
            if kind == "Gopuzen":
                out[f"{p}{name}.b"] = ((w,), "bias")
        if kind == "Gopuzen":
            for n in "12":
                out[p + "ls" + n] = ((w,), "norm")
                out[p + "canon" + n] = ((w, cfg["canon"]["taps"]), "filter")

        def matrices(prefix, bias=False, **rows):
            for name, count in rows.items():
                out[prefix + name] = ((count, w), "matrix")
                if bias:
                    out[f"{prefix}{name}.b"] = ((count,), "bias")

        def softmax(prefix, m, bias=False, gate=0):
            q, k, v = m["heads"] * m["dim"], m["kv_heads"] * m["dim"], m["kv_heads"] * m["vdim"]
            matrices(prefix, bias, q=q)
            if m.get("kv_from") is None:
                matrices(prefix, bias, k=k)
                if "softcap" not in m:
                    matrices(prefix, bias, v=v)
            if gate:
                matrices(prefix, g=gate)
            out[prefix + "o"] = ((w, m["heads"] * m["vdim"]), "matrix")
            return q, k

        def recurrent(prefix, m):
            qk, v = m["kv_heads"] * m["dim"], m["heads"] * m["vdim"]
            for name, rows in (("q", qk), ("k", qk), ("v", v)):
                matrices(prefix, **{name: rows})
                out[f"{prefix}{name}.conv"] = ((rows, m["conv"]), "filter")
            matrices(prefix, b=m["heads"])
            out[prefix + "A_log"] = ((m["heads"],), "rate")
            out[prefix + "norm"] = ((m["vdim"],), "norm")
            out[prefix + "o"] = ((w, v), "matrix")
            return v
        s = p + "mix."
        if layer["type"] == "delta":
            v = recurrent(s, m)
            matrices(s, a=m["heads"], g=v)
            out[s + "dt_bias"] = ((m["heads"],), "step")
        elif layer["type"] == "mlstm":
            qk, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            matrices(s, q=qk, k=qk, v=v, g=v, i=m["heads"], f=m["heads"])
            out[s + "i.b"] = ((m["heads"],), "bias")
            out[s + "f.b"] = ((m["heads"],), "forget")
            out[s + "norm"] = ((v,), "norm")
            out[s + "o"] = ((w, v), "matrix")
        elif layer["type"] == "mamba2":
            inner = m["heads"] * m["vdim"]
            channels = inner + 2 * m["groups"] * m["state"]
            matrices(s, **{"in": inner + channels + m["heads"]})
            out[s + "conv"] = ((channels, m["conv"]), "filter")
            out[s + "conv.b"] = ((channels,), "bias")
            out[s + "dt_bias"] = ((m["heads"],), "step")
            out[s + "A_log"] = ((m["heads"],), "rate")
            out[s + "D"] = ((m["heads"],), "norm")
            out[s + "norm"] = ((inner,), "norm")
            out[s + "o"] = ((w, inner), "matrix")
        elif layer["type"] == "latent_attention":
            H, d, r, e, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            if "q_rank" in m:
                matrices(s, dq=m["q_rank"])
                out[s + "dq.norm"] = ((m["q_rank"],), "norm")
                out[s + "uq"] = ((H * (d + r), m["q_rank"]), "matrix")
            else:
                matrices(s, q=H * (d + r))
            if m.get("kv_from") is None:
                matrices(s, dkv=rank + r)
                out[s + "dkv.norm"] = ((rank,), "norm")
            out[s + "uk"], out[s + "uv"] = ((H * d, rank), "matrix"), ((H * e, rank), "matrix")
            out[s + "sink"] = ((H,), "sink")
            matrices(s, g=H if kind == "Zadenex" else H * e)
            out[s + "o"] = ((w, H * e), "matrix")
        elif layer["type"] == "parallel" and kind == "Gopuzen":
            softmax(s + "left.", m["left"])
            r = m["right"]
            qk, v = r["heads"] * r["dim"], r["heads"] * r["vdim"]
            matrices(s + "right.", q=qk, k=qk, v=v, g=v)
            out[s + "right.norm"] = ((v,), "norm")
            out[s + "right.o"] = ((w, v), "matrix")
        elif layer["type"] == "parallel":
            left, right = m["left"], m["right"]
            q, k = softmax(s + "left.", left)
            out[s + "left.q.norm"], out[s + "left.k.norm"] = ((q,), "norm"), ((k,), "norm")
            v = recurrent(s + "right.", right)
            decays, rank = right["heads"] * right["dim"], right["dim"]
            out[s + "right.dt_bias"] = ((decays,), "step")
            matrices(s + "right.", a1=rank, g1=rank)
            out[s + "right.a2"] = ((decays, rank), "matrix")
            out[s + "right.g2"] = ((v, rank), "matrix")
        else:
            q, k = softmax(s, m, bias=kind in ("Tirurax", "Zadenex", "Dazapel"),
                           gate={"Vafepel": m["heads"] * m["vdim"], "Gopuzen": m["heads"],
                                 "Dazapel": m["heads"] * m["vdim"]}.get(kind, 0))
            if kind == "Tirurax":
                out[s + "q.norm"], out[s + "k.norm"] = ((q,), "norm"), ((k,), "norm")
            if kind == "Vafepel":
                out[s + "q.norm"], out[s + "k.norm"] = ((m["dim"],), "norm"), ((m["dim"],), "norm")
                out[s + "vmix"] = ((), "mix")
            if kind in ("Tirurax", "Vafepel"):
                out[s + "sink"] = ((m["heads"],), "sink")
            if kind == "Zadenex":
                out[s + "talk"] = ((m["heads"], m["heads"]), "talk")
            if kind in ("Zadenex", "Dazapel"):
                out[s + "o.b"] = ((w,), "bias")
        if layer["type"] == "parallel":
            out[s + "left.out"] = out[s + "right.out"] = ((w,), "norm")
        feed_forward_shapes(out, p, w, layer["mlp"], bias=kind in ("Zadenex", "Gopuzen"))
    if kind == "Tirurax":       # an ungated feed-forward
        out = {n: s for n, s in out.items() if not n.endswith("mlp.gate")}
    return out


def shapes_of(case, cfg):
    return qwen_shapes(cfg) if case["model"] in QWEN else design_shapes(cfg)


def make_weights(case, cfg, seed):
    """Every tensor of the checkpoint, bfloat16 on the GPU, of order-one signal."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(shape, scale=1.0):
        return torch.randn(shape, generator=g, device=DEVICE, dtype=BF16).mul_(scale)

    def uniform(shape, low, high):
        return (torch.rand(shape, generator=g, device=DEVICE) * (high - low) + low).to(BF16)
    # the directions that mark the classes of tokens
    width = cfg.get("width", 8)
    classes = torch.randn((CLASSES, width), generator=g, device=DEVICE)

    def router(outputs, values):
        """Rows whose product with a row of class c is about values[:, c]."""
        return ((values @ classes) / width).to(BF16)

    def shuffled(values):
        order = torch.rand((CLASSES, len(values)), generator=g, device=DEVICE).argsort(dim=1)
        return torch.tensor(values, device=DEVICE)[order].t()
    out = {}
    for name, (shape, law) in shapes_of(case, cfg).items():
        if law == "small":
            value = normal(shape, 0.02)
        elif law == "deep":
            value = normal(shape, 0.02 * (2.0 * cfg["num_hidden_layers"]) ** -0.5)
        elif law == "matrix":
            value = normal(shape, shape[1] ** -0.5)
        elif law == "table":
            value = normal(shape)
        elif law == "classes":
            of = torch.arange(shape[0], device=DEVICE) % CLASSES
            value = normal(shape) + (4.0 * classes[of]).to(BF16)
        elif law == "router":
            count = shape[0]
            value = router(count, shuffled([4.0 * e / (count - 1) - 2.0 for e in range(count)]))
        elif law == "grouped_router":       # four groups of four, two of them well ahead
            best = shuffled([1.5, 0.7, -0.8, -1.6]).repeat_interleave(4, dim=0)
            within = torch.cat([shuffled([-0.9, -0.3, 0.3, 0.9]) for _ in range(4)])
            value = router(shape[0], best + within)
        elif law == "correction":
            value = normal(shape, 0.01)
        elif law in ("norm", "offset", "wide_norm"):
            mean = {"norm": 1.0, "offset": 0.0, "wide_norm": 4.0}[law]
            value = uniform(shape, mean - 0.1, mean + 0.1)
        elif law == "bias":
            value = normal(shape, 0.1)
        elif law == "filter":
            value = normal(shape, 0.5)
        elif law == "rate":
            value = uniform(shape, -3.0, 0.5)
        elif law == "step":
            value = uniform(shape, -4.0, 0.0)
        elif law == "forget":
            value = uniform(shape, 1.0, 4.0)
        elif law == "sink":
            value = uniform(shape, -1.0, 1.0)
        elif law == "mix":
            value = uniform(shape, 0.1, 0.6)
        elif law == "talk":
            value = torch.eye(shape[0], device=DEVICE, dtype=BF16) + normal(shape, 0.1)
        out[name] = value
    return out


# ---------------------------------------------------------------------------- cases
def listed():
    return [
        # one decoded token of a batch, drawn as the README's example draws (temperature 0.7, top 20)
        {"name": "sample-b8", "kind": "sample", "batch": 8, "vocab": QWEN_VOCAB, "temperature": 0.7,
         "top_p": 1.0, "top_k": 20},
        # a chat turn on the small model: a short question, an answer at batch 1 (launches count)
        {"name": "qwen3-0.6b-chat", "kind": "serve", "model": "qwen3-0.6b", "dtype": "bf16", "batch": 1,
         "prompt": 23, "ragged": False, "new": 32},
        # the small model behind a server: unequal prompts that start together
        {"name": "qwen3-0.6b-serve-b32", "kind": "serve", "model": "qwen3-0.6b", "dtype": "bf16",
         "batch": 32, "prompt": 2048, "ragged": True, "new": 16},
        # the 32-bit path, odd sizes
        {"name": "qwen3-0.6b-f32", "kind": "serve", "model": "qwen3-0.6b", "dtype": "fp32", "batch": 3,
         "prompt": 301, "ragged": True, "new": 8},
        # the headline: decoding at batch 8 on the 8B shape
        {"name": "qwen3-8b-decode-b8", "kind": "serve", "model": "qwen3-8b", "dtype": "bf16", "batch": 8,
         "prompt": 256, "ragged": False, "new": 32},
        # the headline's prompt: a long document read once, one token after it
        {"name": "qwen3-8b-prefill", "kind": "serve", "model": "qwen3-8b", "dtype": "bf16", "batch": 1,
         "prompt": 2048, "ragged": False, "new": 1},
        # the other architectures: prompts and decoding in one request, at different batches
        {"name": "tirurax-b1", "kind": "serve", "model": "tirurax", "dtype": "bf16", "batch": 1,
         "prompt": 2048, "ragged": False, "new": 16},
        {"name": "zadenex-b8", "kind": "serve", "model": "zadenex", "dtype": "bf16", "batch": 8,
         "prompt": 512, "ragged": False, "new": 16},
        {"name": "vafepel-b2", "kind": "serve", "model": "vafepel", "dtype": "bf16", "batch": 2,
         "prompt": 1777, "ragged": False, "new": 16},
        {"name": "gopuzen-b1", "kind": "serve", "model": "gopuzen", "dtype": "bf16", "batch": 1,
         "prompt": 2048, "ragged": False, "new": 16},
        {"name": "dazapel-b16", "kind": "serve", "model": "dazapel", "dtype": "bf16", "batch": 16,
         "prompt": 300, "ragged": True, "new": 16},
        {"name": "lemotar-b4", "kind": "serve", "model": "lemotar", "dtype": "bf16", "batch": 4,
         "prompt": 1024, "ragged": True, "new": 16},
    ]


def draw(rng):
    def spread(low, high):
        return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))
    model = rng.choice(["sample", "qwen3-0.6b", "qwen3-0.6b", "qwen3-0.6b-f32", "qwen3-8b", "qwen3-8b",
                        *DESIGNS])
    if model == "sample":
        return {"kind": "sample", "batch": spread(1, 64), "vocab": rng.choice([VOCAB, QWEN_VOCAB]),
                "temperature": rng.choice([0.0, 0.7, 1.0]), "top_p": rng.choice([0.9, 1.0]),
                "top_k": spread(2, 200)}
    if model == "qwen3-8b":
        batch = spread(1, 64)
        return {"kind": "serve", "model": model, "dtype": "bf16", "batch": batch,
                "prompt": spread(16, 2048 // batch), "ragged": rng.random() < 0.5,
                "new": rng.randint(0, 16)}
    if model == "qwen3-0.6b-f32":
        batch = spread(1, 16)
        return {"kind": "serve", "model": "qwen3-0.6b", "dtype": "fp32", "batch": batch,
                "prompt": spread(16, 1024 // batch), "ragged": rng.random() < 0.5,
                "new": rng.randint(0, 8)}
    batch = spread(1, 64)
    if model in DESIGNS and rng.random() < 0.2:
        return {"kind": "serve", "model": model, "dtype": "fp32", "batch": batch,
                "prompt": spread(16, 1024 // batch), "ragged": rng.random() < 0.5,
                "new": rng.randint(0, 8)}
    return {"kind": "serve", "model": model, "dtype": "bf16", "batch": batch,
            "prompt": spread(16, min(2048, 8192 // batch)), "ragged": rng.random() < 0.5,
            "new": rng.randint(0, 32)}


def tokens_of(case, vocab, seed):
    """(prompts, the tokens after them) as lists of ids; ragged prompts are uniform in
    [prompt / 32, prompt] (the generation workload's 64 to 2,048)."""
    g = torch.Generator().manual_seed(seed)
    longest = case["prompt"]
    lengths = [longest] * case["batch"]
    if case["ragged"]:
        lengths = torch.randint(max(1, longest // 32), longest + 1, (case["batch"],), generator=g).tolist()
    ids = [torch.randint(0, vocab, (n + case["new"],), generator=g).tolist() for n in lengths]
    return [i[:n] for i, n in zip(ids, lengths)], [i[n:] for i, n in zip(ids, lengths)]


def model_type(case):
    return f"{'qwen3' if case['model'] in QWEN else case['model']}_{case['dtype']}"


def prepare(case, seed):
    if case["kind"] == "sample":
        g = torch.Generator(device=DEVICE).manual_seed(seed)
        logits = torch.randn((case["batch"], case["vocab"]), generator=g, device=DEVICE) * 2.0
        return {"logits": logits, "sampler": Sampler(DEVICE),
                "params": SamplingParams(temperature=case["temperature"], top_p=case["top_p"],
                                         top_k=case["top_k"], seed=seed),
                "streams": list(range(case["batch"])), "counters": [17] * case["batch"]}
    cfg = config_of(case)
    model = Model(cfg, make_weights(case, cfg, seed), model_type(case))
    prompts, after = tokens_of(case, model.decoder.spec.vocab_size, seed)
    session = model.new_session(capacity=case["prompt"] + max(1, case["new"]), max_batch=case["batch"])
    return {"session": session, "prompts": prompts, "after": after}


def run(state):
    if "sampler" in state:
        return state["sampler"](state["logits"], state["params"], state["streams"], state["counters"])
    session, after = state["session"], state["after"]
    slots = [session.begin() for _ in after]
    logits = [session.step([(slot, ids, [len(ids) - 1]) for slot, ids in zip(slots, state["prompts"])])]
    for t in range(len(after[0])):
        logits.append(session.step([(slot, [ids[t]], [0]) for slot, ids in zip(slots, after)]))
    for slot in slots:
        session.end(slot)
    return logits


# ---------------------------------------------------------------------------- what a pass needs
def state_elements(cfg):
    """Floats of fixed-size state that a sequence's decode step reads and writes."""
    total = 0
    for layer in cfg.get("layers", ()):
        m = layer["mixer"]
        if layer["type"] == "parallel":
            m = m["right"]
        elif layer["type"] not in ("delta", "mlstm", "mamba2"):
            continue
        total += m["heads"] * m["vdim"] * m.get("state", m.get("dim"))
    return total


def attention_layers(cfg):
    """(heads, key size, value size, cached elements a token, window or None) of every one."""
    if "layers" not in cfg:
        d, g = cfg["head_dim"], cfg["num_key_value_heads"]
        return [(cfg["num_attention_heads"], d, d, 2 * g * d, None)] * cfg["num_hidden_layers"]
    out = []
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "parallel":
            m = m["left"]
        window = (m.get("mask") or {}).get("size")
        if layer["type"] == "latent_attention":
            out.append((m["heads"], m["dim"] + m["rot_dim"], m["vdim"], m["kv_rank"] + m["rot_dim"], window))
        elif "kv_heads" in m and "conv" not in m:
            out.append((m["heads"], m["dim"], m["vdim"], m["kv_heads"] * (m["dim"] + m["vdim"]), window))
    return out


def work(case):
    """Weights read once a step (of the experts those that its rows choose), the cache and the
    state of the live sequences, the logits; two operations a weight and row, the visible
    pairs of attention, the state's update and read-out."""
    if case["kind"] == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 4 * n, "flops": 2 * n}
    cfg = config_of(case)
    item = 2 if case["dtype"] == "bf16" else 4
    prompts, _ = tokens_of(case, QWEN_VOCAB, 1)
    lengths = [len(p) for p in prompts]
    head = case_vocab = cfg.get("vocab_size", cfg.get("vocab"))
    head *= cfg.get("hidden_size", cfg.get("width"))
    dense, expert, top, experts = 0, 0, 1, 1
    for name, (shape, _) in shapes_of(case, cfg).items():
        if len(shape) != 2 or name in ("embed", "head", "model.embed_tokens.weight", "lm_head.weight"):
            continue
        if ".mlp.e" in name:
            expert += shape[0] * shape[1]
        else:
            dense += shape[0] * shape[1]
    for layer in cfg.get("layers", ()):
        if layer["mlp"]["kind"] == "moe":
            top, experts = layer["mlp"]["router"]["top"], layer["mlp"]["router"]["experts"]
    nbytes = flops = 0
    for step in range(1 + case["new"]):
        rows = sum(lengths) if step == 0 else case["batch"]
        touched = 1.0 - (1.0 - top / experts) ** min(rows, CLASSES)
        nbytes += item * (dense + head + expert * touched) + 4 * case["batch"] * case_vocab
        flops += 2 * rows * (dense + expert * top / experts) + 2 * case["batch"] * head
        states = state_elements(cfg)
        nbytes += 4 * case["batch"] * states * (1 if step == 0 else 2)
        flops += 8 * rows * states
        for heads, key, value, cached, window in attention_layers(cfg):
            for n in lengths:
                if step == 0:
                    near = n if window is None else min(n, window)
                    pairs = near * (near + 1) / 2 + (n - near) * near
                    nbytes += item * n * cached
                else:
                    pairs = n + step if window is None else min(n + step, window)
                    nbytes += item * pairs * cached
                flops += 2 * heads * (key + value) * pairs
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    # four times what the path was measured to be off the 64-bit results
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": {"vafepel": 0.008, "gopuzen": 0.018, "dazapel": 0.008, "lemotar": 0.024}.get(
        case["model"], 0.03)}


# ---------------------------------------------------------------------------- in 64 bits
def rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def silu(x):
    return x * torch.sigmoid(x)


class Plain:
    """A model in 64 bits: whole sequences side by side, padded behind their ends (every
    mechanism is causal), recurrences token by token."""

    def __init__(self, case, cfg, weights):
        self.case, self.cfg, self.w = case, cfg, weights
        self.eps = cfg["norm"]["eps"] if "norm" in cfg else cfg["rms_norm_eps"]
        self.first_values = None
        self.kept = {}

    def get(self, name):
        return self.w[name].to(F64)

    def linear(self, x, name):
        y = x @ self.get(name).T
        return y + self.get(name + ".b") if name + ".b" in self.w else y

    def norm(self, x, name, offset=0.0):
        return rms(x, self.eps) * (self.get(name) + offset)

    def layer_norm(self, x, name):
        x = x - x.mean(dim=-1, keepdim=True)
        return rms(x, self.eps) * self.get(name) + self.get(name + ".b")

    @staticmethod
    def rotate(x, freqs, neighbours=False, magnitude=1.0):
        """x [B, T, heads, dim]: pairs of its first elements turn by position * frequency."""
        angle = torch.arange(x.shape[1], device=x.device, dtype=F64)[:, None] * freqs[None, :].to(F64)
        cos, sin = (magnitude * f(angle)[None, :, None, :] for f in (torch.cos, torch.sin))
        half, out = freqs.numel(), x.clone()
        a, b = ((slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if neighbours
                else (slice(0, half), slice(half, 2 * half)))
        out[..., a], out[..., b] = x[..., a] * cos - x[..., b] * sin, x[..., b] * cos + x[..., a] * sin
        return out

    @staticmethod
    def frequencies(rot):
        """(frequencies, what cosine and sine are multiplied by)."""
        base, dims, scaling = float(rot["base"]), rot["dims"], rot.get("scaling")
        f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
        magnitude = 1.0
        if scaling and "low" in scaling:
            def bent(v):
                length = 2.0 * math.pi / v
                low, high, original = scaling["low"], scaling["high"], scaling["original"]
                if length < original / high:
                    return v
                if length > original / low:
                    return v / scaling["factor"]
                s = (original / length - low) / (high - low)
                return (1.0 - s) * v / scaling["factor"] + s * v
            f = [bent(v) for v in f]
        elif scaling:
            def pair_of(turns):
                return dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
            low = max(math.floor(pair_of(scaling["fast"])), 0)
            high = min(math.ceil(pair_of(scaling["slow"])), dims - 1)
            ramp = [min(max((i - low) / max(high - low, 0.001), 0.0), 1.0) for i in range(len(f))]
            f = [v / scaling["factor"] * r + v * (1.0 - r) for v, r in zip(f, ramp)]
            magnitude = 0.1 * math.log(scaling["factor"]) + 1.0
        return torch.tensor(f, dtype=F64, device=DEVICE), magnitude

    def softmax(self, q, k, v, scale, visible, extra=None, talk=None, cap=None, slopes=None, pool=None):
        """q [B, T, H, d], k [B, T, G, d], v [B, T, G, e] -> [B, T, H e]; `extra` [H]: a score
        that only enters the denominator; `pool` (window, block): blocks' means before it."""
        B, T, H, _ = q.shape
        share = H // k.shape[2]
        out = torch.empty(B, T, H, v.shape[3], dtype=F64, device=q.device)
        at = torch.arange(T, device=q.device)
        for b in range(B):
            keys, values, seen = k[b], v[b], visible
            if pool is not None and T // pool[1]:
                window, size = pool
                count = T // size
                mean = [x[:count * size].reshape(count, size, *x.shape[1:]).mean(dim=1) for x in (keys, values)]
                keys, values = torch.cat([keys, mean[0]]), torch.cat([values, mean[1]])
                ends = torch.arange(count, device=q.device) * size + size - 1
                seen = torch.cat([visible, ends[None, :] <= at[:, None] - window], dim=1)
            groups = range(1) if talk is not None else range(k.shape[2])
            for g in groups:
                if talk is not None:
                    heads = slice(0, H)
                    scores = torch.matmul(q[b].transpose(0, 1), keys.repeat_interleave(share, dim=1).permute(1, 2, 0))
                    scores = torch.tensordot(talk, scores * scale, dims=([1], [0]))
                else:
                    heads = slice(g * share, (g + 1) * share)
                    scores = torch.matmul(q[b, :, heads].transpose(0, 1), keys[:, g].T) * scale
                if cap is not None:
                    scores = cap * torch.tanh(scores / cap)
                if slopes is not None:
                    scores = scores - slopes[heads, None, None] * (at[:, None] - at[None, :])
                scores = scores.masked_fill(~seen[None], -math.inf)
                if extra is not None:
                    scores = torch.cat([scores, extra[heads, None, None].expand(-1, T, 1)], dim=2)
                weights = torch.softmax(scores, dim=-1)
                if extra is not None:
                    weights = weights[..., :-1]
                if talk is not None:
                    read = torch.matmul(weights, values.repeat_interleave(share, dim=1).transpose(0, 1))
                else:
                    read = torch.matmul(weights, values[:, g])
                out[b, :, heads] = read.transpose(0, 1)
        return out.reshape(B, T, -1)

    def visible(self, T, window=None, chunk=None, keep=0):
        at = torch.arange(T, device=DEVICE)
        seen = at[None, :] <= at[:, None]
        if window is not None:
            seen = seen & ((at[:, None] - at[None, :] < window) | (at[None, :] < keep))
        if chunk is not None:
            seen = seen & (at[None, :] // chunk == at[:, None] // chunk)
        return seen

    @staticmethod
    def causal_filter(x, taps):
        """sum_j taps[:, j] x[t - J + 1 + j], zeros before the start."""
        count = taps.shape[1]
        padded = torch.nn.functional.pad(x, (0, 0, count - 1, 0))
        return sum(padded[:, j:j + x.shape[1]] * taps[:, j] for j in range(count))

    def split(self, x, heads):
        return x.reshape(*x.shape[:2], heads, -1)

    # -- mixers ---------------------------------------------------------------------------
    def delta(self, h, s, m, channel):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]

        def convolved(name, heads):
            return self.split(silu(self.causal_filter(self.linear(h, s + name), self.get(f"{s}{name}.conv"))), heads)

        def unit(x):
            return x / torch.sqrt((x * x).sum(dim=-1, keepdim=True) + 1e-6)
        q = (unit(convolved("q", G)) * d ** -0.5).repeat_interleave(H // G, dim=2)
        k = unit(convolved("k", G)).repeat_interleave(H // G, dim=2)
        v = convolved("v", H)
        beta = torch.sigmoid(self.linear(h, s + "b"))
        rate = torch.exp(self.get(s + "A_log"))
        if channel:
            z = self.linear(self.linear(h, s + "a1"), s + "a2") + self.get(s + "dt_bias")
            decay = torch.exp(-rate[:, None] * torch.nn.functional.softplus(self.split(z, H)))
            gate = torch.sigmoid(self.linear(self.linear(h, s + "g1"), s + "g2"))
        else:
            z = self.linear(h, s + "a") + self.get(s + "dt_bias")
            decay = torch.exp(-rate * torch.nn.functional.softplus(z))[..., None].expand(*z.shape, d)
            gate = silu(self.linear(h, s + "g"))
        state = torch.zeros(h.shape[0], H, d, v.shape[3], dtype=F64, device=DEVICE)
        out = torch.empty_like(v)
        for t in range(h.shape[1]):
            state = state * decay[:, t, :, :, None]
            u = beta[:, t, :, None] * (v[:, t] - (state * k[:, t, :, :, None]).sum(dim=2))
            state = state + k[:, t, :, :, None] * u[:, :, None, :]
            out[:, t] = (state * q[:, t, :, :, None]).sum(dim=2)
        out = self.norm(out, s + "norm").reshape(gate.shape) * gate
        return self.linear(out, s + "o")

    def mlstm(self, h, s, m):
        H, d, cap = m["heads"], m["dim"], m["gate_cap"]
        q, k, v = (self.split(self.linear(h, s + n), H) for n in "qkv")
        q = q * d ** -0.5
        log_in = cap * torch.tanh(self.linear(h, s + "i") / cap)
        log_forget = torch.nn.functional.logsigmoid(cap * torch.tanh(self.linear(h, s + "f") / cap))
        S = torch.zeros(h.shape[0], H, d, m["vdim"], dtype=F64, device=DEVICE)
        n = torch.zeros(h.shape[0], H, d, dtype=F64, device=DEVICE)
        top = torch.zeros(h.shape[0], H, dtype=F64, device=DEVICE)
        out = torch.empty_like(v)
        for t in range(h.shape[1]):
            new = torch.maximum(log_forget[:, t] + top, log_in[:, t])
            keep, take = torch.exp(log_forget[:, t] + top - new), torch.exp(log_in[:, t] - new)
            S = keep[..., None, None] * S + take[..., None, None] * k[:, t, :, :, None] * v[:, t, :, None, :]
            n = keep[..., None] * n + take[..., None] * k[:, t]
            top = new
            bottom = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
            out[:, t] = (S * q[:, t, :, :, None]).sum(dim=2) / bottom[..., None]
        out = rms(out, self.eps).reshape(*h.shape[:2], -1) * self.get(s + "norm")
        return self.linear(out * torch.sigmoid(self.linear(h, s + "g")), s + "o")

    def mamba2(self, h, s, m):
        H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * P
        z, xbc, dt = self.linear(h, s + "in").split([inner, inner + 2 * G * N, H], dim=-1)
        xbc = silu(self.causal_filter(xbc, self.get(s + "conv")) + self.get(s + "conv.b"))
        x = self.split(xbc[..., :inner], H)
        Bs = self.split(xbc[..., inner:inner + G * N], G).repeat_interleave(H // G, dim=2)
        Cs = self.split(xbc[..., inner + G * N:], G).repeat_interleave(H // G, dim=2)
        dt = torch.nn.functional.softplus(dt + self.get(s + "dt_bias"))
        decay = torch.exp(-torch.exp(self.get(s + "A_log")) * dt)
        S = torch.zeros(h.shape[0], H, N, P, dtype=F64, device=DEVICE)
        y = torch.empty_like(x)
        for t in range(h.shape[1]):
            S = decay[:, t, :, None, None] * S + (dt[:, t, :, None] * Bs[:, t])[..., None] * x[:, t, :, None, :]
            y[:, t] = (S * Cs[:, t, :, :, None]).sum(dim=2)
        y = (y + self.get(s + "D")[:, None] * x).reshape(*h.shape[:2], inner) * silu(z)
        y = rms(self.split(y, m["norm_groups"]), self.eps).reshape(y.shape) * self.get(s + "norm")
        return self.linear(y, s + "o")

    def lightning(self, h, s, m):
        H = m["heads"]
        q, k, v = (self.split(silu(self.linear(h, s + n)), H) for n in "qkv")
        decay = torch.tensor(m["decay"], dtype=F64, device=DEVICE)[:, None, None]
        S = torch.zeros(h.shape[0], H, m["dim"], m["vdim"], dtype=F64, device=DEVICE)
        out = torch.empty_like(v)
        for t in range(h.shape[1]):
            S = decay * S + k[:, t, :, :, None] * v[:, t, :, None, :]
            out[:, t] = (S * q[:, t, :, :, None]).sum(dim=2)
        out = self.norm(out.reshape(*h.shape[:2], -1), s + "norm") * torch.sigmoid(self.linear(h, s + "g"))
        return self.linear(out, s + "o")

    def latent(self, h, s, m, index):
        H, d, rank = m["heads"], m["dim"], m["kv_rank"]
        neighbours = self.cfg["architecture"] == "Zadenex"
        freqs, magnitude = self.frequencies(m["rot"])
        q = (self.linear(self.norm(self.linear(h, s + "dq"), s + "dq.norm"), s + "uq") if s + "dq" in self.w
             else self.linear(h, s + "q"))
        q = self.split(q, H)
        if m.get("kv_from") is None:
            down = self.linear(h, s + "dkv")
            self.kept[index] = (self.norm(down[..., :rank], s + "dkv.norm"),
                                self.rotate(down[:, :, None, rank:], freqs, neighbours, magnitude))
        latent, turned = self.kept[m.get("kv_from", index)]
        k = torch.cat([self.split(self.linear(latent, s + "uk"), H), turned.expand(-1, -1, H, -1)], dim=3)
        q = torch.cat([q[..., :d], self.rotate(q[..., d:], freqs, neighbours, magnitude)], dim=3)
        seen = self.visible(h.shape[1], window=(m.get("mask") or {}).get("size"))
        out = self.softmax(q, k, self.split(self.linear(latent, s + "uv"), H), m["scale"], seen,
                           extra=self.get(s + "sink"))
        gate = torch.sigmoid(self.linear(h, s + "g"))
        if gate.shape[-1] == H:
            gate = gate.repeat_interleave(m["vdim"], dim=-1)
        return self.linear(out * gate, s + "o")

    def attention(self, h, s, m, index):
        kind, T = self.cfg["architecture"], h.shape[1]
        H, G = m["heads"], m["kv_heads"]
        zero = torch.zeros(H, dtype=F64, device=DEVICE)
        window = (m.get("mask") or {}).get("size")
        q = self.linear(h, s + "q")
        k = self.linear(h, s + "k") if s + "k" in self.w else None
        if kind == "Lemotar":
            v = self.split(k, G)
            freqs, _ = self.frequencies(m["rot"])
            q = self.rotate(self.split(self.norm(q, s + "q.norm"), H), freqs, True)
            k = self.rotate(self.split(self.norm(k, s + "k.norm"), G), freqs, True)
            return self.linear(self.softmax(q, k, v, m["scale"], self.visible(T, window), extra=zero,
                                            cap=m["softcap"]), s + "o")
        v = self.split(self.linear(h, s + "v"), G) if s + "v" in self.w else None
        if kind == "Tirurax":
            q, k = self.norm(q, s + "q.norm"), self.norm(k, s + "k.norm")
            slopes = torch.tensor([2.0 ** (-8.0 * (a + 1) / H) for a in range(H)], dtype=F64, device=DEVICE)
            return self.linear(self.softmax(self.split(q, H), self.split(k, G), v, m["scale"],
                                            self.visible(T, chunk=window), extra=self.get(s + "sink"),
                                            slopes=slopes), s + "o")
        q = self.split(q, H)
        k = None if k is None else self.split(k, G)
        if kind == "Zadenex":
            return self.linear(self.softmax(q, k, v, m["scale"], self.visible(T, window), extra=zero,
                                            talk=self.get(s + "talk")), s + "o")
        if "q_temp" in m:
            steps = (torch.arange(T, device=DEVICE) + 1) // m["q_temp"]["every"]
            q = q * (1.0 + m["q_temp"]["coef"] * torch.log(steps.to(F64) + 1.0))[:, None, None]
            return self.linear(self.softmax(q, k, v, m["scale"], self.visible(T)), s + "o")
        freqs, magnitude = self.frequencies(m["rot"])
        if kind == "Gopuzen":
            q = self.rotate(q, freqs, True)
            if m.get("kv_from") is None:
                self.kept[index] = (self.rotate(k, freqs, True), v)
            k, v = self.kept[m.get("kv_from", index)]
            out = self.softmax(q, k, v, m["scale"], self.visible(T, window), pool=(window, m["mask"]["pool"]))
            gate = torch.sigmoid(self.linear(h, s + "g")).repeat_interleave(m["vdim"], dim=-1)
            return self.linear(out * gate, s + "o")
        if kind == "Dazapel":
            q, k = (rms(self.rotate(x, freqs, False, magnitude), self.eps) for x in (q, k))
            out = self.softmax(q, k, v, m["scale"], self.visible(T, window, keep=m["mask"]["keep_first"]))
        else:       # Vafepel
            q = self.rotate(self.norm(q, s + "q.norm"), freqs)
            k = self.rotate(self.norm(k, s + "k.norm"), freqs)
            if self.first_values is None:
                self.first_values = v
            else:
                share = self.get(s + "vmix")
                v = (1.0 - share) * v + share * self.first_values
            out = self.softmax(q, k, v, m["scale"], self.visible(T, window), extra=self.get(s + "sink"))
        return self.linear(out * torch.sigmoid(self.linear(h, s + "g")), s + "o")

    def mixer(self, h, index, layer):
        s, m, kind = f"l{index}.mix.", layer["mixer"], layer["type"]
        if kind == "parallel":
            left = self.attention(h, s + "left.", m["left"], index)
            right = (self.lightning(h, s + "right.", m["right"]) if "decay" in m["right"]
                     else self.delta(h, s + "right.", m["right"], True))
            return 0.5 * (self.norm(left, s + "left.out") + self.norm(right, s + "right.out"))
        if kind == "delta":
            return self.delta(h, s, m, False)
        if kind == "latent_attention":
            return self.latent(h, s, m, index)
        if kind == "attention":
            return self.attention(h, s, m, index)
        return getattr(self, kind)(h, s, m)

    # -- feed-forwards ----------------------------------------------------------------------
    def gated(self, h, name, act):
        return self.linear(act(self.linear(h, name + "gate"), self.linear(h, name + "up")), name + "down")

    def feed_forward(self, h, index, mlp):
        kind, s = self.cfg["architecture"], f"l{index}.mlp."

        def clamped(limit):
            def act(g, u):
                g = g.clamp(max=limit)
                return g * torch.sigmoid(1.702 * g) * (u.clamp(min=-limit, max=limit) + 1.0)
            return act
        if kind == "Tirurax":
            return self.linear(torch.relu(self.linear(h, s + "up")) ** 2, s + "down")
        if mlp["kind"] == "dense":
            act = {"Zadenex": lambda g, u: torch.nn.functional.gelu(g, approximate="tanh") * u,
                   "Vafepel": clamped(mlp.get("limit"))}.get(kind, lambda g, u: silu(g) * u)
            return self.gated(h, s, act)
        router, experts = mlp["router"], mlp["router"]["experts"]
        logits = self.linear(h, s + "router")
        act = lambda g, u: silu(g) * u  # noqa: E731
        if kind == "Vafepel":
            top, chosen = torch.topk(logits, router["top"], dim=-1)
            weights = torch.softmax(top, dim=-1)
        elif kind == "Gopuzen":
            scores = torch.softmax(logits, dim=-1)
            chosen = torch.topk(scores + self.get(s + "correction"), router["top"], dim=-1).indices
            weights = torch.gather(scores, -1, chosen)
        else:
            act = clamped(mlp["expert"]["limit"])
            scores = torch.sigmoid(logits)
            count, keep = router["groups"]["count"], router["groups"]["keep"]
            groups = torch.topk(scores.reshape(*scores.shape[:-1], count, -1), 2, dim=-1).values.sum(-1)
            kept = torch.zeros_like(groups, dtype=torch.bool).scatter_(
                -1, torch.topk(groups, keep, dim=-1).indices, True).repeat_interleave(experts // count, dim=-1)
            chosen = torch.topk(scores.masked_fill(~kept, -1.0), router["top"], dim=-1).indices
            picked = torch.gather(scores, -1, chosen)
            weights = picked / (picked.sum(-1, keepdim=True) + 1e-20) * router["scale"]
        shares = torch.zeros_like(logits).scatter_(-1, chosen, weights)
        out = h * shares[..., experts:].sum(-1, keepdim=True)          # (the identity experts)
        for e in range(experts):
            rows = shares[..., e] > 0
            if bool(rows.any()):
                out[rows] += shares[rows][:, e:e + 1] * self.gated(h[rows], f"{s}e{e}.", act)
        if mlp.get("shared"):
            out = out + self.gated(h, s + "shared.", clamped(mlp["shared"]["limit"]))
        return out

    # -- whole models -----------------------------------------------------------------------
    def qwen(self, ids):
        cfg = self.cfg
        H, G, d, T = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], ids.shape[1]
        # the architecture's angles are 32-bit products of position and frequency
        exponent = torch.arange(0, d, 2, dtype=torch.float32, device=DEVICE) / d
        freqs = 1.0 / torch.pow(torch.tensor(cfg["rope_theta"], dtype=torch.float32, device=DEVICE), exponent)
        angle = (torch.arange(T, dtype=torch.float32, device=DEVICE)[:, None] * freqs[None, :]).to(F64)
        cos, sin = torch.cos(angle)[None, :, None, :], torch.sin(angle)[None, :, None, :]

        def turned(x):
            u, v = x[..., :d // 2], x[..., d // 2:]
            return torch.cat([u * cos - v * sin, v * cos + u * sin], dim=-1)
        x = self.w["model.embed_tokens.weight"][ids].to(F64)
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.norm(x, p + "input_layernorm.weight")
            q = turned(self.norm(self.split(self.linear(h, p + "self_attn.q_proj.weight"), H),
                                 p + "self_attn.q_norm.weight"))
            k = turned(self.norm(self.split(self.linear(h, p + "self_attn.k_proj.weight"), G),
                                 p + "self_attn.k_norm.weight"))
            v = self.split(self.linear(h, p + "self_attn.v_proj.weight"), G)
            x = x + self.linear(self.softmax(q, k, v, d ** -0.5, self.visible(T)), p + "self_attn.o_proj.weight")
            h = self.norm(x, p + "post_attention_layernorm.weight")
            act = silu(self.linear(h, p + "mlp.gate_proj.weight")) * self.linear(h, p + "mlp.up_proj.weight")
            x = x + self.linear(act, p + "mlp.down_proj.weight")
        return x

    def design(self, ids):
        cfg, kind = self.cfg, self.cfg["architecture"]
        start = x = self.w["embed"][ids].to(F64) * (cfg.get("embedding") or {"scale": 1.0})["scale"]
        if kind == "Vafepel":
            x = self.norm(x, "embed.norm")
        for i, layer in enumerate(cfg["layers"]):
            p = f"l{i}."
            if cfg.get("loop") and i == cfg["loop"]["start"]:       # (one pass)
                if kind == "Zadenex":
                    x = self.linear(torch.cat([x, start], dim=-1), "loop.in")
                x = x + self.get("loop.step")[0]
            for n, sublayer in (("1", lambda h: self.mixer(h, i, layer)),
                                ("2", lambda h: self.feed_forward(h, i, layer["mlp"]))):
                if kind == "Tirurax":
                    x = x + self.norm(sublayer(x), p + "norm" + n)
                elif kind == "Lemotar":
                    x = self.norm(cfg["postln_alpha"] * x + sublayer(x), p + "norm" + n, 1.0)
                elif kind == "Vafepel":
                    x = x + sublayer(self.norm(x, p + "norm" + n))
                elif kind == "Gopuzen":
                    h = self.layer_norm(x, p + "norm" + n)
                    h = h + self.causal_filter(h, self.get(p + "canon" + n))
                    x = x + self.layer_norm(sublayer(h), f"{p}norm{n}b") * self.get(p + "ls" + n)
                else:
                    x = x + cfg["residual_mult"] * self.norm(sublayer(self.norm(x, p + "norm" + n)), f"{p}norm{n}b")
        return x

    def logits(self, x):
        cfg = self.cfg
        if "architecture" not in cfg:
            tied = cfg["tie_word_embeddings"]
            return self.linear(self.norm(x, "model.norm.weight"),
                               "model.embed_tokens.weight" if tied else "lm_head.weight")
        kind = cfg["architecture"]
        x = (self.layer_norm(x, "final.norm") if kind == "Gopuzen"
             else self.norm(x, "final.norm", 1.0 if kind == "Lemotar" else 0.0))
        out = self.linear(x, "head" if "head" in self.w else "embed") * cfg.get("logit_scale", 1.0)
        cap = cfg.get("logit_softcap")
        return out if cap is None else cap * torch.tanh(out / cap)


def exact(case, seed):
    if case["kind"] == "sample":
        return None             # drawn tokens: whole values
    cfg = config_of(case)
    plain = Plain(case, cfg, make_weights(case, cfg, seed))
    prompts, after = tokens_of(case, cfg.get("vocab_size", cfg.get("vocab")), seed)
    lengths = [len(p) for p in prompts]
    ids = torch.zeros((case["batch"], max(lengths) + case["new"]), dtype=torch.long)
    for row, (p, a) in enumerate(zip(prompts, after)):
        ids[row, :len(p) + len(a)] = torch.tensor(p + a)
    ids = ids.to(DEVICE)
    x = plain.qwen(ids) if case["model"] in QWEN else plain.design(ids)
    rows = torch.arange(case["batch"], device=DEVICE)
    last = torch.tensor(lengths, device=DEVICE) - 1
    return [plain.logits(x[rows, last + t]) for t in range(1 + case["new"])]
