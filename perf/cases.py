"""What this framework is timed on: whole passes of its decoders through the public entry points.

A case names a design, its layer sizes, the type of the weights and activations, and one of four things
that a serving program does with a model:

* ``prefill``: the prompts of new sequences in one step, the last row's logits of each;
* ``continue``: more tokens of sequences that the cache already holds (a kept prefix, a next turn);
* ``decode``: steps of one token a sequence through the decode loop, greedy choice on the device and
  back to the host every step, the logits of the last step.  The tokens fed are given, so that a
  near tie in one step does not change what the next one computes;
* ``generate``: the generation loop from prompts to tokens, following a given transcript, with every
  step's logits (and, in float32, where near ties do not flip, the sampler's own choices).

Layer sizes are those of the Qwen2.5 family and of the design benchmark's layers; the weights are random.  Designs with routed experts are not among
them: where a router's two best scores nearly tie, two correct implementations take different experts,
and whole outputs then say nothing about either.
"""
import math
import random

import numpy as np
import torch

from sonicboom_amd.api import Model
from sonicboom_amd.config.registry import architecture_of
from sonicboom_amd.engine import DecoderModel, generate
from sonicboom_amd.parts import Runtime
from sonicboom_amd.sampling import Sampler, SamplingParams

# (layers, width, heads, kv heads, inner width, tied head)
QWEN = {
    "0.5b": (24, 896, 14, 2, 4864, True),
    "1.5b": (28, 1536, 12, 2, 8960, True),
    "3b": (36, 2048, 16, 2, 11008, True),
    "7b": (28, 3584, 28, 4, 18944, False),
}
DESIGN_WIDTHS = {"2048": 2048, "4096": 4096}
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
MOST_FLOPS = 2.7e14          # of the largest listed case
MOST_EXACT_FLOPS = 4e14      # what 64-bit arithmetic does in some seconds


def listed():
    def case(name, do, size, batch, shortest, longest, new=1, design="qwen2", dtype="bfloat16"):
        return {"name": name, "do": do, "design": design, "size": size, "dtype": dtype, "batch": batch,
                "shortest": shortest, "longest": longest, "new": new}
    return [
        # one user of a small model, a short chat: latency and launches
        case("decode_05b_b1", "decode", "0.5b", 1, 137, 137, 12),
        # a few short prompts that arrive together
        case("prefill_05b_short", "prefill", "0.5b", 5, 9, 130),
        # the benchmark's decode step: eight sequences with prompts of 2,048 tokens
        case("decode_7b_b8", "decode", "7b", 8, 2048, 2048, 8),
        # a busy server: many sequences of every length
        case("decode_15b_b41_ragged", "decode", "1.5b", 41, 60, 3000, 8),
        # two long documents being asked about
        case("decode_3b_b2_long", "decode", "3b", 2, 17000, 21000, 8),
        # the benchmark's prompt
        case("prefill_7b_2048", "prefill", "7b", 1, 2048, 2048),
        # a server's prompt step: prompts of many lengths end to end
        case("prefill_3b_ragged", "prefill", "3b", 9, 90, 1900),
        # one long document
        case("prefill_7b_16384", "prefill", "7b", 1, 16384, 16384),
        # the next turn of conversations whose earlier turns are kept
        case("continue_15b", "continue", "1.5b", 3, 400, 900, 61),
        # attention beside retention, gated linear attention: prompts and tokens
        case("generate_dudatar", "generate", "2048", 3, 150, 1100, 24, design="dudatar"),
        # gated recurrences and latent attention: a long prompt
        case("prefill_rasizen", "prefill", "2048", 1, 4001, 4001, design="rasizen"),
        # the float32 path: checking a model's tokens
        case("generate_05b_float32", "generate", "0.5b", 3, 40, 260, 8, dtype="float32"),
    ]


def draw(rng):
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    while True:
        design = rng.choices(["qwen2", "dudatar", "rasizen"], [6, 1, 1])[0]
        dtype = "float32" if design == "qwen2" and rng.random() < 0.12 else "bfloat16"
        size = "0.5b" if dtype == "float32" else rng.choice(sorted(QWEN)) if design == "qwen2" else rng.choice(sorted(DESIGN_WIDTHS))
        do = rng.choice(["prefill", "decode", "continue", "generate"]) if design == "qwen2" else rng.choice(["prefill", "generate"])
        batch = between(1, 4 if dtype == "float32" else 48)
        longest = between(8, 300 if dtype == "float32" else 16384)
        shortest = min(longest, between(4, longest))
        most = 8 if dtype == "float32" else 24
        new = {"prefill": 1, "decode": rng.randint(4, most // 2), "continue": between(2, 300), "generate": rng.randint(4, most)}[do]
        case = {"do": do, "design": design, "size": size, "dtype": dtype, "batch": batch, "shortest": shortest,
                "longest": longest, "new": new}
        if do == "generate" and batch > 12:
            continue
        share = 0.05 if do == "generate" else 1.0 if design == "qwen2" else 0.2       # a drawn case takes no longer than a listed one
        if _model_flops(case, lengths_of(case), [0] * batch) <= MOST_FLOPS * share:
            return case


def lengths_of(case):
    """The prompts' lengths: spread over the range's logarithm, the two ends among them."""
    lo, hi, n = case["shortest"], case["longest"], case["batch"]
    rng = random.Random("%d %d %d" % (lo, hi, n))
    got = [int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) for _ in range(n)]
    got[0] = hi
    if n > 1:
        got[-1] = lo
    return got


# ---- models -----------------------------------------------------------------------------------------

def config_of(case):
    if case["design"] == "qwen2":
        layers, width, heads, kv, inner, tied = QWEN[case["size"]]
        return {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "num_hidden_layers": layers,
                "hidden_size": width, "num_attention_heads": heads, "num_key_value_heads": kv,
                "intermediate_size": inner, "vocab_size": 151936 if tied else 152064, "rope_theta": 1000000.0,
                "rms_norm_eps": 1e-6, "max_position_embeddings": 131072, "tie_word_embeddings": tied,
                "use_sliding_window": False, "hidden_act": "silu"}
    width = DESIGN_WIDTHS[case["size"]]
    heads = width // 128
    if case["design"] == "rasizen":
        att = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
               "mask": {"size": 4096}, "rot": {"base": 1e6, "dims": 64}}
        layers = []
        for _ in range(2):
            own = len(layers) + 1
            ff = {"kind": "dense", "ff": 4 * width}
            layers += [{"type": "mingru", "mixer": {"width": 2 * width}, "mlp": None},
                       {"type": "latent_attention", "mixer": dict(att), "mlp": ff},
                       {"type": "latent_attention", "mixer": dict(att, kv_from=own), "mlp": ff},
                       {"type": "mingru", "mixer": {"width": 2 * width}, "mlp": None}]
        return {"architecture": "Rasizen", "vocab": 32768, "width": width, "residual_mult": 0.5,
                "norm": {"eps": 1e-5, "groups": 2}, "layers": layers}
    right = max(1, heads // 2)
    ff = {"kind": "dense", "ff": (8 * width // 3 + 255) // 256 * 256}
    both = {"type": "parallel", "mlp": ff, "mixer": {
        "left": {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                 "rot": {"base": 1e6, "dims": 64}},
        "right": {"heads": right, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5 - 5.0 * i / right) for i in range(right)],
                  "rot": {"base": 1e6, "dims": 128}}}}
    linear = {"type": "gla", "mlp": ff, "mixer": {"heads": heads, "dim": 128, "vdim": 128, "tau": 16.0, "rank": 16}}
    return {"architecture": "Dudatar", "vocab": 32768, "width": width, "logit_softcap": 30.0, "norm": {"eps": 1e-6},
            "loop": {"start": 1, "stop": 3, "times": 3}, "layers": [both, both, linear, both]}


def vocab_of(cfg):
    return cfg.get("vocab_size") or cfg["vocab"]


def tensors_of(cfg):
    """(name, shape, mean, spread) of every tensor of a model of this configuration."""
    out = []

    def add(name, *shape, mean=0.0, std=0.02):
        out.append((name, shape, mean, std))

    if "architectures" in cfg:
        # what joins the stream is drawn narrower by the depth, as decoders are initialised
        d, ff, v = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
        hd = d // cfg["num_attention_heads"]
        kv = cfg["num_key_value_heads"] * hd
        joins = 0.02 / math.sqrt(2.0 * cfg["num_hidden_layers"])
        add("model.embed_tokens.weight", v, d, std=0.1 if cfg["tie_word_embeddings"] else 0.5)
        for i in range(cfg["num_hidden_layers"]):
            p = "model.layers.%d." % i
            add(p + "input_layernorm.weight", d, mean=1.0)
            for name, n in (("q", d), ("k", kv), ("v", kv)):
                add(p + "self_attn.%s_proj.weight" % name, n, d)
                add(p + "self_attn.%s_proj.bias" % name, n)
            add(p + "self_attn.o_proj.weight", d, d, std=joins)
            add(p + "post_attention_layernorm.weight", d, mean=1.0)
            add(p + "mlp.gate_proj.weight", ff, d)
            add(p + "mlp.up_proj.weight", ff, d)
            add(p + "mlp.down_proj.weight", d, ff, std=joins)
        add("model.norm.weight", d, mean=1.0)
        if not cfg["tie_word_embeddings"]:
            add("lm_head.weight", v, d)
        return out
    d = cfg["width"]
    add("embed", cfg["vocab"], d)
    add("final.norm", d, mean=1.0)
    if cfg["architecture"] == "Rasizen":
        for i, layer in enumerate(cfg["layers"]):
            p, mx = "l%d." % i, layer["mixer"]
            add(p + "norm1", d, mean=1.0)
            if layer["type"] == "mingru":
                for name in ("z", "x"):
                    add(p + "mix." + name, mx["width"], d)
                    add(p + "mix." + name + ".b", mx["width"])
                add(p + "mix.g", mx["width"], d)
                add(p + "mix.o", d, mx["width"])
            else:
                h, rank = mx["heads"], mx["kv_rank"]
                add(p + "mix.q", h * (mx["dim"] + mx["rot_dim"]), d)
                add(p + "mix.uk", h * mx["dim"], rank)
                add(p + "mix.uv", h * mx["vdim"], rank)
                add(p + "mix.g", h * mx["vdim"], d)
                add(p + "mix.o", d, h * mx["vdim"])
                if mx.get("kv_from") is None:
                    add(p + "mix.dkv", rank + mx["rot_dim"], d)
                    add(p + "mix.dkv.norm", rank, mean=1.0)
            if layer["mlp"]:
                add(p + "norm2", d, mean=1.0)
                add(p + "mlp.up", layer["mlp"]["ff"], d)
                add(p + "mlp.down", d, layer["mlp"]["ff"])
                add(p + "mlp.act", 2, std=0.5)
        return out
    add("head", cfg["vocab"], d)
    add("loop.in", d, 2 * d)
    add("loop.step", cfg["loop"]["times"], d, std=0.1)
    for i, layer in enumerate(cfg["layers"]):
        p, mx, ff = "l%d." % i, layer["mixer"], layer["mlp"]["ff"]
        add(p + "norm1", d, mean=1.0)
        if layer["type"] == "parallel":
            a, b = mx["left"], mx["right"]
            for name, n in (("q", a["heads"] * a["dim"]), ("k", a["kv_heads"] * a["dim"]), ("v", a["kv_heads"] * a["vdim"]), ("g", a["heads"])):
                add(p + "mix.left." + name, n, d)
            add(p + "mix.left.o", d, a["heads"] * a["vdim"])
            add(p + "mix.left.out", d, mean=1.0)
            p_mix, mx = p + "mix.right.", b
            add(p + "mix.right.out", d, mean=1.0)
        else:
            p_mix = p + "mix."
            add(p_mix + "norm", mx["vdim"], mean=1.0)
            add(p_mix + "a1", mx["rank"], d)
            add(p_mix + "a2", mx["heads"] * mx["dim"], mx["rank"], std=0.2)
            add(p_mix + "a2.b", mx["heads"] * mx["dim"], mean=2.0, std=1.0)
        for name, n in (("q", mx["heads"] * mx["dim"]), ("k", mx["heads"] * mx["dim"]), ("v", mx["heads"] * mx["vdim"]), ("g", mx["heads"] * mx["vdim"])):
            add(p_mix + name, n, d)
        add(p_mix + "o", d, mx["heads"] * mx["vdim"])
        for name in ("gate", "up"):
            add(p + "mlp." + name, ff, d)
        add(p + "mlp.down", d, ff)
    return out


def weights_of(cfg, seed, device="cuda:0"):
    """The weights as a bfloat16 checkpoint holds them."""
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed) * 1000003 + 17)
    got = {}
    for name, shape, mean, std in tensors_of(cfg):
        got[name] = torch.empty(shape, dtype=torch.bfloat16, device=device).normal_(mean, std, generator=gen)
    return got


def tokens_of(case, cfg, seed):
    """(prompts, the tokens that follow each): lists of ids."""
    rng = np.random.default_rng([int(seed), 5])
    vocab = vocab_of(cfg)
    prompts = [rng.integers(0, vocab, size=n).tolist() for n in lengths_of(case)]
    after = [rng.integers(0, vocab, size=case["new"]).tolist() for _ in prompts]
    return prompts, after


class _Transcript:
    """A sampler that keeps the logits and its own choices, and goes on with given tokens."""

    def __init__(self, follow, params):
        self.follow, self.own = follow, Sampler(params)
        self.logits, self.chosen = [], []

    def pick(self, logits, positions, histories):
        step = len(self.logits)
        self.logits.append(logits.clone())
        self.chosen.append(self.own.pick(logits, positions, histories))
        return [tokens[step] for tokens in self.follow]


def prepare(case, seed):
    cfg = config_of(case)
    dtype = DTYPES[case["dtype"]]
    tensors = weights_of(cfg, seed)
    if dtype != torch.bfloat16:
        tensors = {name: t.to(dtype) for name, t in tensors.items()}
    arch = architecture_of(cfg)
    typed = arch.config_class.from_dict(cfg)
    decoder = DecoderModel(arch.build_spec(typed), tensors, Runtime(torch.device("cuda:0"), dtype), typed)
    del tensors
    prompts, after = tokens_of(case, cfg, seed)
    room = sum((len(p) + case["new"] + 127) // 64 * 64 for p in prompts)
    session = Model(decoder).session(max_tokens=room, max_slots=len(prompts))
    state = {"case": case, "session": session, "prompts": prompts, "after": after, "slots": None}
    if case["do"] in ("decode", "continue"):
        slots = [session.alloc_slot() for _ in prompts]
        session.step([(s, p, ()) for s, p in zip(slots, prompts)])
        state["slots"] = slots
    return state


def run(state):
    case, session, prompts, after = state["case"], state["session"], state["prompts"], state["after"]
    do = case["do"]
    if do == "prefill":
        slots = [session.alloc_slot() for _ in prompts]
        logits = session.step([(s, p, (len(p) - 1,)) for s, p in zip(slots, prompts)])
        for s in slots:
            session.free_slot(s)
        return {"logits": logits}
    if do == "generate":
        sampler = _Transcript(after, SamplingParams(temperature=0.8, top_p=0.95, top_k=50, seed=7))
        generate(session.engine, prompts, SamplingParams(max_tokens=case["new"]), stop_tokens=(), max_batch=len(prompts),
                 sampler=sampler)
        out = {"logits": sampler.logits}
        if case["dtype"] == "float32":
            out["chosen"] = np.asarray(sampler.chosen, dtype=np.int64)
        return out
    slots = state["slots"]
    if do == "continue":
        logits = session.step([(s, t, (len(t) - 1,)) for s, t in zip(slots, after)])
        out = {"logits": logits}
    else:
        loop = session.engine.decode_loop()
        steps = list(zip(*after))
        for fed in steps[:-1]:
            loop.start(slots, fed)
            loop.step()
        loop.start(slots, steps[-1])
        out = {"logits": loop.step_logits().clone()}
    for s, p in zip(slots, prompts):
        session.engine.cache.truncate(s, len(p))
    return out


# ---- the work a pass cannot do without ------------------------------------------------------------------

def _params(case):
    """(weights that every row meets, weights of the head) of the case's model."""
    cfg = config_of(case)
    total = head = 0
    for name, shape, _, _ in tensors_of(cfg):
        n = int(np.prod(shape))
        if name in ("model.embed_tokens.weight", "embed", "lm_head.weight", "head"):
            head = n
        else:
            total += n
    if case["design"] == "dudatar":          # the layers of the loop run several times
        again = sum(int(np.prod(s)) for name, s, _, _ in tensors_of(cfg) if name.split(".")[0] in ("l1", "l2"))
        return total, total + (cfg["loop"]["times"] - 1) * again, head
    return total, total, head


def _attention(case):
    """(layers that attend, query numbers, key and value numbers a token, multiply-adds a query row and key, window)"""
    cfg = config_of(case)
    if case["design"] == "qwen2":
        hd = cfg["hidden_size"] // cfg["num_attention_heads"]
        return cfg["num_hidden_layers"], 2 * cfg["num_key_value_heads"] * hd, 2 * cfg["num_attention_heads"] * hd, 0
    heads = cfg["width"] // 128
    if case["design"] == "rasizen":
        return 4, 576 // 2, heads * (192 + 128), 4096
    return 5, 2 * max(1, heads // 4) * 128, heads * 256, 0


def _model_flops(case, n_new, n_before):
    _, used, head = _params(case)
    layers, _, madds, window = _attention(case)
    rows = sum(n_new)
    pairs = 0
    for n, b in zip(n_new, n_before):
        pairs += n * b + n * (n + 1) // 2 if not window else sum(min(window, b + i + 1) for i in range(n))
    return 2.0 * used * rows + 2.0 * layers * madds * pairs + 2.0 * head * len(n_new)


def work(case):
    size = 4 if case["dtype"] == "float32" else 2
    lengths, new, n = lengths_of(case), case["new"], case["batch"]
    stored, _, head = _params(case)
    layers, per_token, _, window = _attention(case)

    def step(n_new, n_before):
        """One step: every weight once, the cached keys and values once, the new ones and the logits written."""
        seen = sum(min(window, b) if window else b for b in n_before)
        nbytes = (stored + head) * size + layers * per_token * size * (seen + sum(n_new)) + n * (head // config_width(case)) * 4
        return nbytes, _model_flops(case, n_new, n_before)

    if case["do"] == "prefill":
        parts = [step(lengths, [0] * n)]
    elif case["do"] == "continue":
        parts = [step([new] * n, lengths)]
    else:
        parts = [step([1] * n, [k + i for k in lengths]) for i in range(new if case["do"] == "decode" else new - 1)]
        if case["do"] == "generate":
            parts.append(step(lengths, [0] * n))
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


def config_width(case):
    cfg = config_of(case)
    return cfg.get("hidden_size") or cfg["width"]


def tolerance(case):
    # About four times what the same weights and tokens give with sums in another order (prompts cut into
    # portions, other product kernels): 0.004 to 0.006 of the result at the smallest sizes and with
    # gated recurrences, 0.009 to 0.014 elsewhere, and in float32 the distance from 64 bits, 3e-6.
    if case["dtype"] == "float32":
        return {"rel": 1.6e-5, "max": 2e-4, "differ": 0.01}
    if case["design"] == "rasizen" or case["size"] == "0.5b":
        return {"rel": 0.022, "max": 0.12}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits ---------------------------------------------------------------------------------

F64 = torch.float64


def _lin(x, w):
    return x @ w.to(F64).T


def _rms(v, eps):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)


def _layer_norm(v, w, eps):
    d = v - v.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w.to(F64)


def _turn_halves(v, dims, base):
    """v [n, heads, m]: pairs (i, i + dims/2) of the first ``dims`` numbers turn with the row's number."""
    half = dims // 2
    f = base ** (-2.0 * torch.arange(half, dtype=F64, device=v.device) / dims)
    a = torch.arange(v.shape[0], dtype=F64, device=v.device)[:, None, None] * f
    c, s = torch.cos(a), torch.sin(a)
    x, y = v[..., :half], v[..., half:dims]
    return torch.cat([x * c - y * s, y * c + x * s, v[..., dims:]], -1)


def _turn_pairs(v, dims, base):
    """v [n, heads, m]: the pairs (2i, 2i + 1) turn instead."""
    half = dims // 2
    f = base ** (-2.0 * torch.arange(half, dtype=F64, device=v.device) / dims)
    a = torch.arange(v.shape[0], dtype=F64, device=v.device)[:, None, None] * f
    c, s = torch.cos(a), torch.sin(a)
    x, y = v[..., 0:dims:2], v[..., 1:dims:2]
    return torch.cat([torch.stack([x * c - y * s, y * c + x * s], -1).flatten(-2), v[..., dims:]], -1)


def _attend(q, k, v, scale, window=0):
    """q [n, H, d], k [n, G, d], v [n, G, e]: causal softmax attention, query head a reads head a // (H / G)."""
    n, H, _ = q.shape
    G = k.shape[1]
    out = torch.empty((n, H, v.shape[-1]), dtype=F64, device=q.device)
    at = torch.arange(n, device=q.device)
    for t in range(0, n, 4096):
        end = min(n, t + 4096)
        first = max(0, t - window + 1) if window else 0
        hidden = at[None, first:end] > at[t:end, None]
        if window:
            hidden |= at[None, first:end] <= at[t:end, None] - window
        for a in range(H):
            g = a * G // H
            s = (q[t:end, a] @ k[first:end, g].T) * scale
            s.masked_fill_(hidden, -math.inf)
            out[t:end, a] = torch.softmax(s, -1) @ v[first:end, g]
    return out


def _rows_of(lengths):
    first = 0
    for n in lengths:
        yield slice(first, first + n)
        first += n


def _exact_qwen(cfg, w, ids, lengths):
    d, H, G, eps = cfg["hidden_size"], cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    hd = d // H
    x = w["model.embed_tokens.weight"][ids].to(F64)
    for i in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % i
        h = _rms(x, eps) * w[p + "input_layernorm.weight"].to(F64)
        q, k, v = (_lin(h, w[p + "self_attn.%s_proj.weight" % r]) + w[p + "self_attn.%s_proj.bias" % r].to(F64) for r in "qkv")
        y = torch.empty_like(q)
        for rows in _rows_of(lengths):
            qs = _turn_halves(q[rows].unflatten(1, (H, hd)), hd, cfg["rope_theta"])
            ks = _turn_halves(k[rows].unflatten(1, (G, hd)), hd, cfg["rope_theta"])
            y[rows] = _attend(qs, ks, v[rows].unflatten(1, (G, hd)), hd ** -0.5).flatten(1)
        x = x + _lin(y, w[p + "self_attn.o_proj.weight"])
        h = _rms(x, eps) * w[p + "post_attention_layernorm.weight"].to(F64)
        for a in range(0, x.shape[0], 8192):
            b = h[a:a + 8192]
            mid = torch.nn.functional.silu(_lin(b, w[p + "mlp.gate_proj.weight"])) * _lin(b, w[p + "mlp.up_proj.weight"])
            x[a:a + 8192] += _lin(mid, w[p + "mlp.down_proj.weight"])
    head = w["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"]
    return lambda rows: _lin(_rms(x[rows], eps) * w["model.norm.weight"].to(F64), head)


def _scan(q, k, v, decay):
    """S_t = decay_t S_(t-1) + k_t v_t^T, o_t = S_t^T q_t a head; q, k, decay [n, H, D], v [n, H, E]."""
    S = torch.zeros((k.shape[1], k.shape[2], v.shape[2]), dtype=F64, device=k.device)
    out = torch.empty((k.shape[0], k.shape[1], v.shape[2]), dtype=F64, device=k.device)
    for t in range(k.shape[0]):
        S = torch.baddbmm(S * decay[t][:, :, None], k[t][:, :, None].contiguous(), v[t][:, None, :].contiguous())
        out[t] = torch.bmm(q[t][:, None, :].contiguous(), S)[:, 0]
    return out


def _exact_dudatar(cfg, w, ids, lengths):
    eps, d = cfg["norm"]["eps"], cfg["width"]
    silu = torch.nn.functional.silu
    x0 = w["embed"][ids].to(F64)
    x = x0.clone()

    def by_sequence(h, f):
        return torch.cat([f(h[rows]) for rows in _rows_of(lengths)])

    def left(mx, p, h):
        n, H, G = h.shape[0], mx["heads"], mx["kv_heads"]
        dims, base = mx["rot"]["dims"], mx["rot"]["base"]
        q = _rms(_turn_halves(_lin(h, w[p + "q"]).view(n, H, -1), dims, base), eps)
        k = _rms(_turn_halves(_lin(h, w[p + "k"]).view(n, G, -1), dims, base), eps)
        y = _attend(q, k, _lin(h, w[p + "v"]).view(n, G, -1), mx["scale"])
        return _lin((y * torch.sigmoid(_lin(h, w[p + "g"]))[..., None]).flatten(1), w[p + "o"])

    def right(mx, p, h):
        n, H, D = h.shape[0], mx["heads"], mx["dim"]
        dims, base = mx["rot"]["dims"], mx["rot"]["base"]
        q = _turn_halves(_lin(h, w[p + "q"]).view(n, H, D), dims, base)
        k = _turn_halves(_lin(h, w[p + "k"]).view(n, H, D), dims, base) * D ** -0.5
        decay = torch.tensor(mx["decay"], dtype=F64, device=h.device)[None, :, None].expand(n, H, D)
        y = _scan(q, k, _lin(h, w[p + "v"]).view(n, H, -1), decay)
        return _lin(_rms(y, eps).flatten(1) * silu(_lin(h, w[p + "g"])), w[p + "o"])

    def linear_attention(mx, p, h):
        n, H, D = h.shape[0], mx["heads"], mx["dim"]
        q = _lin(h, w[p + "q"]).view(n, H, D) * D ** -0.5
        k, v = _lin(h, w[p + "k"]).view(n, H, D), _lin(h, w[p + "v"]).view(n, H, -1)
        alpha = torch.sigmoid(_lin(_lin(h, w[p + "a1"]), w[p + "a2"]) + w[p + "a2.b"].to(F64)) ** (1.0 / mx["tau"])
        y = _rms(_scan(q, k, v, alpha.view(n, H, D)), eps) * w[p + "norm"].to(F64)
        return _lin(y.flatten(1) * silu(_lin(h, w[p + "g"])), w[p + "o"])

    loop = cfg["loop"]
    order = [(0, None)] + [(i, s if i == loop["start"] else None) for s in range(loop["times"]) for i in range(loop["start"], loop["stop"])]
    order += [(i, None) for i in range(loop["stop"], len(cfg["layers"]))]
    for i, turn in order:
        if turn is not None:
            x = _lin(torch.cat([x, x0], 1), w["loop.in"]) + w["loop.step"][turn].to(F64)
        lay, p = cfg["layers"][i], "l%d." % i
        mx = lay["mixer"]
        h = _layer_norm(x, w[p + "norm1"], eps)
        if lay["type"] == "parallel":
            a = by_sequence(h, lambda r: left(mx["left"], p + "mix.left.", r))
            b = by_sequence(h, lambda r: right(mx["right"], p + "mix.right.", r))
            y = 0.5 * (_rms(a, eps) * w[p + "mix.left.out"].to(F64) + _rms(b, eps) * w[p + "mix.right.out"].to(F64))
        else:
            y = by_sequence(h, lambda r: linear_attention(mx, p + "mix.", r))
        gate = torch.nn.functional.gelu(_lin(h, w[p + "mlp.gate"]), approximate="tanh")
        x = x + y + _lin(gate * _lin(h, w[p + "mlp.up"]), w[p + "mlp.down"])
    cap = cfg["logit_softcap"]
    return lambda rows: cap * torch.tanh(_lin(_layer_norm(x[rows], w["final.norm"], eps), w["head"]) / cap)


def _exact_rasizen(cfg, w, ids, lengths):
    eps, groups, m = cfg["norm"]["eps"], cfg["norm"]["groups"], cfg["residual_mult"]
    silu = torch.nn.functional.silu

    def norm(v, weight):
        return _rms(v.unflatten(1, (groups, -1)), eps).flatten(1) * weight.to(F64)

    def recurrence(z, cand):
        s = torch.zeros_like(z[0])
        out = torch.empty_like(z)
        for t in range(z.shape[0]):
            s = torch.addcmul((1.0 - z[t]) * s, z[t], cand[t])
            out[t] = s
        return out

    x = w["embed"][ids].to(F64)
    kept = {}
    for i, lay in enumerate(cfg["layers"]):
        p, mx = "l%d." % i, lay["mixer"]
        q_name = p + "mix."
        h = norm(x, w[p + "norm1"])
        if lay["type"] == "mingru":
            z = torch.sigmoid(_lin(h, w[q_name + "z"]) + w[q_name + "z.b"].to(F64))
            u = _lin(h, w[q_name + "x"]) + w[q_name + "x.b"].to(F64)
            cand = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
            s = torch.cat([recurrence(z[rows], cand[rows]) for rows in _rows_of(lengths)])
            y = _lin(s * silu(_lin(h, w[q_name + "g"])), w[q_name + "o"])
        else:
            H, dim, rot, rank = mx["heads"], mx["dim"], mx["rot_dim"], mx["kv_rank"]
            dims, base = mx["rot"]["dims"], mx["rot"]["base"]
            if mx.get("kv_from") is None:
                both = _lin(h, w[q_name + "dkv"])
                kept[i] = (_rms(both[:, :rank], eps) * w[q_name + "dkv.norm"].to(F64), both[:, rank:])
            else:
                kept[i] = kept[mx["kv_from"]]
            c, r = kept[i]
            q = _lin(h, w[q_name + "q"]).unflatten(1, (H, dim + rot))
            ys = []
            for rows in _rows_of(lengths):
                n = rows.stop - rows.start
                part = _turn_pairs(r[rows][:, None, :], dims, base).expand(n, H, rot)
                keys = torch.cat([_lin(c[rows], w[q_name + "uk"]).view(n, H, dim), part], -1)
                queries = torch.cat([q[rows][..., :dim], _turn_pairs(q[rows][..., dim:], dims, base)], -1)
                values = _lin(c[rows], w[q_name + "uv"]).view(n, H, -1)
                ys.append(_attend(queries, keys, values, mx["scale"], mx["mask"]["size"]).flatten(1))
            y = _lin(torch.cat(ys) * torch.sigmoid(_lin(h, w[q_name + "g"])), w[q_name + "o"])
        x = x + m * y
        if lay["mlp"]:
            up = _lin(norm(x, w[p + "norm2"]), w[p + "mlp.up"])
            a, b = torch.nn.functional.softplus(w[p + "mlp.act"].to(F64))
            neg = torch.clamp(up, max=0.0)
            mid = torch.where(up > 0, a * up * up + up / 2, (0.5 + b) * (torch.expm1(neg) - neg) + up / 2)
            x = x + m * _lin(mid, w[p + "mlp.down"])
    return lambda rows: _lin(norm(x[rows], w["final.norm"]), w["embed"])


EXACT = {"qwen2": _exact_qwen, "dudatar": _exact_dudatar, "rasizen": _exact_rasizen}


def exact(case, seed):
    cfg = config_of(case)
    lengths, new, n = lengths_of(case), case["new"], case["batch"]
    do = case["do"]
    fed = 0 if do == "prefill" else new - 1 if do == "generate" else new
    whole = [k + fed for k in lengths]
    if _model_flops(case, whole, [0] * n) > MOST_EXACT_FLOPS or (case["design"] != "qwen2" and sum(whole) > 12000):
        return None
    w = weights_of(cfg, seed)
    prompts, after = tokens_of(case, cfg, seed)
    ids = torch.tensor([t for p, a in zip(prompts, after) for t in p + a[:fed]], device="cuda:0")
    logits = EXACT[case["design"]](cfg, w, ids, whole)
    ends = [rows.stop for rows in _rows_of(whole)]
    if do != "generate":
        return {"logits": logits(torch.tensor([e - 1 for e in ends], device="cuda:0"))}
    out = {"logits": [logits(torch.tensor([e - new + i for e in ends], device="cuda:0")) for i in range(new)]}
    if case["dtype"] == "float32":
        out["chosen"] = None
    return out
