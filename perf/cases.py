"""What is measured: passes of the step function over the work that a user of this engine has it do.

A case names a model (a named shape of the package, its layers and the type it computes in) and what one pass
brings: `decode` requests that bring one token each at about `depth` positions, a prompt of `prompt` tokens (whole, or
in portions of at most `portion`) whose last `want` places are scored, or both in one step.  A pass is what a server
does between two answers: pages are reserved, the step is packed, launched and replayed from its recording where the
engine records it, and its float32 logits are the outputs.  Decoding requests go on from where the last pass left them; a prompt is admitted, run and
released in the pass.

Weights are normal values made on the GPU from the seed and loaded through the engine's own loading of a weight
source; `exact` makes the same weights and works the whole sequences out in 64 bits with torch alone.
"""
from __future__ import annotations

import hashlib
import math
import random

import torch

PORTION = 4096          # the engine's default number of prompt tokens in a step
BLOCK = 64              # positions in a page


# ----------------------------------------------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------------------------------------------
def case(name, model, layers, dtype="bfloat16", decode=0, depth=0, prompt=0, portion=PORTION, want=16):
    return {"name": name, "model": model, "layers": layers, "dtype": dtype, "decode": decode, "depth": depth,
            "prompt": prompt, "portion": portion, "want": min(want, prompt)}


def listed():
    a27b, a14b = "qwen1.5-moe-a2.7b", "qwen2-57b-a14b"
    return [
        # the benchmark's model, all layers, decoding behind 2k prompts: one user (latency), the headline batch, a full server
        case("decode_1", a27b, 24, decode=1, depth=2060),
        case("decode_8", a27b, 24, decode=8, depth=2060),
        case("decode_64", a27b, 24, decode=64, depth=2060),
        # its prompts: a short question of odd length, and the benchmark's 2k prompt
        case("prefill_117", a27b, 24, prompt=117),
        case("prefill_2048", a27b, 24, prompt=2048),
        # continuous batching: a portion of a prompt beside the requests that decode
        case("mixed_15_497", a27b, 24, decode=15, depth=1540, prompt=497, want=1),
        # the larger model of the family, a long document in the engine's default portions (four of its equal layers)
        case("long_prompt_16k", a14b, 4, prompt=16384),
        # and its decoding, a batch between the usual ones
        case("large_decode_12", a14b, 4, decode=12, depth=2060),
        # the true 32-bit path, as used to check a model: a prompt, and decoding
        case("float32_prefill_700", a27b, 6, dtype="float32", prompt=700),
        case("float32_decode_4", a27b, 6, dtype="float32", decode=4, depth=1030),
        # latent attention and attention beside a delta rule, dense feed-forwards: an odd prompt, and a small batch
        case("fokinex_prefill_1337", "fokinex-2k", 8, prompt=1337),
        case("fokinex_decode_8", "fokinex-2k", 8, decode=8, depth=2060),
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], spread over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "mixed", "large", "float32", "fokinex"))
    c = dict(model="qwen1.5-moe-a2.7b", layers=24, dtype="bfloat16", decode=0, depth=0, prompt=0, portion=PORTION, want=0)
    if kind == "decode":
        c.update(decode=_spread(rng, 1, 64), depth=_spread(rng, 40, 2500))
    elif kind == "prefill":
        c.update(prompt=_spread(rng, 5, 4000))
    elif kind == "mixed":
        c.update(decode=_spread(rng, 1, 24), depth=_spread(rng, 100, 2000), prompt=_spread(rng, 30, 1000))
    elif kind == "large":
        c.update(model="qwen2-57b-a14b", layers=4)
        if rng.random() < 0.5:
            c.update(prompt=_spread(rng, 300, 12000))
        else:
            c.update(decode=_spread(rng, 1, 32), depth=_spread(rng, 300, 3000))
    elif kind == "float32":
        c.update(layers=6, dtype="float32")
        if rng.random() < 0.5:
            c.update(prompt=_spread(rng, 20, 1500))
        else:
            c.update(decode=_spread(rng, 1, 16), depth=_spread(rng, 40, 1500))
    else:
        c.update(model="fokinex-2k", layers=8)
        if rng.random() < 0.5:
            c.update(prompt=_spread(rng, 20, 4000))
        else:
            c.update(decode=_spread(rng, 1, 32), depth=_spread(rng, 40, 2500))
    if c["prompt"]:                          # generation reads the last place, scoring an answer its places
        c.update(want=rng.choice((1, 16)) if c["prompt"] >= 16 else 1)
    return c


# ----------------------------------------------------------------------------------------------------------------
# inputs from the seed
# ----------------------------------------------------------------------------------------------------------------
def _config(c):
    from ferrox_amd.config import presets
    cfg = presets.load(c["model"])
    if "num_hidden_layers" in cfg:
        cfg = dict(cfg, num_hidden_layers=c["layers"])
    else:
        cfg = dict(cfg, layers=cfg["layers"][:c["layers"]])
    return cfg


def _vocab(cfg):
    return cfg["vocab_size"] if "vocab_size" in cfg else cfg["vocab"]


def _values(name, shape, seed, dtype, scale):
    """The weights of one tensor: of a size that keeps every product's output of order one, as in a trained model."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int.from_bytes(hashlib.sha256(f"{seed}:{name}".encode()).digest()[:7], "little"))
    last = name.split(".")[-1]
    owner = name.split(".")[-2] if last in ("weight", "bias") else last
    t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    if "norm" in owner:
        return t.mul_(0.1).add_(1.0)
    if last == "A_log":                      # decays of 0.8 to 0.97: tens of tokens are remembered
        return t.mul_(0.5).sub_(2.0)
    if last == "sink":
        return t.add_(1.0)
    if last in ("dt_bias", "conv"):
        return t.mul_(0.5)
    if last == "bias":
        return t.mul_(0.02)
    if owner == "embed_tokens":
        return t.mul_(0.02)
    if last == "embed":
        return t.mul_(1.0 / scale)
    return t.mul_(0.9 / math.sqrt(shape[-1]))


class _Weights:
    """A weight source over `_values`, as a checkpoint folder is one."""

    def __init__(self, cfg, seed, dtype):
        self.seed, self.dtype = seed, dtype
        self.scale = (cfg.get("embedding") or {}).get("scale", 1.0)
        self.specs = {}

    def expect(self, specs):
        self.specs = dict(specs)

    def names(self):
        return list(self.specs)

    def info(self, name):
        return self.dtype, tuple(self.specs[name].shape)

    def tensor(self, name):
        return _values(name, tuple(self.specs[name].shape), self.seed, self.dtype, self.scale)


def _depths(c):
    """Where each decoding request stands: no two servers' requests are of one length."""
    return [c["depth"] - (37 * i) % (c["depth"] // 4 + 1) for i in range(c["decode"])]


def _tokens(c, seed, vocab):
    """(what each decoding request has behind it, what it brings pass after pass, the prompt)"""
    rng = random.Random(seed * 7919 + 13)
    behind = [[rng.randrange(vocab) for _ in range(d)] for d in _depths(c)]
    brings = [[rng.randrange(vocab) for _ in range(512)] for _ in behind]
    return behind, brings, [rng.randrange(vocab) for _ in range(c["prompt"])]


class _State:
    """A server's engine with requests in it."""

    def __init__(self, c, seed):
        from ferrox_amd.engine.api import Engine
        from ferrox_amd.engine.loading import parse_dtype
        from ferrox_amd.engine.model import Model
        from ferrox_amd.models.registry import resolve
        raw, dtype = _config(c), parse_dtype(c["dtype"])
        arch = resolve(raw)
        cfg = arch.config_class.from_dict(raw)
        model = Model(arch.build_spec(cfg, None))
        model.config = cfg
        model.load(_Weights(raw, seed, dtype), dtype, "cuda:0")
        self.behind, self.brings, self.prompt = _tokens(c, seed, _vocab(raw))
        self.room = c["depth"] + (4096 if c["decode"] <= 16 else 700)
        pages = c["decode"] * (self.room // BLOCK + 2) + c["prompt"] // BLOCK + 2
        self.engine = Engine(model=model, block_size=BLOCK, num_pages=pages, max_seqs=c["decode"] + 1)
        self.portion, self.want = c["portion"], c["want"]
        self.at = [0] * len(self.behind)
        self.fill()

    def fill(self):
        """Every decoding request behind its context, as many of them in a step as fit, and one decoded token on."""
        from ferrox_amd.engine.runner import StepEntry
        runner = self.engine.runner
        part, size = [], 0
        for i, tokens in enumerate(self.behind):
            runner.release(i)
            if not runner.admit(i):
                raise RuntimeError("no slot for a request")
            for o in range(0, len(tokens), PORTION):
                piece = tokens[o:o + PORTION]
                if part and size + len(piece) > PORTION:
                    self.engine.step(part)
                    part, size = [], 0
                if not runner.reserve(i, len(piece)):
                    raise RuntimeError("no pages for a request")
                part.append(StepEntry(i, piece, []))
                size += len(piece)
            self.at[i] = 0
        if part:
            self.engine.step(part)
        if self.behind:
            self.engine.step(self.decoding())

    def decoding(self):
        from ferrox_amd.engine.runner import StepEntry
        out = []
        for i, brings in enumerate(self.brings):
            if not self.engine.runner.reserve(i, 1):
                raise RuntimeError("no pages for a decoded token")
            out.append(StepEntry(i, [brings[self.at[i] % len(brings)]], [0]))
            self.at[i] += 1
        return out


def prepare(c, seed):
    return _State(c, seed)


def run(state):
    from ferrox_amd.engine.runner import StepEntry
    engine, runner = state.engine, state.engine.runner
    if state.behind and max(len(b) + a for b, a in zip(state.behind, state.at)) >= state.room:
        state.fill()
    entries = state.decoding() if state.behind else []
    if not state.prompt:
        return {"logits": engine.step(entries)}
    if not runner.admit("prompt"):
        raise RuntimeError("no slot for the prompt")
    for o in range(0, len(state.prompt), state.portion):
        piece = state.prompt[o:o + state.portion]
        if not runner.reserve("prompt", len(piece)):
            raise RuntimeError("no pages for the prompt")
        end = o + len(piece) == len(state.prompt)
        logits = engine.step(entries + [StepEntry("prompt", piece, list(range(len(piece) - state.want, len(piece))) if end else [])])
        entries = state.decoding() if entries and not end else []
    runner.release("prompt")
    return {"logits": logits}


# ----------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------------------------
def _layer_sizes(cfg, i):
    """Of layer i: weights that every token meets, weights of an expert, experts, experts a token takes, key/value
    numbers a position keeps, multiplications per pair of positions, numbers of a recurrent state per sequence."""
    if "num_hidden_layers" in cfg:
        H, hd = cfg["hidden_size"], cfg["hidden_size"] // cfg["num_attention_heads"]
        qw, kw = cfg["num_attention_heads"] * hd, cfg["num_key_value_heads"] * hd
        dense = (qw + 2 * kw) * H + H * qw + cfg["num_experts"] * H + 3 * cfg["shared_expert_intermediate_size"] * H
        return dense, 3 * cfg["moe_intermediate_size"] * H, cfg["num_experts"], cfg["num_experts_per_tok"], 2 * kw, 2 * qw, 0
    H, m = cfg["width"], cfg["layers"][i]["mixer"]
    dense = 3 * H * cfg["layers"][i]["mlp"]["ff"]
    if "kv_rank" in m:
        nh, d, v, own = m["heads"], m["dim"], m["vdim"], m["kv_rank"] + m["rot_dim"] if m.get("kv_from") is None else 0
        dense += H * m["q_rank"] + m["q_rank"] * nh * (d + m["rot_dim"]) + m["kv_rank"] * nh * (d + v) + nh * v * H + H * own
        return dense, 0, 1, 0, own, nh * (d + m["rot_dim"] + v), 0
    a, r = m["left"], m["right"]
    dense += H * (3 * a["heads"] * a["dim"] + a["kv_heads"] * a["dim"])
    dense += H * (2 * r["kv_heads"] * r["dim"] + 3 * r["heads"] * r["vdim"] + 2 * r["heads"])
    return dense, 0, 1, 0, 2 * a["kv_heads"] * a["dim"], 2 * a["heads"] * a["dim"], r["heads"] * r["dim"] * r["vdim"]


def work(c):
    cfg, es = _config(c), 2 if c["dtype"] == "bfloat16" else 4
    H = cfg["hidden_size"] if "hidden_size" in cfg else cfg["width"]
    V, depths = _vocab(cfg), _depths(c)
    tokens, rows = c["prompt"] + c["decode"], c["decode"] + c["want"]
    pairs = sum(d + 1 for d in depths) + c["prompt"] * (c["prompt"] + 1) / 2
    numbers, flops = V * H + tokens * H, 2.0 * rows * V * H
    moved = 4.0 * rows * V
    for i in range(c["layers"]):
        dense, expert, E, top, kept, pair, state = _layer_sizes(cfg, i)
        numbers += dense + expert * E * (1.0 - (1.0 - top / E) ** tokens) + kept * (sum(depths) + tokens)
        moved += 8.0 * state * (c["decode"] + (0.5 if c["prompt"] else 0.0))
        flops += 2.0 * (dense + top * expert) * tokens + 2.0 * pair * pairs + 8.0 * state * tokens
    return {"bytes": numbers * es + moved, "flops": flops}


def tolerance(c):
    # measured against `exact`: 2.3e-6 in 32 bits (sums of 2,048 and more terms in another order), 4e-3 to 1e-2 in bfloat16
    # (where two experts stand close, a rounding decides which of them a token takes)
    return {"rel": 1e-5} if c["dtype"] == "float32" else {"rel": 0.03}


# ----------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ----------------------------------------------------------------------------------------------------------------
def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _angles(pos, freqs):
    """Positions times frequencies as a 32-bit implementation has them, [tokens, 1, pairs] in 64 bits."""
    f = torch.tensor(freqs, dtype=torch.float64, device="cuda").float()
    return (pos.float()[:, None] * f).double()[:, None]


def _turn_halves(x, pos, base):
    d = x.shape[-1]
    a = _angles(pos, [base ** (-2.0 * i / d) for i in range(d // 2)])
    u, v = x[..., :d // 2], x[..., d // 2:]
    return torch.cat((u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()), -1)


def _turn_pairs(x, pos, freqs, magnitude=1.0):
    a = _angles(pos, freqs)
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack((u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()), -1).flatten(-2) * magnitude


def _by_pair(rot):
    """Frequencies blended by the pair's index, and the magnitude of the turned vector."""
    dims, base, s = rot["dims"], rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not s:
        return f, 1.0

    def index(turns):
        return dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

    lo, hi = max(math.floor(index(s["fast"])), 0), min(math.ceil(index(s["slow"])), dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [x / s["factor"] * r + x * (1.0 - r) for x, r in zip(f, ramp)], 0.1 * math.log(s["factor"]) + 1.0


def _attend(q, k, v, cuts, scale, sink=None, cap=None, slopes=None):
    """Causal attention within each sequence: q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H, V]."""
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
    share = q.shape[1] // k.shape[1]
    for a, b in cuts:
        for h in range(q.shape[1]):
            kk, vv = k[a:b, h // share], v[a:b, h // share]
            for o in range(a, b, 2048):
                e = min(o + 2048, b)
                s = (q[o:e, h] @ kk[:e - a].T) * scale
                if cap:
                    s = cap * torch.tanh(s / cap)
                apart = torch.arange(o - a, e - a, device=q.device)[:, None] - torch.arange(e - a, device=q.device)
                if slopes is not None:
                    s = s - slopes[h] * apart
                s = s.masked_fill(apart < 0, -math.inf)
                top = s.max(-1, keepdim=True).values
                if sink is not None:
                    top = torch.maximum(top, sink[h])
                p = torch.exp(s - top)
                total = p.sum(-1, keepdim=True)
                if sink is not None:
                    total = total + torch.exp(sink[h] - top)
                out[o:e, h] = (p / total) @ vv[:e - a]
    return out.flatten(1)


def _conv_silu(x, taps, cuts):
    y, n = torch.zeros_like(x), taps.shape[1]
    for a, b in cuts:
        for j in range(min(n, b - a)):
            y[a + j:b] += taps[:, n - 1 - j] * x[a:b - j]
    return y * torch.sigmoid(y)


def _delta(h, W, p, m, eps, cuts):
    """The gated delta rule with one decay per head."""
    T, H, G, D, V = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]

    def conv(x):
        return _conv_silu(h @ W(p + x).T, W(p + x + ".conv"), cuts)

    def unit(x):
        return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)

    q = (unit(conv("q").view(T, G, D)) * D ** -0.5).repeat_interleave(H // G, 1)
    k = unit(conv("k").view(T, G, D)).repeat_interleave(H // G, 1)
    v = conv("v").view(T, H, V)
    beta = torch.sigmoid(h @ W(p + "b").T)
    gate = torch.nn.functional.silu(h @ W(p + "g").T)
    g = torch.exp(-torch.exp(W(p + "A_log")) * torch.nn.functional.softplus(h @ W(p + "a").T + W(p + "dt_bias")))
    out = torch.empty(T, H, V, dtype=h.dtype, device=h.device)
    # sequences of one length side by side
    for length in sorted({b - a_ for a_, b in cuts}):
        first = torch.tensor([a_ for a_, b in cuts if b - a_ == length], device=h.device)
        S = torch.zeros(len(first), H, D, V, dtype=h.dtype, device=h.device)
        for t in range(length):
            at = first + t
            S = g[at][..., None, None] * S
            kt = k[at][..., None]
            u = beta[at][..., None, None] * (v[at][..., None, :] - (S * kt).sum(-2, keepdim=True))
            S = S + kt * u
            out[at] = (S * q[at][..., None]).sum(-2)
    out = _rms(out, W(p + "norm"), eps).flatten(1) * gate
    return out @ W(p + "o").T


def _experts(x, ids, weights, n, expert):
    out = torch.zeros_like(x)
    for e in range(n):
        at, slot = (ids == e).nonzero(as_tuple=True)
        if len(at):
            out.index_add_(0, at, expert(e, x[at]) * weights[at, slot][:, None])
    return out


def _qwen2_moe(cfg, W, tokens, pos, cuts, rows):
    nh, nkv, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    T, silu = len(tokens), torch.nn.functional.silu
    h = W("model.embed_tokens.weight", tokens)
    for l in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{l}."
        x = _rms(h, W(p + "input_layernorm.weight"), eps)
        q, k, v = (x @ W(p + f"self_attn.{n}_proj.weight").T + W(p + f"self_attn.{n}_proj.bias") for n in "qkv")
        q, k, v = q.view(T, nh, -1), k.view(T, nkv, -1), v.view(T, nkv, -1)
        q, k = _turn_halves(q, pos, cfg["rope_theta"]), _turn_halves(k, pos, cfg["rope_theta"])
        h = h + _attend(q, k, v, cuts, q.shape[-1] ** -0.5) @ W(p + "self_attn.o_proj.weight").T
        x = _rms(h, W(p + "post_attention_layernorm.weight"), eps)
        if l == cfg["num_hidden_layers"] - 1:         # nothing reads the last layer's other rows
            h, x = h[rows], x[rows]

        def mlp(p, x):
            return (silu(x @ W(p + "gate_proj.weight").T) * (x @ W(p + "up_proj.weight").T)) @ W(p + "down_proj.weight").T

        weights, ids = torch.softmax(x @ W(p + "mlp.gate.weight").T, -1).topk(cfg["num_experts_per_tok"], -1)
        h = h + _experts(x, ids, weights, cfg["num_experts"], lambda e, z: mlp(p + f"mlp.experts.{e}.", z))
        h = h + torch.sigmoid(x @ W(p + "mlp.shared_expert_gate.weight").T) * mlp(p + "mlp.shared_expert.", x)
    return _rms(h, W("model.norm.weight"), eps) @ W("lm_head.weight").T


def _fokinex(cfg, W, tokens, pos, cuts, rows):
    eps, T = cfg["norm"]["eps"], len(tokens)
    x = W("embed", tokens) * cfg["embedding"]["scale"]
    kept = {}
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        h = _rms(x, W(p + "norm1"), eps)
        if layer["type"] == "latent_attention":
            H, D, R = m["heads"], m["dim"], m["kv_rank"]
            f, mag = _by_pair(m["rot"])
            if m.get("kv_from") is None:
                down = h @ W(p + "mix.dkv").T
                kept[i] = _rms(down[:, :R], W(p + "mix.dkv.norm"), eps), _turn_pairs(down[:, None, R:], pos, f, mag)
            c, k_rot = kept[i if m.get("kv_from") is None else m["kv_from"]]
            q = (_rms(h @ W(p + "mix.dq").T, W(p + "mix.dq.norm"), eps) @ W(p + "mix.uq").T).view(T, H, -1)
            q = torch.cat((q[..., :D], _turn_pairs(q[..., D:], pos, f, mag)), -1)
            k = torch.cat(((c @ W(p + "mix.uk").T).view(T, H, D), k_rot.expand(T, H, -1)), -1)
            y = _attend(q, k, (c @ W(p + "mix.uv").T).view(T, H, -1), cuts, m["scale"], sink=W(p + "mix.sink")) @ W(p + "mix.o").T
        else:
            a = m["left"]
            H, G, q, k = a["heads"], a["kv_heads"], h @ W(p + "mix.left.q").T, h @ W(p + "mix.left.k").T
            y = _attend(_rms(q, W(p + "mix.left.q.norm"), eps).view(T, H, -1), _rms(k, W(p + "mix.left.k.norm"), eps).view(T, G, -1),
                        k.view(T, G, -1), cuts, a["scale"], cap=a["softcap"], slopes=[2.0 ** (-8.0 * (j + 1) / H) for j in range(H)])
            y = m["left_scale"] * ((y * torch.sigmoid(h @ W(p + "mix.left.g").T)) @ W(p + "mix.left.o").T)
            y = y + m["right_scale"] * _delta(h, W, p + "mix.right.", m["right"], eps, cuts)
        f = p + "mlp."
        y = y + (torch.nn.functional.silu(h @ W(f + "gate").T) * (h @ W(f + "up").T)) @ W(f + "down").T
        x = x + y
    return _rms(x[rows], W("final.norm"), eps) @ W("head").T


def exact(c, seed):
    """The first pass on a new state: whole sequences from their first position, without a cache."""
    cfg = _config(c)
    depths = _depths(c)
    whole = dict(c, decode=0, prompt=sum(d + 2 for d in depths) + c["prompt"])
    if work(whole)["flops"] > 2e14:                   # over about 20 seconds in 64 bits
        return None
    from ferrox_amd.engine.model import Model         # the names and shapes of a model's tensors
    from ferrox_amd.models.registry import resolve
    arch = resolve(cfg)
    source = _Weights(cfg, seed, torch.bfloat16 if c["dtype"] == "bfloat16" else torch.float32)
    source.expect(Model(arch.build_spec(arch.config_class.from_dict(cfg), None)).named_params())

    def W(name, rows=None):
        t = source.tensor(name)
        return (t if rows is None else t[rows]).double()

    behind, brings, prompt = _tokens(c, seed, _vocab(cfg))
    sequences = [b + t[:2] for b, t in zip(behind, brings)] + ([prompt] if prompt else [])
    cuts, flat = [], []
    for s in sequences:
        cuts.append((len(flat), len(flat) + len(s)))
        flat += s
    tokens = torch.tensor(flat, device="cuda")
    pos = torch.cat([torch.arange(b - a, device="cuda") for a, b in cuts])
    wants = [1] * len(behind) + ([c["want"]] if prompt else [])
    rows = torch.tensor([b - n + j for (_, b), n in zip(cuts, wants) for j in range(n)], device="cuda")
    forward = _fokinex if c["model"].startswith("fokinex") else _qwen2_moe
    with torch.no_grad():
        return {"logits": forward(cfg, W, tokens, pos, cuts, rows)}
