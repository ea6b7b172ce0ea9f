"""What is measured: requests and prompts of whole models, as a program that uses this library
runs them on one GPU.

A pass takes a batch of prompts of unequal length through one step (``Engine.step``'s two
halves, so that the sampler gets the batch's keys), draws each one's first token, lets a
``DecodeSession`` draw the next ones, feeds the last token in a step of its own, whose logits
show everything that the session left in the cache, and gives the slots back.  A case without
new tokens is the prompt step alone.

Weights are random, drawn from the seed.  Three things are as in a trained model and not as in
plain noise, because with plain noise the results would hang on ties that two correct
implementations decide differently: the next token is clear (the head's rows follow the
embedding's), a router separates the experts that it chooses (tokens come in clusters, and each
cluster has its experts in every layer), and a sublayer's result is small beside the stream.
"""
import math
import random
import zlib

import torch

import gpt_fast_amd as gfa
from gpt_fast_amd.engine.decode import DecodeSession
from gpt_fast_amd.sampling import SamplingParams, sample
from gpt_fast_amd.weights.bindings import dtype_for_role

DEVICE = "cuda:0"
CLUSTERS = 64
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
# layers that are run of the two stacks whose presets have 32 of them
LAYERS = {"vusenex-4096": 8, "refolix-4096": 8}


# --------------------------------------------------------------------------- the cases
def _case(model, dtype, batch, shortest, longest, new, sampled=False, name=None):
    c = dict(model=model, dtype=dtype, batch=batch, shortest=shortest, longest=longest, new=new,
             sampled=sampled)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest: a small model answers a few words; launches and the host count
        _case("stories110M", "bfloat16", 1, 5, 5, 8, name="110M short request"),
        # the float32 engine, which users take to check results: a few requests of a small model
        _case("stories110M", "float32", 4, 20, 200, 12, name="110M float32 requests"),
        # one user at an 8B model: a question, an answer drawn token by token
        _case("llama-3.1-8b", "bfloat16", 1, 200, 200, 24, name="8B one request"),
        # a few users together, sampled as the command line does by default
        _case("llama-3.1-8b", "bfloat16", 8, 60, 400, 16, sampled=True, name="8B eight requests"),
        # a full batch of a throughput run
        _case("llama-3.1-8b", "bfloat16", 64, 50, 180, 12, name="8B full batch"),
        # time to the first token: a chat turn's prompt, the benchmark's prompt, prompts of
        # unequal length in one step
        _case("llama-3.1-8b", "bfloat16", 1, 300, 300, 0, name="8B chat prompt"),
        _case("llama-3.1-8b", "bfloat16", 1, 2048, 2048, 0, name="8B prompt of 2048"),
        _case("llama-3.1-8b", "bfloat16", 8, 16, 1024, 0, name="8B unequal prompts"),
        # a long document and the first words of an answer
        _case("llama-3.1-8b", "bfloat16", 1, 6001, 6001, 8, name="8B long document"),
        # mixtures of experts with latent attention and attention with a sink
        _case("vusenex-4096", "bfloat16", 16, 40, 200, 12, name="vusenex requests"),
        _case("vusenex-4096", "bfloat16", 1, 1777, 1777, 0, name="vusenex prompt"),
        # mixtures of gated experts with retention, windowed attention and the delta rule
        _case("refolix-4096", "bfloat16", 4, 150, 900, 12, name="refolix requests"),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    model = rng.choice(["llama-3.1-8b"] * 6 + ["vusenex-4096", "refolix-4096"] * 2 + ["stories110M"] * 2)
    dtype = "float32" if model == "stories110M" and rng.random() < 0.5 else "bfloat16"
    batch = 1 if rng.random() < 0.4 else _log_uniform(rng, 2, 64)
    # prompt tokens of one step at most, and of one sequence
    most, alone = {"llama-3.1-8b": (7000, 6001), "stories110M": (4000, 900)}.get(model, (4000, 2048))
    longest = _log_uniform(rng, 5, min(alone, most // batch))
    shortest = longest if batch == 1 else _log_uniform(rng, max(3, longest // 16), longest)
    new = 0 if rng.random() < 0.4 else _log_uniform(rng, 2, 16)
    return _case(model, dtype, batch, shortest, longest, new, sampled=new > 0 and rng.random() < 0.35)


def _lengths(case):
    rng = random.Random(f"{case['batch']} {case['shortest']} {case['longest']}")
    out = [rng.randint(case["shortest"], case["longest"]) for _ in range(case["batch"])]
    out[-1] = case["longest"]
    return out


def _prompts(case, seed, vocab):
    rng = random.Random(f"prompts {seed}")
    return [[rng.randrange(vocab) for _ in range(n)] for n in _lengths(case)]


def _config(case):
    """(architecture, typed configuration, its config.json dictionary)."""
    arch, config = gfa.find_preset(case["model"])
    raw = arch.config_dict(config)
    if case["model"] in LAYERS:
        raw["layers"] = raw["layers"][:LAYERS[case["model"]]]
        raw["max_positions"] = 8192
        config = arch.read_config(raw)
    return arch, config, raw


# --------------------------------------------------------------------------- the weights
class Weights:
    """Checkpoint tensors by name, each drawn from (seed, name)."""

    def __init__(self, raw, dtype, seed):
        self.raw, self.dtype, self.seed = raw, DTYPES[dtype], seed

    def _randn(self, name, shape, dtype):
        g = torch.Generator(device=DEVICE)
        g.manual_seed(zlib.crc32(f"{self.seed} {name}".encode()))
        return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)

    def _embedding(self, shape):
        own = self._randn("embedding", shape, self.dtype)
        if "layers" not in self.raw:
            return own
        centers = self._randn("centers", (CLUSTERS, shape[1]), self.dtype)
        kind = torch.arange(shape[0], device=DEVICE) % CLUSTERS
        return own.mul_(0.8).add_(centers[kind].mul_(0.6))

    def _router(self, name, shape):
        """Every cluster of tokens has its experts: half of them in each of two groups."""
        layer = self.raw["layers"][int(name[1:name.index(".")])]
        r = layer["mlp"]["router"]
        groups, keep = r["groups"]["count"], r["groups"]["keep"]
        size, each = shape[0] // groups, r["top"] // keep
        rng = random.Random(f"{self.seed} {name}")
        gain = torch.zeros(shape[0], CLUSTERS)
        for c in range(CLUSTERS):
            for g in rng.sample(range(groups), keep):
                for e in rng.sample(range(size), each):
                    gain[g * size + e, c] = rng.uniform(2.5, 4.5)
        centers = self._randn("centers", (CLUSTERS, shape[1]), self.dtype)
        return (gain.to(DEVICE) @ centers.float() / (0.6 * shape[1])).to(self.dtype)

    def __call__(self, name, shape, init="linear", dtype=None):
        dtype = dtype or self.dtype
        if name in ("embed", "model.embed_tokens.weight"):
            return self._embedding(shape)
        if name in ("head", "lm_head.weight"):          # the next token is the current one plus one
            return self._embedding(shape).roll(1, 0).mul_(0.02)
        if name.endswith("mlp.router"):
            return self._router(name, shape)
        t = self._randn(name, shape, dtype)
        if init == "linear":
            std = 0.02
            if name.endswith(("o_proj.weight", "down_proj.weight")):
                std /= math.sqrt(2.0 * self.raw["num_hidden_layers"])
            return t.mul_(std)
        if init == "unit":
            return t
        if name.endswith("correction"):
            return t.mul_(0.03)
        t = t.mul_(0.1) if init == "around_zero" else t.mul_(0.1).add_(1.0)
        if init == "positive":
            return t.abs_()
        own = name.split(".")[-1]
        if "layers" in self.raw and name.count(".") == 1:    # factors on a sublayer's result
            if own in ("ls1", "ls2"):
                return t.mul_(0.3)
            if own in ("norm1", "norm2") and len(shape) == 0:
                return t.mul_(0.15)
        return t


# --------------------------------------------------------------------------- the pass
def prepare(case, seed):
    arch, config, raw = _config(case)
    draw_weight = Weights(raw, case["dtype"], seed)
    compute = DTYPES[case["dtype"]]
    parameters = {}
    for b in arch.bindings(config).bindings:
        parts = [draw_weight(s.name, s.shape, s.init, dtype_for_role(b.role, compute)) for s in b.sources]
        parameters[b.target] = (b.combine(parts) if b.combine else parts[0]).contiguous()
    pages = sum((n + case["new"] + 2 + 63) // 64 + 1 for n in _lengths(case))
    engine = gfa.Engine.from_plan(arch.plan(config), parameters, case["dtype"], DEVICE,
                                  max_tokens=64 * pages, max_sequences=case["batch"])
    params = SamplingParams(temperature=0.8, top_k=200, seed=seed) if case["sampled"] \
        else SamplingParams(temperature=0.0)
    return {"engine": engine, "prompts": _prompts(case, seed, engine.vocab_size), "params": params,
            "new": case["new"]}


def run(state):
    engine, params, new = state["engine"], state["params"], state["new"]
    slots = [engine.start_sequence() for _ in state["prompts"]]
    entries = [gfa.Entry(s, p, want=[len(p) - 1], key=i) for i, (s, p) in enumerate(zip(slots, state["prompts"]))]
    if not new:
        out = {"first_logits": engine.step(entries)}
    else:
        with torch.no_grad():
            batch = engine.prepare(entries)
            first = engine.model.forward(batch, engine.cache)
            token = sample(first, params, batch.row_keys, batch.want_pos, position_offset=1)
        session = DecodeSession(engine, slots, [e.key for e in entries], token, params, max_new_tokens=new)
        tokens, under_way = [token.tolist()], None
        for _ in range(new - 1):
            handle = session.launch()
            if under_way is not None:                    # read one step late, as generate() does
                tokens.append(session.collect(under_way))
            under_way = handle
        tokens.append(session.collect(under_way))
        session.close()
        last = engine.step([gfa.Entry(s, [t], want=[0], key=i) for i, (s, t) in enumerate(zip(slots, tokens[-1]))])
        out = {"first_logits": first, "tokens": torch.tensor(tokens), "last_logits": last}
    for s in slots:
        engine.end_sequence(s)
    return out


# --------------------------------------------------------------------------- what it costs
def _sizes(raw):
    """(weights every token is multiplied with, weights of one expert, experts, chosen, heads x size of
    every layer with attention over all keys, cached numbers per token, vocabulary x width)."""
    if "layers" not in raw:
        D, H, L = raw["hidden_size"], raw["num_attention_heads"], raw["num_hidden_layers"]
        G, hd, inner = raw["num_key_value_heads"], raw["head_dim"], raw["intermediate_size"]
        dense = L * (D * (H + 2 * G) * hd + H * hd * D + 3 * D * inner)
        return dense, 0, 0, 0, L * H * hd, L * 2 * G * hd, raw["vocab_size"] * D
    D = raw["width"]
    dense = expert = experts = chosen = scores = cached = 0
    for l in raw["layers"]:
        m, f = l["mixer"], l["mlp"]
        if l["type"] == "parallel":
            a, r = m["left"], m["right"]
            dense += D * a["dim"] * (2 * a["heads"] + 2 * a["kv_heads"])
            dense += D * r["dim"] * (2 * r["kv_heads"] + 3 * r["heads"])
            scores += a["heads"] * a["dim"]
            cached += 2 * a["kv_heads"] * a["dim"]
        elif l["type"] == "retention":
            dense += 5 * D * m["heads"] * m["dim"]
        elif l["type"] == "latent_attention":
            dense += D * (2 * m["heads"] * m["dim"] + m["kv_rank"]) + 2 * m["heads"] * m["dim"] * m["kv_rank"]
            scores += m["heads"] * m["dim"]
            cached += m["kv_rank"]
        else:
            dense += D * m["dim"] * (2 * m["heads"] + m["kv_heads"])
            scores += m["heads"] * m["dim"]
            cached += 2 * m["kv_heads"] * m["dim"]
        gated = raw["architecture"] == "Refolix"
        dense += (3 if gated else 2) * D * f["shared"]["ff"] + D * f["router"]["experts"]
        if not gated:
            dense += 2 * D * D                           # the gates on both sublayers' results
        expert = (3 if gated else 2) * D * f["expert"]["ff"]
        experts, chosen = f["router"]["experts"], f["router"]["top"]
    return dense, expert, experts, chosen, scores, cached, raw["vocab"] * D


def work(case):
    raw = _config(case)[2]
    dense, expert, experts, chosen, scores, cached, head = _sizes(raw)
    layers = len(raw["layers"]) if "layers" in raw else 0
    size = 2 if case["dtype"] == "bfloat16" else 4
    n_bytes = flops = 0.0
    lengths = _lengths(case)
    # the prompt step, then `new` steps of one token per sequence
    for step in range(1 + case["new"]):
        new = lengths if step == 0 else [1] * len(lengths)
        held = [0] * len(lengths) if step == 0 else [n + step - 1 for n in lengths]
        tokens, rows = sum(new), len(lengths)
        read = experts * (1.0 - (1.0 - chosen / experts) ** tokens) if experts else 0.0
        keys = sum(t * h + t * (t + 1) / 2 for t, h in zip(new, held))
        n_bytes += size * (dense + layers * read * expert + head)
        n_bytes += size * cached * (sum(held) + tokens) + 4 * rows * (head // raw.get("hidden_size", raw.get("width")))
        flops += 2.0 * tokens * (dense + layers * chosen * expert) + 2.0 * rows * head + 4.0 * scores * keys
    return {"bytes": n_bytes, "flops": flops}


def tolerance(case):
    """About four times what two correct implementations differ by: each is off the result in 64
    bits by (measured) 5e-7 in float32, 2e-3 in bfloat16 through 8 to 12 layers, 8e-3 through 32."""
    if case["dtype"] == "float32":
        return {"rel": 4e-6}
    return {"rel": 2.5e-2 if case["model"] == "llama-3.1-8b" else 8e-3}


# --------------------------------------------------------------------------- in 64 bits
F = torch.float64


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, eps):
    x = x - x.mean(-1, keepdim=True)
    return _rms(x, eps) * w


def _silu(z):
    return z * torch.sigmoid(z)


def _half_turn(x, positions, freqs, dims, grow=1.0):
    """x [T, heads, d]: pairs (i, i + dims / 2) of the first dims elements turned."""
    a = positions.to(F)[:, None] * freqs[None, :]
    c, s = (a.cos() * grow)[:, None, :], (a.sin() * grow)[:, None, :]
    u, v, rest = x[..., :dims // 2], x[..., dims // 2:dims], x[..., dims:]
    return torch.cat([u * c - v * s, v * c + u * s, rest], -1)


def _pair_turn(x, positions, freqs, dims, grow=1.0):
    """x [T, heads, d]: pairs (2 i, 2 i + 1) of the first dims elements turned."""
    a = positions.to(F)[:, None] * freqs[None, :]
    c, s = (a.cos() * grow)[:, None, :], (a.sin() * grow)[:, None, :]
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    turned = torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
    return torch.cat([turned, x[..., dims:]], -1)


def _ladder(dims, base):
    return torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F, device=DEVICE)


def _llama_ladder(raw, dims):
    f = _ladder(dims, raw["rope_theta"])
    sc = raw.get("rope_scaling")
    if not sc:
        return f
    length = 2.0 * math.pi / f
    low = sc["original_max_position_embeddings"] / sc["low_freq_factor"]
    high = sc["original_max_position_embeddings"] / sc["high_freq_factor"]
    mix = (sc["original_max_position_embeddings"] / length - sc["low_freq_factor"]) / (
        sc["high_freq_factor"] - sc["low_freq_factor"])
    between = (1.0 - mix) * f / sc["factor"] + mix * f
    return torch.where(length > low, f / sc["factor"], torch.where(length < high, f, between))


def _ramped_ladder(rot):
    """(frequencies, factor on cos and sin): the slow end of the ladder divided along a ramp."""
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    f = _ladder(dims, base)
    if not sc:
        return f, 1.0

    def place(turns):
        return dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(place(sc["fast"])), 0), min(math.ceil(place(sc["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, device=DEVICE).to(F) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


class _Packed:
    """Whole sequences, packed back to back."""

    def __init__(self, sequences):
        self.tokens = torch.tensor([t for s in sequences for t in s], device=DEVICE)
        self.lengths = [len(s) for s in sequences]
        self.ranges, n = [], 0
        for length in self.lengths:
            self.ranges.append((n, n + length))
            n += length
        self.positions = torch.cat([torch.arange(n, device=DEVICE) for n in self.lengths])

    def attention(self, q, k, v, scale, scores=None, window=None, sink=False):
        """Causal attention with grouped keys; ``scores(head, s, distance)`` changes a head's scores."""
        H, G = q.shape[1], k.shape[1]
        out = torch.empty(q.shape[0], H, v.shape[2], dtype=F, device=DEVICE)
        for a, b in self.ranges:
            i = torch.arange(b - a, device=DEVICE)
            distance = i[:, None] - i[None, :]
            hidden = distance < 0 if window is None else (distance < 0) | (distance >= window)
            for h in range(H):
                g = h // (H // G)
                s = (q[a:b, h] @ k[a:b, g].T) * scale
                if scores is not None:
                    s = scores(h, s, distance)
                s = s.masked_fill_(hidden, -math.inf)
                if sink:                                 # one more key of score 0 without a value
                    m = s.max(-1, keepdim=True).values.clamp_(min=0.0)
                    e = torch.exp(s - m)
                    out[a:b, h] = (e @ v[a:b, g]) / (torch.exp(-m) + e.sum(-1, keepdim=True))
                else:
                    out[a:b, h] = torch.softmax(s, -1) @ v[a:b, g]
        return out


def _llama(raw, W, x, seqs):
    D, H, G, hd = raw["hidden_size"], raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"]
    inner, eps, T = raw["intermediate_size"], raw["rms_norm_eps"], x.shape[0]
    freqs = _llama_ladder(raw, hd)

    def turn(t):
        return _half_turn(t, seqs.positions, freqs, hd)
    for i in range(raw["num_hidden_layers"]):
        p = f"model.layers.{i}."

        def lin(h, name, n_out, n_in):
            return h @ W(p + name + ".weight", (n_out, n_in)).to(F).T
        h = _rms(x, eps) * W(p + "input_layernorm.weight", (D,), "norm", torch.float32)
        q = turn(lin(h, "self_attn.q_proj", H * hd, D).view(T, H, hd))
        k = turn(lin(h, "self_attn.k_proj", G * hd, D).view(T, G, hd))
        v = lin(h, "self_attn.v_proj", G * hd, D).view(T, G, hd)
        o = seqs.attention(q, k, v, hd ** -0.5)
        x = x + lin(o.view(T, H * hd), "self_attn.o_proj", D, H * hd)
        h = _rms(x, eps) * W(p + "post_attention_layernorm.weight", (D,), "norm", torch.float32)
        h = _silu(lin(h, "mlp.gate_proj", inner, D)) * lin(h, "mlp.up_proj", inner, D)
        x = x + lin(h, "mlp.down_proj", D, inner)
    return _rms(x, eps) * W("model.norm.weight", (D,), "norm", torch.float32)


def _chosen_experts(scores, choice, group_score, r):
    """(experts [T, top], weights [T, top]): the best groups, then the best of their experts."""
    T, E = scores.shape
    count, keep = r["groups"]["count"], r["groups"]["keep"]
    best = group_score.topk(keep, dim=-1).indices
    open_ = torch.zeros(T, count, dtype=torch.bool, device=DEVICE).scatter_(1, best, True)
    open_ = open_[:, :, None].expand(T, count, E // count).reshape(T, E)
    chosen = choice.masked_fill(~open_, -math.inf).topk(r["top"], dim=-1).indices
    picked = scores.gather(1, chosen)
    return chosen, picked / (picked.sum(-1, keepdim=True) + 1e-20)


def _experts(h, chosen, weights, one):
    y = torch.zeros_like(h)
    for e in torch.unique(chosen).tolist():
        row, place = (chosen == e).nonzero(as_tuple=True)
        y.index_add_(0, row, one(h[row], e) * weights[row, place][:, None])
    return y


def _vusenex(raw, W, x, seqs):
    D, eps, T = raw["width"], raw["norm"]["eps"], x.shape[0]
    f32 = torch.float32
    pair = raw["embedding"]["bigram"]
    before = seqs.tokens.roll(1)
    row = (before * pair["mul_prev"] + seqs.tokens * pair["mul_cur"]) % pair["buckets"]
    row = torch.where(seqs.positions == 0, pair["buckets"], row)
    x = x + W("bigram", (pair["buckets"] + 1, D))[row].to(F) + W("pos", (raw["max_positions"], D))[seqs.positions].to(F)

    def gelu(z):
        return 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0)))
    for i, layer in enumerate(raw["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        H, d = m["heads"], m["dim"]

        def lin(h, name, n_out, n_in):
            return h @ W(p + name, (n_out, n_in)).to(F).T

        def vec(name, n, init="norm"):
            return W(p + name, (n,), init, f32).to(F)

        def joined(x, y, gate, norm):
            y = y * torch.sigmoid(lin(x, gate, D, D) + vec(gate + ".b", D, "around_zero"))
            return x + _rms(y, eps) * W(p + norm, (), "norm", f32).to(F)
        if layer["type"] == "latent_attention":
            R = m["kv_rank"]
            c = _rms(lin(x, "mix.dkv", R, D), eps) * vec("mix.dkv.norm", R)
            q, k = lin(x, "mix.q", H * d, D), lin(c, "mix.uk", H * d, R)
            v = lin(c, "mix.uv", H * d, R)
            o = seqs.attention(q.view(T, H, d), k.view(T, H, d), v.view(T, H, d), m["scale"])
        else:
            G = m["kv_heads"]
            q = lin(x, "mix.q", H * d, D) + vec("mix.q.b", H * d, "around_zero")
            v = lin(x, "mix.k", G * d, D) + vec("mix.k.b", G * d, "around_zero")
            q, k = _rms(q, eps) * vec("mix.q.norm", H * d), _rms(v, eps) * vec("mix.k.norm", G * d)
            t = m["q_temp"]
            turns = torch.div(seqs.positions + 1, t["every"], rounding_mode="floor") + 1
            q = q * (1.0 + t["coef"] * turns.to(F).log())[:, None]
            r1, r2 = vec("mix.r1", H, "positive"), vec("mix.r2", H, "positive")
            o = seqs.attention(q.view(T, H, d), k.view(T, G, d), v.view(T, G, d), m["scale"], sink=True,
                               scores=lambda h, s, dist: s - r1[h] * torch.log1p(r2[h] * dist.clamp(min=0).to(F)))
        x = joined(x, lin(o.reshape(T, H * d), "mix.o", D, H * d), "rg1", "norm1")
        r, ff, shared = f["router"], f["expert"]["ff"], f["shared"]["ff"]
        s = torch.softmax(lin(x, "mlp.router", r["experts"], D), -1)
        chosen, weights = _chosen_experts(s, s, s.view(T, r["groups"]["count"], -1).max(-1).values, r)
        y = _experts(x, chosen, weights,
                     lambda h, e: lin(gelu(lin(h, f"mlp.e{e}.up", ff, D)), f"mlp.e{e}.down", D, ff))
        y = y + lin(gelu(lin(x, "mlp.shared.up", shared, D)), "mlp.shared.down", D, shared)
        x = joined(x, y, "rg2", "norm2")
    return _rms(x, eps) * W("final.norm", (), "norm", f32).to(F)


def _delta_rule(q, k, v, g, beta, seqs):
    """Per head S <- g S;  S <- S + k (beta (v - S^T k))^T;  o = S^T q, all sequences side by side."""
    H, B, most = v.shape[1], len(seqs.lengths), max(seqs.lengths)
    k, q = (t.repeat_interleave(H // t.shape[1], 1) for t in (k, q))

    def padded(t):
        out = torch.zeros(most, B, *t.shape[1:], dtype=F, device=DEVICE)
        for n, (a, b) in enumerate(seqs.ranges):
            out[:b - a, n] = t[a:b]
        return out
    q, k, v, g, beta = (padded(t) for t in (q, k, v, g, beta))
    S = torch.zeros(B, H, k.shape[3], v.shape[3], dtype=F, device=DEVICE)
    o = torch.empty_like(v)
    for t in range(most):
        S = g[t][..., None, None] * S
        u = beta[t][..., None] * (v[t] - (k[t][..., None, :] @ S)[..., 0, :])
        S = S + k[t][..., :, None] * u[..., None, :]
        o[t] = (q[t][..., None, :] @ S)[..., 0, :]
    return torch.cat([o[:n, i] for i, n in enumerate(seqs.lengths)])


def _refolix(raw, W, x, seqs):
    D, eps, alpha, T = raw["width"], raw["norm"]["eps"], raw["postln_alpha"], x.shape[0]
    f32 = torch.float32
    x = x * raw["embedding"]["scale"]
    for i, layer in enumerate(raw["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]

        def lin(h, name, n_out, n_in):
            return h @ W(p + name, (n_out, n_in)).to(F).T

        def vec(name, shape, init="norm"):
            return W(p + name, shape if isinstance(shape, tuple) else (shape,), init, f32).to(F)

        def convolved(name, n, taps):
            t, w = lin(x, "mix.right." + name, n, D), vec(f"mix.right.{name}.conv", (n, taps), "unit")
            out = t * w[:, -1]
            for back in range(1, taps):
                moved = torch.where((seqs.positions >= back)[:, None], t.roll(back, 0), 0.0)
                out = out + moved * w[:, taps - 1 - back]
            return _silu(out)
        if layer["type"] == "parallel":
            a, r = m["left"], m["right"]
            H, G, d = a["heads"], a["kv_heads"], a["dim"]
            freqs, grow = _ramped_ladder(a["rot"])
            q, k = (_pair_turn(_rms(lin(x, "mix.left." + n, heads * d, D).view(T, heads, d), eps)
                               * vec(f"mix.left.{n}.norm", d), seqs.positions, freqs, a["rot"]["dims"], grow)
                    for n, heads in (("q", H), ("k", G)))
            v = lin(x, "mix.left.v", G * d, D).view(T, G, d)
            o = seqs.attention(q, k, v, a["scale"], window=a["mask"]["size"],
                               scores=lambda h, s, dist: a["softcap"] * torch.tanh(s / a["softcap"]))
            left = lin(o.reshape(T, H * d), "mix.left.o", D, H * d)
            H, G, d, taps = r["heads"], r["kv_heads"], r["dim"], r["conv"]
            q, k = (convolved(n, G * d, taps).view(T, G, d) for n in ("q", "k"))
            v = convolved("v", H * d, taps).view(T, H, d)
            q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            beta = torch.sigmoid(lin(x, "mix.right.b", H, D))
            z = lin(x, "mix.right.a", H, D) + vec("mix.right.dt_bias", H, "around_zero")
            g = torch.exp(-torch.exp(vec("mix.right.A_log", H, "around_zero")) * torch.nn.functional.softplus(z))
            o = _rms(_delta_rule(q * d ** -0.5, k, v, g, beta, seqs), eps) * vec("mix.right.norm", d)
            o = o.reshape(T, H * d) * _silu(lin(x, "mix.right.g", H * d, D))
            right = lin(o, "mix.right.o", D, H * d)
            y = 0.5 * (_rms(left, eps) * vec("mix.left.out", D) + _rms(right, eps) * vec("mix.right.out", D))
        else:
            H, d = m["heads"], m["dim"]
            freqs, grow = _ramped_ladder(m["rot"])
            q, k = (_half_turn(lin(x, "mix." + n, H * d, D).view(T, H, d), seqs.positions, freqs, m["rot"]["dims"],
                               grow) for n in ("q", "k"))
            v = lin(x, "mix.v", H * d, D).view(T, H, d)
            o = torch.empty(T, H, d, dtype=F, device=DEVICE)
            for a, b in seqs.ranges:
                n = torch.arange(b - a, device=DEVICE)
                back = (n[:, None] - n[None, :]).to(F)
                for h in range(H):
                    held = torch.where(back >= 0, float(m["decay"][h]) ** back.clamp(min=0.0), 0.0)
                    o[a:b, h] = ((q[a:b, h] @ k[a:b, h].T) * d ** -0.5 * held) @ v[a:b, h]
            y = lin(_rms(o, eps).reshape(T, H * d) * _silu(lin(x, "mix.g", H * d, D)), "mix.o", D, H * d)
        x = _layer_norm(alpha * x + vec("ls1", D) * y, vec("norm1", D), eps)
        r, ff, shared = f["router"], f["expert"]["ff"], f["shared"]["ff"]
        s = torch.sigmoid(lin(x, "mlp.router", r["experts"], D))
        choice = s + vec("mlp.correction", r["experts"], "around_zero")
        by_group = choice.view(T, r["groups"]["count"], -1).topk(2, dim=-1).values.sum(-1)
        chosen, weights = _chosen_experts(s, choice, by_group, r)

        def gated(h, name, n):
            return lin(_silu(lin(h, name + ".gate", n, D)) * lin(h, name + ".up", n, D), name + ".down", D, n)
        y = _experts(x, chosen, weights, lambda h, e: gated(h, f"mlp.e{e}", ff))
        y = y + torch.sigmoid(lin(x, "mlp.shared.sg", 1, D)) * gated(x, "mlp.shared", shared)
        x = _layer_norm(alpha * x + vec("ls2", D) * y, vec("norm2", D), eps)
    return _layer_norm(x, W("final.norm", (D,), "norm", f32).to(F), eps)


@torch.no_grad()
def exact(case, seed):
    """The tokens are whole numbers and have no value here; the last logits are those behind the
    tokens that follow each other, which is what every pass draws."""
    raw = _config(case)[2]
    W = Weights(raw, case["dtype"], seed)
    V, D = raw.get("vocab_size", raw.get("vocab")), raw.get("hidden_size", raw.get("width"))
    prompts, new = _prompts(case, seed, V), case["new"]
    seqs = _Packed([p + [(p[-1] + 1 + j) % V for j in range(new)] for p in prompts])
    llama = "layers" not in raw
    x = W("model.embed_tokens.weight" if llama else "embed", (V, D))[seqs.tokens].to(F)
    x = (_llama if llama else _vusenex if raw["architecture"] == "Vusenex" else _refolix)(raw, W, x, seqs)
    head = W("lm_head.weight" if llama else "head", (V, D)).to(F)

    def logits(back):
        z = x[[b - 1 - back for _, b in seqs.ranges]] @ head.T
        cap = raw.get("logit_softcap")
        return cap * torch.tanh(z / cap) if cap else z
    out = {"first_logits": logits(new)}
    if new:
        follow = all((logits(j).argmax(-1) == torch.tensor([(p[-1] + 1 + new - j) % V for p in prompts],
                                                           device=DEVICE)).all() for j in range(1, new + 1))
        out.update(tokens=None, last_logits=logits(0) if follow else None)
    return out
