"""The work that users of this library have it do, as cases that can be timed and checked.

A case is one pass of a serving or scoring program through the public entry points:

* "decode": a batch of running sequences gets its next STEPS tokens, the way the generation loop asks for them
  (`Engine.decode_and_choose_many`), greedily or sampled.  The sequences go on from pass to pass; when they reach the end
  of their room they end and the same requests start again, as in a server.
* "prefill": new requests' prompts go through in one step (`Engine.step`), the logits of their last tokens come back.
* "score": the model is called on token ids and gives the logits of every place.

Sizes: the Llama-3-8B, Llama-2-7B and micro shapes of the library's registry and of its benchmark (fewer layers, all of
one shape, so that a pass stays short), and its Zodolorn "4b-a1b" (attention over a latent, experts) and Defapel "3b-a1b"
(windowed attention beside a delta rule, experts) variants, likewise.  Weights are random: the library's rule, a
function of the seed and a tensor's name, with an embedding that stays visible through the layers and a head that follows
it, so that every next token has a clear winner, as in a trained model (a near tie would let rounding choose another
continuation).  `exact` computes the same numbers from the same rule in float64, in plain torch.
"""

from __future__ import annotations

import hashlib
import math

import numpy as np
import torch

import fms_amd
from fms_amd.architectures import variant_config
from fms_amd.engine import Engine
from fms_amd.sampling import SamplingParams, choose, request_seed

STEPS = 4  # decode steps of a pass: as many as the generation loop runs before it looks at the tokens
ROOM = 1024  # tokens that a running sequence may grow by before its request ends

# model -> (architecture, variant, overrides, factor on the embedding's 0.02)
MODELS = {
    "llama-micro": ("llama", "micro", {}, 50.0),
    "llama-3-8b": ("llama", "3-8b", {"max_expected_seq_len": 8192}, 100.0),
    "llama-2-7b": ("llama", "2-7b", {"max_expected_seq_len": 4096}, 100.0),
    # With experts the embedding is most of the stream: a router's near tie, which rounding may turn either way, then
    # moves a token's logits by two per cent and not by ten.  (Zodolorn's embedding is scaled by sqrt(width) as well.)
    "zodolorn-4b-a1b": ("zodolorn", "4b-a1b", {}, 16.0),
    "defapel-3b-a1b": ("defapel", "3b-a1b", {}, 600.0),
}
MAX_LEN = {"llama-micro": 1024, "llama-2-7b": 4096}


def _case(name, model, layers, what, batch, shortest, longest, dtype="bf16", sampled=False):
    c = dict(model=model, layers=layers, what=what, batch=batch, shortest=shortest, longest=longest, dtype=dtype, sampled=sampled)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a chat with a model so small that only launches and latency count
        _case("micro_decode_1", "llama-micro", 5, "decode", 1, 64, 64),
        # one user at a terminal: a token of one sequence reads every weight once
        _case("8b_decode_1", "llama-3-8b", 8, "decode", 1, 1024, 1024),
        # the benchmark's headline: a small serving batch with contexts of all lengths
        _case("8b_decode_8", "llama-3-8b", 8, "decode", 8, 128, 2048),
        # a full serving batch that samples (top_k 10, the default of generate)
        _case("8b_decode_64_sampled", "llama-3-8b", 8, "decode", 64, 128, 2048, sampled=True),
        # long documents: the cache is as much to read as the weights
        _case("8b_decode_8_long", "llama-3-8b", 8, "decode", 8, 6900, 7000),
        # a prompt of the benchmark's size
        _case("8b_prefill_2048", "llama-3-8b", 8, "prefill", 1, 2048, 2048),
        # a batch of unequal prompts in one ragged step
        _case("8b_prefill_ragged", "llama-3-8b", 8, "prefill", 9, 17, 1025),
        # scoring a text in float32: logits of every place
        _case("7b_score_f32", "llama-2-7b", 4, "score", 1, 301, 301, dtype="fp32"),
        # a mixture of experts with attention over a latent: a prompt, and a serving batch
        _case("zodolorn_prefill_2048", "zodolorn-4b-a1b", 4, "prefill", 1, 2048, 2048),
        _case("zodolorn_decode_32", "zodolorn-4b-a1b", 4, "decode", 32, 128, 2048),
        # a recurrent model with a mixture of experts: two prompts of odd lengths, and a small serving batch
        _case("defapel_prefill_2", "defapel-3b-a1b", 4, "prefill", 2, 777, 1500),
        _case("defapel_decode_8", "defapel-3b-a1b", 4, "decode", 8, 128, 2048),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["llama_decode", "llama_decode", "llama_prefill", "llama_prefill", "score_f32", "family_prefill", "family_decode"])
    llama = rng.choice(["llama-3-8b", "llama-3-8b", "llama-2-7b"])
    family = rng.choice(["zodolorn-4b-a1b", "defapel-3b-a1b"])
    if kind == "llama_decode":
        batch = _log_int(rng, 1, 64)
        longest = _log_int(rng, 128, min(2900, 16 * 7000 // batch))
        return _case(None, llama, 8, "decode", batch, _log_int(rng, 64, longest), longest, sampled=rng.random() < 0.5)
    if kind == "llama_prefill":
        total = _log_int(rng, 16, 4600)
        batch = rng.randint(1, max(1, min(9, total // 16)))
        longest = max(1, min(2900, total * 3 // (2 * batch)) if batch > 1 else min(2900, total))
        return _case(None, llama, 8, "prefill", batch, max(1, min(longest, 2 * total // batch - longest)), longest)
    if kind == "score_f32":
        n = _log_int(rng, 8, 301)
        return _case(None, "llama-2-7b", 4, "score", 1, n, n, dtype="fp32")
    if kind == "family_prefill":
        longest = _log_int(rng, 32, 2048)
        batch = rng.randint(1, max(1, min(4, 2400 // longest)))
        return _case(None, family, 4, "prefill", batch, longest if batch == 1 else rng.randint(1 + longest // 2, longest), longest)
    batch = _log_int(rng, 1, 32)
    longest = _log_int(rng, 128, 2048)
    return _case(None, family, 4, "decode", batch, _log_int(rng, 64, longest), longest)


def _lengths(case):
    n, lo, hi = case["batch"], case["shortest"], case["longest"]
    return [hi] if n == 1 else [lo + i * (hi - lo) // (n - 1) for i in range(n)]


def _config(case):
    arch, variant, overrides, _ = MODELS[case["model"]]
    if arch == "llama":
        return variant_config(arch, variant, nlayers=case["layers"], **overrides)
    full = variant_config(arch, variant)
    return variant_config(arch, variant, layers=full.layers[: case["layers"]])


def _vocab(config):
    return getattr(config, "src_vocab_size", None) or config.vocab


def _prompts(case, seed, vocab):
    rng = np.random.default_rng([seed, 17])
    return [[int(t) for t in rng.integers(0, vocab, n)] for n in _lengths(case)]


def _followers(vocab, seed):
    """before[v]: the token that v follows."""
    return torch.from_numpy(np.random.default_rng([seed, 23]).permutation(vocab))


def _names(case):
    """(embedding, head or None if it is the embedding)"""
    arch = MODELS[case["model"]][0]
    return {"llama": ("base_model.embedding.weight", "head.weight"), "zodolorn": ("embed.weight", "head.weight"),
            "defapel": ("embed.weight", None)}[arch]


# ---- the program's side ------------------------------------------------------------------------------------------
def _model(case, seed):
    config = _config(case)
    arch, _, _, factor = MODELS[case["model"]]
    model = fms_amd.from_config(config, arch, data_type=case["dtype"], random_seed=seed)
    tensors = model.state_dict()
    embed, head = _names(case)
    if head is not None:
        tensors[head].copy_(tensors[embed][_followers(_vocab(config), seed).to(tensors[embed].device)])
    tensors[embed].mul_(factor)
    for name, t in tensors.items():
        if name.endswith("conv.weight"):
            t.mul_(16.0)
    return model


def _start(state):
    """The requests' prompts go through, one after the other, and their first tokens are chosen."""
    engine, tokens = state["engine"], []
    state["slots"] = [engine.new_sequence() for _ in state["prompts"]]
    for r, (slot, prompt) in enumerate(zip(state["slots"], state["prompts"])):
        logits = engine.step([slot], [prompt], "last")
        tokens += choose(logits, state["sampling"], [state["seeds"][r]], [0]).tolist()
    state["tokens"], state["done"] = tokens, 1


def _decode(state):
    if max(len(p) for p in state["prompts"]) + state["done"] + STEPS > state["end"]:
        for slot in state["slots"]:
            state["engine"].end_sequence(slot)
        _start(state)
    counters = [state["done"]] * len(state["slots"])
    chosen = state["engine"].decode_and_choose_many(state["slots"], state["tokens"], state["sampling"], state["seeds"], counters, steps=STEPS)
    state["tokens"] = chosen[-1]
    state["done"] += STEPS
    return chosen


def prepare(case, seed):
    model = _model(case, seed)
    state = {"what": case["what"], "model": model}
    prompts = _prompts(case, seed, model.spec.vocab)
    if case["what"] == "score":
        state["ids"] = torch.tensor(prompts)
        return state
    state["prompts"] = prompts
    decode = case["what"] == "decode"
    top = MAX_LEN.get(case["model"], 8192)
    state["end"] = min(max(len(p) for p in prompts) + ROOM, top)
    room = sum(-(-(len(p) + (ROOM if decode else 0)) // 64) * 64 for p in prompts)
    state["engine"] = Engine(model, max_tokens=room, max_slots=len(prompts))
    state["sampling"] = SamplingParams(do_sample=case["sampled"], temperature=1.0, top_k=10)
    state["seeds"] = [request_seed(seed, r) for r in range(len(prompts))]
    if decode:  # a server that is running: the requests are in the cache and their first STEPS tokens are out
        _start(state)
        _decode(state)
    return state


def run(state):
    if state["what"] == "score":
        return {"logits": state["model"](state["ids"])}
    engine = state["engine"]
    if state["what"] == "prefill":
        slots = [engine.new_sequence() for _ in state["prompts"]]
        logits = engine.step(slots, state["prompts"], "last")
        for slot in slots:
            engine.end_sequence(slot)
        return {"logits": logits}
    chosen = _decode(state)
    return {"tokens": np.array(chosen), "logits": engine.last_graph.logits[: len(chosen[0])]}


# ---- what a pass cannot do without -----------------------------------------------------------------------------
def work(case):
    config = _config(case)
    size = 4 if case["dtype"] == "fp32" else 2
    lengths = _lengths(case)
    decode = case["what"] == "decode"
    rows = len(lengths) if decode else sum(lengths)  # tokens of a step
    wanted = sum(lengths) if case["what"] == "score" else len(lengths)
    arch = MODELS[case["model"]][0]
    vocab, width = _vocab(config), (config.emb_dim if arch == "llama" else config.width)
    weights = vocab * width  # the head; of the embedding only the tokens' rows
    flops = 2.0 * wanted * vocab * width
    other = rows * width * size + wanted * vocab * 4.0  # embedding rows, logits

    def product(out, inner, used=1.0):
        nonlocal weights, flops
        weights += used * out * inner
        flops += 2.0 * rows * out * inner

    def keys(window=0):  # (pairs of query and key, keys that are read) of one layer
        seen = (lambda n: min(n, window)) if window else (lambda n: n)
        if decode:
            return sum(seen(n + STEPS) for n in lengths), sum(seen(n + STEPS) for n in lengths)
        return sum(seen(i + 1) for n in lengths for i in range(n)), sum(lengths)

    def attention(score_width, value_width, key_size, window=0):
        nonlocal flops, other
        pairs, read = keys(window)
        flops += 2.0 * pairs * (score_width + value_width)
        other += (read if decode else 0) * key_size * size + rows * key_size * size  # a prompt's keys are written, not read

    def experts(mlp, ff):
        nonlocal weights, flops
        n, top = mlp["router"]["experts"], mlp["router"]["top"]
        weights += n * (1.0 - (1.0 - top / n) ** rows) * 3 * ff * width + n * width
        flops += 2.0 * rows * (top * 3 * ff + n) * width

    if arch == "llama":
        h, k, d, f = config.nheads, config.kv_heads, config.head_dim, config.ffn_hidden_dim
        for _ in range(config.nlayers):
            product((h + 2 * k) * d, width)
            product(width, h * d)
            product(3 * f, width)
            attention(h * d, h * d, 2 * k * d)
    elif arch == "zodolorn":
        for layer in config.layers:
            m, mlp = layer["mixer"], layer["mlp"]
            h, d, p, v, r, q = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
            product(q + h + (0 if "kv_from" in m else r + p), width)
            product(h * (d + p), q)
            product(width, h * v)
            product(h * (d + v), r)
            attention(h * (d + p), h * v, r + p)
            if mlp["kind"] == "dense":
                product(2 * mlp["ff"], width)
            else:
                experts(mlp, mlp["expert"]["ff"])
                product(3 * mlp["shared"]["ff"], width)
    else:
        for layer in config.layers:
            m = layer["mixer"]
            if layer["type"] == "parallel":
                a, m = m["left"], m["right"]
                h, g, d, v = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
                product(h * (d + 2 * v) + g * (d + v), width)
                attention(h * d, h * v, g * (d + v), a["mask"]["size"])
            h, g, d, v = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            low = m.get("decay_rank")
            product(2 * g * d + 2 * h * v + h + (2 * low - h * v if low else h), width)
            if low:
                product(h * (d + v), low)
            product(width, h * v)
            flops += 6.0 * rows * h * d * v  # the recurrence
            other += 2 * 4.0 * len(lengths) * h * d * v
            experts(layer["mlp"], layer["mlp"]["expert"]["ff"])
    passes = STEPS if decode else 1
    return {"bytes": passes * (weights * size + other), "flops": passes * flops}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 2e-4}  # 32-bit sums of up to 11008 products
    # bfloat16 activations: `exact` is 0.007 to 0.011 away from 8 layers, 0.002 where the embedding is most of the stream,
    # and 0.02 where a token's router is near a tie and takes the other expert
    return {"rel": 0.03, "max": 0.3, "differ": 0.0}


# ---- the same in float64 -----------------------------------------------------------------------------------------
class _Weights:
    """The weights that `_model` puts in place: N(0, 0.02) from a generator seeded by (seed, name), rounded to the model's type."""

    def __init__(self, case, seed):
        self.seed, self.device = seed, torch.device("cuda")
        self.dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        self.factor = MODELS[case["model"]][3]
        self.names = _names(case)

    def raw(self, name, shape):
        digest = hashlib.sha256(f"{self.seed}:{name}".encode()).digest()
        gen = torch.Generator(device=self.device)
        gen.manual_seed(int.from_bytes(digest[:8], "little") & 0x7FFFFFFFFFFFFFFF)
        return (torch.randn(shape, generator=gen, device=self.device, dtype=torch.float32) * 0.02).to(self.dtype)

    def __call__(self, name, *shape):
        t = self.raw(name, shape)
        if name.endswith("conv.weight"):
            t.mul_(16.0)
        return t.double()

    def embedding(self, vocab, width):
        return self.raw(self.names[0], (vocab, width)).mul_(self.factor)

    def head(self, vocab, width):
        if self.names[1] is None:
            return self.embedding(vocab, width)
        return self.raw(self.names[0], (vocab, width))[_followers(vocab, self.seed).to(self.device)]


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate(x, positions, freqs):
    """x [T, heads, D]: the first 2 len(freqs) entries in adjacent pairs, by float32 angles."""
    n = 2 * len(freqs)
    angle = (positions.float()[:, None] * freqs.float()[None, :]).double()[:, None, :]
    cos, sin, u, v = torch.cos(angle), torch.sin(angle), x[..., 0:n:2], x[..., 1:n:2]
    out = x.clone()
    out[..., 0:n:2], out[..., 1:n:2] = u * cos - v * sin, v * cos + u * sin
    return out


def _frequencies(dims, base, scaling, device):
    f = float(base) ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device=device) / dims)
    if scaling:
        wave = 2.0 * math.pi / f
        s = ((scaling["original"] / wave - scaling["low"]) / (scaling["high"] - scaling["low"])).clamp(0.0, 1.0)
        f = (1.0 - s) * f / scaling["factor"] + s * f
    return f


def _attend(q, k, v, spans, scale, window=0, cap=0.0, sink=None):
    """Causal softmax attention of every span of rows on its own; q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H, V]."""
    H, G = q.shape[1], k.shape[1]
    out = torch.empty(q.shape[0], H, v.shape[2], dtype=q.dtype, device=q.device)
    for a, b in spans:
        for at in range(a, b, 512):
            to = min(at + 512, b)
            lo = max(a, at - window + 1) if window else a
            i, j = torch.arange(at, to, device=q.device)[:, None], torch.arange(lo, to, device=q.device)[None, :]
            hidden = (j > i) | (i - j >= window) if window else j > i
            for g in range(G):
                rows = slice(g * (H // G), (g + 1) * (H // G))
                s = torch.matmul(q[at:to, rows].transpose(0, 1).contiguous(), k[lo:to, g].T.contiguous()) * scale
                s = cap * torch.tanh(s / cap) if cap else s
                s = s.masked_fill_(hidden, float("-inf"))
                if sink is not None:
                    s = torch.cat([s, sink[rows, None, None].expand(-1, to - at, 1)], dim=2)
                p = torch.softmax(s, dim=2)[:, :, : to - lo].contiguous()
                out[at:to, rows] = torch.matmul(p, v[lo:to, g].contiguous()).transpose(0, 1)
    return out


def _silu(x):
    return x * torch.sigmoid(x)


def _llama(W, config, x, positions, spans):
    E, H, K, D, F = config.emb_dim, config.nheads, config.kv_heads, config.head_dim, config.ffn_hidden_dim
    freqs = 1.0 / (config.rope_theta ** (torch.arange(0, D, 2).float() / D)).to(x.device)
    for i in range(config.nlayers):
        p = f"base_model.layers.{i}."
        h = _rms(x, config.norm_eps)
        q, k, v = (h @ W(p + "attn.in_proj.qkv_fused.weight", (H + 2 * K) * D, E).T).split([H * D, K * D, K * D], dim=1)
        q, k = _rotate(q.view(-1, H, D), positions, freqs), _rotate(k.view(-1, K, D), positions, freqs)
        y = _attend(q, k, v.reshape(-1, K, D), spans, D ** -0.5)
        x = x + y.reshape(-1, H * D) @ W(p + "attn.dense.weight", E, H * D).T
        g, u = (_rms(x, config.norm_eps) @ W(p + "ff_sub_layer.wg1_fused.weight", 2 * F, E).T).chunk(2, dim=1)
        x = x + (_silu(g) * u) @ W(p + "ff_sub_layer.w2.weight", E, F).T
    return _rms(x, config.norm_eps)


def _run_experts(W, p, mlp, x, width, ids, act, scale_in=None, scale_out=None):
    E, F = mlp["router"]["experts"], mlp["expert"]["ff"]
    gate, up, down = W(p + "experts.gate", E, F, width), W(p + "experts.up", E, F, width), W(p + "experts.down", E, width, F)
    out = torch.zeros_like(x)
    for e in range(E):
        t, j = torch.where(ids == e)
        if len(t):
            z = x[t] if scale_in is None else x[t] * scale_in[t, j, None]
            y = act(z @ gate[e].T, z @ up[e].T) @ down[e].T
            out.index_add_(0, t, y if scale_out is None else y * scale_out[t, j, None])
    return out


def _zodolorn(W, config, x, positions, spans):
    eps, width = config.norm["eps"], config.width
    x = x * config.embedding["scale"]
    for i, layer in enumerate(config.layers):
        m, mlp, p = layer["mixer"], layer["mlp"], f"l{i}."
        H, D, P, V, R, Q = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
        freqs = _frequencies(m["rot"]["dims"], m["rot"]["base"], None, x.device)
        h = _rms(x, eps)
        own = "kv_from" not in m
        cq, gate, down = (h @ W(p + "mix.down.weight", Q + H + (R + P if own else 0), width).T).split([Q, H, R + P if own else 0], dim=1)
        if own:
            latent, shared = _rms(down[:, :R], eps), _rotate(down[:, None, R:], positions, freqs)
        q = (_rms(cq, eps) @ W(p + "mix.uq.weight", H * (D + P), Q).T).view(-1, H, D + P)
        q = torch.cat([q[..., :D], _rotate(q[..., D:], positions, freqs)], dim=2)
        k = (latent @ W(p + "mix.uk.weight", H * D, R).T).view(-1, H, D)
        v = (latent @ W(p + "mix.uv.weight", H * V, R).T).view(-1, H, V)
        y = _attend(q, torch.cat([k, shared.expand(-1, H, -1)], dim=2), v, spans, m["scale"], sink=torch.zeros(H, dtype=x.dtype, device=x.device))
        y = (y * torch.sigmoid(gate)[:, :, None]).reshape(-1, H * V)
        x = x + _rms(y @ W(p + "mix.o.weight", width, H * V).T, eps)
        h = _rms(x, eps)
        if mlp["kind"] == "dense":
            y = torch.nn.functional.gelu(h @ W(p + "mlp.up.weight", mlp["ff"], width).T) @ W(p + "mlp.down.weight", width, mlp["ff"]).T
        else:
            def act(g, u, limit=mlp["expert"]["limit"]):
                g = g.clamp(max=limit)
                return g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1.0)

            router = h @ W(p + "mlp.router.weight", mlp["router"]["experts"] + 1, width).T
            best, ids = torch.topk(router[:, :-1], mlp["router"]["top"], dim=1)
            y = _run_experts(W, p + "mlp.", mlp, h, width, ids, act, scale_out=torch.softmax(best, dim=1))
            S = mlp["shared"]["ff"]
            z = act(*(h @ W(p + "mlp.shared.gate_up.weight", 2 * S, width).T).chunk(2, dim=1), limit=mlp["shared"]["limit"])
            y = y + z @ W(p + "mlp.shared.down.weight", width, S).T * torch.sigmoid(router[:, -1:])
        x = x + _rms(y, eps)
    return _rms(x, eps)


def _delta(W, p, m, h, width, spans, eps):
    H, G, D, V, taps, low = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"], m.get("decay_rank") or 0
    cols = [2 * G * D + H * V, H, low or H, m.get("gate_rank") or H * V]
    qkv, beta, a, gate = (h @ W(p + "in_proj.weight", sum(cols), width).T).split(cols, dim=1)
    if low:
        a, gate = a @ W(p + "decay_up.weight", H * D, low).T, torch.sigmoid(gate @ W(p + "gate_up.weight", H * V, m["gate_rank"]).T)
        decay = torch.exp(-torch.nn.functional.softplus(a)).view(-1, H, D)
    else:
        gate, decay = _silu(gate), torch.exp(-torch.nn.functional.softplus(a))[:, :, None]
    beta, conv = torch.sigmoid(beta), W(p + "conv.weight", cols[0], taps)
    out = torch.empty(h.shape[0], H, V, dtype=h.dtype, device=h.device)
    for a, b in spans:
        x = torch.cat([torch.zeros(taps - 1, cols[0], dtype=h.dtype, device=h.device), qkv[a:b]])
        x = _silu(sum(x[j : j + b - a] * conv[:, j] for j in range(taps)))
        q, k, v = x.split([G * D, G * D, H * V], dim=1)
        q, k = (t.reshape(-1, G, D) / torch.sqrt((t.reshape(-1, G, D) ** 2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = (q * D ** -0.5).repeat_interleave(H // G, dim=1), k.repeat_interleave(H // G, dim=1)
        v, S = v.reshape(-1, H, V), torch.zeros(H, D, V, dtype=h.dtype, device=h.device)
        for t in range(b - a):  # S <- decay S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q
            S = S * decay[a + t, :, :, None]
            u = beta[a + t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1))
            S = S + k[t, :, :, None] * u[:, None, :]
            out[a + t] = (S * q[t, :, :, None]).sum(1)
    return (_rms(out, eps).reshape(-1, H * V) * gate) @ W(p + "out.weight", width, H * V).T


def _defapel(W, config, x, positions, spans):
    eps, width = config.norm["eps"], config.width
    for i, layer in enumerate(config.layers):
        m, mlp, p = layer["mixer"], layer["mlp"], f"l{i}."
        h = _rms(x, eps)
        if layer["type"] == "parallel":
            a = m["left"]
            H, G, D, V, q = a["heads"], a["kv_heads"], a["dim"], a["vdim"], p + "mix.left."
            freqs = _frequencies(a["rot"]["dims"], a["rot"]["base"], a["rot"].get("scaling"), x.device)
            cols = [H * D, G * D, G * V, H * V]
            queries, keys, values, gate = (h @ W(q + "in_proj.qkv_fused.weight", sum(cols), width).T).split(cols, dim=1)
            queries = _rotate(_rms(queries, eps).view(-1, H, D), positions, freqs)
            keys = _rotate(_rms(keys, eps).view(-1, G, D), positions, freqs)
            y = _attend(queries, keys, values.reshape(-1, G, V), spans, a["scale"], window=a["mask"]["size"], cap=a["softcap"])
            left = (y.reshape(-1, H * V) * torch.sigmoid(gate)) @ W(q + "dense.weight", width, H * V).T
            x = x + m["left_scale"] * left + m["right_scale"] * _delta(W, p + "mix.right.", m["right"], h, width, spans, eps)
        else:
            x = x + _delta(W, p + "mix.", m, h, width, spans, eps)
        h = _rms(x, eps)
        best, ids = torch.topk(torch.sigmoid(h @ W(p + "mlp.router.weight", mlp["router"]["experts"], width).T), mlp["router"]["top"], dim=1)
        x = x + _run_experts(W, p + "mlp.", mlp, h, width, ids, lambda g, u: _silu(g) * u, scale_in=best)
    return _rms(x, eps)


def exact(case, seed):
    config = _config(case)
    vocab = _vocab(config)
    W = _Weights(case, seed)
    prompts = _prompts(case, seed, vocab)
    decode = case["what"] == "decode"
    fed = 2 * STEPS if decode else 0  # tokens after the prompt: those of the prepared steps and of the pass
    before = _followers(vocab, seed)
    after = torch.empty_like(before)
    after[before] = torch.arange(vocab)
    if W.names[1] is None:
        after = torch.arange(vocab)
    rows, spans, ids = [], [], []
    for prompt in prompts:
        for _ in range(fed):  # the clear winner of every step; the logits below say whether it was
            prompt = prompt + [int(after[prompt[-1]])]
        spans.append((len(ids), len(ids) + len(prompt)))
        ids += prompt
        rows += range(len(ids) - len(prompt), len(ids)) if case["what"] == "score" else range(len(ids) - fed - 1, len(ids))
    ids = torch.tensor(ids)
    positions = torch.cat([torch.arange(b - a) for a, b in spans]).to(W.device)
    layers = {"llama": _llama, "zodolorn": _zodolorn, "defapel": _defapel}[MODELS[case["model"]][0]]
    width = config.emb_dim if hasattr(config, "emb_dim") else config.width
    x = W.embedding(vocab, width)[ids.to(W.device)].double()
    x = layers(W, config, x, positions, spans)[torch.tensor(list(rows), device=W.device)]
    logits = torch.cat([x @ part.double().T for part in W.head(vocab, width).split(16384)], dim=1)
    if case["what"] == "score":
        return {"logits": logits.view(len(prompts), -1, vocab)}
    if not decode:
        return {"logits": logits}
    logits = logits.view(len(prompts), fed + 1, vocab)
    chosen = logits.argmax(-1).cpu()
    if not torch.equal(chosen[:, :-1], torch.stack([ids[b - fed : b] for _, b in spans])):
        return None  # not the continuation that was assumed
    return {"tokens": chosen[:, fed + 1 - STEPS :].T.numpy(), "logits": logits[:, -1]}
