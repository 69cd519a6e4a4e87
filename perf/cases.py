"""What a program that serves with this engine has it do, as measurable cases.

A case of kind "steps" is the life of one batch of requests on the step function: the prompts go in (in steps of at
most ``BUDGET`` tokens, as the scheduler would deal them out), every request is decoded greedily ``new`` tokens further
(several steps to a graph launch in bfloat16, step by step in float32), and the requests end.  It returns the logits
behind the prompts, the chosen tokens and the logits of the last step, which depend on every key and value stored on the
way.  ``new`` 0 is a prompt alone (the time to a first token).  A case of kind "generate" is a queue of requests through
``LLM.generate``: scheduler, mixed steps of prompt portions beside decoding, sampler.

Weights are random, drawn on the GPU from the seed, with the spread of a usual initialisation (0.02 at a width of 896,
less in wider models, the products that end a sublayer divided by sqrt(2 layers)), embedding rows that stay visible in
the residual stream behind all layers, and a head that holds the embedding's rows moved by a fixed number of tokens (a
tied head holds them as they are).  So the largest logit of a row stands as far above the others as a trained model's
does, and a greedy or drawn continuation does not hang on rounding.
"""
from __future__ import annotations

import math
import random

import torch

import llm_infrence_engine_amd as eng
from llm_infrence_engine_amd.config import config_from_dict, preset
from llm_infrence_engine_amd.engine import ModelRunner, StepEntry
from llm_infrence_engine_amd.parts.base import Runtime
from llm_infrence_engine_amd.parts.model import Model

PAGE = 16               # tokens per cache page
BUDGET = 4096           # most tokens of one step
PER_LAUNCH = 8          # most decode steps of one graph launch
SHIFT = 7919            # an untied head answers token t with token t + SHIFT
DEVICE = "cuda:0"
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


# --------------------------------------------------------------------------------------------------------- the cases
def _case(name, model, batch, prompt, spread, new, dtype="bfloat16", layers=0, kind="steps"):
    """``prompt``: tokens of the longest prompt; the others are up to ``spread`` shorter, drawn from the seed's own
    generator.  ``layers`` 0: all of the configuration's."""
    c = {"kind": kind, "model": model, "dtype": dtype, "layers": layers, "batch": batch, "prompt": prompt,
         "spread": spread, "new": new}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user, a short question and a short answer: nothing but latency, one row in every product
        _case("reply_0.5b", "0.5b", 1, 33, 0, 33),
        # the batch that the headline is quoted on: 8 requests behind 512-token prompts
        _case("batch8_0.5b", "0.5b", 8, 512, 0, 65),
        # a full batch with prompts of ragged lengths
        _case("batch64_0.5b", "0.5b", 64, 131, 64, 33),
        # two long documents read in portions, and answers behind them: attention over thousands of keys
        _case("documents_0.5b", "0.5b", 2, 7600, 333, 33),
        # the time to a first token: a short ragged batch of prompts, and the 2,048-token prompt at both widths
        _case("first_token_0.5b", "0.5b", 3, 171, 80, 0),
        _case("prompt_0.5b", "0.5b", 1, 2048, 0, 0),
        _case("prompt_7b", "7b", 1, 2048, 0, 0),
        # the 7B sizes serving a full batch; decoding is bound by reading the weights, the prompts by products
        _case("batch64_7b", "7b", 64, 130, 64, 33),
        # the largest configuration, one user: every step reads 64 GB of weights
        _case("reply_32b", "32b", 1, 200, 0, 17),
        # the true 32-bit path, which results are checked with
        _case("check_float32", "0.5b", 3, 130, 41, 9, dtype="float32"),
        # the second architecture (delta rule, attention through a latent) at the size its benchmark has
        _case("gemadra_0.5b", "gemadra-0.5b", 4, 512, 64, 33, layers=4),
        # a queue through the whole engine: ragged prompts, half of the requests draw their tokens
        _case("serve_0.5b", "0.5b", 24, 900, 880, 40, kind="generate"),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    """One more case of the same ranges: kinds, models, batch sizes, prompt lengths and continuations as above."""
    kind = rng.choices(["decode", "prompt", "documents", "7b", "32b", "float32", "gemadra", "generate"],
                       [5, 4, 1, 3, 1, 1, 2, 2])[0]
    new = rng.randint(9, 70)
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        prompt = _log_int(rng, 16, min(2048, 16384 // batch))
        return _case("", "0.5b", batch, prompt, rng.randint(0, prompt // 2), new)
    if kind == "prompt":
        model = rng.choice(["0.5b", "0.5b", "7b"])
        batch = _log_int(rng, 1, 8)
        prompt = _log_int(rng, 17, 4096 // batch)
        return _case("", model, batch, prompt, rng.randint(0, prompt // 2), 0)
    if kind == "documents":
        prompt = _log_int(rng, 2500, 7600)
        return _case("", "0.5b", rng.randint(1, 2), prompt, rng.randint(0, 500), rng.randint(9, 40))
    if kind == "7b":
        batch = _log_int(rng, 1, 64)
        prompt = _log_int(rng, 16, min(1024, 8192 // batch))
        return _case("", "7b", batch, prompt, rng.randint(0, prompt // 2), rng.randint(9, 33))
    if kind == "32b":
        return _case("", "32b", 1, _log_int(rng, 16, 300), 0, rng.randint(5, 16))
    if kind == "float32":
        return _case("", "0.5b", rng.randint(1, 4), _log_int(rng, 17, 130), rng.randint(0, 16), rng.randint(3, 9), dtype="float32")
    if kind == "gemadra":
        batch = _log_int(rng, 1, 8)
        prompt = _log_int(rng, 20, 2048 // batch)
        return _case("", "gemadra-0.5b", batch, prompt, rng.randint(0, prompt // 2), rng.choice([0, new]), layers=4)
    prompt = _log_int(rng, 60, 900)
    return _case("", "0.5b", rng.randint(3, 24), prompt, prompt - 20, rng.randint(9, 40), kind="generate")


# ------------------------------------------------------------------------------------------------------------ weights
def _config(case) -> dict:
    d = preset(case["model"])
    if case["layers"]:
        if "layers" in d:
            d["layers"] = d["layers"][:case["layers"]]
        else:
            d["num_hidden_layers"] = case["layers"]
    return d


def _tensors(d: dict) -> list:
    """(name, shape, what it is) of every tensor of a configuration, in a fixed order."""
    out = []
    if "layers" in d:
        W = d["width"]
        out.append(("embed", (d["vocab"], W), "embedding"))
        for i, e in enumerate(d["layers"]):
            m, p = e["mixer"], f"l{i}."
            out += [(p + "norm1", (W,), "norm0"), (p + "canon1", (W, d["canon"]["taps"]), "taps")]
            H, D, E = m["heads"], m["dim"], m["vdim"]
            if e["type"] == "channel_delta":
                G, t = m["kv_heads"], m["conv"]
                for n, c in (("q", G * D), ("k", G * D), ("v", H * E)):
                    out += [(p + "mix." + n, (c, W), "matrix"), (p + f"mix.{n}.conv", (c, t), "taps")]
                out += [(p + "mix.a1", (m["decay_rank"], W), "matrix"), (p + "mix.a2", (H * D, m["decay_rank"]), "matrix"),
                        (p + "mix.dt_bias", (H * D,), "dt"), (p + "mix.A_log", (H,), "bias"), (p + "mix.b", (H, W), "matrix"),
                        (p + "mix.g1", (m["gate_rank"], W), "matrix"), (p + "mix.g2", (H * E, m["gate_rank"]), "matrix"),
                        (p + "mix.norm", (E,), "norm")]
            else:
                R, C, Q = m["rot_dim"], m["kv_rank"], m["q_rank"]
                out += [(p + "mix.dq", (Q, W), "matrix"), (p + "mix.dq.norm", (Q,), "norm"),
                        (p + "mix.uq", (H * (D + R), Q), "matrix"), (p + "mix.dkv", (C + R, W), "matrix"),
                        (p + "mix.dkv.norm", (C,), "norm"), (p + "mix.uk", (H * D, C), "matrix"),
                        (p + "mix.uv", (H * E, C), "matrix"), (p + "mix.sink", (H,), "bias"), (p + "mix.g", (H * E, W), "matrix")]
            ff = e["mlp"]["ff"]
            out += [(p + "mix.o", (W, H * E), "end"), (p + "norm2", (W,), "norm0"), (p + "mlp.up", (ff, W), "matrix"),
                    (p + "mlp.act", (2,), "bias"), (p + "mlp.down", (W, ff), "end")]
        return out + [("final.norm", (W,), "final0"), ("head", (d["vocab"], W), "head")]
    H, I, V, nkv = d["hidden_size"], d["intermediate_size"], d["vocab_size"], d["num_key_value_heads"]
    hd = H // d["num_attention_heads"]
    out.append(("model.embed_tokens.weight", (V, H), "embedding"))
    for i in range(d["num_hidden_layers"]):
        p = f"model.layers.{i}."
        out.append((p + "input_layernorm.weight", (H,), "norm"))
        for n, r in (("q", H), ("k", nkv * hd), ("v", nkv * hd)):
            out += [(p + f"self_attn.{n}_proj.weight", (r, H), "matrix"), (p + f"self_attn.{n}_proj.bias", (r,), "bias")]
        out += [(p + "self_attn.o_proj.weight", (H, H), "end"), (p + "post_attention_layernorm.weight", (H,), "norm"),
                (p + "mlp.gate_proj.weight", (I, H), "matrix"), (p + "mlp.up_proj.weight", (I, H), "matrix"),
                (p + "mlp.down_proj.weight", (H, I), "end")]
    out.append(("model.norm.weight", (H,), "final"))
    return out if d["tie_word_embeddings"] else out + [("lm_head.weight", (V, H), "head")]


class _Weights:
    """Stands where a checkpoint reader stands: every tensor is drawn on the GPU when it is asked for."""

    def __init__(self, d: dict, seed: int, dtype: torch.dtype):
        tensors = _tensors(d)
        self.layers = len(d["layers"]) if "layers" in d else d["num_hidden_layers"]
        self.shapes = {n: (i, s, w) for i, (n, s, w) in enumerate(tensors)}
        self.seed, self.dtype, self.embedding = seed, dtype, tensors[0][0]
        self.std = 0.02 * math.sqrt(896 / tensors[0][1][1])

    def check(self, wanted, ignorable=()):
        names = {s.name: tuple(s.shape) for s in wanted}
        if names != {n: tuple(s) for n, (_, s, _) in self.shapes.items()}:
            raise ValueError("the model wants other tensors than were drawn")

    def close(self):
        pass

    def get(self, name):
        i, shape, what = self.shapes[name]
        if what == "head":
            return torch.roll(self.get(self.embedding), SHIFT, 0)
        g = torch.Generator(device=DEVICE).manual_seed(self.seed * 1000003 + i)
        std, mean = {"matrix": (self.std, 0.0), "end": (self.std / math.sqrt(2 * self.layers), 0.0), "embedding": (0.2, 0.0),
                     "bias": (0.1, 0.0), "dt": (0.5, -3.0), "taps": (0.3, 0.0), "norm": (0.1, 1.0), "norm0": (0.1, 0.0),
                     "final": (0.015, 0.15), "final0": (0.015, -0.85)}[what]
        keep = self.dtype if what in ("matrix", "end", "embedding") else torch.float32
        out = torch.empty(shape, dtype=keep, device=DEVICE)
        flat = out.view(-1)
        for a in range(0, flat.numel(), 1 << 26):
            b = min(flat.numel(), a + (1 << 26))
            flat[a:b].copy_(torch.randn(b - a, generator=g, device=DEVICE).mul_(std).add_(mean))
        return out


def _prompts(case, seed):
    rng = random.Random(seed)
    d = _config(case)
    vocab = d["vocab"] if "layers" in d else d["vocab_size"]
    lens = [case["prompt"] - (rng.randint(0, case["spread"]) if i else 0) for i in range(case["batch"])]
    return [[rng.randrange(vocab) for _ in range(n)] for n in lens]


# ------------------------------------------------------------------------------------------------------ prepare, run
def prepare(case, seed):
    d = _config(case)
    cfg = config_from_dict(d)
    dtype = DTYPES[case["dtype"]]
    model = Model(cfg.to_spec())
    model.config = cfg
    model.load(_Weights(d, seed, dtype), Runtime(torch.device(DEVICE), dtype))
    prompts = _prompts(case, seed)
    state = {"case": case, "prompts": prompts, "model": model}
    longest = case["prompt"] + case["new"]
    if case["kind"] == "generate":
        state["llm"] = eng.LLM(model, max_seqs=16, max_len=1024, max_num_batched_tokens=BUDGET,
                               decode_steps_per_launch=PER_LAUNCH)
        state["params"] = [eng.SamplingParams(max_new_tokens=case["new"] - i % 9,
                                              **({"temperature": 0.8, "top_k": 50, "top_p": 0.9, "seed": i} if i % 2 else {}))
                           for i in range(len(prompts))]
        return state
    graphs = dtype == torch.bfloat16
    max_len = -(-longest // PAGE) * PAGE
    runner = ModelRunner(model, PAGE, len(prompts) * (max_len // PAGE), len(prompts), max_len, hip_graphs=graphs)
    state["steps"] = _portions([len(p) for p in prompts])
    if graphs:     # what these requests will need, as an engine captures it before it serves
        runner.graphs.warm_up(_launches(case["new"]) or [1], batch_sizes=[len(prompts)] if case["new"] else [],
                              portion_tokens=[sum(b - a for _, a, b in step) for step in state["steps"]])
    state["runner"] = runner
    return state


def _portions(lens):
    """The prompts dealt out over steps of at most ``BUDGET`` tokens: [(request, from, to)] per step."""
    steps, room = [[]], BUDGET
    for r, n in enumerate(lens):
        at = 0
        while at < n:
            if room == 0:
                steps.append([])
                room = BUDGET
            take = min(room, n - at)
            steps[-1].append((r, at, at + take))
            at, room = at + take, room - take
    return steps


def _launches(new):
    """Decode steps of each graph launch: as many as allowed, powers of two, the last step by itself."""
    out, left, k = [], new - 1, PER_LAUNCH
    while left > 0:
        while k > left:
            k //= 2
        out.append(k)
        left -= k
    return out + [1] if new else []


def run(state):
    case, prompts = state["case"], state["prompts"]
    if case["kind"] == "generate":
        return [torch.tensor(o.token_ids) for o in state["llm"].generate(prompts, state["params"])]
    runner = state["runner"]
    R = range(len(prompts))
    rows = []
    for step in state["steps"]:
        rows.append(runner.step([StepEntry(r, prompts[r][a:b], [b - a - 1] if b == len(prompts[r]) else [])
                                 for r, a, b in step]))
    first = torch.cat(rows)
    out = {"first": first}
    if case["new"]:
        last = first.argmax(-1).tolist()
        chosen = [last]
        if runner.graphs is not None:
            for k in _launches(case["new"])[:-1]:
                chosen += runner.decode_steps([StepEntry(r, [last[r]]) for r in R], k)
                last = chosen[-1]
        else:
            for _ in range(case["new"] - 1):
                last = runner.step([StepEntry(r, [last[r]], [0]) for r in R]).argmax(-1).tolist()
                chosen.append(last)
        logits = runner.step([StepEntry(r, [last[r]], [0]) for r in R]).clone()
        out.update(tokens=torch.tensor(chosen), last=logits)
    for r in R:
        runner.free_request(r)
    return out


# -------------------------------------------------------------------------------------------------- what it must cost
def _sizes(case):
    """(values of the matrices every token passes, of the head, vocabulary, cache values a token keeps, multiply-adds per
    visible key, per token beside the matrices, window) of a case's model."""
    d = _config(case)
    t = _tensors(d)
    body = sum(s[0] * s[1] for _, s, w in t if len(s) == 2 and w in ("matrix", "end"))
    vocab, width = t[0][1]
    if "layers" in d:
        kv = key = rec = 0
        for e in d["layers"]:
            m = e["mixer"]
            if e["type"] == "channel_delta":
                rec += 3 * m["heads"] * m["dim"] * m["vdim"]
            else:
                kv += m["kv_rank"] + m["rot_dim"]
                key += m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        return body, vocab * width, vocab, kv, key, rec, 1024
    hd = width // d["num_attention_heads"]
    L = d["num_hidden_layers"]
    return body, vocab * width, vocab, 2 * L * d["num_key_value_heads"] * hd, 2 * L * width, 0, 1 << 30


def work(case):
    """Every weight once for the prompts and once for every decode step (a step needs the token before it), every live
    key and value once a step, logits where they are wanted; two operations a multiply-add."""
    body, head, vocab, kv, key, rec, window = _sizes(case)
    size = 4 if case["dtype"] == "float32" else 2
    mean = case["prompt"] - case["spread"] / 2
    B, T = case["batch"], case["new"]
    steps = T if case["kind"] == "steps" else T * -(-B // 16)
    seen = sum(min(mean + t, window) for t in range(1, T + 1))             # keys a request's decoded tokens see
    past = min(mean, window)
    in_prompt = past * (past + 1) / 2 + (mean - past) * window
    nbytes = (1 + steps) * (body + head) * size + B * (seen + mean + T) * kv * size + B * vocab * 4 * (1 + bool(T))
    macs = B * ((mean + T) * (body + rec) + (1 + T) * head + (in_prompt + seen) * key)
    return {"bytes": nbytes, "flops": 2 * macs}


def tolerance(case):
    """Logits: four times what this engine was seen to lie away from 64 bits (activations rounded to bfloat16 between all
    products: 0.0037 of the norm, Gemadra 0.006; in 32 bits 1.5e-6).  Tokens are whole numbers; a draw can fall on a
    boundary."""
    if case["kind"] == "generate":
        return {"rel": 0.0, "differ": 0.005}
    if case["dtype"] == "float32":
        return {"rel": 6e-6, "max": 6e-5, "differ": 0.0}
    rel = 0.024 if case["model"].startswith("gemadra") else 0.015
    return {"rel": rel, "max": 6 * rel, "differ": 0.005}


# ------------------------------------------------------------------------------------------------------ in 64 bits
def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, scale, window=None, sink=None):
    """q [H, T, D], k [G, T, D], v [G, T, E] of one sequence from its start -> [T, H * E]."""
    H, T, _ = q.shape
    per = H // k.shape[0]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    pos = torch.arange(T, device=q.device)
    for a in range(0, T, 1024):
        b = min(T, a + 1024)
        lo = 0 if window is None else max(0, a - window + 1)
        hidden = pos[None, lo:b] > pos[a:b, None]
        if window is not None:
            hidden |= pos[None, lo:b] <= pos[a:b, None] - window
        for h in range(H):
            s = (q[h, a:b] @ k[h // per, lo:b].t() * scale).masked_fill_(hidden, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(b - a, 1)], 1)
            p = s.softmax(-1)
            out[a:b, h] = p[:, :b - lo] @ v[h // per, lo:b]
    return out.reshape(T, -1)


def _conv(x, w):
    """Causal, per channel: w's last column meets the current token."""
    taps = w.shape[1]
    wide = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return sum(wide[j:j + x.shape[0]] * w[:, j] for j in range(taps))


def _turn(x, first, second, base, dims, pos):
    """x [T, H, D]: entries ``first`` turn with ``second`` by pos * base^(-2i/dims)."""
    f = base ** (-2.0 * torch.arange(dims // 2, dtype=x.dtype, device=x.device) / dims)
    a = (pos[:, None] * f)[:, None]
    out = x.clone()
    u, w = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * a.cos() - w * a.sin(), w * a.cos() + u * a.sin()
    return out


def _qwen2_layer(d, w, p, xs):
    nh, nkv, eps = d["num_attention_heads"], d["num_key_value_heads"], d["rms_norm_eps"]
    hd = d["hidden_size"] // nh
    wq, wk, wv = (w(p + f"self_attn.{n}_proj.weight") for n in "qkv")
    bq, bk, bv = (w(p + f"self_attn.{n}_proj.bias") for n in "qkv")
    g1, g2, wo = w(p + "input_layernorm.weight"), w(p + "post_attention_layernorm.weight"), w(p + "self_attn.o_proj.weight")
    wg, wu, wd = (w(p + f"mlp.{n}_proj.weight") for n in ("gate", "up", "down"))
    for x in xs:
        T = x.shape[0]
        pos = torch.arange(T, dtype=x.dtype, device=x.device)
        h = _rms(x, g1, eps)
        q, k, v = ((h @ m.t() + b).reshape(T, -1, hd) for m, b in ((wq, bq), (wk, bk), (wv, bv)))
        lo, hi = slice(0, hd // 2), slice(hd // 2, hd)
        q, k = (_turn(t, lo, hi, d["rope_theta"], hd, pos) for t in (q, k))
        x += _attend(*(t.transpose(0, 1).contiguous() for t in (q, k, v)), hd ** -0.5) @ wo.t()
        h = _rms(x, g2, eps)
        x += (torch.nn.functional.silu(h @ wg.t()) * (h @ wu.t())) @ wd.t()


def _gemadra_layer(d, w, p, xs, e):
    F = torch.nn.functional
    m, eps = e["mixer"], d["norm"]["eps"]
    H, D, E = m["heads"], m["dim"], m["vdim"]
    t = {n[len(p):]: w(n) for n in (n for n, _, _ in _tensors(d)) if n.startswith(p)}
    for x in xs:
        T = x.shape[0]
        n = _rms(x, 1 + t["norm1"], eps)
        h = n + _conv(n, t["canon1"])
        if e["type"] == "channel_delta":
            G = m["kv_heads"]
            q, k, v = (F.silu(_conv(h @ t["mix." + c].t(), t[f"mix.{c}.conv"])) for c in "qkv")
            q, k, v = q.reshape(T, G, D), k.reshape(T, G, D), v.reshape(T, H, E)
            q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
            k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            q, k = (c.repeat_interleave(H // G, 1) for c in (q, k))
            beta = torch.sigmoid(h @ t["mix.b"].t())
            a = (h @ t["mix.a1"].t()) @ t["mix.a2"].t() + t["mix.dt_bias"]
            g = torch.exp(-torch.exp(t["mix.A_log"])[:, None] * F.softplus(a.reshape(T, H, D)))
            S, o = x.new_zeros(H, D, E), x.new_empty(T, H, E)
            for i in range(T):
                S = g[i, :, :, None] * S
                u = beta[i, :, None] * (v[i] - (S * k[i, :, :, None]).sum(1))
                S = S + k[i, :, :, None] * u[:, None]
                o[i] = (S * q[i, :, :, None]).sum(1)
            gate = torch.sigmoid((h @ t["mix.g1"].t()) @ t["mix.g2"].t()).reshape(T, H, E)
            y = (_rms(o, t["mix.norm"], eps) * gate).reshape(T, -1)
        else:
            C, R, rot = m["kv_rank"], m["rot_dim"], m["rot"]
            pos = torch.arange(T, dtype=x.dtype, device=x.device)
            even, odd = slice(0, rot["dims"], 2), slice(1, rot["dims"], 2)
            q = (_rms(h @ t["mix.dq"].t(), t["mix.dq.norm"], eps) @ t["mix.uq"].t()).reshape(T, H, D + R)
            q = torch.cat([q[..., :D], _turn(q[..., D:], even, odd, rot["base"], rot["dims"], pos)], -1)
            kv = h @ t["mix.dkv"].t()
            c = _rms(kv[:, :C], t["mix.dkv.norm"], eps)
            kr = _turn(kv[:, None, C:], even, odd, rot["base"], rot["dims"], pos).expand(T, H, R)
            k = torch.cat([(c @ t["mix.uk"].t()).reshape(T, H, D), kr], -1)
            v = (c @ t["mix.uv"].t()).reshape(T, H, E)
            o = _attend(*(z.transpose(0, 1).contiguous() for z in (q, k, v)), m["scale"], m["mask"]["size"], t["mix.sink"])
            y = o * torch.sigmoid(h @ t["mix.g"].t())
        u = _rms(x, 1 + t["norm2"], eps) @ t["mlp.up"].t()
        up, un = F.softplus(t["mlp.act"][0]), 0.5 + F.softplus(t["mlp.act"][1])
        u = torch.where(u > 0, up * u * u, un * (torch.expm1(u.clamp(max=0.0)) - u)) + 0.5 * u
        x += y @ t["mix.o"].t() + u @ t["mlp.down"].t()


@torch.no_grad()
def exact(case, seed):
    """The logits of ``run`` in 64 bits.  The continuation is the one the head was made for, and is checked to be it."""
    if case["kind"] == "generate":
        return None
    d = _config(case)
    source = _Weights(d, seed, DTYPES[case["dtype"]])
    w = lambda name: source.get(name).double()      # noqa: E731
    vocab = source.shapes[source.embedding][1][0]
    step = 0 if d.get("tie_word_embeddings") else SHIFT
    prompts, T = _prompts(case, seed), case["new"]
    seqs = [p + [(p[-1] + step * (i + 1)) % vocab for i in range(T)] for p in prompts]
    table = source.get(source.embedding)
    xs = [table[torch.tensor(s, device=DEVICE)].double() for s in seqs]
    for i in range(source.layers):
        if "layers" in d:
            _gemadra_layer(d, w, f"l{i}.", xs, d["layers"][i])
        else:
            _qwen2_layer(d, w, f"model.layers.{i}.", xs)
    eps, norm = (d["norm"]["eps"], 1 + w("final.norm")) if "layers" in d else (d["rms_norm_eps"], w("model.norm.weight"))
    head = torch.roll(table, step, 0).double()
    logits = [_rms(x[len(p) - 1:], norm, eps) @ head.t() for x, p in zip(xs, prompts)]
    for s, p, rows in zip(seqs, prompts, logits):
        if rows[:T].argmax(-1).tolist() != s[len(p):]:
            raise ValueError("the continuation is not the one that the head was made for")
    out = {"first": torch.stack([r[0] for r in logits])}
    if T:
        out.update(tokens=None, last=torch.stack([r[-1] for r in logits]))
    return out
