"""What this engine's speed is measured on: the steps that a serving or scoring program asks of
it, through ``ModelRunner.step``, the one forward path under the engine, the command line, the
replay program and the perplexity tool.

Three things are done here, as ``do`` names them:

* ``decode``: requests whose contexts lie in the cache go on for a few steps of one given token
  each (replaying a transcript, scoring continuations).  Every pass forks the cached requests,
  decodes on the children and frees them, so that a pass can be repeated.
* ``step``: one step that brings portions of prompts (whole prompts, or new tokens on cached
  ones), beside decoding requests or alone; logits for the last token of every request, or for
  the second half of every portion, as perplexity windows ask for them.
* ``generate``: prompts to greedy tokens, the sampled tokens fed back.

Models have the shapes of the package's presets with random weights, prompts are uniform random
token ids, as in ``bench.py``.  The 8B shape runs with a quarter of its layers: every layer does
the same work."""
import math

import torch

from rust_llm_inference_server_amd.config import preset_dict
from rust_llm_inference_server_amd.engine import ModelRunner, StepEntry
from rust_llm_inference_server_amd.models import Model
from rust_llm_inference_server_amd.registry import architecture_of
from rust_llm_inference_server_amd.sampling import SamplingParams
from rust_llm_inference_server_amd.sampling.sampler import Sampler, sample_on_device

PAGE = 16
FILL_TOKENS = 8192              # tokens per step while the cached contexts are made
CHILD = 1_000_000               # ids of forked requests
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
LAYERS = {"llama-3.1-8b": 8}


def listed():
    def decode(name, model, requests, context, steps, spread=0.0, dtype="bfloat16"):
        return {"name": name, "do": "decode", "model": model, "dtype": dtype,
                "requests": requests, "context": context, "spread": spread, "steps": steps}

    def step(name, model, portions, new, cached=0, spread=0.0, singles=0, context=0,
             want="last", dtype="bfloat16"):
        return {"name": name, "do": "step", "model": model, "dtype": dtype,
                "portions": portions, "new": new, "cached": cached, "spread": spread,
                "requests": singles, "context": context, "want": want}

    return [
        # A chat with one user: each token waits for one step.
        decode("1b-decode-1", "llama-3.2-1b", 1, 640, 8),
        # The headline: eight requests near the benchmark's context of 4,096.
        decode("1b-decode-8", "llama-3.2-1b", 8, 4096, 8),
        # A busy server: as many requests as it admits, contexts of all ages.
        decode("1b-decode-64", "llama-3.2-1b", 64, 640, 4, spread=1.0),
        # The same at the wider shape, a batch that fills no power of two.
        decode("3b-decode-27", "llama-3.2-3b", 27, 1200, 4, spread=1.0),
        # Few requests with long documents in the cache.
        decode("8b-decode-4-long", "llama-3.1-8b", 4, 14000, 6, spread=0.5),
        # The prompt that the headline's prefill figure is quoted on.
        step("1b-prefill-2048", "llama-3.2-1b", 1, 2048),
        # Short chat prompts of odd lengths that arrive together.
        step("1b-prefill-short", "llama-3.2-1b", 3, 127, spread=1.0),
        # A long document in one step.
        step("8b-prefill-8192", "llama-3.1-8b", 1, 8192),
        # Continuous batching under a token budget of 512: a portion of a long prompt beside
        # decoding requests.
        step("3b-mixed-512", "llama-3.2-3b", 1, 464, cached=2000, singles=48, context=1000,
             spread=1.0),
        # A window of a perplexity run: logits for half of it.
        step("1b-score-512", "llama-3.2-1b", 1, 512, want="half"),
        # The 32-bit path, as parity runs against other implementations use it: a few prompts and
        # the greedy tokens behind them.
        {"name": "1b-generate-f32", "do": "generate", "model": "llama-3.2-1b",
         "dtype": "float32", "requests": 4, "prompt": 96, "spread": 1.0, "steps": 6},
        # The smallest model that ships, in 32 bits: every kernel is a few microseconds.
        {"name": "tiny-generate-f32", "do": "generate", "model": "tiny-b", "dtype": "float32",
         "requests": 3, "prompt": 24, "spread": 1.0, "steps": 8},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(["llama-3.2-1b"] * 3 + ["llama-3.2-3b", "llama-3.1-8b"])
    spread = round(rng.uniform(0.0, 1.0), 2)
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "mixed", "score", "f32",
                       "f32", "tiny"])
    if kind == "tiny":
        return {"do": "generate", "model": rng.choice(["tiny-a", "tiny-b"]), "dtype": "float32",
                "requests": rng.randint(1, 5), "prompt": rng.randint(3, 40), "spread": spread,
                "steps": rng.randint(4, 12)}
    if kind == "decode":
        requests = log(1, 64)
        return {"do": "decode", "model": model, "dtype": "bfloat16", "requests": requests,
                "context": log(32, min(14000, 49152 // requests)), "spread": spread,
                "steps": rng.randint(3, 6)}
    if kind == "f32" and rng.random() < 0.7:
        if rng.random() < 0.5:
            return {"do": "generate", "model": "llama-3.2-1b", "dtype": "float32",
                    "requests": rng.randint(1, 6), "prompt": log(4, 120), "spread": spread,
                    "steps": rng.randint(2, 6)}
        return {"do": "decode", "model": "llama-3.2-1b", "dtype": "float32",
                "requests": log(1, 16), "context": log(32, 600), "spread": spread, "steps": 2}
    case = {"do": "step", "model": model, "dtype": "bfloat16", "portions": 1, "new": 0,
            "cached": 0, "spread": spread, "requests": 0, "context": 0, "want": "last"}
    if kind == "prefill":
        case["portions"] = rng.randint(1, 4)
        case["new"] = log(16, 4096 // case["portions"])
        if rng.random() < 0.4:
            case["cached"] = log(64, 8000)
    elif kind == "mixed":
        case.update(requests=rng.randint(1, 63), context=log(64, 1500), new=log(24, 480),
                    cached=log(32, 4000))
    elif kind == "score":
        case.update(new=log(64, 1024), want="half", portions=rng.randint(1, 2))
    else:
        case.update(model="llama-3.2-1b", dtype="float32", new=log(8, 400),
                    want=rng.choice(["last", "half"]))
    return case


# ------------------------------------------------------------------------------- sizes
def _spread(n, mean, spread, unit=1):
    """``n`` lengths around ``mean``, evenly from ``(1 - spread / 2) mean`` to ``(1 + spread / 2)
    mean``, the longest first, in multiples of ``unit``."""
    out = [mean * (1.0 + spread * ((i + 0.5) / n - 0.5)) for i in range(n)]
    return sorted((max(1, int(round(v / unit))) * unit for v in out), reverse=True)


def _config(case):
    cfg = preset_dict(case["model"])
    cfg["num_hidden_layers"] = LAYERS.get(case["model"], cfg["num_hidden_layers"])
    return cfg


def _lengths(case):
    """Per request (cached positions, new tokens, wanted indices of the new tokens): requests
    that bring one token at a time first."""
    if case["do"] == "generate":
        return [(0, n, [n - 1]) for n in _spread(case["requests"], case["prompt"], case["spread"])]
    # whole pages, so that what a child writes never falls on a page that it shares
    singles = _spread(case["requests"], case["context"], case["spread"], PAGE) \
        if case["requests"] else []
    if case["do"] == "decode":
        return [(n, case["steps"], list(range(case["steps"]))) for n in singles]
    out = [(n, 1, [0]) for n in singles]
    new = _spread(case["portions"], case["new"], case["spread"])
    cached = _spread(case["portions"], case["cached"], case["spread"], PAGE) \
        if case["cached"] else [0] * case["portions"]
    for c, n in zip(cached, new):
        out.append((c, n, list(range(n // 2, n)) if case["want"] == "half" else [n - 1]))
    return out


# ------------------------------------------------------------------------------ inputs
def _weights(cfg, dtype, seed):
    arch = architecture_of(cfg)
    spec = arch.build_spec(arch.parse_config(cfg))
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)
    weights = {}
    for t in spec.tensor_specs():
        mean = 1.0 if t.init == "ones_normal" else 0.0
        w = torch.empty(tuple(t.shape), dtype=dtype, device="cuda")
        weights[t.name] = w.normal_(mean, t.std, generator=gen)
    return spec, weights


def _tokens(case, vocab, seed):
    """Per request its cached and its new token ids."""
    gen = torch.Generator().manual_seed(int(seed) * 2)
    return [(torch.randint(0, vocab, (c,), generator=gen).tolist(),
             torch.randint(0, vocab, (n,), generator=gen).tolist()) for c, n, _ in _lengths(case)]


class _State:
    pass


def prepare(case, seed):
    """A loaded model, its runner and cache, and requests whose contexts have been computed."""
    cfg = _config(case)
    dtype = DTYPES[case["dtype"]]
    lengths = _lengths(case)
    steps = case["steps"] if case["do"] == "generate" else 0
    longest = max(c + n for c, n, _ in lengths) + steps
    spec, weights = _weights(cfg, dtype, seed)
    model = Model(spec, weights, dtype, torch.device("cuda", torch.cuda.current_device()), longest)
    s = _State()
    s.case, s.lengths = case, lengths
    s.ids = _tokens(case, cfg["vocab_size"], seed)
    pages = sum(-(-c // PAGE) + -(-(c + n + steps) // PAGE) + 1 for c, n, _ in lengths) + 8
    s.runner = ModelRunner(model, num_pages=pages, page_size=PAGE, max_num_seqs=len(lengths),
                           max_batched_tokens=max(FILL_TOKENS, sum(n for _, n, _ in lengths)))
    if case["do"] != "step":
        s.runner.capture_decode_steps(longest, sampled=False)    # as a server does at its start
    # the cached contexts, several requests to a step
    entries, room = [], FILL_TOKENS
    for i, (old, _) in enumerate(s.ids):
        if old:
            s.runner.reserve(i, len(old))
        at = 0
        while at < len(old):
            part = old[at:at + room]
            entries.append(StepEntry(i, part, []))
            at, room = at + len(part), room - len(part)
            if room == 0:
                s.runner.step(entries)
                entries, room = [], FILL_TOKENS
    if entries:
        s.runner.step(entries)
    return s


# -------------------------------------------------------------------------------- pass
def run(s):
    r = s.runner
    steps = s.case["steps"] if s.case["do"] == "generate" else 0
    live = []
    for i, (c, n, _) in enumerate(s.lengths):
        seq = CHILD + i
        if c:
            r.fork(i, seq)
        r.reserve(seq, c + n + steps)
        live.append(seq)
    if s.case["do"] == "decode":
        out = [r.step([StepEntry(seq, [new[t]], [0]) for seq, (_, new) in zip(live, s.ids)])
               for t in range(s.case["steps"])]
    elif s.case["do"] == "step":
        out = [r.step([StepEntry(seq, new, want)
                       for seq, (_, new), (_, _, want) in zip(live, s.ids, s.lengths)])]
    else:
        sampler = Sampler(SamplingParams.greedy(steps))
        out, picked = [], []
        entries = [StepEntry(seq, new, want)
                   for seq, (_, new), (_, _, want) in zip(live, s.ids, s.lengths)]
        for t in range(steps):
            out.append(r.step(entries))
            picked.append(sample_on_device(out[-1], [sampler.device_mode(n + t)
                                                     for _, n, _ in s.lengths]))
            entries = [StepEntry(seq, [tok], [0]) for seq, tok in zip(live, picked[-1])]
        out.append(torch.tensor(picked))
    for seq in live:
        r.free(seq)
    return out


# ------------------------------------------------------------------------- work, limits
def work(case):
    cfg = _config(case)
    elem = DTYPES[case["dtype"]].itemsize
    L, H, I, V, d = (cfg["num_hidden_layers"], cfg["hidden_size"], cfg["intermediate_size"],
                     cfg["vocab_size"], cfg["head_dim"])
    nh, nkv = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    params = L * ((nh + 2 * nkv) * d * H + H * nh * d + 3 * H * I + 2 * H)
    head = V * H + H
    kv = 2 * L * nkv * d * elem                                # bytes of one cached position
    nbytes = flops = 0.0

    def one(parts):
        """A step of (cached, new, wanted rows) per request."""
        nonlocal nbytes, flops
        T, rows = sum(n for _, n, _ in parts), sum(w for _, _, w in parts)
        nbytes += (params + head) * elem + T * H * elem + rows * V * 4
        nbytes += kv * sum(c + n for c, n, _ in parts)
        flops += 2.0 * params * T + 2.0 * V * H * rows
        flops += 4.0 * L * nh * d * sum(n * c + n * (n + 1) / 2 for c, n, _ in parts)

    lengths = _lengths(case)
    if case["do"] == "decode":
        for t in range(case["steps"]):
            one([(c + t, 1, 1) for c, _, _ in lengths])
    elif case["do"] == "step":
        one([(c, n, len(w)) for c, n, w in lengths])
    else:
        one([(0, n, 1) for _, n, _ in lengths])
        for t in range(1, case["steps"]):
            one([(n + t - 1, 1, 1) for _, n, _ in lengths])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # About four times the error against ``exact``: in bfloat16 0.016 to 0.026 at the 1B shape and
    # at eight layers of the 8B shape, 0.035 to 0.037 at the 28 layers of the 3B shape; in 32 bits
    # 8e-6 to 9e-6 at the 1B shape, 2e-7 to 5e-7 at the tiny ones.
    if case["dtype"] == "bfloat16":
        return {"rel": 0.1, "max": 0.6}
    return {"rel": 4e-5, "max": 4e-4, "differ": 0.02}


# ------------------------------------------------------------------------------- 64 bits
def _frequencies(cfg):
    d, scaling = cfg["head_dim"], cfg.get("rope_scaling")
    out = []
    for j in range(d // 2):
        f = cfg["rope_theta"] ** (-2.0 * j / d)
        if scaling:
            old, lo, hi = (scaling["original_max_position_embeddings"],
                           scaling["low_freq_factor"], scaling["high_freq_factor"])
            turns = old * f / (2.0 * math.pi)
            share = min(1.0, max(0.0, (turns - lo) / (hi - lo)))
            f = share * f + (1.0 - share) * f / scaling["factor"]
        out.append(f)
    return torch.tensor(out, dtype=torch.float64, device="cuda")


def _norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _by_rows(f, x, rows=8192):
    return torch.cat([f(x[i:i + rows]) for i in range(0, x.shape[0], rows)])


def _attend(q, k, v, scale, rows=512):
    """Causal attention of one sequence; q (T, heads, d), k and v (T, kv heads, d)."""
    T, nh, d = q.shape
    group = nh // k.shape[1]
    out = torch.empty_like(q)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    for i in range(0, T, rows):
        e = min(T, i + rows)
        qi = q[i:e].reshape(e - i, -1, group, d).permute(1, 2, 0, 3).reshape(-1, group * (e - i), d)
        s = torch.bmm(qi, kt[:, :, :e].contiguous()) * scale
        mask = torch.arange(e, device="cuda")[None, :] > torch.arange(i, e, device="cuda")[:, None]
        s = s.view(-1, group, e - i, e).masked_fill_(mask, -math.inf)
        p = torch.softmax(s, -1).view(-1, group * (e - i), e)
        o = torch.bmm(p, vt[:, :e].contiguous()).view(-1, group, e - i, d)
        out[i:e] = o.permute(2, 0, 1, 3).reshape(e - i, nh, d)
    return out


def _logits64(cfg, w, seqs, wanted):
    """Float64 logits of whole token sequences at their wanted positions, one tensor each."""
    H, d, eps = cfg["hidden_size"], cfg["head_dim"], cfg["rms_norm_eps"]
    nh, nkv = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    lens = [len(t) for t in seqs]
    pos = torch.cat([torch.arange(n, dtype=torch.float64) for n in lens]).cuda()
    angle = pos[:, None, None] * _frequencies(cfg)[None, None, :]
    cos, sin = angle.cos(), angle.sin()

    def turn(x):
        a, b = x[..., : d // 2], x[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    ids = torch.cat([torch.tensor(t) for t in seqs]).cuda()
    x = w["model.embed_tokens.weight"][ids].double()
    T = x.shape[0]
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."

        def mat(name):
            return w[p + name + ".weight"].double().t()

        h = _norm(x, w[p + "input_layernorm.weight"], eps)
        q = turn((h @ mat("self_attn.q_proj")).view(T, nh, d))
        k = turn((h @ mat("self_attn.k_proj")).view(T, nkv, d))
        v = (h @ mat("self_attn.v_proj")).view(T, nkv, d)
        del h
        a = torch.cat([_attend(*t, d ** -0.5) for t in zip(q.split(lens), k.split(lens),
                                                           v.split(lens))])
        x = x + a.reshape(T, nh * d) @ mat("self_attn.o_proj")
        del q, k, v, a
        gate, up, down = (mat("mlp." + n) for n in ("gate_proj", "up_proj", "down_proj"))

        def unit(rows):
            g = _norm(rows, w[p + "post_attention_layernorm.weight"], eps)
            return rows + (torch.nn.functional.silu(g @ gate) * (g @ up)) @ down

        x = _by_rows(unit, x)
    head = w["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"]
    head = head.double().t()
    return [_norm(xs[rows], w["model.norm.weight"], eps) @ head
            for xs, rows in zip(x.split(lens), wanted)]


def exact(case, seed):
    cfg = _config(case)
    lengths = _lengths(case)
    total = sum(c + n for c, n, _ in lengths)
    if total * cfg["num_hidden_layers"] * cfg["hidden_size"] ** 2 > 4e13:
        return None                                          # some 15 seconds in 64 bits
    _, w = _weights(cfg, DTYPES[case["dtype"]], seed)
    ids = _tokens(case, cfg["vocab_size"], seed)
    if case["do"] == "generate":
        seqs, out, picked = [list(new) for _, new in ids], [], []
        for _ in range(case["steps"]):
            rows = _logits64(cfg, w, seqs, [[len(t) - 1] for t in seqs])
            out.append(torch.cat(rows))
            picked.append(out[-1].argmax(-1).tolist())
            for t, tok in zip(seqs, picked[-1]):
                t.append(tok)
        return out + [torch.tensor(picked)]
    rows = _logits64(cfg, w, [old + new for old, new in ids],
                     [[c + i for i in want] for c, _, want in lengths])
    if case["do"] == "decode":
        return [torch.stack([r[t] for r in rows]) for t in range(case["steps"])]
    return [torch.cat(rows)]
