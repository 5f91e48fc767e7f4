"""The work a user of this engine has it do, as cases that can be timed: steps of the engine's step function on whole models.

A case names a model, a data type and one kind of work:

  decode   every one of `batch` requests on its own context brings one token and wants its logits: a step of text generation.
           The contexts are ragged (between a quarter and all of `context`) unless `even` says otherwise.
  prompt   one request's whole prompt of `tokens` tokens in one step, from an empty cache: the wait for a first token.  `want` says
           whose logits are asked for: the last token's (generation) or all (scoring a text, replaying a trace).
  mixed    a step of the continuous-batching scheduler: `batch` decoding requests, the rest of one prompt that began in an earlier
           step, and the beginning of another, `rows` rows in all.
  request  whole requests, for models with memories that cannot be rewound: `batch` prompts of `tokens` tokens in one step, then
           `steps` steps of one given token each; the logits of all of them.

The models are those of the repository's benchmark: the Llama 3.2 1B and 3B and the Llama 3.1 8B shapes of `configs/`, whole, and
the Rigalorn model of `bench.py --rigalorn --sizes 1b` (delta-rule memories, attention through latents, windowed attention).
Weights are random: matrices N(0, 0.02), norm weights 1 + 0.1 N(0, 1), and a memory's decay parameters, step sizes and taps as such
layers are initialised for training.  Token ids are uniform.
"""
import math
import random
import zlib

import torch

from geneinfer_amd.config import parse_config
from geneinfer_amd.engine import DecoderModel, Runner, StepEntry

PAGE = 16
_LLAMA3_ROPE = dict(rope_type="llama3", low_freq_factor=1.0, high_freq_factor=4.0, original_max_position_embeddings=8192)


def _llama(hidden, ff, layers, heads, dim, factor, tied):
    return dict(architectures=["LlamaForCausalLM"], hidden_size=hidden, intermediate_size=ff, num_hidden_layers=layers, num_attention_heads=heads,
                num_key_value_heads=8, head_dim=dim, vocab_size=128256, max_position_embeddings=131072, rope_theta=500000.0, rms_norm_eps=1e-5,
                tie_word_embeddings=tied, rope_scaling=dict(_LLAMA3_ROPE, factor=factor))


def _rigalorn(width, heads, groups, dim, ff, vocab, layers, max_positions=8192):
    mlp = dict(kind="dense", ff=ff)
    delta = dict(type="delta", mlp=mlp, mixer=dict(heads=heads // 4, kv_heads=heads // 8, dim=dim, vdim=2 * dim, conv=4))
    latent = dict(type="latent_attention", mlp=mlp, mixer=dict(heads=heads, dim=dim, rot_dim=dim // 2, vdim=dim, q_rank=12 * dim, kv_rank=4 * dim,
                                                               scale=(1.5 * dim) ** -0.5, rot=dict(dims=dim // 2, base=500000.0), mask=dict(size=1024)))
    blended = dict(type="attention", mlp=mlp, mixer=dict(heads=heads, kv_heads=groups, dim=dim, vdim=dim, scale=dim ** -0.5, v_mix=True,
                                                         mask=dict(size=1024), rot=dict(dims=dim // 2, base=10000.0, scaling=dict(
                                                             factor=4.0, original=4096, fast=16.0, slow=2.0))))
    return dict(architecture="Rigalorn", vocab=vocab, width=width, embedding=dict(scale=width ** 0.5), norm=dict(eps=1e-5), max_positions=max_positions,
                layers=([delta, latent, blended, delta] * layers)[:layers])


MODELS = {
    "llama-3.2-1b": _llama(2048, 8192, 16, 32, 64, 32.0, True),
    "llama-3.2-3b": _llama(3072, 8192, 28, 24, 128, 32.0, True),
    "llama-3.1-8b": _llama(4096, 14336, 32, 32, 128, 8.0, False),
    "rigalorn-1b": _rigalorn(2048, 32, 8, 64, 8192, 32000, 8),
}


# ------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # one user at a terminal: the latency of a token
        dict(name="decode_1b_b1", kind="decode", model="llama-3.2-1b", dtype="bfloat16", batch=1, context=700, even=True),
        # the benchmark's decode step
        dict(name="decode_1b_b8", kind="decode", model="llama-3.2-1b", dtype="bfloat16", batch=8, context=2048, even=True),
        # a full server: as many requests as the benchmark's largest batch, at contexts of their own
        dict(name="decode_1b_b64", kind="decode", model="llama-3.2-1b", dtype="bfloat16", batch=64, context=2048, even=False),
        # the largest model, a small batch: bound by its weights
        dict(name="decode_8b_b8", kind="decode", model="llama-3.1-8b", dtype="bfloat16", batch=8, context=1500, even=False),
        # a chat message
        dict(name="prompt_1b_131", kind="prompt", model="llama-3.2-1b", dtype="bfloat16", tokens=131, want="last"),
        # the benchmark's prompt
        dict(name="prompt_1b_2048", kind="prompt", model="llama-3.2-1b", dtype="bfloat16", tokens=2048, want="last"),
        # a long document read by the largest model
        dict(name="prompt_8b_8192", kind="prompt", model="llama-3.1-8b", dtype="bfloat16", tokens=8192, want="last"),
        # the scheduler's step under the benchmark's mixed workload (budget of 2,048 rows)
        dict(name="mixed_3b_2048", kind="mixed", model="llama-3.2-3b", dtype="bfloat16", batch=24, context=3000, rows=2048),
        # the 32-bit path: a text's logits at every position, as the replay tool dumps them
        dict(name="score_1b_f32_301", kind="prompt", model="llama-3.2-1b", dtype="float32", tokens=301, want="all"),
        # and its decode step
        dict(name="decode_1b_f32_b3", kind="decode", model="llama-3.2-1b", dtype="float32", batch=3, context=600, even=False),
        # another architecture: a long prompt, and a few requests from prompt to last token
        dict(name="prompt_rigalorn_1777", kind="request", model="rigalorn-1b", dtype="bfloat16", batch=1, tokens=1777, steps=0),
        dict(name="request_rigalorn_b5", kind="request", model="rigalorn-1b", dtype="bfloat16", batch=5, tokens=200, steps=24),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "mixed", "f32_decode", "f32_prompt", "request", "request"])
    if kind == "decode":
        model = rng.choice(["llama-3.2-1b", "llama-3.2-1b", "llama-3.2-3b", "llama-3.1-8b"])
        batch = _log_int(rng, 1, 64)
        most = {"llama-3.2-1b": 131072, "llama-3.2-3b": 32768, "llama-3.1-8b": 16384}[model] // batch
        return dict(kind="decode", model=model, dtype="bfloat16", batch=batch, context=_log_int(rng, 64, min(4000, most)), even=rng.random() < 0.3)
    if kind == "prompt":
        model = rng.choice(["llama-3.2-1b", "llama-3.2-1b", "llama-3.2-3b", "llama-3.1-8b"])
        return dict(kind="prompt", model=model, dtype="bfloat16", tokens=_log_int(rng, 16, 8000), want="last")
    if kind == "mixed":
        return dict(kind="mixed", model=rng.choice(["llama-3.2-1b", "llama-3.2-3b"]), dtype="bfloat16", batch=_log_int(rng, 1, 48),
                    context=_log_int(rng, 200, 3000), rows=_log_int(rng, 256, 2048))
    if kind == "f32_decode":
        return dict(kind="decode", model="llama-3.2-1b", dtype="float32", batch=_log_int(rng, 1, 8), context=_log_int(rng, 64, 1000), even=rng.random() < 0.3)
    if kind == "f32_prompt":
        return dict(kind="prompt", model="llama-3.2-1b", dtype="float32", tokens=_log_int(rng, 16, 600), want=rng.choice(["last", "all"]))
    if rng.random() < 0.5:
        return dict(kind="request", model="rigalorn-1b", dtype="bfloat16", batch=1, tokens=_log_int(rng, 64, 2048), steps=0)
    return dict(kind="request", model="rigalorn-1b", dtype="bfloat16", batch=_log_int(rng, 1, 8), tokens=_log_int(rng, 16, 256), steps=rng.randint(8, 32))


def _plan(case):
    """What every request of the case brings: [(positions in the cache beforehand, tokens in the step, places whose logits are wanted)].
    The ragged lengths come from the case's own numbers, not from the seed: the work of a case is the same for every input."""
    if case["kind"] == "decode":
        top, rng = case["context"], random.Random("%d %d" % (case["batch"], case["context"]))
        return [(top if case["even"] or i == 0 else rng.randint(max(1, top // 4), top), 1, (0,)) for i in range(case["batch"])]
    if case["kind"] == "prompt":
        n = case["tokens"]
        return [(0, n, (n - 1,) if case["want"] == "last" else tuple(range(n)))]
    if case["kind"] == "mixed":
        top, rng = case["context"], random.Random("%d %d %d" % (case["batch"], case["context"], case["rows"]))
        left = case["rows"] - case["batch"]
        rest = left - left // 3                                     # the end of one prompt, then the beginning of another
        return ([(rng.randint(max(1, top // 8), top), 1, (0,)) for _ in range(case["batch"])]
                + [(rng.randint(top // 4, top // 2), rest, (rest - 1,)), (0, left - rest, ())])
    n = case["tokens"]
    return [(0, n, (n - 1,)) for _ in range(case["batch"])]


# ------------------------------------------------------------------------------------------ inputs
def _shapes(cfg):
    """Name -> (shape, kind of values) of the model's tensors."""
    out = {}
    if "architectures" in cfg:
        D, F, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
        A, KV = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
        out["model.embed_tokens.weight"] = ((V, D), "matrix")
        for i in range(cfg["num_hidden_layers"]):
            p = "model.layers.%d." % i
            for name, shape in (("self_attn.q_proj", (A, D)), ("self_attn.k_proj", (KV, D)), ("self_attn.v_proj", (KV, D)), ("self_attn.o_proj", (D, A)),
                                ("mlp.gate_proj", (F, D)), ("mlp.up_proj", (F, D)), ("mlp.down_proj", (D, F))):
                out[p + name + ".weight"] = (shape, "matrix")
            out[p + "input_layernorm.weight"] = out[p + "post_attention_layernorm.weight"] = ((D,), "norm")
        out["model.norm.weight"] = ((D,), "norm")
        if not cfg["tie_word_embeddings"]:
            out["lm_head.weight"] = ((V, D), "matrix")
        return out
    D, V = cfg["width"], cfg["vocab"]
    out["embed"], out["head"], out["final.norm"] = ((V, D), "matrix"), ((V, D), "matrix"), ((D,), "norm")
    blended = 0
    for i, layer in enumerate(cfg["layers"]):
        m, x, ff = layer["mixer"], "l%d.mix." % i, layer["mlp"]["ff"]
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        out["l%d.norm1" % i] = ((D,), "norm")
        if layer["type"] == "delta":
            G = m["kv_heads"]
            for name, n in (("q", G * d), ("k", G * d), ("v", H * dv)):
                out[x + name], out[x + name + ".conv"] = ((n, D), "matrix"), ((n, m["conv"]), "taps")
            out[x + "a"], out[x + "b"], out[x + "g"], out[x + "o"] = ((H, D), "matrix"), ((H, D), "matrix"), ((H * dv, D), "matrix"), ((D, H * dv), "matrix")
            out[x + "A_log"], out[x + "dt_bias"], out[x + "norm"] = ((H,), "decay"), ((H,), "step"), ((dv,), "norm")
        elif layer["type"] == "latent_attention":
            r, rank = m["rot_dim"], m["kv_rank"]
            for name, shape in (("dq", (m["q_rank"], D)), ("uq", (H * (d + r), m["q_rank"])), ("dkv", (rank + r, D)), ("uk", (H * d, rank)), ("uv", (H * dv, rank)),
                                ("o", (D, H * dv))):
                out[x + name] = (shape, "matrix")
            out[x + "dq.norm"], out[x + "dkv.norm"] = ((m["q_rank"],), "norm"), ((rank,), "norm")
        else:
            G = m["kv_heads"]
            for name, n in (("q", H * d), ("k", G * d), ("v", G * dv)):
                out[x + name], out[x + name + ".b"] = ((n, D), "matrix"), ((n,), "matrix")
            out[x + "o"] = ((D, H * dv), "matrix")
            if blended:
                out[x + "vmix"] = ((), "blend")
            blended += 1
        out["l%d.mlp.up" % i], out["l%d.mlp.down" % i], out["l%d.mlp.act" % i] = ((ff, D), "matrix"), ((D, ff), "matrix"), ((2,), "activation")
    return out


def _tensor(name, shape, kind, seed, dtype):
    gen = torch.Generator(device="cuda").manual_seed(zlib.crc32(name.encode()) * 100003 + seed)
    if kind == "matrix" and len(shape) == 2:                        # (in pieces of rows: the widened numbers of a whole table need not lie about)
        out = torch.empty(shape, dtype=dtype, device="cuda")
        step = max(1, (1 << 28) // shape[1])
        for a in range(0, shape[0], step):
            piece = out[a:a + step]
            piece.copy_(torch.randn(piece.shape, generator=gen, device="cuda") * 0.02)
        return out
    if kind == "activation":                                        # slopes of 0.8 on both sides
        return torch.tensor([math.log(math.expm1(0.8)), math.log(math.expm1(0.3))], device="cuda").to(dtype)
    if kind == "blend":
        return torch.tensor(0.5, device="cuda").to(dtype)
    if kind in ("matrix", "norm"):
        z = torch.randn(shape, generator=gen, device="cuda")
        return (0.02 * z if kind == "matrix" else 1.0 + 0.1 * z).to(dtype)
    u = torch.rand(shape, generator=gen, device="cuda")
    if kind == "taps":
        return (u - 0.5).to(dtype)
    if kind == "decay":                                             # decay rates between 1 and 16 a unit of step size
        return torch.log(1.0 + 15.0 * u).to(dtype)
    step = torch.exp(math.log(1e-3) + u * math.log(100.0))          # step sizes between 0.001 and 0.1
    return torch.log(torch.expm1(step)).to(dtype)


def _weights(case, seed):
    dtype = getattr(torch, case["dtype"])
    return {name: _tensor(name, shape, kind, seed, dtype) for name, (shape, kind) in _shapes(MODELS[case["model"]]).items()}


def _vocab(cfg):
    return cfg.get("vocab_size") or cfg["vocab"]


def _tokens(case, seed):
    """Per request: the tokens its cache holds beforehand, and those it brings (a `request` case: the prompt's and the steps')."""
    rng, vocab, steps = random.Random("tokens %d" % seed), _vocab(MODELS[case["model"]]), case.get("steps", 0)
    return [([rng.randrange(vocab) for _ in range(past)], [rng.randrange(vocab) for _ in range(n + steps)]) for past, n, _ in _plan(case)]


def prepare(case, seed):
    cfg, plan, tokens, steps = MODELS[case["model"]], _plan(case), _tokens(case, seed), case.get("steps", 0)
    config = parse_config(cfg)
    model = DecoderModel(config.model_spec(), _weights(case, seed), getattr(torch, case["dtype"]), "cuda:0")
    model.config = config
    lengths = [past + n + steps for past, n, _ in plan]
    rows = max(2048, sum(n for _, n, _ in plan))
    runner = Runner(model, page_size=PAGE, max_tokens=sum(-(-(n + 1) // PAGE) * PAGE for n in lengths), max_requests=len(plan), max_rows=rows,
                    max_positions=max(lengths) + 1)
    keeps = case["kind"] in ("decode", "mixed")                     # (their requests live on from pass to pass)
    if keeps:
        for i, (past, _) in enumerate(tokens):
            runner.open(i)
            for a in range(0, len(past), 2048):
                runner.step([StepEntry(i, past[a:a + 2048])])
    entries = [StepEntry(i, t[:n], want) for i, ((_, n, want), (_, t)) in enumerate(zip(plan, tokens))]
    later = [[StepEntry(i, [t[n + s]], (0,)) for i, ((_, n, _), (_, t)) in enumerate(zip(plan, tokens))] for s in range(steps)]
    return dict(runner=runner, entries=entries, later=later, lengths=[past for past, _, _ in plan], keeps=keeps)


def run(state):
    runner, entries = state["runner"], state["entries"]
    if state["keeps"]:
        for e, length in zip(entries, state["lengths"]):            # back to where the step begins
            runner.truncate(e.request, length)
        return runner.step(entries)
    for e in entries:
        runner.open(e.request)
    logits = runner.step(entries)
    if state["later"]:
        logits = [logits.clone()] + [runner.step(step).clone() for step in state["later"]]
    for e in entries:
        runner.close(e.request)
    return logits


# -------------------------------------------------------------------------------------------- work
def work(case):
    cfg, plan, steps = MODELS[case["model"]], _plan(case), case.get("steps", 0)
    elem = 2 if case["dtype"] == "bfloat16" else 4
    shapes = _shapes(cfg)
    table = {"model.embed_tokens.weight", "embed"}
    head = "model.embed_tokens.weight" if cfg.get("tie_word_embeddings") else ("lm_head.weight" if "architectures" in cfg else "head")
    layer_weights = sum(math.prod(s) for name, (s, _) in shapes.items() if name not in table and name != head)
    head_weights = math.prod(shapes[head][0])
    D, V = shapes[head][0][1], shapes[head][0][0]
    bytes_, flops = 0.0, 0.0
    # (positions before, rows, wanted) of every step of the pass
    passes = [plan] + [[(past + n + s, 1, (0,)) for past, n, _ in plan] for s in range(steps)]
    for entries in passes:
        rows, wanted = sum(n for _, n, _ in entries), sum(len(w) for _, _, w in entries)
        bytes_ += elem * (layer_weights + (head_weights if wanted else 0) + rows * D) + 4.0 * wanted * V
        flops += 2.0 * rows * layer_weights + 2.0 * wanted * head_weights
        for past, n, _ in entries:
            for mixer in _mixers(cfg):
                if mixer["kind"] == "memory":
                    bytes_ += 2 * 4.0 * mixer["state"]                                             # the memory, read and written, 32-bit
                    flops += 8.0 * n * mixer["state"]                                              # decayed, read twice, written
                    continue
                w = mixer["window"] or 1 << 60
                seen = sum(min(past + i + 1, w) for i in range(n)) if n <= 64 or w < past + n else n * past + n * (n + 1) / 2
                bytes_ += elem * mixer["per_position"] * (min(past + n, w + n - 1) + n)            # read once, the new ones written
                flops += 2.0 * mixer["per_pair"] * seen
    return dict(bytes=bytes_, flops=flops)


def _mixers(cfg):
    if "architectures" in cfg:
        H, G, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        return [dict(kind="attention", per_position=2 * G * d, per_pair=2 * H * d, window=None)] * cfg["num_hidden_layers"]
    out = []
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "delta":
            out.append(dict(kind="memory", state=m["heads"] * m["dim"] * m["vdim"]))
        elif layer["type"] == "latent_attention":
            out.append(dict(kind="attention", per_position=m["kv_rank"] + m["rot_dim"], per_pair=m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), window=m["mask"]["size"]))
        else:
            out.append(dict(kind="attention", per_position=m["kv_heads"] * (m["dim"] + m["vdim"]), per_pair=m["heads"] * (m["dim"] + m["vdim"]), window=m["mask"]["size"]))
    return out


def tolerance(case):
    """From the distance to `exact`.  bfloat16: 0.016 to 0.019 at the 1B shape, 0.03 at 3B, 0.04 at 8B (twice the layers), 0.005 for Rigalorn;
    two implementations that round at the same places are far nearer to each other than to it.  32-bit: 9e-6."""
    if case["dtype"] == "float32":
        return {"rel": 3e-5}
    return {"rel": 0.02} if case["model"].startswith("rigalorn") else {"rel": 0.03}


# ------------------------------------------------------------------------------------------- exact
def exact(case, seed):
    """The logits in 64 bits, from the same weights and tokens: whole sequences, no cache, ordinary torch."""
    rows = sum(past + n + case.get("steps", 0) for past, n, _ in _plan(case))
    cfg, tokens, steps = MODELS[case["model"]], _tokens(case, seed), case.get("steps", 0)
    if rows * sum(math.prod(s) for s, _ in _shapes(cfg).values()) > 1.6e14:           # (some 20 seconds in 64 bits)
        return None
    w = _weights(case, seed)
    sequences = [past + brought for past, brought in tokens]
    wanted = [[past + place for place in want] + [past + n + s for s in range(steps)] for past, n, want in _plan(case)]
    picked = (_exact_llama if "architectures" in cfg else _exact_rigalorn)(cfg, w, sequences, wanted)
    if case["kind"] != "request":
        return torch.cat(picked)
    steps_first = [torch.stack([p[s] for p in picked]) for s in range(steps + 1)]
    return steps_first if steps else steps_first[0]


def _times(x, weight):
    """x @ weight^T in 64 bits, some rows at a time."""
    weight, out = weight.double(), torch.empty((x.shape[0], weight.shape[0]), dtype=torch.float64, device=x.device)
    for a in range(0, x.shape[0], 16384):
        torch.mm(x[a:a + 16384], weight.t(), out=out[a:a + 16384])
    return out


def _rms_norm(x, weight, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight.double()


def _softmax_attention(q, k, v, scale, window=None):
    """q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H * dv], causal; a head and some rows at a time."""
    T, H, _ = q.shape
    G, out = k.shape[1], torch.empty((T, H, v.shape[2]), dtype=torch.float64, device=q.device)
    for h in range(H):
        kh, vh = k[:, h * G // H].contiguous(), v[:, h * G // H].contiguous()
        for a in range(0, T, 2048):
            b = min(T, a + 2048)
            first = max(0, a - window + 1) if window else 0
            s = torch.mm(q[a:b, h], kh[first:b].t()) * scale
            i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(first, b, device=q.device)[None, :]
            hidden = j > i if window is None else (j > i) | (i - j >= window)
            out[a:b, h] = torch.mm(torch.softmax(s.masked_fill_(hidden, float("-inf")), -1), vh[first:b])
    return out.reshape(T, -1)


def _turn(u, v, frequencies, magnitude=1.0):
    """The pairs (u, v) [T, heads, pairs] turned by position times frequency."""
    angle = torch.arange(u.shape[0], dtype=torch.float64, device=u.device)[:, None] * torch.tensor(frequencies, dtype=torch.float64, device=u.device)[None]
    cos, sin = (torch.cos(angle) * magnitude)[:, None], (torch.sin(angle) * magnitude)[:, None]
    return u * cos - v * sin, v * cos + u * sin


def _turn_halves(x, frequencies, magnitude=1.0):
    n = len(frequencies)
    return torch.cat([*_turn(x[..., :n], x[..., n:2 * n], frequencies, magnitude), x[..., 2 * n:]], -1)


def _turn_neighbours(x, frequencies):
    u, v = _turn(x[..., 0::2], x[..., 1::2], frequencies)
    return torch.stack([u, v], -1).flatten(-2)


def _spans(sequences):
    at, out = 0, []
    for s in sequences:
        out.append((at, at + len(s)))
        at += len(s)
    return out


def _pick(x, spans, wanted, norm, eps, head):
    places = [a + p for (a, _), ps in zip(spans, wanted) for p in ps]
    logits = _times(_rms_norm(x[torch.tensor(places, device=x.device)], norm, eps), head)
    return list(torch.split(logits, [len(ps) for ps in wanted]))


def _exact_llama(cfg, w, sequences, wanted):
    D, H, G, d, eps = cfg["hidden_size"], cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    rope, frequencies = cfg["rope_scaling"], []
    for i in range(d // 2):
        f = cfg["rope_theta"] ** (-2.0 * i / d)
        length, original = 2.0 * math.pi / f, rope["original_max_position_embeddings"]
        if length > original / rope["low_freq_factor"]:
            f /= rope["factor"]
        elif length >= original / rope["high_freq_factor"]:
            share = (original / length - rope["low_freq_factor"]) / (rope["high_freq_factor"] - rope["low_freq_factor"])
            f = (1.0 - share) * f / rope["factor"] + share * f
        frequencies.append(f)
    spans = _spans(sequences)
    x = w["model.embed_tokens.weight"][torch.tensor([t for s in sequences for t in s], device="cuda")].double()
    for i in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % i
        h = _rms_norm(x, w[p + "input_layernorm.weight"], eps)
        q, k, v = (_times(h, w[p + "self_attn.%s_proj.weight" % n]).view(len(h), -1, d) for n in "qkv")
        mixed = [_softmax_attention(_turn_halves(q[a:b], frequencies), _turn_halves(k[a:b], frequencies), v[a:b], d ** -0.5) for a, b in spans]
        x += _times(torch.cat(mixed), w[p + "self_attn.o_proj.weight"])
        h = _rms_norm(x, w[p + "post_attention_layernorm.weight"], eps)
        for a in range(0, len(x), 32768):
            gate, up = (_times(h[a:a + 32768], w[p + "mlp.%s_proj.weight" % n]) for n in ("gate", "up"))
            x[a:a + 32768] += _times(torch.nn.functional.silu(gate).mul_(up), w[p + "mlp.down_proj.weight"])
    head = w["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"]
    return _pick(x, spans, wanted, w["model.norm.weight"], eps, head)


def _exact_rigalorn(cfg, w, sequences, wanted):
    eps, softplus = cfg["norm"]["eps"], lambda z: torch.logaddexp(z, torch.zeros_like(z))
    spans = _spans(sequences)
    x = w["embed"][torch.tensor([t for s in sequences for t in s], device="cuda")].double() * cfg["embedding"]["scale"]
    first_values = None
    for i, layer in enumerate(cfg["layers"]):
        m = layer["mixer"]
        p = {name[len("l%d." % i):]: t.double() for name, t in w.items() if name.startswith("l%d." % i)}
        h, H, d, dv = _rms_norm(x, p["norm1"], eps), m["heads"], m["dim"], m["vdim"]
        if layer["type"] == "delta":
            mixed = torch.cat([_exact_delta(h[a:b], p, m, eps, softplus) for a, b in spans])
        elif layer["type"] == "latent_attention":
            r, rank, T = m["rot_dim"], m["kv_rank"], len(h)
            frequencies = [m["rot"]["base"] ** (-2.0 * j / r) for j in range(r // 2)]
            q = _times(_rms_norm(_times(h, p["mix.dq"]), p["mix.dq.norm"], eps), p["mix.uq"]).view(T, H, d + r)
            down = _times(h, p["mix.dkv"])
            c = _rms_norm(down[:, :rank], p["mix.dkv.norm"], eps)
            k, v, mixed = _times(c, p["mix.uk"]).view(T, H, d), _times(c, p["mix.uv"]).view(T, H, dv), []
            for a, b in spans:
                turned = _turn_neighbours(down[a:b, None, rank:], frequencies)
                mixed.append(_softmax_attention(torch.cat([q[a:b, :, :d], _turn_neighbours(q[a:b, :, d:], frequencies)], -1),
                                                torch.cat([k[a:b], turned.expand(b - a, H, r)], -1), v[a:b], m["scale"], m["mask"]["size"]))
            mixed = torch.cat(mixed)
        else:
            q, k, v = ((_times(h, p["mix." + n]) + p["mix." + n + ".b"]).view(len(h), -1, size) for n, size in (("q", d), ("k", d), ("v", dv)))
            rot, n = m["rot"], m["rot"]["dims"]
            s = rot["scaling"]
            index = lambda turns: n * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
            low, high = max(math.floor(index(s["fast"])), 0), min(math.ceil(index(s["slow"])), n - 1)
            ramp = [min(max((j - low) / max(high - low, 0.001), 0.0), 1.0) for j in range(n // 2)]
            frequencies = [rot["base"] ** (-2.0 * j / n) * (1.0 - g + g / s["factor"]) for j, g in enumerate(ramp)]
            magnitude = 0.1 * math.log(s["factor"]) + 1.0
            if first_values is None:
                first_values = v
            else:
                v = (1.0 - p["mix.vmix"]) * v + p["mix.vmix"] * first_values
            mixed = torch.cat([_softmax_attention(_turn_halves(q[a:b], frequencies, magnitude), _turn_halves(k[a:b], frequencies, magnitude), v[a:b],
                                                  m["scale"], m["mask"]["size"]) for a, b in spans])
        z, act = _times(h, p["mlp.up"]), p["mlp.act"]
        z = 0.5 * z + torch.where(z > 0, softplus(act[0]) * z * z, (0.5 + softplus(act[1])) * (torch.expm1(z.clamp(max=0.0)) - z))
        x = x + _times(mixed, p["mix.o"]) + _times(z, p["mlp.down"])
    return _pick(x, spans, wanted, w["final.norm"], eps, w["head"])


def _exact_delta(h, p, m, eps, softplus):
    T, H, G, dk, dv = len(h), m["heads"], m["kv_heads"], m["dim"], m["vdim"]

    def conv(name):
        z, taps = _times(h, p["mix." + name]), p["mix." + name + ".conv"]
        n = taps.shape[1]
        z = torch.cat([z.new_zeros(n - 1, z.shape[1]), z])
        return torch.nn.functional.silu(sum(z[j:j + T] * taps[:, j] for j in range(n)))

    unit = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
    q = (unit(conv("q").view(T, G, dk)) * dk ** -0.5).repeat_interleave(H // G, 1)
    k = unit(conv("k").view(T, G, dk)).repeat_interleave(H // G, 1)
    v = conv("v").view(T, H, dv)
    beta = torch.sigmoid(_times(h, p["mix.b"]))[:, :, None]
    decay = torch.exp(-torch.exp(p["mix.A_log"]) * softplus(_times(h, p["mix.a"]) + p["mix.dt_bias"]))[:, :, None, None]
    S, out = h.new_zeros(H, dk, dv), torch.empty((T, H, dv), dtype=torch.float64, device=h.device)
    for t in range(T):
        S = S * decay[t]
        S = S + k[t][:, :, None] * (beta[t] * (v[t] - (S * k[t][:, :, None]).sum(1)))[:, None]
        out[t] = (S * q[t][:, :, None]).sum(1)
    out = _rms_norm(out, p["mix.norm"], eps)
    return out.reshape(T, -1) * torch.nn.functional.silu(_times(h, p["mix.g"]))
