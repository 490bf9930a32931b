"""What this library is timed on: the work that its users have it do, through Engine.step and generate.

Five kinds of pass:
  decode    one step of sequences that already hold a context (a token each, from the cache); every pass goes on by
            one token, as generation does, so the context grows a little while a case is timed
  prompt    requests of whole prompts: started, stepped, given back
  trace     requests from prompt to end with given tokens (what bin/trace_run replays): the prompts, then steps of one
            token each, the logits of every step
  score     the probability of every token of a text (perplexity)
  generate  generate() with greedy sampling, the tokens and the logits they were drawn from

In bfloat16 the tokens are given, not drawn: two logits may lie closer together than its rounding, and which of them
is drawn would decide everything behind it.  For the same reason the designs whose layers choose experts are not here
in bfloat16.  Sampling runs in the generate cases, in float32.

The model shapes are bench.py's (the Mistral-7B and Llama-3.2-3B shapes, four layers of the Rekirax design at width
4,096) and a small one of the tests.  Weights are drawn from the seed: matrices uniform in +-1/sqrt(inputs) and stored
in the compute dtype, embeddings normal, norm weights about one.  `layers` keeps the first layers of a shape where all
of them would make the preparation slow; the step's other kernels and each layer's stay what they are."""
import hashlib
import math

import torch

from yalm_amd import Engine, Model, Sampler, config_from_dict, generate

DEVICE = "cuda:0"

MISTRAL_7B = {
    "architectures": ["MistralForCausalLM"], "hidden_size": 4096, "intermediate_size": 14336,
    "num_hidden_layers": 32, "num_attention_heads": 32, "num_key_value_heads": 8, "head_dim": 128,
    "vocab_size": 32000, "max_position_embeddings": 32768, "rope_theta": 1000000.0, "rms_norm_eps": 1e-5,
    "hidden_act": "silu", "tie_word_embeddings": False,
}
LLAMA_3B = {
    "architectures": ["LlamaForCausalLM"], "hidden_size": 3072, "intermediate_size": 8192,
    "num_hidden_layers": 28, "num_attention_heads": 24, "num_key_value_heads": 8, "head_dim": 128,
    "vocab_size": 128256, "max_position_embeddings": 131072, "rope_theta": 500000.0, "rms_norm_eps": 1e-5,
    "rope_scaling": {"rope_type": "llama3", "factor": 32.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                     "original_max_position_embeddings": 8192},
    "hidden_act": "silu", "tie_word_embeddings": True,
}
SMALL = {
    "architectures": ["LlamaForCausalLM"], "hidden_size": 256, "intermediate_size": 640,
    "num_hidden_layers": 2, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 128,
    "vocab_size": 512, "max_position_embeddings": 512, "rope_theta": 10000.0, "rms_norm_eps": 1e-5,
    "hidden_act": "silu", "tie_word_embeddings": False,
}


def _rekirax():
    width, heads = 4096, 32
    left = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1536},
            "rot": {"dims": 64, "base": 500000.0}}
    side = {"type": "parallel", "mixer": {"left": left, "right": {"heads": heads, "dim": 128, "vdim": 128}},
            "mlp": {"kind": "dense", "ff": width * 7 // 2}}
    window = {"type": "attention", "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128,
                                             "scale": 128 ** -0.5, "softcap": 30.0, "mask": {"size": 1024}},
              "mlp": {"kind": "dense", "ff": width * 7 // 2}}
    return {"architecture": "Rekirax", "vocab": 32000, "width": width, "norm": {"eps": 1e-5}, "canon": {"taps": 4},
            "loop": {"start": 1, "stop": 3, "times": 1}, "layers": [side, window, side, side]}


SHAPES = {"mistral-7b-v0.2": MISTRAL_7B, "mistral-7b-v0.1": dict(MISTRAL_7B, rope_theta=10000.0, sliding_window=4096),
          "llama-3.2-3b": LLAMA_3B, "small": SMALL, "rekirax": _rekirax()}
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
SPARE = 4096             # positions that a decode case has left to go on into


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    """batch, context (tokens held before the step) or tokens (of a prompt); spread: a sequence has down to (1 - spread)
    of that many; new: steps of one token behind the prompt."""
    return [
        # the smallest calls: a few requests on a small model, where launches and the host's work are all there is
        dict(name="generate_small", kind="generate", shape="small", layers=2, dtype="fp32", batch=3, tokens=20, spread=0.9, new=16),
        # one chat user in the middle of a long answer: every weight is read for a single token
        dict(name="decode_b1", kind="decode", shape="mistral-7b-v0.2", layers=32, dtype="bf16", batch=1, context=3056, spread=0.0),
        # the benchmark's headline: eight users in step
        dict(name="decode_b8", kind="decode", shape="mistral-7b-v0.2", layers=32, dtype="bf16", batch=8, context=3056, spread=0.0),
        # a full server whose requests differ in length: keys and values outweigh the weights
        dict(name="decode_b64_ragged", kind="decode", shape="mistral-7b-v0.2", layers=8, dtype="bf16", batch=64, context=3041, spread=0.65),
        # an odd number of users of the smaller shape: narrower layers, a head four times as wide, tied
        dict(name="decode_b13_3b", kind="decode", shape="llama-3.2-3b", layers=28, dtype="bf16", batch=13, context=4347, spread=0.1),
        # one reader of a long document: a single sequence's keys are the larger part of the work
        dict(name="decode_b1_long", kind="decode", shape="mistral-7b-v0.2", layers=8, dtype="bf16", batch=1, context=28000, spread=0.0),
        # the benchmark's prompt
        dict(name="prompt_2048", kind="prompt", shape="mistral-7b-v0.2", layers=32, dtype="bf16", batch=1, tokens=2048, spread=0.0),
        # a short question: the time to the first token of a chat turn
        dict(name="prompt_33", kind="prompt", shape="mistral-7b-v0.2", layers=32, dtype="bf16", batch=1, tokens=33, spread=0.0),
        # requests of unequal lengths that arrive together
        dict(name="prompts_ragged_3b", kind="prompt", shape="llama-3.2-3b", layers=28, dtype="bf16", batch=7, tokens=991, spread=0.95),
        # a document beyond the window of a model that keeps one
        dict(name="prompt_6000_window", kind="prompt", shape="mistral-7b-v0.1", layers=8, dtype="bf16", batch=1, tokens=6000, spread=0.0),
        # a text's perplexity in the true float32 path
        dict(name="score_fp32", kind="score", shape="llama-3.2-3b", layers=4, dtype="fp32", batch=1, tokens=701, spread=0.0),
        # requests from prompt to end on layers with a recurrence, chunked and windowed attention
        dict(name="trace_rekirax", kind="trace", shape="rekirax", layers=4, dtype="bf16", batch=5, tokens=509, spread=0.5, new=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same kinds over their ranges."""
    kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "prompt", "score", "trace", "generate"])
    spread = rng.choice([0.0, round(rng.uniform(0.05, 0.95), 2)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "bf16", "fp32"])
    shape = rng.choice(["mistral-7b-v0.2", "mistral-7b-v0.2", "mistral-7b-v0.1", "llama-3.2-3b"])
    layers = rng.randint(2, 8)
    if kind == "decode":
        batch = _log(rng, 1, 96)
        context = _log(rng, 16, min(24000, 120000 // batch))
        if dtype == "fp32":              # the float32 path serves few sequences
            batch, context, layers = min(batch, 16), min(context, 4000), min(layers, 4)
        return dict(kind=kind, shape=shape, layers=layers, dtype=dtype, batch=batch, context=context, spread=spread)
    if kind == "prompt":
        total = _log(rng, 1, 9000)
        batch = min(total, rng.choice([1, 1, 1, rng.randint(2, 16)]))
        if dtype == "fp32":
            total, layers = min(total, 1000), min(layers, 4)
            batch = min(batch, total)
        return dict(kind=kind, shape=shape, layers=layers, dtype=dtype, batch=batch, tokens=max(1, total // batch), spread=spread)
    if kind == "score":
        tokens = _log(rng, 16, 700 if dtype == "fp32" else 3000)
        return dict(kind=kind, shape=shape, layers=min(layers, 4), dtype=dtype, batch=1, tokens=tokens, spread=0.0)
    if kind == "trace":
        batch = rng.randint(1, 9)
        return dict(kind=kind, shape=rng.choice([shape, "rekirax", "rekirax"]), layers=4, dtype="bf16", batch=batch,
                    tokens=_log(rng, 4, 2400 // batch), spread=spread, new=rng.randint(2, 16))
    return dict(kind=kind, shape="small", layers=2, dtype="fp32", batch=rng.randint(1, 12), tokens=_log(rng, 2, 300),
                spread=spread, new=rng.randint(4, 32))


# ------------------------------------------------------------------------------------------------ inputs from the seed
def _number(seed, name):
    return int.from_bytes(hashlib.blake2b(("%d/%s" % (seed, name)).encode(), digest_size=7).digest(), "little")


def _tensors(case):
    """{name of a model folder: (shape, how its values are drawn)} of the case's model."""
    cfg, out = SHAPES[case["shape"]], {}

    def matrix(name, rows, cols):
        out[name] = ((rows, cols), "matrix")

    def vector(name, n, how):
        out[name] = ((n,), how)
    if case["shape"] == "rekirax":
        D, V = cfg["width"], cfg["vocab"]
        out["embed"] = ((V, D), "embedding")
        vector("embed.norm", D, "offset")
        vector("final.norm", D, "offset")
        matrix("loop.in", D, 2 * D)
        out["loop.step"] = ((1, D), "bias")
        for i, layer in enumerate(cfg["layers"]):
            p, m = "l%d." % i, layer["mixer"]
            vector(p + "norm1", D, "offset")
            vector(p + "norm2", D, "offset")
            out[p + "canon1"] = ((D, cfg["canon"]["taps"]), "taps")
            a, q = (m["left"], p + "mix.left.") if layer["type"] == "parallel" else (m, p + "mix.")
            H, G, d = a["heads"], a["kv_heads"], a["dim"]
            matrix(q + "q", H * d, D)
            matrix(q + "k", G * d, D)
            matrix(q + "o", D, H * d)
            if layer["type"] == "parallel":
                matrix(q + "v", G * d, D)
                matrix(q + "g", H * d, D)
                vector(q + "q.norm", H * d, "norm")
                vector(q + "k.norm", G * d, "norm")
                r, R = p + "mix.right.", m["right"]["heads"] * m["right"]["dim"]
                for n in ("q", "f", "v"):
                    matrix(r + n, R, D)
                matrix(r + "o", D, R)
                vector(r + "f.b", R, "bias")
                vector(r + "lower", R, "fraction")
                vector(r + "norm", m["right"]["vdim"], "norm")
                vector(p + "mix.left.out", D, "norm")
                vector(p + "mix.right.out", D, "norm")
            else:
                vector(q + "q.norm", d, "norm")
                vector(q + "k.norm", d, "norm")
                vector(q + "r1", H, "fraction")
                vector(q + "r2", H, "fraction")
            F = layer["mlp"]["ff"]
            for n in ("gate", "up"):
                matrix(p + "mlp." + n, F, D)
                vector(p + "mlp." + n + ".b", F, "bias")
            matrix(p + "mlp.down", D, F)
            vector(p + "mlp.down.b", D, "bias")
        return out
    D, F, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
    Q, K = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
    # a tied head reads the embedding's table: the embedding is then drawn as a head's matrix is
    out["model.embed_tokens.weight"] = ((V, D), "matrix" if cfg["tie_word_embeddings"] else "embedding")
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        for name, rows, cols in (("self_attn.q_proj", Q, D), ("self_attn.k_proj", K, D), ("self_attn.v_proj", K, D),
                                 ("self_attn.o_proj", D, Q), ("mlp.gate_proj", F, D), ("mlp.up_proj", F, D), ("mlp.down_proj", D, F)):
            matrix(p + name + ".weight", rows, cols)
        vector(p + "input_layernorm.weight", D, "norm")
        vector(p + "post_attention_layernorm.weight", D, "norm")
    vector("model.norm.weight", D, "norm")
    if not cfg["tie_word_embeddings"]:
        matrix("lm_head.weight", V, D)
    return out


def _values(case, seed):
    """get(name): a tensor of the case's model on the device, as stored (matrices in the compute dtype, vectors in 32 bits)."""
    table, dtype = _tensors(case), DTYPES[case["dtype"]]

    def get(name):
        shape, how = table[name]
        g = torch.Generator(device=DEVICE).manual_seed(_number(seed, name))
        t = torch.empty(shape, dtype=torch.float32 if len(shape) == 1 else dtype, device=DEVICE)
        if how == "embedding":
            return t.normal_(0.0, 1.0, generator=g)
        low, high = {"matrix": (-1.0 / math.sqrt(shape[-1]), 1.0 / math.sqrt(shape[-1])), "norm": (0.9, 1.1), "offset": (-0.1, 0.1),
                     "bias": (-0.5, 0.5), "taps": (-0.8, 0.8), "fraction": (0.1, 0.9)}[how]
        return t.uniform_(low, high, generator=g)
    return get


def _lengths(case):
    """Tokens of each sequence: evenly from (1 - spread) of the longest to it, in no order of size."""
    n, B = case.get("context") or case["tokens"], case["batch"]
    lens = [max(1, n - int(round(case["spread"] * n * i / max(1, B - 1)))) for i in range(B)]
    return [lens[(i * 7 + 3) % B] for i in range(B)] if B % 7 else lens


def _texts(case, seed):
    """Each sequence's tokens: its prompt, and the ones given behind it."""
    cfg = SHAPES[case["shape"]]
    V = cfg.get("vocab_size") or cfg["vocab"]
    g = torch.Generator().manual_seed(_number(seed, "texts"))
    lens, more = _lengths(case), case.get("new", 1)
    flat = torch.randint(0, V, (sum(lens) + more * len(lens),), generator=g).tolist()
    out, at = [], 0
    for n in lens:
        out.append((flat[at:at + n], flat[at + n:at + n + more]))
        at += n + more
    return out


class _Keeping(Sampler):
    """A sampler that keeps the logits it drew from."""

    def draw(self, logits, temperature, request_ids, steps):
        self.kept.append(logits.clone())
        return super().draw(logits, temperature, request_ids, steps)


def prepare(case, seed):
    cfg = config_from_dict(SHAPES[case["shape"]])
    spec = cfg.to_spec()
    if case["layers"] < len(spec.layers) and case["shape"] != "rekirax":
        spec.layers = spec.layers[:case["layers"]]
        spec.schedule = spec.schedule[:case["layers"]]
    model = Model(spec, cfg).load(_values(case, seed), DTYPES[case["dtype"]], DEVICE)
    texts = _texts(case, seed)
    B, lens = case["batch"], [len(p) for p, _ in texts]
    spare = min(SPARE, spec.max_positions - max(lens)) if case["kind"] == "decode" else case.get("new", 0) + 1
    engine = Engine(model, max_tokens=sum((n + spare + 63) // 64 * 64 for n in lens), max_batch=B)
    state = {"case": case, "engine": engine, "texts": texts}
    if case["kind"] == "decode":
        ragged = B > 1 and max(lens) - sum(lens) / B >= max(128, 0.2 * max(lens))
        engine.warmup([B], min_len=max(lens) + 1, max_len=max(lens) + spare, ragged=ragged)
        slots = state["slots"] = engine.start(B)
        at = 0
        while at < B:                       # the contexts, some sequences at a time
            end, total = at, 0
            while end < B and (end == at or total + lens[end] <= 16384):
                total += lens[end]
                end += 1
            engine.step(slots[at:end], [p for p, _ in texts[at:end]])
            at = end
    elif case.get("new"):
        engine.warmup(range(1, B + 1) if case["kind"] == "generate" else [B], min_len=max(lens) + 1, max_len=max(lens) + case["new"] + 1)
    return state


def run(state):
    case, engine, texts = state["case"], state["engine"], state["texts"]
    kind, B = case["kind"], case["batch"]
    if kind == "decode":
        return engine.step(state["slots"], [new for _, new in texts])
    prompts = [p for p, _ in texts]
    if kind == "generate":
        sampler = _Keeping(0)
        sampler.kept = []
        tokens = generate(engine, prompts, max_new_tokens=case["new"], temperature=0.0, stop_ids=(), sampler=sampler)
        return {"tokens": torch.tensor(tokens), "logits": torch.stack(sampler.kept)}
    slots = engine.start(B)
    if kind == "prompt":
        out = engine.step(slots, prompts)
    elif kind == "score":
        n = len(prompts[0])
        out = engine.step(slots, prompts, [list(range(n - 1))], [prompts[0][1:]])
    else:
        out = [engine.step(slots, prompts).clone()]
        for i in range(case["new"]):
            out.append(engine.step(slots, [[new[i]] for _, new in texts]).clone())
        out = torch.stack(out)
    engine.release(slots)
    return out


# ------------------------------------------------------------------------------------------------ what a pass needs
def _layer_costs(case):
    """(weights of the layers' matrices, [(window or chunk or 0, elements of a key and its value, elements of a query and its
    result, states of a recurrence) of each layer], head matrix elements, width, vocab)"""
    cfg = SHAPES[case["shape"]]
    if case["shape"] == "rekirax":
        D, V, weights, layers = cfg["width"], cfg["vocab"], 2 * cfg["width"] ** 2, []
        for layer in cfg["layers"]:
            a = layer["mixer"].get("left", layer["mixer"])
            q, k = a["heads"] * a["dim"], a["kv_heads"] * a["dim"]
            both = layer["type"] == "parallel"
            weights += D * (2 * q + k) + (D * (k + q) + 4 * D * q if both else 0) + 3 * D * layer["mlp"]["ff"]
            layers.append((a["mask"]["size"], both, 2 * k, 2 * q, q * a["dim"] if both else 0))
        return weights, layers, D, V
    D, F, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
    q, k = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
    layers = [(cfg.get("sliding_window") or 0, False, 2 * k, 2 * q, 0)] * case["layers"]
    return case["layers"] * (D * (2 * q + 2 * k) + 3 * D * F), layers, D, V


def work(case):
    """Every weight read once a step and an embedding row a token, the visible keys and values read once and the new ones
    written, the logits written (the probabilities of a score); a multiplication and an addition for each weight and token,
    each visible key and query, each element of a recurrence's state and token."""
    weights, layers, D, V = _layer_costs(case)
    size = 2 if case["dtype"] == "bf16" else 4
    lens = _lengths(case)
    nbytes = flops = 0

    def visible(pos, window, chunk):                       # keys that the token at `pos` sees
        return pos % window + 1 if chunk else min(pos + 1, window) if window else pos + 1

    def steps(brought, rows, out_bytes):
        """brought: (first position, tokens) of each sequence."""
        nonlocal nbytes, flops
        T = sum(n for _, n in brought)
        nbytes += (weights + V * D + T * D) * size + out_bytes
        flops += 2 * (weights * T + rows * V * D)
        for window, chunk, kv, q, state in layers:
            for start, n in brought:
                if n == 1:
                    seen = read = visible(start, window, chunk)
                else:
                    seen = sum(visible(p, window, chunk) for p in range(start, start + n))
                    read = 0
                nbytes += (read + n) * kv * size + 8 * state       # the state is read and written in 32 bits
                flops += 2 * seen * q + 4 * n * state
    if case["kind"] == "decode":
        steps([(n, 1) for n in lens], len(lens), 4 * V * len(lens))
    elif case["kind"] == "score":
        steps([(0, lens[0])], lens[0] - 1, 4 * (lens[0] - 1))
    else:
        steps([(0, n) for n in lens], len(lens), 4 * V * len(lens))
        more = {"prompt": 0, "trace": case.get("new", 0), "generate": case.get("new", 1) - 1}[case["kind"]]
        for i in range(more):
            steps([(n + i, 1) for n in lens], len(lens), 4 * V * len(lens))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what run() is off exact() by: 1.2e-7 to 1.5e-6 in float32, 1.8e-3 to 4.7e-3 in bfloat16 (a normal
    spread's largest of 100,000 values is five times its size).  No whole values but the tokens drawn in float32."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    return {"rel": 0.02, "max": 0.1}


# ------------------------------------------------------------------------------------------------ 64 bits
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, positions, freq):
    """x [T, heads, d]: element i of a head's first 2 len(freq) turns with element i + len(freq)."""
    n = freq.numel()
    angle = positions.to(torch.float64)[:, None, None] * freq
    a, b = x[..., :n], x[..., n:2 * n]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), x[..., 2 * n:]], -1)


def _attention(q, k, v, sees, scale, shape_score=None, first=0):
    """q [T, H, d] from position `first`, k and v [S, G, d]; sees(i, j): the visible pairs.  Some queries at a time."""
    T, H, d = q.shape
    S, G, _ = k.shape
    kt = k.permute(1, 2, 0).contiguous()                                       # [G, d, S]
    vs = v.permute(1, 0, 2).contiguous()                                       # [G, S, d]
    out = torch.empty_like(q)
    block = max(1, min(T, (1 << 28) // (H * S)))
    j = torch.arange(S, device=q.device)
    for a in range(0, T, block):
        b = min(T, a + block)
        i = torch.arange(first + a, first + b, device=q.device)[:, None]
        s = (q[a:b].permute(1, 0, 2).reshape(G, H // G * (b - a), d) @ kt).mul_(scale).reshape(H, b - a, S)
        if shape_score is not None:
            s = shape_score(s, (i - j).to(torch.float64))
        s = torch.softmax(s.masked_fill_(~sees(i, j), float("-inf")), -1)
        out[a:b] = (s.reshape(G, H // G * (b - a), S) @ vs).reshape(H, b - a, d).permute(1, 0, 2)
    return out.reshape(T, H * d)


def _frequencies(cfg):
    d = cfg["head_dim"]
    f = float(cfg["rope_theta"]) ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEVICE) / d)
    rs = cfg.get("rope_scaling")
    if rs:
        length = 2 * math.pi / f
        lo, hi, L = rs["low_freq_factor"], rs["high_freq_factor"], rs["original_max_position_embeddings"]
        s = ((L / length - lo) / (hi - lo)).clamp(0.0, 1.0)
        f = (1 - s) * f / rs["factor"] + s * f
    return f


def _llama(case, W, texts, wanted):
    """The hidden rows behind the last norm at the wanted places of each text."""
    cfg = SHAPES[case["shape"]]
    H, G, d, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    freq, window = _frequencies(cfg), cfg.get("sliding_window") or 0

    def sees(i, j):
        return (j <= i) & (i - j < window) if window else j <= i
    table = W("model.embed_tokens.weight")
    xs = [table[torch.tensor(t, device=DEVICE)] for t in texts]
    del table
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        wq, wk, wv, wo = (W(p + "self_attn.%s_proj.weight" % n) for n in "qkvo")
        n1, n2 = W(p + "input_layernorm.weight"), W(p + "post_attention_layernorm.weight")
        wg, wu, wd = (W(p + "mlp.%s_proj.weight" % n) for n in ("gate", "up", "down"))
        for s, x in enumerate(xs):
            at = torch.arange(x.shape[0], device=DEVICE)
            h = _rms(x, eps) * n1
            q = _turn((h @ wq.T).reshape(-1, H, d), at, freq)
            k = _turn((h @ wk.T).reshape(-1, G, d), at, freq)
            if i == case["layers"] - 1:               # behind the last attention only the wanted rows go on
                lo = min(wanted[s])
                x, q = x[lo:], q[lo:]
                wanted[s] = [w - lo for w in wanted[s]]
            else:
                lo = 0
            x = x + _attention(q, k, (h @ wv.T).reshape(-1, G, d), sees, d ** -0.5, first=lo) @ wo.T
            h = _rms(x, eps) * n2
            g = h @ wg.T
            xs[s] = x + ((g * torch.sigmoid(g)) * (h @ wu.T)) @ wd.T
    norm = W("model.norm.weight")
    return [_rms(x[w], eps) * norm for x, w in zip(xs, wanted)]


def _rekirax_rows(case, W, texts, wanted):
    cfg = SHAPES["rekirax"]
    eps, taps = cfg["norm"]["eps"], cfg["canon"]["taps"]
    table, en = W("embed"), 1.0 + W("embed.norm")
    xs = [_rms(table[torch.tensor(t, device=DEVICE)], eps) * en for t in texts]
    del table
    x0 = list(xs)
    for i, layer in enumerate(cfg["layers"]):
        if i == cfg["loop"]["start"]:
            m, b = W("loop.in"), W("loop.step")[0]
            xs = [torch.cat([x, e], -1) @ m.T + b for x, e in zip(xs, x0)]
        p = "l%d." % i
        w = {n[len(p):]: W(n) for n in _tensors(case) if n.startswith(p)}
        for s, x in enumerate(xs):
            T = x.shape[0]
            at = torch.arange(T, device=DEVICE)
            h = _rms(x, eps) * (1.0 + w["norm1"])
            padded = torch.cat([torch.zeros((taps - 1, h.shape[1]), dtype=h.dtype, device=DEVICE), h])
            h = h + sum(w["canon1"][:, j] * padded[j:j + T] for j in range(taps))
            if layer["type"] == "parallel":
                a = layer["mixer"]["left"]
                H, G, d, size = a["heads"], a["kv_heads"], a["dim"], a["mask"]["size"]
                q = (_rms(h @ w["mix.left.q"].T, eps) * w["mix.left.q.norm"]).reshape(T, H, d)
                k = (_rms(h @ w["mix.left.k"].T, eps) * w["mix.left.k.norm"]).reshape(T, G, d)
                n = a["rot"]["dims"]
                f = float(a["rot"]["base"]) ** (-torch.arange(0, n, 2, dtype=torch.float64, device=DEVICE) / n)
                o = _attention(_turn(q, at, f), _turn(k, at, f), (h @ w["mix.left.v"].T).reshape(T, G, d),
                               lambda i, j: (j <= i) & (i // size == j // size), a["scale"])
                left = (o * torch.sigmoid(h @ w["mix.left.g"].T)) @ w["mix.left.o"].T
                H, d, dv = (layer["mixer"]["right"][n] for n in ("heads", "dim", "vdim"))
                q = h @ w["mix.right.q"].T
                q = (q * torch.sigmoid(q)).reshape(T, H, d)
                low = w["mix.right.lower"]
                f = (low + (1.0 - low) * torch.sigmoid(h @ w["mix.right.f"].T + w["mix.right.f.b"])).reshape(T, H, d)
                v = (h @ w["mix.right.v"].T).reshape(T, H, dv)
                S = torch.zeros((H, d, dv), dtype=torch.float64, device=DEVICE)
                o = torch.empty((T, H, dv), dtype=torch.float64, device=DEVICE)
                for t in range(T):
                    S = f[t][:, :, None] * S + (1.0 - f[t])[:, :, None] * v[t][:, None, :]
                    o[t] = (S * q[t][:, :, None]).sum(1)
                right = (_rms(o, eps) * w["mix.right.norm"]).reshape(T, H * dv) @ w["mix.right.o"].T
                y = 0.5 * (_rms(left, eps) * w["mix.left.out"] + _rms(right, eps) * w["mix.right.out"])
            else:
                a = layer["mixer"]
                H, G, d, size, cap = a["heads"], a["kv_heads"], a["dim"], a["mask"]["size"], a["softcap"]
                q = _rms((h @ w["mix.q"].T).reshape(T, H, d), eps) * w["mix.q.norm"]
                raw = (h @ w["mix.k"].T).reshape(T, G, d)
                r1, r2 = w["mix.r1"][:, None, None], w["mix.r2"][:, None, None]
                y = _attention(q, _rms(raw, eps) * w["mix.k.norm"], raw, lambda i, j: (j <= i) & (i - j < size), a["scale"],
                               lambda s, far: cap * torch.tanh(s / cap) - r1 * torch.log(1.0 + r2 * far.clamp(min=0.0))) @ w["mix.o"].T
            x = x + y
            h = _rms(x, eps) * (1.0 + w["norm2"])
            g = h @ w["mlp.gate"].T + w["mlp.gate.b"]
            g = 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))
            xs[s] = x + (g * (h @ w["mlp.up"].T + w["mlp.up.b"])) @ w["mlp.down"].T + w["mlp.down.b"]
    norm = 1.0 + W("final.norm")
    return [_rms(x[at], eps) * norm for x, at in zip(xs, wanted)]


def exact(case, seed):
    """What run() gives, in 64 bits: whole texts without a cache.  None where the products alone would take long."""
    lens, more = _lengths(case), case.get("new", 1)
    weights = _layer_costs(case)[0]
    if 2 * weights * (sum(lens) + more * len(lens)) > 4e14:
        return None
    get = _values(case, seed)

    def W(name):
        return get(name).to(torch.float64)
    rows = _rekirax_rows if case["shape"] == "rekirax" else _llama
    cfg = SHAPES[case["shape"]]
    tied = case["shape"] == "rekirax" or cfg["tie_word_embeddings"]
    head = W("embed" if case["shape"] == "rekirax" else "model.embed_tokens.weight" if tied else "lm_head.weight")
    texts, kind = _texts(case, seed), case["kind"]
    prompts = [list(p) for p, _ in texts]
    if kind == "generate":
        tokens, logits = [[] for _ in prompts], []
        for _ in range(more):
            seen = [p + t for p, t in zip(prompts, tokens)]
            logits.append(torch.cat(rows(case, W, seen, [[len(t) - 1] for t in seen])) @ head.T)
            for t, best in zip(tokens, logits[-1].argmax(-1).tolist()):
                t.append(best)
        return {"tokens": torch.tensor(tokens), "logits": torch.stack(logits)}
    if kind == "score":
        n = lens[0]
        h = rows(case, W, prompts, [list(range(n - 1))])[0]
        p = torch.cat([torch.softmax(h[a:a + 128] @ head.T, -1) for a in range(0, n - 1, 128)])
        return p[torch.arange(n - 1, device=DEVICE), torch.tensor(prompts[0][1:], device=DEVICE)]
    if kind == "prompt":
        return torch.cat(rows(case, W, prompts, [[n - 1] for n in lens])) @ head.T
    if kind == "decode":
        return torch.cat(rows(case, W, [p + new for p, new in texts], [[n] for n in lens])) @ head.T
    h = torch.stack(rows(case, W, [p + new for p, new in texts], [list(range(n - 1, n + more)) for n in lens]))
    return (h @ head.T).transpose(0, 1)
