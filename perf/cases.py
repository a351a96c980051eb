"""What this engine is asked to do in earnest, as cases that can be timed and checked.

A case is a model, a data type, and what one pass brings to ``Engine.step``:

* ``requests`` requests that decode, each with up to ``context`` cached tokens (their lengths
  differ), one token each in every step of the pass;
* ``prompts`` new prompts of up to ``tokens`` tokens each (their lengths differ), opened, computed
  in steps of at most ``budget`` rows beside the decoding requests, and closed again.

A pass returns the float32 logits of every step's wanted rows: those of every decoded token and of
the last token of every prompt.  A decoding request grows by its tokens, as it does in a server; one
that has reached the longest length of its slot makes room for the same request anew.

The sizes are those of ``bench.py``: the layer sizes of the Qwen2.5 checkpoints and the Vivevik design.
The weights are random, drawn on the GPU from the seed; so are the tokens.
"""
import math

import torch

import llm_inference_lab_amd as lab

PAGE = 64               # cache page of bench.py
FILL_TOKENS = 8192      # rows of the steps that fill the caches before a pass
ROOM = 1024             # tokens that a decoding request can grow by before it is opened anew
DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}

# width, heads, kv heads, head size, feed-forward width, layers, vocabulary, head tied to the embedding
QWEN2 = {
    "0.5b": (896, 14, 2, 64, 4864, 24, 151936, True),
    "1.5b": (1536, 12, 2, 128, 8960, 28, 151936, True),
    "3b": (2048, 16, 2, 128, 11008, 36, 151936, True),
    "7b": (3584, 28, 4, 128, 18944, 28, 152064, False),
}
ROPE_THETA = 1e6
# gated linear attention, then attention with keys of its own, then attention that reads them, in turn
VIVEVIK = {
    "vivevik_small": (896, 14, 2, 64, 4864, 12, 32000, True),
    "vivevik_medium": (2048, 16, 2, 128, 11008, 12, 32000, True),
}
WINDOW, KEEP = 1024, 8
GLA_DIM, GLA_VDIM, GLA_RANK, GLA_TAU = 64, 128, 32, 8.0
EPS = 1e-6


def _case(model, dtype="bf16", requests=0, context=0, prompts=0, tokens=0, budget=FILL_TOKENS):
    return {"model": model, "dtype": dtype, "requests": requests, "context": context, "prompts": prompts,
            "tokens": tokens, "budget": budget}


def listed():
    return [
        # one user's chat on the small model: the smallest step there is, a chain of launches
        dict(_case("0.5b", requests=1, context=600), name="decode_1"),
        # a few users with long histories: the repository's headline point (bench.py's default)
        dict(_case("0.5b", requests=8, context=4096), name="decode_8"),
        # a busy server of the small model
        dict(_case("0.5b", requests=64, context=2000), name="decode_64"),
        # the 32-bit mode, for users who compare against another implementation
        dict(_case("0.5b", dtype="f32", requests=8, context=1000), name="decode_8_f32"),
        # one prompt in one step: time to the first token (bench.py's prefill)
        dict(_case("0.5b", prompts=1, tokens=2048), name="prompt_2048"),
        # the same in the 32-bit mode, at a length that fills no tile
        dict(_case("0.5b", dtype="f32", prompts=1, tokens=1531), name="prompt_1531_f32"),
        # continuous batching at the default budget of 512 rows: a prompt's portions beside decodes
        dict(_case("0.5b", requests=48, context=1500, prompts=1, tokens=1801, budget=512), name="mixed_48"),
        # a larger model, few users with long histories: bound by its weights
        dict(_case("7b", requests=8, context=4096), name="decode_8_7b"),
        # a larger model with many users
        dict(_case("7b", requests=128, context=512), name="decode_128_7b"),
        # time to the first token of the larger model, several prompts at once in one step
        dict(_case("7b", prompts=3, tokens=1000), name="prompts_3_7b"),
        # the other kind of layers: a recurrence beside windowed attention, prompt and decode
        dict(_case("vivevik_small", prompts=1, tokens=1900), name="prompt_1900_vivevik"),
        dict(_case("vivevik_medium", requests=16, context=1500), name="decode_16_vivevik"),
    ]


def draw(rng):
    """A case of the same ranges: any of the models, decode, prompts or both; sizes over their logarithm;
    at most the cost of the largest listed case."""
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    most = max(_seconds(c) for c in listed())
    while True:
        model = rng.choice(["0.5b", "0.5b", "1.5b", "3b", "7b", "7b", "vivevik_small", "vivevik_medium"])
        dtype = "f32" if model == "0.5b" and rng.random() < 0.3 else "bf16"
        kind = rng.choice(["decode", "decode", "prompts", "prompts", "mixed"])
        case = _case(model, dtype)
        if kind != "prompts":
            case.update(requests=spread(1, 128), context=spread(64, 4096))
            if case["requests"] * case["context"] > 140000:      # (the caches of a state are filled in under a second)
                continue
        if kind != "decode":
            case.update(prompts=rng.choice([1, 1, 2, 3, 5]), tokens=spread(32, 4096))
        if kind == "mixed":
            case["budget"] = rng.choice([512, 1024, 2048])
        if _rows(case) <= FILL_TOKENS and _seconds(case) <= most:
            return case


# ------------------------------------------------------------------------------------ shapes of a case
def _sizes(case):
    return (QWEN2.get(case["model"]) or VIVEVIK[case["model"]])


def _layers(case):
    """The mixer of every layer: "full", "gla", "window" (keys of its own) or "shared" (the keys of the layer
    before)."""
    n = _sizes(case)[5]
    return ["full"] * n if case["model"] in QWEN2 else [("gla", "window", "shared")[i % 3] for i in range(n)]


def _contexts(case):
    """Cached tokens of every decoding request: from three quarters of the context to all of it."""
    c = case["context"]
    return [c - i * 97 % (c // 4 + 1) for i in range(case["requests"])]


def _lengths(case):
    """Tokens of every prompt: from half of the case's to all of them."""
    t = case["tokens"]
    return [t - i * 211 % (t // 2 + 1) for i in range(case["prompts"])]


def _rows(case):
    return sum(_lengths(case)) if case["budget"] >= FILL_TOKENS else case["budget"]


def _plan(case):
    """The steps of a pass: for each the portions ``(prompt, first, end)`` beside the decoded tokens."""
    room = case["budget"] - case["requests"]
    steps, free = [[]], room
    for p, length in enumerate(_lengths(case)):
        at = 0
        while at < length:
            if free == 0:
                steps.append([])
                free = room
            n = min(free, length - at)
            steps[-1].append((p, at, at + n))
            at, free = at + n, free - n
    return steps


def _parameters(case):
    """Numbers of a layer's matrices in turn, and of the head."""
    w, heads, kv, dim, ff, _, vocab, _ = _sizes(case)
    per = {
        "full": w * (heads + 2 * kv) * dim + heads * dim * w + 3 * w * ff,
        "gla": w * (w // GLA_VDIM) * (2 * GLA_DIM + 3 * GLA_VDIM) + GLA_RANK * (w + (w // GLA_VDIM) * GLA_DIM),
        "window": w * (heads + 2 * kv) * dim + heads * dim * w + 2 * w * ff,
        "shared": w * heads * dim + heads * dim * w + 2 * w * ff,
    }
    return [per[kind] for kind in _layers(case)], w * vocab


def work(case):
    """Per step: every weight once, the keys and values that are seen read and the new ones written, the
    recurrent states both ways, the logits written."""
    w, heads, kv, dim, ff, _, vocab, _ = _sizes(case)
    width = 2 if case["dtype"] == "bf16" else 4
    per_layer, head = _parameters(case)
    nbytes = flops = 0
    for s, portions in enumerate(_plan(case)):
        entries = [(c + s, c + s + 1, True) for c in _contexts(case)]
        entries += [(a, b, b == _lengths(case)[p]) for p, a, b in portions]
        rows, wanted = sum(b - a for a, b, _ in entries), sum(want for _, _, want in entries)
        nbytes += width * (sum(per_layer) + head + rows * w) + 4 * wanted * vocab
        flops += 2 * (rows * sum(per_layer) + wanted * head)
        for kind in _layers(case):
            for a, b, _ in entries:
                if kind == "gla":
                    state = (w // GLA_VDIM) * GLA_DIM * GLA_VDIM
                    nbytes += 8 * state
                    flops += 4 * state * (b - a)
                    continue
                most = b if kind == "full" else WINDOW + KEEP
                pairs = sum(min(i + 1, most) for i in range(a, b))
                flops += 4 * pairs * heads * dim
                nbytes += width * 2 * kv * dim * (min(b, most + b - a) + (b - a if kind != "shared" else 0))
    return {"bytes": nbytes, "flops": flops}


def _seconds(case):
    """About how long a pass takes: to compare the cost of cases."""
    w = work(case)
    return len(_plan(case)) * 5e-4 + w["bytes"] / 4e12 + w["flops"] / (7e14 if case["dtype"] == "bf16" else 8e13)


def tolerance(case):
    """Measured, about four times what another order of the sums and ``exact`` show (the residual sums of up
    to 36 layers of random weights).  bfloat16: its activations are rounded once per kernel."""
    return {"rel": 2e-5, "max": 4e-4} if case["dtype"] == "f32" else {"rel": 0.03, "max": 0.6}


# ------------------------------------------------------------------------------------ weights and tokens
def _weights(case, seed):
    """``(name, tensor)`` of the model file, drawn on the GPU: matrices, biases and learned vectors around
    zero, the weights of norms around one; bfloat16 in the file, as the checkpoints are.  The spread of a
    matrix keeps the size of what it multiplies at every width (0.02 at 896), and what adds into the stream
    is smaller by the root of the number of its terms, as in models that train: all terms together weigh
    what one does."""
    w, heads, kv, dim, ff, layers, vocab, tied = _sizes(case)
    spread = 0.6 / math.sqrt(w)
    into = spread / math.sqrt(2 * layers)
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(1_000_003 * int(seed) + 11)

    def normal(*shape, mean=0.0, std=spread):
        return torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(mean, std, generator=gen)

    def norm(n):
        return normal(n, mean=1.0, std=0.1)

    if case["model"] in QWEN2:
        yield "model.embed_tokens.weight", normal(vocab, w)
        for i in range(len(_layers(case))):
            at = f"model.layers.{i}."
            yield at + "input_layernorm.weight", norm(w)
            for name, rows in (("q", heads * dim), ("k", kv * dim), ("v", kv * dim)):
                yield at + f"self_attn.{name}_proj.weight", normal(rows, w)
                yield at + f"self_attn.{name}_proj.bias", normal(rows)
            yield at + "self_attn.o_proj.weight", normal(w, heads * dim, std=into)
            yield at + "post_attention_layernorm.weight", norm(w)
            yield at + "mlp.gate_proj.weight", normal(ff, w)
            yield at + "mlp.up_proj.weight", normal(ff, w)
            yield at + "mlp.down_proj.weight", normal(w, ff, std=into)
        yield "model.norm.weight", norm(w)
        if not tied:
            yield "lm_head.weight", normal(vocab, w)
        return
    yield "embed", normal(vocab, w)
    gla_heads = w // GLA_VDIM
    for i, kind in enumerate(_layers(case)):
        at = f"l{i}."
        if kind == "gla":
            for name, rows in (("q", GLA_DIM), ("k", GLA_DIM), ("v", GLA_VDIM), ("g", GLA_VDIM)):
                yield at + f"mix.{name}", normal(gla_heads * rows, w)
            yield at + "mix.a1", normal(GLA_RANK, w)
            yield at + "mix.a2", normal(gla_heads * GLA_DIM, GLA_RANK)
            yield at + "mix.a2.b", normal(gla_heads * GLA_DIM)
            yield at + "mix.norm", norm(GLA_VDIM)
            yield at + "mix.o", normal(w, gla_heads * GLA_VDIM, std=into)
        else:
            yield at + "mix.q", normal(heads * dim, w)
            yield at + "mix.q.norm", norm(heads * dim)
            if kind == "window":
                yield at + "mix.k", normal(kv * dim, w)
                yield at + "mix.k.norm", norm(kv * dim)
                yield at + "mix.v", normal(kv * dim, w)
            yield at + "mix.sink", normal(heads)
            yield at + "mix.o", normal(w, heads * dim, std=into)
        yield at + "norm1", norm(w)
        if kind != "gla":
            yield at + "mlp.up", normal(ff, w)
            yield at + "mlp.down", normal(w, ff, std=into)
            yield at + "norm2", norm(w)
    yield "final.norm", norm(w)


def _config(case):
    w, heads, kv, dim, ff, layers, vocab, tied = _sizes(case)
    if case["model"] in QWEN2:
        return lab.Qwen2Config.from_dict(dict(
            architectures=["Qwen2ForCausalLM"], model_type="qwen2", vocab_size=vocab, hidden_size=w, intermediate_size=ff,
            num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=kv, head_dim=dim, rms_norm_eps=EPS,
            rope_theta=ROPE_THETA, max_position_embeddings=32768, use_sliding_window=False, tie_word_embeddings=tied))
    listed_layers = []
    for i, kind in enumerate(_layers(case)):
        if kind == "gla":
            listed_layers.append(dict(type="gla", mlp=None, mixer=dict(
                heads=w // GLA_VDIM, dim=GLA_DIM, vdim=GLA_VDIM, tau=GLA_TAU, rank=GLA_RANK)))
            continue
        mixer = dict(heads=heads, kv_heads=kv, dim=dim, vdim=dim, scale=dim ** -0.5,
                     mask=dict(size=WINDOW, keep_first=KEEP))
        if kind == "shared":
            mixer["kv_from"] = i - 1
        listed_layers.append(dict(type="attention", mixer=mixer, mlp=dict(kind="dense", ff=ff)))
    return lab.VivevikConfig.from_dict(dict(architecture="Vivevik", vocab=vocab, width=w, norm=dict(eps=EPS),
                                            layers=listed_layers))


def _tokens(case, seed):
    """The decoding requests' tokens (cached and still to come) and the prompts', as lists of whole numbers."""
    gen = torch.Generator().manual_seed(7_919 * int(seed) + 5)
    vocab = _sizes(case)[6]

    def some(n):
        return torch.randint(0, vocab, (n,), generator=gen).tolist()
    return [some(c + ROOM) for c in _contexts(case)], [some(n) for n in _lengths(case)]


# ------------------------------------------------------------------------------------ a user's program
class _Server:
    """An engine with its decoding requests in flight."""

    def __init__(self, case, seed):
        self.case, self.plan = case, _plan(case)
        self.decoding, self.prompts = _tokens(case, seed)
        self.contexts = _contexts(case)
        longest = max([c + ROOM for c in self.contexts] + _lengths(case))
        pages = sum(-(-n // PAGE) for n in [c + ROOM for c in self.contexts] + _lengths(case))
        self.engine = lab.Engine(config=_config(case), tensors=_weights(case, seed), dtype=case["dtype"], device=DEVICE,
                                 page_size=PAGE, num_pages=pages, max_requests=case["requests"] + case["prompts"],
                                 max_batch_tokens=FILL_TOKENS, max_seq_len=longest, graph="auto")
        self.handles = []
        self.fill()

    def fill(self):
        """Open the decoding requests and compute their cached tokens."""
        for h in self.handles:
            self.engine.close(h)
        self.handles = [self.engine.open(i) for i in range(len(self.contexts))]
        self.at = 0
        entries, free = [], FILL_TOKENS
        for h, tokens, length in zip(self.handles, self.decoding, self.contexts):
            first = 0
            while first < length:
                n = min(free, length - first)
                entries.append(lab.StepEntry(h, tokens[first:first + n]))
                first, free = first + n, free - n
                if free == 0:
                    self.engine.step(entries)
                    entries, free = [], FILL_TOKENS
        if entries:
            self.engine.step(entries)


def prepare(case, seed):
    return _Server(case, seed)


def run(state):
    if state.at + len(state.plan) > ROOM:
        state.fill()
    opened = [state.engine.open(("prompt", p)) for p in range(len(state.prompts))]
    out = []
    for portions in state.plan:
        entries = [lab.StepEntry(h, [tokens[c + state.at]], (0,))
                   for h, tokens, c in zip(state.handles, state.decoding, state.contexts)]
        for p, a, b in portions:
            last = b == len(state.prompts[p])
            entries.append(lab.StepEntry(opened[p], state.prompts[p][a:b], (b - a - 1,) if last else ()))
        logits = state.engine.step(entries)
        if logits is not None:
            out.append(logits if len(state.plan) == 1 else logits.clone())      # (the next step writes over them)
        state.at += 1
    for h in opened:
        state.engine.close(h)
    return out


# ------------------------------------------------------------------------------------ the same in 64 bits
EXACT_FLOPS = 5e14      # about 15 seconds of 64-bit products


def _linear(x, weight, bias=None):
    y = torch.cat([part @ weight.T for part in x.split(16384)])
    return y if bias is None else y + bias


def _rms(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight


def _layer_norm(x, weight):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], weight, None, EPS)


def _gated(h, gate, up, down):
    return (torch.nn.functional.silu(h @ gate.T) * (h @ up.T)) @ down.T


def _turn(x, base):
    """Channel ``i`` of a head with channel ``i + d / 2``, by position times ``base ** (-2 i / d)``."""
    t, _, d = x.shape
    where = torch.arange(t, device=x.device, dtype=x.dtype)
    angle = where[:, None] * base ** (-2.0 * torch.arange(d // 2, device=x.device, dtype=x.dtype) / d)
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    lo, hi = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _attend(q, k, v, sink=None, window=None):
    """One sequence: ``q [T, heads, d]``, ``k, v [T, kv heads, d]``; ``sink``: one more term per head in the
    softmax's denominator; ``window``: only so many positions back, and the first ``KEEP``."""
    t, heads, d = q.shape
    group = heads // k.shape[1]
    i = torch.arange(t, device=q.device)
    hidden = i[None] > i[:, None]
    if window is not None:
        hidden |= (i[:, None] - i[None] >= window) & (i[None] >= KEEP)
    out = torch.empty_like(q)
    for h in range(heads):
        s = (q[:, h] @ k[:, h // group].T.contiguous()) * d ** -0.5
        s.masked_fill_(hidden, -math.inf)
        m = s.amax(-1, keepdim=True)
        if sink is not None:
            m = torch.maximum(m, sink[h])
        e = (s - m).exp_()
        below = e.sum(-1, keepdim=True)
        if sink is not None:
            below = below + (sink[h] - m).exp()
        out[:, h] = (e @ v[:, h // group]) / below
    return out


def _recur(q, k, v, decay):
    """``S = decay_t S + k_t v_t^T``, ``o_t = S^T q_t`` for every head, token by token."""
    state = torch.zeros(q.shape[1], GLA_DIM, GLA_VDIM, dtype=q.dtype, device=q.device)
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        state = torch.addcmul(k[t, :, :, None] * v[t, :, None, :], decay[t, :, :, None], state)
        out[t] = (q[t, :, None, :] @ state)[:, 0]
    return out


def _forward(case, seed, sequences, wanted):
    """Logits at the ``wanted`` last positions of every sequence: the formulas of the model, in 64 bits."""
    w, heads, kv, dim, ff, _, vocab, tied = _sizes(case)
    # (in order: drawn a second time as the layers come, since all of them in 64 bits need not fit)
    source = iter(_weights(case, seed))

    def take(*names):
        got = []
        for name in names:
            found, tensor = next(source)
            assert found.endswith(name), (found, name)
            got.append(tensor.double())
        return got if len(got) > 1 else got[0]

    lengths = [len(s) for s in sequences]
    qwen = case["model"] in QWEN2
    embed = take("embed_tokens.weight" if qwen else "embed")
    x = embed[torch.tensor([t for s in sequences for t in s], device=DEVICE)]
    if not tied:
        del embed

    def per_sequence(fn, *rows):
        return torch.cat([fn(*part) for part in zip(*(r.split(lengths) for r in rows))])

    for kind in _layers(case):
        if kind == "full":
            n1, wq, bq, wk, bk, wv, bv, wo, n2, wg, wu, wd = take(
                "input_layernorm.weight", "q_proj.weight", "q_proj.bias", "k_proj.weight", "k_proj.bias", "v_proj.weight",
                "v_proj.bias", "o_proj.weight", "post_attention_layernorm.weight", "gate_proj.weight", "up_proj.weight",
                "down_proj.weight")
            h = _rms(x, n1)
            q, k, v = (_linear(h, m, b).unflatten(-1, (-1, dim)) for m, b in ((wq, bq), (wk, bk), (wv, bv)))
            o = per_sequence(lambda q, k, v: _attend(_turn(q, ROPE_THETA), _turn(k, ROPE_THETA), v), q, k, v)
            x = x + _linear(o.flatten(1), wo)
            x = torch.cat([part + _gated(_rms(part, n2), wg, wu, wd) for part in x.split(8192)])
            continue
        if kind == "gla":
            wq, wk, wv, wg, a1, a2, a2b, on, wo, n1 = take("q", "k", "v", "g", "a1", "a2", "a2.b", "mix.norm", "o", "norm1")
            q, k, v = (_linear(x, m).unflatten(-1, (-1, d)) for m, d in ((wq, GLA_DIM), (wk, GLA_DIM), (wv, GLA_VDIM)))
            decay = (_linear(_linear(x, a1), a2, a2b).sigmoid() ** (1 / GLA_TAU)).unflatten(-1, (-1, GLA_DIM))
            o = per_sequence(_recur, q * GLA_DIM ** -0.5, k, v, decay)
            y = _linear(_rms(o, on).flatten(1) * torch.nn.functional.silu(_linear(x, wg)), wo)
            x = x + _layer_norm(y, n1)
            continue
        wq, qn = take("mix.q", "q.norm")
        if kind == "window":
            wk, kn, wv = take("mix.k", "k.norm", "mix.v")
            k = _rms(_linear(x, wk), kn).unflatten(-1, (-1, dim))
            v = _linear(x, wv).unflatten(-1, (-1, dim))
        sink, wo, n1, up, down, n2 = take("sink", "mix.o", "norm1", "up", "down", "norm2")
        q = _rms(_linear(x, wq), qn).unflatten(-1, (-1, dim))
        o = per_sequence(lambda q, k, v: _attend(q, k, v, sink, WINDOW), q, k, v)
        x = x + _layer_norm(_linear(o.flatten(1), wo), n1)
        x = torch.cat([part + _layer_norm((part @ up.T).relu().square() @ down.T, n2) for part in x.split(8192)])
    last = take("norm.weight" if qwen else "final.norm")
    head = embed if tied else take("lm_head.weight")
    rows = [r for part, n in zip(x.split(lengths), wanted) for r in part[len(part) - n:].unbind()]
    x = torch.stack(rows)
    logits = _linear(_rms(x, last) if qwen else _layer_norm(x, last), head)
    return logits.split(wanted)


def exact(case, seed):
    plan = _plan(case)
    decoding, prompts = _tokens(case, seed)
    sequences = [t[:c + len(plan)] for t, c in zip(decoding, _contexts(case))] + prompts
    rows = sum(len(s) for s in sequences)
    if 2 * rows * sum(_parameters(case)[0]) > EXACT_FLOPS:
        return None
    if "gla" in _layers(case) and rows > 30000:       # (token by token)
        return None
    logits = _forward(case, seed, sequences, [len(plan)] * len(decoding) + [1] * len(prompts))
    out = []
    for s, portions in enumerate(plan):
        step = [logits[i][s] for i in range(len(decoding))]
        step += [logits[len(decoding) + p][0] for p, _, b in portions if b == len(prompts[p])]
        if step:
            out.append(torch.stack(step))
    return out
