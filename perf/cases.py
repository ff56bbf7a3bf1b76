"""What a user of this engine has it do, as cases that can be measured and checked.

A case is either ``traffic``: requests with given prompts that generate a number of tokens each through the engine's step
function (``Executor.step``), with given ids in the place of chosen ones, so that every pass and every implementation runs
the same steps; or ``choose``: a step's tokens chosen from its logits (``DevicePicker``).

traffic   model, layers       one of MODELS below (layer sizes of this repository's configurations), with so many layers
          dtype               "bfloat16" (what serving uses) or "float32" (the 32-bit path)
          requests, first     how many requests, and how many of them come with the first step ...
          every               ... one more with every so many steps
          shortest, longest   lengths of their prompts, spread over this range by the seed
          new                 tokens a request generates: its prompt's last logits and new - 1 steps of one token
          portion             a prompt goes in portions of so many tokens beside the others' tokens (0: whole)
choose    rows, vocab         rows of logits; every fifth one greedy, the others with a temperature, a top-k, a top-p, both
"""
import math
import random

import torch

LLAMA_KEYS = ("vocab_size", "hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size",
              "rope_theta", "rms_norm_eps", "max_position_embeddings", "tie_word_embeddings")


def _llama(*values):
    return dict(zip(LLAMA_KEYS, values), architectures=["LlamaForCausalLM"], model_type="llama")


MODELS = {
    "tiny-a": _llama(256, 64, 4, 2, 16, 176, 10000.0, 1e-5, 128, False),
    "tiny-b": _llama(384, 96, 3, 3, 32, 256, 500000.0, 1e-6, 256, True),
    "tinyllama-1.1b": _llama(32000, 2048, 32, 4, 64, 5632, 10000.0, 1e-5, 2048, False),
    "llama-2-7b": _llama(32000, 4096, 32, 32, 128, 11008, 10000.0, 1e-5, 4096, False),
    "llama-3-8b": _llama(128256, 4096, 32, 8, 128, 14336, 500000.0, 1e-5, 8192, False),
    # every third layer a recurrent one without a feed-forward, the others latent attention with a dense feed-forward
    "mamenex-2k": dict(architecture="Mamenex", vocab=32000, width=2048, norm=dict(eps=1e-5), canon=dict(taps=3)),
}
MAMENEX_ATTENTION = dict(type="latent_attention", mlp=dict(kind="dense", ff=8192), mixer=dict(
    heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5, rot=dict(base=10000.0, dims=64)))
MAMENEX_RECURRENT = dict(type="rglru", mlp=None, mixer=dict(width=2560, blocks=10, conv=4))
PAGE = 64


def _traffic(name, model, layers, dtype, requests, shortest, longest, new, portion=0, first=None, every=0):
    case = dict(kind="traffic", model=model, layers=layers, dtype=dtype, requests=requests, shortest=shortest, longest=longest,
                new=new, portion=portion, first=requests if first is None else first, every=every)
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest run there is, three short prompts on two narrow layers: launches and the host are all of it
        _traffic("tiny_f32", "tiny-a", 2, "float32", 3, 1, 33, 16),
        # one user at a prompt: 16 tokens in, 32 out
        _traffic("chat_b1", "tinyllama-1.1b", 22, "bfloat16", 1, 16, 16, 32),
        # eight requests decoding at 512 to 576 tokens of context
        _traffic("decode_b8", "tinyllama-1.1b", 22, "bfloat16", 8, 512, 512, 64),
        # a full batch of short chats
        _traffic("chat_b64", "tinyllama-1.1b", 22, "bfloat16", 64, 16, 64, 64),
        # time to the first token of one long prompt
        _traffic("prompt_2048", "tinyllama-1.1b", 22, "bfloat16", 1, 2048, 2048, 1),
        # requests that come one after the other: most steps hold a prompt, or a portion of one, beside decoded tokens
        _traffic("arrivals", "tinyllama-1.1b", 22, "bfloat16", 16, 24, 700, 24, portion=256, first=4, every=2),
        # the same at wide layers and long prompts in portions of 512
        _traffic("serve_wide", "llama-3-8b", 8, "bfloat16", 8, 128, 4096, 24, portion=512),
        # every head with keys of its own at 1,000 tokens of context: the cache is what a step reads most
        _traffic("decode_mha", "llama-2-7b", 8, "bfloat16", 16, 900, 1024, 48),
        # the 32-bit path: a prompt, and eight requests decoding
        _traffic("prompt_f32", "tinyllama-1.1b", 22, "float32", 1, 1000, 1000, 1),
        _traffic("decode_f32", "tinyllama-1.1b", 22, "float32", 8, 24, 100, 32),
        # latent attention and recurrent layers
        _traffic("mamenex", "mamenex-2k", 6, "bfloat16", 8, 100, 700, 48),
        # a full batch's tokens chosen from its logits, requests with options of every kind
        dict(name="choose_64", kind="choose", rows=64, vocab=32000),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over the logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random):
    kind = rng.randrange(11)
    bf16, f32 = "bfloat16", "float32"
    if kind == 0:
        model, layers, most = rng.choice((("tiny-a", 2, 100), ("tiny-b", 3, 200)))
        longest = _spread(rng, 2, most)
        return _traffic(None, model, layers, rng.choice((bf16, f32)), rng.randint(1, 6), rng.randint(1, longest), longest,
                        rng.randint(2, 24), portion=rng.choice((0, 32)))
    if kind in (1, 2):                                      # decoding at any number of requests
        requests = _spread(rng, 1, 64)
        longest = _spread(rng, 8, max(16, min(1400, 16384 // requests)))
        return _traffic(None, "tinyllama-1.1b", 22, bf16, requests, rng.randint(max(1, longest // 2), longest), longest, rng.randint(24, 64))
    if kind in (3, 4):                                      # prompts, whole
        requests = rng.choice((1, 1, 2, 3))
        longest = _spread(rng, 20, 2000)
        return _traffic(None, "tinyllama-1.1b", 22, bf16, requests, rng.randint(max(1, longest // 4), longest), longest, rng.randint(1, 2))
    if kind == 5:                                           # requests that come and go
        longest = _spread(rng, 40, 1000)
        return _traffic(None, "tinyllama-1.1b", 22, bf16, rng.randint(6, 24), rng.randint(8, longest), longest, rng.randint(8, 24),
                        portion=rng.choice((0, 128, 200, 256, 512)), first=rng.randint(1, 6), every=rng.randint(1, 3))
    if kind == 6:
        longest = _spread(rng, 200, 4000)
        return _traffic(None, "llama-3-8b", 8, bf16, rng.randint(1, 7), rng.randint(100, longest), longest, rng.randint(1, 24),
                        portion=rng.choice((0, 256, 512, 1000)))
    if kind == 7:
        requests = _spread(rng, 1, 16)
        longest = _spread(rng, 100, 1000)
        return _traffic(None, "llama-2-7b", 8, bf16, requests, rng.randint(longest // 2, longest), longest, rng.randint(8, 32))
    if kind == 8:
        longest = _spread(rng, 8, 1000)
        requests = max(1, min(_spread(rng, 1, 16), 1000 // longest))
        return _traffic(None, "tinyllama-1.1b", 22, f32, requests, rng.randint(max(1, longest // 2), longest), longest, rng.randint(1, 24),
                        portion=rng.choice((0, 0, 256)))
    if kind == 9:
        requests = _spread(rng, 1, 16)
        longest = _spread(rng, 16, 800)
        return _traffic(None, "mamenex-2k", 6, bf16, requests, rng.randint(max(1, longest // 2), longest), longest, rng.randint(1, 40))
    return dict(kind="choose", rows=_spread(rng, 1, 128), vocab=rng.choice((32000, 128256, rng.randint(1000, 128000))))


# --- what a pass is made of ----------------------------------------------------------

def _config(case):
    raw = dict(MODELS[case["model"]])
    if raw.get("architecture") == "Mamenex":
        raw["layers"] = [MAMENEX_RECURRENT if i % 3 == 0 else MAMENEX_ATTENTION for i in range(case["layers"])]
    else:
        raw["num_hidden_layers"] = case["layers"]
    return raw


def _vocab(case):
    raw = MODELS[case["model"]]
    return raw.get("vocab_size") or raw["vocab"]


def _lengths(case, seed):
    """Prompt lengths: both ends of the range, the rest spread between."""
    rng = random.Random(seed * 7 + 3)
    n = case["requests"]
    got = [case["longest"], case["shortest"]][:n] + [rng.randint(case["shortest"], case["longest"]) for _ in range(n - 2)]
    rng.shuffle(got)
    return got


def _ids(case, seed):
    """Every request's ids: its prompt and the new - 1 tokens that stand for chosen ones."""
    rng = random.Random(seed * 11 + 5)
    vocab = _vocab(case)
    return [[rng.randrange(vocab) for _ in range(n + case["new"] - 1)] for n in _lengths(case, seed)]


def _steps(case, lengths):
    """The steps of a pass: (requests admitted before it, [(request, from, to, whether its last place's logits are wanted)],
    requests that end with it)."""
    new, portion = case["new"], case["portion"]
    at, waiting, live, steps = {}, list(range(len(lengths))), [], []
    while waiting or live:
        n = len(steps)
        due = case["first"] + (n // case["every"] if case["every"] else 0) - (len(lengths) - len(waiting))
        come, waiting = waiting[:max(due, 0)], waiting[max(due, 0):]
        live = live + come
        at.update((r, 0) for r in come)
        entries, gone = [], []
        for r in live:
            a, end = at[r], lengths[r]
            b = a + 1 if a >= end else min(end, a + portion) if portion else end
            entries.append((r, a, b, b >= end))
            at[r] = b
            if b == end + new - 1:
                gone.append(r)
        live = [r for r in live if r not in gone]
        steps.append((come, entries, gone))
    return steps


def _weight_shapes(case):
    """[(name, shape, scale, offset)] of the model's tensors: matrices N(0, 0.02), norms near 1, as configured models have them."""
    raw = _config(case)
    out = []
    mat = lambda name, *shape: out.append((name, shape, 0.02, 0.0))      # noqa: E731
    if "layers" not in raw:
        h, d, f = raw["hidden_size"], raw["head_dim"], raw["intermediate_size"]
        q, kv = raw["num_attention_heads"] * d, raw["num_key_value_heads"] * d
        norm = lambda name: out.append((name, (h,), 0.1, 1.0))      # noqa: E731
        mat("model.embed_tokens.weight", raw["vocab_size"], h)
        for i in range(case["layers"]):
            p = "model.layers.%d." % i
            norm(p + "input_layernorm.weight")
            for name, shape in (("q", (q, h)), ("k", (kv, h)), ("v", (kv, h)), ("o", (h, q))):
                mat(p + "self_attn.%s_proj.weight" % name, *shape)
            norm(p + "post_attention_layernorm.weight")
            for name, shape in (("gate", (f, h)), ("up", (f, h)), ("down", (h, f))):
                mat(p + "mlp.%s_proj.weight" % name, *shape)
        norm("model.norm.weight")
        if not raw["tie_word_embeddings"]:
            mat("lm_head.weight", raw["vocab_size"], h)
        return out
    w = raw["width"]
    vec = lambda name, *shape: out.append((name, shape, 0.1, 0.0))      # noqa: E731
    mat("embed", raw["vocab"], w)
    for i, layer in enumerate(raw["layers"]):
        p, m = "l%d." % i, layer["mixer"]
        vec(p + "norm1", w), vec(p + "norm1b", w), out.append((p + "canon1", (w, raw["canon"]["taps"]), 0.3, 0.0))
        if layer["type"] == "latent_attention":
            H = m["heads"]
            mat(p + "mix.q", H * (m["dim"] + m["rot_dim"]), w), mat(p + "mix.dkv", m["kv_rank"] + m["rot_dim"], w)
            out.append((p + "mix.dkv.norm", (m["kv_rank"],), 0.1, 1.0))
            mat(p + "mix.uk", H * m["dim"], m["kv_rank"]), mat(p + "mix.uv", H * m["vdim"], m["kv_rank"])
            mat(p + "mix.o", w, H * m["vdim"]), vec(p + "mix.sink", H)
        else:
            W, B = m["width"], m["blocks"]
            for name in ("y", "x"):
                mat(p + "mix." + name, W, w), vec(p + "mix.%s.b" % name, W)
            out.append((p + "mix.conv", (W, m["conv"]), 0.3, 0.0)), vec(p + "mix.conv.b", W)
            for name in ("ra", "ri"):
                mat(p + "mix." + name, B, W // B, W // B), vec(p + "mix.%s.b" % name, B, W // B)
            vec(p + "mix.lam", W), mat(p + "mix.o", w, W)
        if layer["mlp"] is not None:
            vec(p + "norm2", w), vec(p + "norm2b", w)
            mat(p + "mlp.up", layer["mlp"]["ff"], w), mat(p + "mlp.down", w, layer["mlp"]["ff"]), vec(p + "mlp.act", 2)
    vec("final.norm", w)
    return out


def _weights(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = getattr(torch, case["dtype"])
    out = {}
    for name, shape, scale, offset in _weight_shapes(case):
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, scale, generator=gen)
        out[name] = (t + offset if offset else t).to(dtype)
    return out


# --- the choosing of tokens -------------------------------------------------------------

OPTIONS = (dict(), dict(temperature=0.8), dict(temperature=0.7, top_k=40), dict(temperature=1.0, top_p=0.9),
           dict(temperature=1.2, top_k=100, top_p=0.95))


class _Uniform:
    """A request's generator of uniform numbers, at the number it is about to give."""
    def __init__(self, u):
        self.u = u

    def uniform(self):
        return self.u


def _logits(case, seed):
    """Rows of logits spread as a trained model's: a few ids stand out of a wide rest."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    z = torch.empty(case["rows"], case["vocab"], dtype=torch.float32, device="cuda").normal_(0.0, 2.0, generator=gen)
    rng = random.Random(seed * 13 + 1)
    return z, [OPTIONS[i % 5] for i in range(case["rows"])], [rng.random() for _ in range(case["rows"])]


# --- a pass -----------------------------------------------------------------------------

def prepare(case, seed):
    if case["kind"] == "choose":
        from bare_cuda_4gib_amd.sampling import DevicePicker, SamplingParams
        logits, options, us = _logits(case, seed)
        return dict(kind="choose", picker=DevicePicker(), logits=logits, params=[SamplingParams(**o) for o in options],
                    rngs=[_Uniform(u) for u in us])
    from bare_cuda_4gib_amd.config import architecture_for
    from bare_cuda_4gib_amd.engine import Executor, Model, Runtime, StepEntry, parse_dtype
    raw = _config(case)
    arch = architecture_for(raw)
    model = Model(arch.describe(arch.config_class.from_dict(raw)))
    model.bind(_weights(case, seed), Runtime(torch.device("cuda:0"), parse_dtype(case["dtype"])))
    lengths, ids = _lengths(case, seed), _ids(case, seed)
    pages = [-(-len(x) // PAGE) for x in ids]
    most = max(max(len(x) for x in ids), min(max(pages) * PAGE, model.max_seq_len))
    executor = Executor(model, num_pages=sum(pages), max_requests=len(ids), max_tokens=most, page_tokens=PAGE)
    steps = [(come, [StepEntry(r, ids[r][a:b], [b - a - 1] if want else []) for r, a, b, want in entries], gone)
             for come, entries, gone in _steps(case, lengths)]
    rows = sum(len(e.want) for _, entries, _ in steps for e in entries)
    return dict(kind="traffic", executor=executor, steps=steps, logits=torch.empty(rows, model.vocab_size, device="cuda"))


def run(state):
    if state["kind"] == "choose":
        return state["picker"].pick(state["logits"], state["params"], state["rngs"])
    executor, out, n = state["executor"], state["logits"], 0
    for come, entries, gone in state["steps"]:
        for r in come:
            executor.admit(r)
        logits = executor.step(entries)
        if logits is not None:                      # (a later step may write the same buffer)
            out[n:n + logits.shape[0]].copy_(logits)
            n += logits.shape[0]
        for r in gone:
            executor.release(r)
    return out


# --- what a pass cannot do without --------------------------------------------------------

def work(case):
    """Per step: the weights it uses read once, the cache of its requests read once, its logits written; the operations of
    its rows. (Lengths at the middle of the case's range.)"""
    if case["kind"] == "choose":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 0.0}
    raw, elem = _config(case), 2 if case["dtype"] == "bfloat16" else 4
    shapes = {name: math.prod(shape) for name, shape, _, _ in _weight_shapes(case)}
    vocab = _vocab(case)
    width = raw.get("hidden_size") or raw["width"]
    head = vocab * width
    table = "model.embed_tokens.weight" if "layers" not in raw else "embed"
    body = sum(n for name, n in shapes.items() if name not in (table, "lm_head.weight"))
    if "layers" not in raw:
        kv = 2 * raw["num_key_value_heads"] * raw["head_dim"] * case["layers"]                      # values a token
        pair = 4 * raw["num_attention_heads"] * raw["head_dim"] * case["layers"]                    # operations a (query, key)
    else:
        at = [layer["mixer"] for layer in raw["layers"] if layer["type"] == "latent_attention"]
        kv = sum(m["kv_rank"] + m["rot_dim"] for m in at)
        pair = sum(2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]) for m in at)
    lengths = [round(case["shortest"] + (case["longest"] - case["shortest"]) * (i + 0.5) / case["requests"]) for i in range(case["requests"])]
    nbytes = flops = 0.0
    for _, entries, _ in _steps(case, lengths):
        rows = sum(b - a for _, a, b, _ in entries)
        wanted = sum(1 for e in entries if e[3])
        nbytes += elem * (body + (head if wanted else 0) + rows * width + kv * sum(b for _, _, b, _ in entries)) + 4.0 * wanted * vocab
        flops += 2.0 * (rows * body + wanted * head) + pair * sum((b - a) * (a + b + 1) / 2 for _, a, b, _ in entries)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "choose":
        return {"rel": 0.0, "differ": 0.01}         # an id may turn where a sum ends within a rounding of the drawn number
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "max": 3e-4}
    return {"rel": 0.03, "max": 0.3}


# --- the same in 64 bits, from the equations -------------------------------------------------

def exact(case, seed):
    if case["kind"] == "choose":
        return _exact_choice(case, seed)
    lengths, ids = _lengths(case, seed), _ids(case, seed)
    weights = _weights(case, seed)
    stack = _exact_mamenex if "layers" in _config(case) else _exact_llama
    wanted = [list(range(n - 1, len(x))) for n, x in zip(lengths, ids)]
    logits = stack(case, weights, ids, wanted)      # per request [new, vocab]
    taken = [0] * len(ids)
    rows = []
    for _, entries, _ in _steps(case, lengths):
        for r, _, _, want in entries:
            if want:
                rows.append(logits[r][taken[r]])
                taken[r] += 1
    return torch.stack(rows)


def _exact_choice(case, seed):
    z, options, us = _logits(case, seed)
    got = []
    for row, o, u in zip(z.double(), options, us):
        if not o:
            got.append(int(row.argmax()))
            continue
        w = torch.exp((row - row.max()) / o["temperature"])
        kept = torch.arange(w.numel(), device=w.device)
        if "top_k" in o or "top_p" in o:
            kept = torch.sort(w, descending=True, stable=True).indices[:o.get("top_k") or w.numel()]
            mass = torch.cumsum(w[kept], 0)
            if "top_p" in o:
                kept = kept[:min(int((mass < o["top_p"] * mass[-1]).sum()) + 1, kept.numel())]
        mass = torch.cumsum(w[kept], 0)
        got.append(int(kept[min(int((mass <= u * mass[-1]).sum()), kept.numel() - 1)]))
    return got


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _angles(n, dims, base):
    t = torch.arange(n, dtype=torch.float64, device="cuda")[:, None]
    return t * base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)[None, :]


def _attend(q, k, v, scale, sink=None):
    """q [H, T, d], k [G, T, d], v [G, T, e]: causal softmax attention, with a sink's weight in the sum. [T, H, e]"""
    H, T, _ = q.shape
    out = torch.empty(T, H, v.shape[2], dtype=torch.float64, device="cuda")
    hidden = torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1)
    for h in range(H):
        g = h * k.shape[0] // H
        s = ((q[h] @ k[g].T) * scale).masked_fill_(hidden, -math.inf)
        norm = torch.logsumexp(s, -1, keepdim=True)
        if sink is not None:
            norm = torch.logaddexp(norm, sink[h])
        out[:, h] = torch.exp(s - norm) @ v[g]
    return out


def _in_rows(ids):
    """All requests' rows one after the other, and where each request's lie."""
    ends = torch.tensor([0] + [len(x) for x in ids]).cumsum(0).tolist()
    return torch.tensor([t for x in ids for t in x], device="cuda"), list(zip(ends, ends[1:]))


def _exact_llama(case, weights, ids, wanted):
    raw = _config(case)
    H, G, d, eps = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"], raw["rms_norm_eps"]
    flat, places = _in_rows(ids)
    x = weights["model.embed_tokens.weight"][flat].double()
    angles = _angles(max(len(r) for r in ids), d, raw["rope_theta"])
    cos, sin = torch.cos(angles), torch.sin(angles)

    def turned(u):                                  # [heads, T, d]: element i is paired with i + d / 2
        a, b = u[..., :d // 2], u[..., d // 2:]
        c, s = cos[:u.shape[1]], sin[:u.shape[1]]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    for i in range(case["layers"]):
        w = {n: weights["model.layers.%d.%s.weight" % (i, n)].double() for n in (
            "input_layernorm", "post_attention_layernorm", "self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj",
            "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")}
        h = _rms(x, eps) * w["input_layernorm"]
        q, k, v = (h @ w["self_attn.%s_proj" % n].T for n in "qkv")
        o = torch.empty_like(q)
        for a, b in places:
            qr, kr, vr = (u[a:b].view(b - a, -1, d).transpose(0, 1) for u in (q, k, v))
            o[a:b] = _attend(turned(qr), turned(kr), vr, d ** -0.5).reshape(b - a, H * d)
        x = x + o @ w["self_attn.o_proj"].T
        h = _rms(x, eps) * w["post_attention_layernorm"]
        x = x + (torch.nn.functional.silu(h @ w["mlp.gate_proj"].T) * (h @ w["mlp.up_proj"].T)) @ w["mlp.down_proj"].T
    head = weights["model.embed_tokens.weight" if raw["tie_word_embeddings"] else "lm_head.weight"].double()
    out = []
    for (a, b), want in zip(places, wanted):
        rows = x[a:b][torch.tensor(want, device="cuda")]
        out.append((_rms(rows, eps) * weights["model.norm.weight"].double()) @ head.T)
    return out


def _convolved(u, w, places):
    """u [rows, C], w [C, taps]: a causal convolution over each request's rows; the last tap is the row's own."""
    out = torch.zeros_like(u)
    taps = w.shape[1]
    for a, b in places:
        for j in range(taps):
            back = taps - 1 - j
            if back < b - a:
                out[a + back:b] += u[a:b - back] * w[:, j]
    return out


def _exact_mamenex(case, weights, ids, wanted):
    raw = _config(case)
    eps = raw["norm"]["eps"]
    W = {n: t.double() for n, t in weights.items()}
    flat, places = _in_rows(ids)
    x = W["embed"][flat]
    longest = max(len(r) for r in ids)
    normed = lambda u, name: _rms(u, eps) * (1.0 + W[name])      # noqa: E731
    softplus = torch.nn.functional.softplus
    for i, layer in enumerate(raw["layers"]):
        p, m = "l%d." % i, layer["mixer"]
        h = normed(x, p + "norm1")
        h = h + _convolved(h, W[p + "canon1"], places)
        if layer["type"] == "latent_attention":
            H, n, r, rank = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
            angles = _angles(longest, r, m["rot"]["base"])

            def turned(u):                          # [T, ..., r]: neighbours are paired
                c, s = (f(angles[:u.shape[0]]).view([u.shape[0]] + [1] * (u.dim() - 2) + [r // 2]) for f in (torch.cos, torch.sin))
                a, b = u[..., 0::2], u[..., 1::2]
                return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)

            q, dkv = (h @ W[p + "mix.q"].T).view(-1, H, n + r), h @ W[p + "mix.dkv"].T
            latent = _rms(dkv[:, :rank], eps) * W[p + "mix.dkv.norm"]
            k, v = (latent @ W[p + "mix.uk"].T).view(-1, H, n), (latent @ W[p + "mix.uv"].T).view(-1, H, m["vdim"])
            y = torch.empty(x.shape[0], H * m["vdim"], dtype=torch.float64, device="cuda")
            for a, b in places:
                qr = torch.cat([q[a:b, :, :n], turned(q[a:b, :, n:])], -1).transpose(0, 1)
                kr = torch.cat([k[a:b], turned(dkv[a:b, rank:])[:, None].expand(-1, H, -1)], -1).transpose(0, 1)
                y[a:b] = _attend(qr, kr, v[a:b].transpose(0, 1), m["scale"], W[p + "mix.sink"]).reshape(b - a, -1)
        else:
            width, blocks = m["width"], m["blocks"]
            gate = torch.nn.functional.gelu(h @ W[p + "mix.y"].T + W[p + "mix.y.b"], approximate="tanh")
            u = _convolved(h @ W[p + "mix.x"].T + W[p + "mix.x.b"], W[p + "mix.conv"], places) + W[p + "mix.conv.b"]
            ub = u.view(-1, blocks, width // blocks).transpose(0, 1)
            r, g = (torch.sigmoid((torch.stack([ub[b] @ W[p + "mix." + n][b].T for b in range(blocks)], 1) + W[p + "mix.%s.b" % n])
                                  .reshape(-1, width)) for n in ("ra", "ri"))
            decay = torch.exp(-8.0 * r * softplus(W[p + "mix.lam"]))
            into = torch.sqrt(1.0 - decay * decay) * g * u
            y = torch.empty_like(u)
            for a, b in places:
                state = torch.zeros(width, dtype=torch.float64, device="cuda")
                for t in range(a, b):
                    state = decay[t] * state + into[t]
                    y[t] = state
            y = y * gate
        x = x + normed(y @ W[p + "mix.o"].T, p + "norm1b")
        if layer["mlp"] is not None:
            z, act = normed(x, p + "norm2") @ W[p + "mlp.up"].T, softplus(W[p + "mlp.act"])
            z = torch.where(z > 0, act[0] * z * z, (0.5 + act[1]) * (torch.expm1(z.clamp(max=0.0)) - z)) + z / 2
            x = x + normed(z @ W[p + "mlp.down"].T, p + "norm2b")
    return [normed(x[a:b][torch.tensor(want, device="cuda")], "final.norm") @ W["embed"].T for (a, b), want in zip(places, wanted)]
