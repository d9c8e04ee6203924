"""What this library's speed is measured at: requests as its users send them, through the step function.

A case is a model and one batch of requests: `batch` prompts of lo..hi tokens that start together in one prompt step, then
`steps` decode steps of one token each, then the sequences are released.  A pass is the whole of that on sequences of its
own (new_sequence, step, step(device_tokens=...), release), so every pass does the same work.  The decoded tokens are given
(as a scorer gives them, and so that two implementations whose logits differ by a rounding stay on the same sequence); they
lie on the device, where a sampler leaves them.  The logits of every wanted place come back.

The models are the benchmark's own configurations (the 8B shape, and the designs at width 2,048 with 12 layers) and the
smallest one of the tests, with random weights made on the device: matrices N(0, 0.02), a half's last matrix by 1 / sqrt(2
layers) less and embedding rows N(0, 1) so that a layer changes the stream by a share, as in a trained model, instead of
replacing it (which would amplify every rounding from layer to layer), norm weights 1, what has a range of its own (decays,
shifts, biases over distance) inside that range.  Mixtures of experts are not among them: with random
routers many choices are near ties, and two correct bf16 implementations then choose differently by more than any
tolerance on their outputs allows.
"""
import math
import random

import torch

DEV = "cuda:0"
F64 = torch.float64

LLAMA_8B = dict(model_type="llama", vocab_size=128256, hidden_size=4096, intermediate_size=14336, num_hidden_layers=32,
                num_attention_heads=32, num_key_value_heads=8, head_dim=128, max_position_embeddings=131072,
                rope_theta=500000.0, rms_norm_eps=1e-5, tie_word_embeddings=False,
                rope_scaling=dict(rope_type="llama3", factor=8.0, low_freq_factor=1.0, high_freq_factor=4.0,
                                  original_max_position_embeddings=8192))
LLAMA_2048 = dict(model_type="llama", vocab_size=32000, hidden_size=2048, intermediate_size=5632, num_hidden_layers=12,
                  num_attention_heads=16, num_key_value_heads=4, head_dim=128, max_position_embeddings=8192,
                  rope_theta=500000.0, rms_norm_eps=1e-5, tie_word_embeddings=False)
LLAMA_TINY = dict(model_type="llama", vocab_size=256, hidden_size=64, intermediate_size=172, num_hidden_layers=2,
                  num_attention_heads=4, num_key_value_heads=2, head_dim=16, max_position_embeddings=512,
                  rope_theta=10000.0, rms_norm_eps=1e-5, tie_word_embeddings=False)


def _sunusun():
    wkv = dict(type="wkv", mixer=dict(heads=32, dim=64, decay_rank=64), mlp=dict(kind="dense", ff=8192))
    par = dict(type="parallel", mlp=dict(kind="dense", ff=8192), mixer=dict(
        left=dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=128 ** -0.5, q_temp=dict(coef=0.1, every=256)),
        right=dict(width=2048)))
    return dict(architecture="Sunusun", vocab=32000, width=2048, norm=dict(eps=1e-6), logit_scale=1.0,
                layers=[par if i % 3 == 2 else wkv for i in range(12)])


def _fazopel():
    lin = dict(heads=16, dim=128, vdim=128, decay=[round(1.0 - 2.0 ** -(5.0 + 3.0 * h / 15), 9) for h in range(16)])
    att = dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=128 ** -0.5, rot=dict(base=500000.0, dims=64))
    mlp = dict(kind="dense", ff=8192)
    return dict(architecture="Fazopel", vocab=32000, width=2048, norm=dict(eps=1e-6),
                layers=[dict(type="attention", mixer=att, mlp=mlp) if i % 3 == 2 else dict(type="lightning", mixer=lin, mlp=mlp)
                        for i in range(12)])


MODELS = {"llama-8b": LLAMA_8B, "llama-2048": LLAMA_2048, "llama-tiny": LLAMA_TINY, "sunusun-2048": _sunusun(),
          "fazopel-2048": _fazopel()}


# ---- the cases -----------------------------------------------------------------------------------------------------

def _case(model, dtype, batch, lo, hi, steps, want=1, name=None):
    c = dict(model=model, dtype=dtype, batch=batch, lo=lo, hi=hi, steps=steps, want=want)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest model there is: launches and host work alone
        _case("llama-tiny", "float32", 1, 5, 5, 16, name="tiny-f32-b1"),
        # one user, one short question, a short answer: what a chat waits for
        _case("llama-8b", "bfloat16", 1, 24, 24, 32, name="8b-chat-b1"),
        # a few users of unequal, odd prompt lengths whose answers are a few words (classification, tool calls)
        _case("llama-8b", "bfloat16", 3, 37, 301, 6, name="8b-short-b3"),
        # the benchmark's batch and prompt lengths
        _case("llama-8b", "bfloat16", 8, 128, 2048, 32, name="8b-serve-b8"),
        # a full batch of shorter prompts: throughput serving
        _case("llama-8b", "bfloat16", 64, 16, 512, 32, name="8b-serve-b64"),
        # a prompt of 2,048 tokens and its first token: time to first token, the benchmark's prefill
        _case("llama-8b", "bfloat16", 1, 2048, 2048, 0, name="8b-prefill-2048"),
        # a long document and a short summary of it
        _case("llama-8b", "bfloat16", 1, 8100, 8100, 16, name="8b-document-b1"),
        # a small model, where launches count, with logits at several places of every prompt (scoring of continuations)
        _case("llama-2048", "bfloat16", 4, 70, 500, 24, want=48, name="2048-score-b4"),
        # float32, the reference precision: one sequence replayed token by token
        _case("llama-2048", "float32", 1, 199, 199, 16, name="2048-f32-b1"),
        # float32: a batch of prompts and the first tokens of their continuations
        _case("llama-2048", "float32", 8, 64, 1024, 8, name="2048-f32-b8"),
        # a recurrent design: a long prompt and a short continuation
        _case("sunusun-2048", "bfloat16", 1, 2048, 2048, 16, name="sunusun-b1"),
        # linear attention beside attention with a sink: a small batch of unequal prompts
        _case("fazopel-2048", "bfloat16", 4, 100, 1500, 24, name="fazopel-b4"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    model, dtype, batches, tokens, longest = rng.choice([
        ("llama-8b", "bfloat16", 64, 16000, 8100), ("llama-8b", "bfloat16", 64, 16000, 8100),
        ("llama-8b", "bfloat16", 64, 16000, 8100), ("llama-2048", "bfloat16", 32, 16000, 8000),
        ("llama-2048", "float32", 16, 4000, 2048), ("sunusun-2048", "bfloat16", 16, 8000, 4096),
        ("fazopel-2048", "bfloat16", 16, 8000, 4096), ("llama-tiny", "float32", 8, 3000, 480)])
    batch = _log_int(rng, 1, batches)
    hi = _log_int(rng, 2, min(longest, tokens // batch))
    lo = _log_int(rng, 2, hi)
    steps = rng.randint(0, 32)
    want = rng.choice([1, 1, 1, min(lo, 256 // batch)])
    return _case(model, dtype, batch, lo, hi, steps, want)


def _lengths(case):
    """The prompts' lengths, a function of the case alone."""
    rnd = random.Random(f"{case['batch']} {case['lo']} {case['hi']}")
    return [rnd.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


# ---- what a pass needs at the least -----------------------------------------------------------------------------------

def _is_llama(raw):
    return raw.get("model_type") == "llama"


def _tensors(raw):
    """name -> (shape, how it is drawn) of every tensor of the model folder."""
    t = {}

    def mat(name, *shape):
        t[name] = (shape, "matrix")

    if _is_llama(raw):
        D, F, V, d = raw["hidden_size"], raw["intermediate_size"], raw["vocab_size"], raw["head_dim"]
        Q, G = raw["num_attention_heads"] * d, raw["num_key_value_heads"] * d
        mat("model.embed_tokens.weight", V, D)
        mat("lm_head.weight", V, D)
        t["model.norm.weight"] = ((D,), "one")
        for i in range(raw["num_hidden_layers"]):
            p = f"model.layers.{i}."
            t[p + "input_layernorm.weight"] = t[p + "post_attention_layernorm.weight"] = ((D,), "one")
            mat(p + "self_attn.q_proj.weight", Q, D)
            mat(p + "self_attn.k_proj.weight", G, D)
            mat(p + "self_attn.v_proj.weight", G, D)
            mat(p + "self_attn.o_proj.weight", D, Q)
            mat(p + "mlp.gate_proj.weight", F, D)
            mat(p + "mlp.up_proj.weight", F, D)
            mat(p + "mlp.down_proj.weight", D, F)
        return t
    D, V, sun = raw["width"], raw["vocab"], raw["architecture"] == "Sunusun"
    mat("embed", V, D)
    mat("head", V, D)
    t["final.norm"] = (() if sun else (D,), "one")
    for i, L in enumerate(raw["layers"]):
        p, m = f"l{i}.", L["mixer"]
        t[p + "norm1"] = t[p + "norm2"] = (() if sun else (D,), "one")
        mat(p + "mlp.up", L["mlp"]["ff"], D)
        mat(p + "mlp.down", D, L["mlp"]["ff"])
        if L["type"] == "wkv":
            W, r = m["heads"] * m["dim"], m["decay_rank"]
            for s in "rkvgw":
                t[p + "mix.mu." + s] = ((D,), "share")
            for s in "rkvg":
                mat(p + "mix." + s, W, D)
            mat(p + "mix.w1", r, D)
            mat(p + "mix.w2", W, r)
            t[p + "mix.w0"] = ((W,), "decay")
            t[p + "mix.u"] = ((m["heads"], m["dim"]), "bonus")
            t[p + "mix.norm"] = ((W,), "one")
            mat(p + "mix.o", D, W)
        elif L["type"] == "parallel":
            a, W = m["left"], m["right"]["width"]
            q = p + "mix.left."
            mat(q + "q", a["heads"] * a["dim"], D)
            mat(q + "k", a["kv_heads"] * a["dim"], D)
            mat(q + "v", a["kv_heads"] * a["vdim"], D)
            mat(q + "o", D, a["heads"] * a["vdim"])
            t[q + "q.norm"] = t[q + "k.norm"] = ((a["dim"],), "one")
            t[q + "r1"] = t[q + "r2"] = ((a["heads"],), "share")
            t[q + "out"] = t[p + "mix.right.out"] = ((D,), "one")
            for s in "zxg":
                mat(p + "mix.right." + s, W, D)
            mat(p + "mix.right.o", D, W)
            t[p + "mix.right.z.b"] = t[p + "mix.right.x.b"] = ((W,), "bias")
        elif L["type"] == "lightning":
            for s, n in (("q", m["dim"]), ("k", m["dim"]), ("v", m["vdim"]), ("g", m["vdim"])):
                mat(p + "mix." + s, m["heads"] * n, D)
            mat(p + "mix.o", D, m["heads"] * m["vdim"])
            t[p + "mix.norm"] = ((m["heads"] * m["vdim"],), "one")
        else:
            mat(p + "mix.q", m["heads"] * m["dim"], D)
            mat(p + "mix.k", m["kv_heads"] * m["dim"], D)
            mat(p + "mix.o", D, m["heads"] * m["dim"])
            t[p + "mix.q.norm"] = t[p + "mix.k.norm"] = ((m["dim"],), "one")
    return t


def _attention_layers(raw):
    """(layers with attention, query heads, numbers cached a token and layer, head size, elements of state of a sequence)."""
    if _is_llama(raw):
        return raw["num_hidden_layers"], raw["num_attention_heads"], 2 * raw["num_key_value_heads"] * raw["head_dim"], raw["head_dim"], 0
    n, H, kv, d, state = 0, 0, 0, 0, 0
    for L in raw["layers"]:
        m = L["mixer"].get("left", L["mixer"])
        if L["type"] in ("attention", "parallel"):
            n, H, d = n + 1, m["heads"], m["dim"]
            kv = (1 if L["type"] == "attention" else 2) * m["kv_heads"] * d      # the values of the first are its keys
            state += L["mixer"]["right"]["width"] if L["type"] == "parallel" else 0
        else:
            state += m["heads"] * m["dim"] * m.get("vdim", m["dim"])
    return n, H, kv, d, state


def work(case):
    """Every matrix once a step (they do not fit into any cache between two steps), the cached keys and values that a step's
    tokens see once, the recurrent states read and written, the logits written; twice the multiply-adds of the products, of
    attention's and of the recurrences'."""
    raw, size = MODELS[case["model"]], 2 if case["dtype"] == "bfloat16" else 4
    lens, B, n = _lengths(case), case["batch"], case["steps"]
    V, D = (raw["vocab_size"], raw["hidden_size"]) if _is_llama(raw) else (raw["vocab"], raw["width"])
    layer_params = sum(math.prod(s) for s, kind in _tensors(raw).values() if kind == "matrix") - 2 * V * D
    layers, H, kv, d, state = _attention_layers(raw)
    tokens = sum(lens) + n * B
    rows = B * case["want"] + n * B
    seen_prompt = sum(lens)                                    # keys that a step reads, each once
    seen_decode = sum(L * n + n * (n + 1) // 2 for L in lens)
    pairs = sum((L + n) * (L + n + 1) // 2 for L in lens)      # (query, key) pairs
    return {"bytes": (n + 1) * (layer_params + V * D) * size + (seen_prompt + seen_decode) * layers * kv * size
            + 8 * state * B * (n + 1) + rows * V * 4 + tokens * D * size,
            "flops": 2.0 * tokens * layer_params + 2.0 * rows * V * D + 4.0 * pairs * H * d * layers + 4.0 * tokens * state}


def tolerance(case):
    """Four times what correct forms of the path differ by: bf16 up to 8e-3 from 64 bits, and 1e-2 between products summed and
    rounded in other places (the library's or this library's, norms folded in or not); float32 1.2e-6 from 64 bits."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 3e-2, "max": 0.2}


# ---- a pass ----------------------------------------------------------------------------------------------------------

LAST_OF_A_HALF = (".o", ".down", "o_proj.weight", "down_proj.weight")


def _draw_tensor(name, shape, kind, layers, gen, dtype):
    if kind == "one":
        return torch.ones(shape, dtype=torch.float32, device=DEV)
    if kind == "matrix":
        std = 1.0 if "embed" in name else 0.02 * (2 * layers) ** -0.5 if name.endswith(LAST_OF_A_HALF) else 0.02
        return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, std, generator=gen).to(dtype)
    t = torch.empty(shape, dtype=torch.float32, device=DEV).uniform_(0.0, 1.0, generator=gen)
    lo, hi = {"share": (0.02, 1.0), "decay": (-6.0, -1.0), "bonus": (-0.5, 0.5), "bias": (-1.0, 1.0)}[kind]
    return lo + (hi - lo) * t


def _inputs(case, seed):
    """(weights on the device, prompts as token lists, the decoded tokens [steps, batch])."""
    raw = MODELS[case["model"]]
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    gen = torch.Generator(device=DEV).manual_seed(seed)
    vocab, layers = (raw["vocab_size"], raw["num_hidden_layers"]) if _is_llama(raw) else (raw["vocab"], len(raw["layers"]))
    weights = {name: _draw_tensor(name, shape, kind, layers, gen, dtype) for name, (shape, kind) in _tensors(raw).items()}
    rnd = random.Random(seed)
    prompts = [[rnd.randrange(vocab) for _ in range(n)] for n in _lengths(case)]
    given = [[rnd.randrange(vocab) for _ in range(case["batch"])] for _ in range(case["steps"])]
    return weights, prompts, given


def prepare(case, seed):
    """The loaded model with its cache, warmed up as a server warms up for the sizes that it expects."""
    import bitnet_c_amd as bn
    from bitnet_c_amd.config import architecture_for
    from bitnet_c_amd.engine import DecoderModel
    raw = MODELS[case["model"]]
    weights, prompts, given = _inputs(case, seed)
    arch = architecture_for(raw)
    plan = arch.build_plan(arch.config_cls.from_dict(raw))
    model = DecoderModel(plan, torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32, DEV)
    model.load(weights)
    del weights
    torch.cuda.empty_cache()
    lens, B, want = _lengths(case), case["batch"], case["want"]
    per_seq = -(-(max(lens) + case["steps"] + 1) // 64) * 64
    engine = bn.Engine(model, max_tokens=max(B * per_seq, 256), max_seq_len=per_seq, max_slots=B + 1)
    llm = bn.LLM(engine)
    if case["steps"] > 0:
        engine.prepare_decode(B)
    slots = [llm.new_sequence() for _ in lens]
    llm.step([bn.StepEntry(s, p, range(len(p) - want, len(p))) for s, p in zip(slots, prompts)])
    for s in slots:
        llm.release(s)
    if max(lens) > 1:
        engine.prepare_prompt(sum(lens), B, B * want)
    return dict(llm=llm, entry=bn.StepEntry, prompts=prompts, want=want,
                given=[torch.tensor(g, dtype=torch.int32, device=DEV) for g in given])


def run(state):
    llm, entry, want = state["llm"], state["entry"], state["want"]
    slots = [llm.new_sequence() for _ in state["prompts"]]
    try:
        first = llm.step([entry(s, p, range(len(p) - want, len(p))) for s, p in zip(slots, state["prompts"])])
        entries = [entry(s, [0], [0]) for s in slots]
        later = [llm.step(entries, device_tokens=tokens) for tokens in state["given"]]
    finally:
        for s in slots:
            llm.release(s)
    return {"prompt": first, "decoded": torch.stack(later)} if later else {"prompt": first}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------
# Positions, frequencies and the angle p * f are 32-bit numbers by the models' definition; everything after that is not.

def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _frequencies(base, dims, scaling=None):
    f = base ** (-2.0 * torch.arange(dims // 2, dtype=F64) / dims)
    if scaling:
        wave = 2.0 * math.pi / f
        orig, low, high = (float(scaling[k]) for k in ("original_max_position_embeddings", "low_freq_factor", "high_freq_factor"))
        s = (orig / wave - low) / (high - low)
        f = torch.where(wave < orig / high, f, torch.where(wave > orig / low, f / scaling["factor"],
                                                          (1.0 - s) * f / scaling["factor"] + s * f))
    return f.to(torch.float32).to(DEV)


def _rotate(x, pos, freq):
    """x [T, heads, d]: dimension i turns with dimension i + n, n frequencies; the rest passes."""
    n = freq.numel()
    a = (pos.to(torch.float32)[:, None] * freq[None, :]).to(F64)[:, None, :]
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * torch.cos(a) - v * torch.sin(a), v * torch.cos(a) + u * torch.sin(a), x[..., 2 * n:]], dim=-1)


def _attend(q, k, v, scale, sink, bias=None):
    """Causal attention of one sequence, a head at a time: q [T, H, d], k, v [T, G, .]; bias: (a, b) per head."""
    T, H = q.shape[:2]
    out = torch.empty(T, H, v.shape[-1], dtype=F64, device=DEV)
    pos = torch.arange(T, device=DEV)
    hidden = pos[:, None] < pos[None, :]
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h].contiguous() @ k[:, g].t().contiguous()) * scale
        if bias is not None:
            s -= bias[0][h] * torch.log1p(bias[1][h] * (pos[:, None] - pos[None, :]).clamp(min=0))
        s.masked_fill_(hidden, -math.inf)
        top = s.max(dim=-1, keepdim=True).values
        if sink:
            top = top.clamp(min=0.0)
        e = torch.exp(s - top)
        z = e.sum(dim=-1, keepdim=True) + (torch.exp(-top) if sink else 0.0)
        out[:, h] = (e @ v[:, g].contiguous()) / z
    return out.reshape(T, -1)


class _Rows:
    """The tokens of all sequences one after another, and the same with a row of its own for every sequence."""

    def __init__(self, lens):
        self.lens, self.T = lens, max(lens)
        self.pos = torch.cat([torch.arange(n) for n in lens]).to(DEV)
        self.place = torch.cat([b * self.T + torch.arange(n) for b, n in enumerate(lens)]).to(DEV)
        self.cuts = [(sum(lens[:b]), sum(lens[:b + 1])) for b in range(len(lens))]

    def padded(self, x):
        out = torch.zeros((len(self.lens) * self.T,) + x.shape[1:], dtype=F64, device=DEV)
        out[self.place] = x
        return out.view((len(self.lens), self.T) + x.shape[1:])

    def flat(self, x):
        return x.reshape((-1,) + x.shape[2:])[self.place]

    def each(self, fn, *xs):
        return torch.cat([fn(*(x[a:b] for x in xs)) for a, b in self.cuts])


def _llama_layers(raw, W, x, rows):
    d, eps = raw["head_dim"], raw["rms_norm_eps"]
    freq = _frequencies(raw["rope_theta"], d, raw.get("rope_scaling"))
    for i in range(raw["num_hidden_layers"]):
        def w(name):
            return W[f"model.layers.{i}.{name}.weight"].to(F64).t()
        h = _unit(x, eps)
        q, k, v = ((h @ w(f"self_attn.{s}_proj")).view(x.shape[0], -1, d) for s in "qkv")
        q, k = _rotate(q, rows.pos, freq), _rotate(k, rows.pos, freq)
        x = x + rows.each(lambda q, k, v: _attend(q, k, v, d ** -0.5, False), q, k, v) @ w("self_attn.o_proj")
        h = _unit(x, eps)
        x = x + (torch.nn.functional.silu(h @ w("mlp.gate_proj")) * (h @ w("mlp.up_proj"))) @ w("mlp.down_proj")
    return _unit(x, eps)


def _wkv(W, p, m, h, rows, eps):
    H, d = m["heads"], m["dim"]
    hp = rows.padded(h)
    before = rows.flat(torch.cat([torch.zeros_like(hp[:, :1]), hp[:, :-1]], dim=1))
    def w(name):
        return W[p + name].to(F64)
    x = {s: h + (before - h) * w("mu." + s) for s in "rkvgw"}
    r, k, v = (rows.padded((x[s] @ w(s).t()).view(-1, H, d)) for s in "rkv")
    gate = torch.nn.functional.silu(x["g"] @ w("g").t())
    decay = torch.exp(-torch.exp(torch.tanh(x["w"] @ w("w1").t()) @ w("w2").t() + w("w0")))
    decay = rows.padded(decay.view(-1, H, d))
    u = w("u")[None, :, :, None]
    S = torch.zeros(r.shape[0], H, d, d, dtype=F64, device=DEV)
    o = torch.empty_like(r)
    for t in range(rows.T):
        kv = k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = (r[:, t, :, :, None] * (S + u * kv)).sum(dim=2)
        S = decay[:, t, :, :, None] * S + kv
    return (_unit(rows.flat(o), eps).reshape(-1, H * d) * gate) @ w("o").t()


def _parallel(W, p, m, h, rows, eps):
    a, n = m["left"], h.shape[0]
    def w(name):
        return W[p + name].to(F64)
    q = _unit((h @ w("left.q").t()).view(n, a["heads"], a["dim"]), eps)
    k = _unit((h @ w("left.k").t()).view(n, a["kv_heads"], a["dim"]), eps)
    v = (h @ w("left.v").t()).view(n, a["kv_heads"], a["vdim"])
    temp = a["q_temp"]
    turns = torch.div(rows.pos + 1, temp["every"], rounding_mode="floor").to(F64)
    q = q * (1.0 + temp["coef"] * torch.log(turns + 1.0))[:, None, None]
    bias = (w("left.r1"), w("left.r2"))
    left = rows.each(lambda q, k, v: _attend(q, k, v, a["scale"], True, bias), q, k, v) @ w("left.o").t()
    z = rows.padded(torch.sigmoid(h @ w("right.z").t() + w("right.z.b")))
    c = h @ w("right.x").t() + w("right.x.b")
    c = rows.padded(torch.where(c >= 0, c + 0.5, torch.sigmoid(c)))
    S, y = torch.zeros_like(z[:, 0]), torch.empty_like(z)
    for t in range(rows.T):
        S = (1.0 - z[:, t]) * S + z[:, t] * c[:, t]
        y[:, t] = S
    right = (rows.flat(y) * torch.nn.functional.silu(h @ w("right.g").t())) @ w("right.o").t()
    return 0.5 * (_unit(left, eps) + _unit(right, eps))


def _sunusun_layers(raw, W, x, rows):
    eps, D = raw["norm"]["eps"], raw["width"]
    freq = (10000.0 ** (-2.0 * torch.arange((D + 1) // 2, dtype=F64) / D)).to(torch.float32).to(DEV)
    angle = (rows.pos.to(torch.float32)[:, None] * freq[None, :]).to(F64)
    x = x + torch.stack([torch.sin(angle), torch.cos(angle)], dim=-1).reshape(x.shape[0], -1)[:, :D]
    for i, L in enumerate(raw["layers"]):
        mixer = _wkv if L["type"] == "wkv" else _parallel
        x = x + mixer(W, f"l{i}.mix.", L["mixer"], _unit(x, eps), rows, eps)
        a = torch.nn.functional.gelu(_unit(x, eps) @ W[f"l{i}.mlp.up"].to(F64).t())
        x = x + a @ W[f"l{i}.mlp.down"].to(F64).t()
    return _unit(x, eps)


def _lightning(W, p, m, h, rows, eps):
    H, d, silu = m["heads"], m["dim"], torch.nn.functional.silu
    q, k, v = (rows.padded(silu(h @ W[p + s].to(F64).t()).view(h.shape[0], H, -1)) for s in "qkv")
    decay = torch.tensor(m["decay"], dtype=F64, device=DEV)[None, :, None, None]
    S, o = torch.zeros(q.shape[0], H, d, v.shape[-1], dtype=F64, device=DEV), torch.empty_like(v)
    for t in range(rows.T):
        S = decay * S + k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = (q[:, t, :, :, None] * S).sum(dim=2)
    y = _unit(rows.flat(o).reshape(h.shape[0], -1), eps) * torch.sigmoid(h @ W[p + "g"].to(F64).t())
    return y @ W[p + "o"].to(F64).t()


def _sink_attention(W, p, m, h, rows, eps):
    n = h.shape[0]
    freq = _frequencies(m["rot"]["base"], m["rot"]["dims"])
    q = _unit((h @ W[p + "q"].to(F64).t()).view(n, m["heads"], m["dim"]), eps)
    v = (h @ W[p + "k"].to(F64).t()).view(n, m["kv_heads"], m["dim"])
    q, k = _rotate(q, rows.pos, freq), _rotate(_unit(v, eps), rows.pos, freq)
    return rows.each(lambda q, k, v: _attend(q, k, v, m["scale"], True), q, k, v) @ W[p + "o"].to(F64).t()


def _fazopel_layers(raw, W, x, rows):
    eps = raw["norm"]["eps"]
    for i, L in enumerate(raw["layers"]):
        mixer = _lightning if L["type"] == "lightning" else _sink_attention
        x = x + _unit(mixer(W, f"l{i}.mix.", L["mixer"], x, rows, eps), eps)
        a = torch.relu(x @ W[f"l{i}.mlp.up"].to(F64).t()) ** 2
        x = x + _unit(a @ W[f"l{i}.mlp.down"].to(F64).t(), eps)
    return _unit(x, eps)


@torch.no_grad()
def exact(case, seed):
    raw = MODELS[case["model"]]
    W, prompts, given = _inputs(case, seed)
    seqs = [p + [g[b] for g in given] for b, p in enumerate(prompts)]
    rows = _Rows([len(s) for s in seqs])
    embed, head = ("model.embed_tokens.weight", "lm_head.weight") if _is_llama(raw) else ("embed", "head")
    x = W[embed][torch.tensor([t for s in seqs for t in s], device=DEV)].to(F64)
    layers = _llama_layers if _is_llama(raw) else _sunusun_layers if raw["architecture"] == "Sunusun" else _fazopel_layers
    x = layers(raw, W, x, rows)
    first = [a + len(p) - case["want"] + j for (a, _), p in zip(rows.cuts, prompts) for j in range(case["want"])]
    later = [a + len(p) + t for t in range(case["steps"]) for (a, _), p in zip(rows.cuts, prompts)]
    W = W[head].to(F64).t()
    out = {"prompt": x[first] @ W}
    if later:
        out["decoded"] = (x[later] @ W).view(case["steps"], case["batch"], -1)
    return out
