"""The work that programs have this engine do, as measurable cases.

A case is one step through `Engine.step`, which is what serving consists of: `decodes` requests that bring one token each to a
cached context, beside `prompts` requests that bring `portion` tokens each behind `start` cached ones.  Or (`rows`) it is one draw
of tokens from logits through `Sampler.sample`.  Weights, tokens and cached keys and values are random, made from the seed alone.
Layer sizes are those of the repository's benchmark (`bench.py`: the dense family's shapes and two of its other designs); the
number of layers is cut where a pass would take long, the sizes of a layer and of the vocabulary are not.

Cached keys and values are drawn from a unit normal law, which is what a per-head norm leaves of keys and close to what random
weights give as values; matrices N(0, 0.02) and norm weights 1 + N(0, 0.1), the law of the repository's random models, but for
what leads into the residual stream: embeddings, the last product of a sub-layer and a norm behind a sub-layer are drawn so that a
layer adds a small share to the stream, as in a trained model (and as the usual initialisation of deep decoders has it).
"""
import hashlib
import math

import torch

PAGE = 16
# name: width, feed-forward, query heads, key heads, layers of the model, logits through the embedding's table
DENSE = {"0.6B": (1024, 3072, 16, 8, 28, True), "1.7B": (2048, 6144, 16, 8, 28, True), "4B": (2560, 9728, 32, 8, 36, True),
         "8B": (4096, 12288, 32, 8, 36, False), "14B": (5120, 17408, 40, 8, 40, False), "32B": (5120, 25600, 64, 8, 64, False)}
DENSE_VOCAB, DENSE_THETA, HEAD = 151936, 1000000.0, 128
DESIGN_VOCAB = 32768
EPS = 1e-6


def _step(name, model, layers, decodes=0, context=0, prompts=0, portion=0, start=0, dtype="bfloat16"):
    return {"name": name, "model": model, "layers": layers, "decodes": decodes, "context": context, "prompts": prompts,
            "portion": portion, "start": start, "dtype": dtype}


def listed():
    return [
        # a draw with the default sampling parameters for every request of a serving batch
        {"name": "sample_24", "rows": 24, "vocab": DENSE_VOCAB, "history": 300},
        # one chat user of a small model: a token at a time, bound by launches and fixed costs
        _step("decode_small_1", "0.6B", 28, decodes=1, context=700),
        # a few users with long contexts: the repository's headline
        _step("decode_8_long", "8B", 12, decodes=8, context=8192),
        # a full serving batch with contexts of all lengths
        _step("decode_64", "8B", 12, decodes=64, context=1500),
        # the first answer of a small model to a short question
        _step("prompt_small", "0.6B", 28, prompts=1, portion=117),
        # several short questions that arrive together
        _step("prompts_3x150", "8B", 12, prompts=3, portion=150),
        # a document in one step, and a long one
        _step("prompt_2048", "8B", 12, prompts=1, portion=2048),
        _step("prompt_8192", "8B", 12, prompts=1, portion=8192),
        # continuous batching: a portion of a prompt beside requests that decode
        _step("mixed_9_512", "14B", 10, decodes=9, context=3100, prompts=1, portion=512, start=1500),
        # the true 32-bit path, for checks against other implementations
        _step("prompt_f32", "8B", 4, prompts=1, portion=555, dtype="float32"),
        # the designs with layers of other kinds: recurrences with matrix states beside window attention with a sink ...
        _step("lofudra_prompt", "lofudra-2k", 6, prompts=1, portion=1500),
        # ... and routed experts behind window attention over caches that layers share
        _step("fisanex_decode", "fisanex-2k", 6, decodes=8, context=2000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "decode", "decode", "prompt", "prompt", "mixed", "f32", "lofudra", "fisanex"])
    if kind == "sample":
        return {"rows": _log(rng, 1, 64), "vocab": DENSE_VOCAB, "history": _log(rng, 1, 4000)}
    model = rng.choice(list(DENSE))
    layers = min(DENSE[model][4], {"8B": 12, "14B": 8, "32B": 6}.get(model, 20))
    if kind == "decode":
        decodes = _log(rng, 1, 64)
        c = _step("", model, layers, decodes=decodes, context=_log(rng, 40, min(16384, 120000 // decodes)))
    elif kind == "prompt":
        prompts = rng.choice([1, 1, 1, 2, 4])
        c = _step("", model, layers, prompts=prompts, portion=_log(rng, 20, 3000 // prompts))
    elif kind == "mixed":
        c = _step("", model, layers, decodes=rng.randint(1, 32), context=_log(rng, 100, 4096), prompts=1,
                  portion=_log(rng, 100, 512), start=rng.choice([0, rng.randint(1, 3500)]))
    elif kind == "f32":
        if rng.random() < 0.5:
            c = _step("", "8B", 4, decodes=rng.randint(1, 16), context=_log(rng, 40, 4096), dtype="float32")
        else:
            c = _step("", rng.choice(["0.6B", "8B"]), 4, prompts=1, portion=_log(rng, 20, 1200), dtype="float32")
    elif kind == "lofudra":
        c = _step("", rng.choice(["lofudra-1k", "lofudra-2k"]), 6, prompts=1, portion=_log(rng, 50, 2048))
    else:
        width = rng.choice(["fisanex-1k", "fisanex-2k"])
        c = (_step("", width, 6, decodes=rng.choice([1, 2, 3, 5, 8, 16, 32]), context=_log(rng, 100, 4096)) if rng.random() < 0.6
             else _step("", width, 6, prompts=1, portion=_log(rng, 50, 2048)))
    del c["name"]
    return c


# ---- configurations -----------------------------------------------------------------------------------------------

def _width(case):
    return {"1k": 1024, "2k": 2048}[case["model"].split("-")[1]]


def _raw(case):
    """config.json of the case's model."""
    model, layers = case["model"], case["layers"]
    if model in DENSE:
        width, ff, heads, kv, _, tied = DENSE[model]
        return dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", vocab_size=DENSE_VOCAB, hidden_size=width,
                    intermediate_size=ff, num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=kv, head_dim=HEAD,
                    rope_theta=DENSE_THETA, rms_norm_eps=EPS, tie_word_embeddings=tied, max_position_embeddings=40960)
    width = _width(case)
    heads = width // 128
    if model.startswith("lofudra"):
        ssm = {"type": "mamba2", "mixer": {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}}
        par = {"type": "parallel",
               "mixer": {"left": {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                                  "mask": {"size": 1024}, "rot": {"base": 500000.0, "dims": 128}},
                         "right": {"heads": heads, "dim": 64, "vdim": 128,
                                   "decay": [1.0 - 2.0 ** (-5 - 5 * i / max(heads - 1, 1)) for i in range(heads)]},
                         "left_scale": 1.0, "right_scale": 1.0}}
        mem = {"type": "mlstm", "mixer": {"heads": max(1, width // 256), "dim": 128, "vdim": 256, "gate_cap": 15.0}}
        return {"architecture": "Lofudra", "vocab": DESIGN_VOCAB, "width": width, "norm": {"eps": EPS},
                "layers": [dict([ssm, par, mem][i % 3], mlp={"kind": "dense", "ff": 4 * width}) for i in range(layers)]}
    mixer = {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 64, "scale": 128 ** -0.5, "mask": {"size": 1024},
             "rot": {"base": 500000.0, "dims": 64}}
    ff = 3 * width // 4 // 64 * 64
    moe = {"kind": "moe", "router": {"experts": 32, "identity": 4, "top": 4}, "expert": {"ff": ff, "limit": 7.0},
           "shared": {"ff": 2 * ff, "limit": 7.0}}
    return {"architecture": "Fisanex", "vocab": DESIGN_VOCAB, "width": width, "norm": {"eps": EPS}, "postln_alpha": 2.0,
            "embedding": {"scale": 8.0}, "logit_scale": 0.5,
            "layers": [{"type": "attention", "mixer": dict(mixer), "mlp": {"kind": "dense", "ff": 3 * width}} if i % 2 == 0 else
                       {"type": "attention", "mixer": dict(mixer, kv_from=i - 1), "mlp": moe} for i in range(layers)]}


def _dtype(case):
    return torch.float32 if case["dtype"] == "float32" else torch.bfloat16


def _generator(seed, name, device="cuda"):
    digest = hashlib.sha256(f"{seed}:{name}".encode()).digest()
    return torch.Generator(device=device).manual_seed(int.from_bytes(digest[:6], "little"))


def _tensor(seed, name, shape, init, dtype):
    """One of the model's tensors, in the precision that the model holds it in."""
    mean, std = (1.0, 0.1) if init == "norm" else (0.0, 0.02)
    if name.endswith(("norm1b", "norm2b")):
        mean, std = 0.2, 0.02
    elif name.endswith(("o_proj.weight", "down_proj.weight")):
        std = 0.003
    elif name == "embed" or name.endswith("embed_tokens.weight"):
        std = 0.5
    return torch.empty(tuple(shape), dtype=dtype, device="cuda").normal_(mean, std, generator=_generator(seed, name))


# ---- the requests of a step -----------------------------------------------------------------------------------------

def _requests(case, seed):
    """(cached tokens, new tokens) of every request: contexts of a batch lie between a third of the longest and the longest."""
    gen = _generator(seed, "tokens", "cpu")
    vocab = DENSE_VOCAB if case["model"] in DENSE else DESIGN_VOCAB
    n, longest, out = case["decodes"], case["context"], []
    for i in range(n):
        cached = longest if n <= 8 else max(1, longest - (2 * longest // 3) * ((i * 7) % n) // n)
        out.append((cached, torch.randint(0, vocab, (1,), generator=gen).tolist()))
    for i in range(case["prompts"]):
        out.append((case["start"], torch.randint(0, vocab, (case["portion"] + 3 * i,), generator=gen).tolist()))
    return out


def _pages(requests):
    return [-(-(cached + len(tokens)) // PAGE) for cached, tokens in requests]


def prepare(case, seed):
    if "rows" in case:
        from inferrs_amd.sampling import Sampler, SamplingParams
        rows, vocab = case["rows"], case["vocab"]
        logits = torch.randn((rows, vocab), generator=_generator(seed, "logits"), device="cuda") * 2.5
        gen = _generator(seed, "history", "cpu")
        history = [torch.randint(0, vocab, (case["history"] + i,), generator=gen).tolist() for i in range(rows)]
        return {"sampler": Sampler("cuda:0"), "logits": logits, "params": [SamplingParams() for _ in range(rows)], "history": history,
                "seeds": torch.randint(0, 1 << 30, (rows,), generator=gen).tolist()}
    from inferrs_amd.config import Qwen3Config
    from inferrs_amd.config.fisanex import FisanexConfig
    from inferrs_amd.config.lofudra import LofudraConfig
    from inferrs_amd.engine import DecoderModel, Engine, Entry
    from inferrs_amd.parts.assemble import generated_tensors
    cls = Qwen3Config if case["model"] in DENSE else LofudraConfig if case["model"].startswith("lofudra") else FisanexConfig
    spec, dtype = cls.from_dict(_raw(case)).to_spec(), _dtype(case)
    tensors = {name: _tensor(seed, name, t.shape, t.init, dtype) for name, t in generated_tensors(spec).items()}
    requests = _requests(case, seed)
    engine = Engine(DecoderModel(spec, tensors, dtype, "cuda:0"), page_size=PAGE, num_pages=sum(_pages(requests)) + 1,
                    max_seqs=len(requests))
    cached = any(c for c, _ in requests)
    if cached:
        for i, a in enumerate(engine.storage.arrays):
            a.normal_(0.0, 1.0, generator=_generator(seed, f"cache{i}"))
    for i, (c, tokens) in enumerate(requests):
        if cached:
            engine.add_request(i)
            if not engine.cache.reserve(i, c + len(tokens)):
                raise RuntimeError("the pages do not hold the case's contexts")
            engine.cache.commit(i, c)
    # prompts without a cached token begin, run and end within a pass; requests with a context take the same step again
    return {"engine": engine, "entries": [Entry(i, tokens, [len(tokens) - 1]) for i, (_, tokens) in enumerate(requests)],
            "again": cached}


def run(state):
    if "sampler" in state:
        return torch.tensor(state["sampler"].sample(state["logits"], state["params"], state["history"], state["seeds"]))
    engine = state["engine"]
    logits = engine.step(state["entries"], commit=not state["again"])
    if not state["again"]:
        for e in state["entries"]:
            engine.end_request(e.seq_id)
    return [logits, list(engine.storage.arrays)]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def work(case):
    if "rows" in case:
        return {"bytes": 4.0 * case["rows"] * (case["vocab"] + 1), "flops": 4.0 * case["rows"] * case["vocab"]}
    requests, size = _requests(case, 0), 4 if case["dtype"] == "float32" else 2
    n, wanted = sum(len(t) for _, t in requests), len(requests)
    raw = _raw(case)
    params, flops, kv = 0.0, 0.0, 0.0

    def attend(heads, key_heads, d, dv, window, owner):
        nonlocal flops, kv
        for cached, tokens in requests:
            m = len(tokens)
            seen = sum(min(cached + j + 1, window) for j in range(m)) if window else m * cached + m * (m + 1) / 2
            flops += 2.0 * (d + dv) * heads * seen
            kv += key_heads * (d + dv) * (min(cached, window) if window else cached) + (key_heads * (d + dv) * m if owner else 0)

    def product(rows, out, inner, used=1.0):
        nonlocal params, flops
        params += used * out * inner
        flops += 2.0 * rows * out * inner

    if case["model"] in DENSE:
        width, ff, heads, kv_heads, _, _ = DENSE[case["model"]]
        for _ in range(case["layers"]):
            product(n, (heads + 2 * kv_heads) * HEAD, width)
            product(n, width, heads * HEAD)
            product(n, 3 * ff, width)
            attend(heads, kv_heads, HEAD, HEAD, None, True)
        product(wanted, DENSE_VOCAB, width)
        vocab = DENSE_VOCAB
    else:
        width, vocab = raw["width"], DESIGN_VOCAB
        for layer in raw["layers"]:
            m, f = layer["mixer"], layer["mlp"]
            if layer["type"] == "mamba2":
                inner = m["heads"] * m["vdim"]
                product(n, 2 * inner + 2 * m["state"] + m["heads"], width)
                product(n, width, inner)
                flops += 4.0 * n * inner * m["state"]
            elif layer["type"] == "mlstm":
                k, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
                product(n, 2 * k + 2 * v + 2 * m["heads"], width)
                product(n, width, v)
                flops += 4.0 * n * k * m["vdim"]
            elif layer["type"] == "parallel":
                le, r = m["left"], m["right"]
                product(n, (le["heads"] + le["kv_heads"]) * le["dim"], width)
                product(n, width, le["heads"] * le["dim"])
                attend(le["heads"], le["kv_heads"], le["dim"], le["dim"], le["mask"]["size"], True)
                product(n, 2 * r["heads"] * (r["dim"] + r["vdim"]), width)
                product(n, width, r["heads"] * r["vdim"])
                flops += 4.0 * n * r["heads"] * r["dim"] * r["vdim"]
            else:
                own = "kv_from" not in m
                d, dv, h, g = m["dim"], m["vdim"], m["heads"], m["kv_heads"]
                product(n, h * (d + dv) + (g * (d + dv) if own else 0), width)
                product(n, width, h * dv)
                attend(h, g, d, dv, m["mask"]["size"], own)
            if f["kind"] == "moe":
                experts, top, outs = f["router"]["experts"], f["router"]["top"], f["router"]["experts"] + f["router"]["identity"]
                product(n, outs, width)
                used = experts * (1.0 - (1.0 - top / outs) ** n)
                params += used * 3 * f["expert"]["ff"] * width
                flops += 2.0 * n * top * experts / outs * 3 * f["expert"]["ff"] * width
                product(n, 3 * f["shared"]["ff"], width)
            else:
                product(n, (3 if case["model"].startswith("fisanex") else 2) * f["ff"], width)
        product(wanted, vocab, width)
    return {"bytes": size * (params + kv + n * width) + 4.0 * wanted * vocab, "flops": flops}


def tolerance(case):
    if "rows" in case:
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 1.2e-5, "max": 1e-3}         # (3e-6 off the 64-bit result, in part by the 32-bit angles of the rotation)
    return {"rel": 0.03, "max": 0.9}                # (0.4 to 1.6 % off the 64-bit result: a stream rounded to bfloat16 twice a layer)


# ---- the same in 64 bits --------------------------------------------------------------------------------------------

class _Weights:
    """The model's tensors in 64 bits, made when they are asked for."""

    def __init__(self, case, seed):
        self.seed, self.dtype = seed, _dtype(case)

    def __call__(self, name, *shape):
        return _tensor(self.seed, name, shape, "matrix", self.dtype).double()

    def norm(self, name, *shape):
        return _tensor(self.seed, name, shape, "norm", self.dtype).double()


def _rms(x, w):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w


def _silu(z):
    return z * torch.sigmoid(z)


def _turn(x, positions, base, dims):
    """x [tokens, heads, d]: feature i of the first `dims` turns with i + dims/2."""
    half = dims // 2
    f = base ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / dims)
    a = positions.double()[:, None, None] * f
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)


def _attention(q, k, v, first, scale, window=None, sink=False):
    """q [n, H, d] at positions first.., k and v [first + n, G, .]: [n, H * dv]."""
    n, H, d = q.shape
    G, total = k.shape[1], k.shape[0]
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    out = torch.empty((n, H, v.shape[-1]), dtype=q.dtype, device=q.device)
    for lo in range(0, n, 512):
        hi = min(n, lo + 512)
        part = q[lo:hi].view(hi - lo, G, H // G, d).permute(1, 2, 0, 3).reshape(G, -1, d)
        s = (part @ kt).view(G, H // G, hi - lo, total) * scale
        far = (first + torch.arange(lo, hi, device=q.device))[:, None] - torch.arange(total, device=q.device)
        s = s.masked_fill(~((far >= 0) if window is None else (far >= 0) & (far < window)), float("-inf"))
        top = s.amax(-1, keepdim=True)
        e = torch.exp(s - top)
        p = e / (e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))
        o = p.reshape(G, -1, total) @ vt
        out[lo:hi] = o.view(G, H // G, hi - lo, -1).permute(2, 0, 1, 3).reshape(hi - lo, H, -1)
    return out.reshape(n, -1)


class _Cache:
    """Cached keys and values by request, where the engine's pages hold them: [pages, G, PAGE, d] for keys, [pages, G, dv, PAGE]
    for values, a request's pages one behind the other."""

    def __init__(self, requests):
        self.requests = requests
        counts = _pages(requests)
        self.first = [sum(counts[:i]) for i in range(len(counts))]
        self.counts = counts

    def get(self, keys, values, r):
        lo, hi, n = self.first[r], self.first[r] + self.counts[r], self.requests[r][0]
        k = keys[lo:hi].permute(0, 2, 1, 3).flatten(0, 1)[:n]
        v = values[lo:hi].permute(0, 3, 1, 2).flatten(0, 1)[:n]
        return k.double(), v.double()

    def put(self, keys, values, r, k, v):
        at = self.requests[r][0] + torch.arange(k.shape[0], device=k.device)
        page, slot = self.first[r] + at // PAGE, at % PAGE
        keys[page, :, slot] = k
        values[page, :, :, slot] = v


def _spans(requests):
    lo = 0
    for r, (cached, tokens) in enumerate(requests):
        yield r, cached, lo, lo + len(tokens)
        lo += len(tokens)


def _exact_dense(case, seed):
    width, ff, heads, kv_heads, _, tied = DENSE[case["model"]]
    requests, W, L, d = _requests(case, seed), _Weights(case, seed), case["layers"], HEAD
    cache, n_cached = _Cache(requests), any(c for c, _ in requests)
    pages = sum(cache.counts) + 1
    shape = (L, 2, pages, kv_heads, PAGE, d)
    storage = torch.zeros(shape, dtype=_dtype(case), device="cuda")
    if n_cached:
        storage.normal_(0.0, 1.0, generator=_generator(seed, "cache0"))
    storage = storage.double()
    ids = torch.tensor([t for _, tokens in requests for t in tokens], device="cuda")
    pos = torch.cat([c + torch.arange(len(t), device="cuda") for c, t in requests])
    embed = _tensor(seed, "model.embed_tokens.weight", (DENSE_VOCAB, width), "matrix", _dtype(case))
    x = embed[ids].double()
    for i in range(L):
        p = f"model.layers.{i}."
        h = _rms(x, W.norm(p + "input_layernorm.weight", width))
        q = (h @ W(p + "self_attn.q_proj.weight", heads * d, width).T).view(-1, heads, d)
        k = (h @ W(p + "self_attn.k_proj.weight", kv_heads * d, width).T).view(-1, kv_heads, d)
        v = (h @ W(p + "self_attn.v_proj.weight", kv_heads * d, width).T).view(-1, kv_heads, d)
        q = _turn(_rms(q, W.norm(p + "self_attn.q_norm.weight", d)), pos, DENSE_THETA, d)
        k = _turn(_rms(k, W.norm(p + "self_attn.k_norm.weight", d)), pos, DENSE_THETA, d)
        keys, values = storage[i, 0], storage[i, 1].view(pages, kv_heads, d, PAGE)
        a = torch.empty_like(q).view(-1, heads * d)
        for r, cached, lo, hi in _spans(requests):
            ck, cv = cache.get(keys, values, r)
            a[lo:hi] = _attention(q[lo:hi], torch.cat([ck, k[lo:hi]]), torch.cat([cv, v[lo:hi]]), cached, d ** -0.5)
            cache.put(keys, values, r, k[lo:hi], v[lo:hi])
        x = x + a @ W(p + "self_attn.o_proj.weight", width, heads * d).T
        h = _rms(x, W.norm(p + "post_attention_layernorm.weight", width))
        act = _silu(h @ W(p + "mlp.gate_proj.weight", ff, width).T) * (h @ W(p + "mlp.up_proj.weight", ff, width).T)
        x = x + act @ W(p + "mlp.down_proj.weight", width, ff).T
    last = torch.tensor([hi - 1 for _, _, _, hi in _spans(requests)], device="cuda")
    head = embed if tied else _tensor(seed, "lm_head.weight", (DENSE_VOCAB, width), "matrix", _dtype(case))
    h = _rms(x[last], W.norm("model.norm.weight", width))
    logits = torch.cat([h @ part.double().T for part in head.split(16384)], 1)
    # (a decode batch that the engine fills up to a size of its captured steps: the filling rows write a page too, which is no result)
    n = case["decodes"]
    filled = case["prompts"] == 0 and n > 8 and n % (2 if n <= 16 else 4 if n <= 32 else 8)
    return [logits, [None if filled else storage]]


def _exact_lofudra(case, seed):
    raw, W = _raw(case), _Weights(case, seed)
    (_, tokens), = _requests(case, seed)
    width, n = raw["width"], len(tokens)
    pos = torch.arange(n, device="cuda")
    x = _tensor(seed, "embed", (DESIGN_VOCAB, width), "matrix", _dtype(case))[torch.tensor(tokens, device="cuda")].double()

    def sums(q, k, v, keep, take=None):
        """S <- keep_t S + take_t k_t v_t^T a head, o_t = S^T q_t: q, k [n, H, d], v [n, H, dv], keep and take [n, H]."""
        S = torch.zeros((q.shape[1], q.shape[2], v.shape[2]), dtype=q.dtype, device=q.device)
        out = torch.empty_like(v)
        if take is not None:
            k = k * take[..., None]
        for t in range(n):
            S.mul_(keep[t][:, None, None]).baddbmm_(k[t][:, :, None], v[t][:, None, :])
            out[t] = torch.bmm(q[t][:, None, :], S)[:, 0]
        return out

    for i, layer in enumerate(raw["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        h = _rms(x, W.norm(f"l{i}.norm1", width))
        if layer["type"] == "mamba2":
            H, dv, N = m["heads"], m["vdim"], m["state"]
            inner = H * dv
            proj = h @ W(p + "in", 2 * inner + 2 * N + H, width).T
            z, xbc, dt = proj.split([inner, inner + 2 * N, H], 1)
            taps, padded = W(p + "conv", inner + 2 * N, m["conv"]), torch.cat([xbc.new_zeros(m["conv"] - 1, inner + 2 * N), xbc])
            xbc = _silu(W(p + "conv.b", inner + 2 * N) + sum(padded[j:j + n] * taps[:, j] for j in range(m["conv"])))
            u, B, C = xbc.split([inner, N, N], 1)
            u = u.reshape(n, H, dv)
            dt = torch.nn.functional.softplus(dt + W(p + "dt_bias", H))
            keep = torch.exp(-torch.exp(W(p + "A_log", H)) * dt)
            y = sums(C[:, None].expand(n, H, N), B[:, None].expand(n, H, N), u, keep, dt) + W.norm(p + "D", H)[:, None] * u
            y = _rms(y.reshape(n, inner) * _silu(z), W.norm(p + "norm", inner)) @ W(p + "o", width, inner).T
        elif layer["type"] == "mlstm":
            H, d, dv, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
            q = (h @ W(p + "q", H * d, width).T).view(n, H, d) * d ** -0.5
            k, v = (h @ W(p + "k", H * d, width).T).view(n, H, d), (h @ W(p + "v", H * dv, width).T).view(n, H, dv)
            gi = cap * torch.tanh((h @ W(p + "i", H, width).T + W(p + "i.b", H)) / cap)
            gf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ W(p + "f", H, width).T + W(p + "f.b", H)) / cap))
            top, tops = torch.zeros(H, dtype=h.dtype, device="cuda"), [torch.zeros(H, dtype=h.dtype, device="cuda")]
            for t in range(n):
                top = torch.maximum(gf[t] + top, gi[t])
                tops.append(top)
            tops = torch.stack(tops)
            keep, take = torch.exp(gf + tops[:-1] - tops[1:]), torch.exp(gi - tops[1:])
            o = sums(q, k, torch.cat([v, torch.ones_like(v[..., :1])], -1), keep, take)   # (the last column: the normaliser)
            o = o[..., :dv] / (torch.maximum(o[..., dv:].abs(), torch.exp(-tops[1:])[..., None]) + 1e-6)
            y = _rms(o, None).reshape(n, H * dv) * W.norm(p + "norm", H * dv) * torch.sigmoid(h @ W(p + "g", H * dv, width).T)
            y = y @ W(p + "o", width, H * dv).T
        else:
            le, r = m["left"], m["right"]
            H, G, d, pl = le["heads"], le["kv_heads"], le["dim"], p + "left."
            q = (h @ W(pl + "q", H * d, width).T + W(pl + "q.b", H * d)).view(n, H, d)
            v = (h @ W(pl + "k", G * d, width).T + W(pl + "k.b", G * d)).view(n, G, d)
            q = _turn(_rms(q, W.norm(pl + "q.norm", d)), pos, le["rot"]["base"], le["rot"]["dims"])
            k = _turn(_rms(v, W.norm(pl + "k.norm", d)), pos, le["rot"]["base"], le["rot"]["dims"])
            y = _attention(q, k, v, 0, le["scale"], le["mask"]["size"], sink=True) @ W(pl + "o", width, H * d).T * m["left_scale"]
            H, d, dv, pr = r["heads"], r["dim"], r["vdim"], p + "right."
            q, k = (h @ W(pr + "q", H * d, width).T).view(n, H, d), (h @ W(pr + "k", H * d, width).T).view(n, H, d) * d ** -0.5
            v = (h @ W(pr + "v", H * dv, width).T).view(n, H, dv)
            o = sums(q, k, v, torch.tensor(r["decay"], dtype=h.dtype, device="cuda").expand(n, H))
            o = _rms(o, None).reshape(n, H * dv) * _silu(h @ W(pr + "g", H * dv, width).T)
            y = y + o @ W(pr + "o", width, H * dv).T * m["right_scale"]
        x = x + _rms(y, W.norm(f"l{i}.norm1b", width))
        h = _rms(x, W.norm(f"l{i}.norm2", width)) @ W(f"l{i}.mlp.up", layer["mlp"]["ff"], width).T
        h = torch.nn.functional.gelu(h) @ W(f"l{i}.mlp.down", width, layer["mlp"]["ff"]).T
        x = x + _rms(h, W.norm(f"l{i}.norm2b", width))
    logits = _rms(x[-1:], W.norm("final.norm", width)) @ W("head", DESIGN_VOCAB, width).T
    return [logits, []]          # (how the states and pages of this design lie is the engine's own business)


def _exact_fisanex(case, seed):
    raw, W, requests = _raw(case), _Weights(case, seed), _requests(case, seed)
    width, cache = raw["width"], _Cache(requests)
    m = raw["layers"][0]["mixer"]
    H, G, d, dv, base, dims = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]["base"], m["rot"]["dims"]
    pages, owners = sum(cache.counts) + 1, [i for i, layer in enumerate(raw["layers"]) if "kv_from" not in layer["mixer"]]
    keys = torch.zeros((len(owners), pages, G, PAGE, d), dtype=_dtype(case), device="cuda")
    values = torch.zeros((len(owners), pages, G, PAGE, dv), dtype=_dtype(case), device="cuda")
    if any(c for c, _ in requests):
        keys.normal_(0.0, 1.0, generator=_generator(seed, "cache0"))
        values.normal_(0.0, 1.0, generator=_generator(seed, "cache1"))
    pos = torch.cat([c + torch.arange(len(t), device="cuda") for c, t in requests])
    ids = torch.tensor([t for _, tokens in requests for t in tokens], device="cuda")
    embed = W("embed", DESIGN_VOCAB, width)
    x = embed[ids] * raw["embedding"]["scale"]
    alpha, seen = raw["postln_alpha"], {}

    def clamped(h, p, ff, limit):
        g = (h @ W(p + "gate", ff, width).T).clamp(max=limit)
        u = (h @ W(p + "up", ff, width).T).clamp(-limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ W(p + "down", width, ff).T

    for i, layer in enumerate(raw["layers"]):
        p, f = f"l{i}.mix.", layer["mlp"]
        if i in owners:
            at = owners.index(i)
            k = (x @ W(p + "k", G * d, width).T).view(-1, G, d)
            k = _turn(_rms(k, W.norm(p + "k.norm", d)), pos, base, dims)
            v = (x @ W(p + "v", G * dv, width).T).view(-1, G, dv)
            both = [cache.get(keys[at], values[at].view(pages, G, dv, PAGE), r) for r in range(len(requests))]
            seen[i] = [(torch.cat([both[r][0], k[lo:hi]]), torch.cat([both[r][1], v[lo:hi]])) for r, _, lo, hi in _spans(requests)]
        src = seen[layer["mixer"].get("kv_from", i)]
        q = (x @ W(p + "q", H * d, width).T).view(-1, H, d)
        q = _turn(_rms(q, W.norm(p + "q.norm", d)), pos, base, dims)
        a = torch.cat([_attention(q[lo:hi], *src[r], cached, m["scale"], m["mask"]["size"]) for r, cached, lo, hi in _spans(requests)])
        a = (a * torch.sigmoid(x @ W(p + "g", H * dv, width).T)) @ W(p + "o", width, H * dv).T
        x = _rms(alpha * x + a, W.norm(f"l{i}.norm1", width))
        p = f"l{i}.mlp."
        if f["kind"] == "dense":
            y = (_silu(x @ W(p + "gate", f["ff"], width).T) * (x @ W(p + "up", f["ff"], width).T)) @ W(p + "down", width, f["ff"]).T
        else:
            experts, top, outs = f["router"]["experts"], f["router"]["top"], f["router"]["experts"] + f["router"]["identity"]
            s = torch.softmax(x @ W(p + "router", outs, width).T, -1)
            chosen = torch.topk(s + W(p + "correction", outs), top, -1).indices
            weight = torch.gather(s, 1, chosen)
            y = clamped(x, p + "shared.", f["shared"]["ff"], f["shared"]["limit"])
            y = y + x * torch.where(chosen >= experts, weight, torch.zeros_like(weight)).sum(-1, keepdim=True)
            for e in range(experts):
                t, j = torch.nonzero(chosen == e, as_tuple=True)
                if t.numel():
                    y[t] += weight[t, j][:, None] * clamped(x[t], f"{p}e{e}.", f["expert"]["ff"], f["expert"]["limit"])
        x = _rms(alpha * x + y, W.norm(f"l{i}.norm2", width))
    last = torch.tensor([hi - 1 for _, _, _, hi in _spans(requests)], device="cuda")
    logits = _rms(x[last], W.norm("final.norm", width)) @ embed.T * raw["logit_scale"]
    return [logits, []]          # (the window gives pages back, so that where keys and values lie is the engine's own business)


def exact(case, seed):
    if "rows" in case:
        return None
    if case["model"] in DENSE:
        return _exact_dense(case, seed)
    return (_exact_lofudra if case["model"].startswith("lofudra") else _exact_fisanex)(case, seed)
