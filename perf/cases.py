"""The work that users of this framework have it do, as cases to be timed and compared.

Three kinds of work make up a deployment: texts are embedded (``EncoderModel.encode_ids``), vectors are searched
(``HipFlatIndex.search``), and a decoder reads prompts (``LLMEngine.forward_step``) and writes tokens (the model's
``forward_decode`` and ``logits`` in a captured graph, as the engines run them).  The decoders are the five registered
families at the layer sizes of their 7B presets.  Each runs four layers, one period of every family's layer pattern, so
that weights are made and 64-bit results are computed in seconds.

Sizes are those of the headline benchmark (128 threads of about 2600 prompt tokens, an index of a million rows), of the
model comparison (128 x 700, 24 x 2800, 32 x 1024, 1 x 2800) and of its latency points (single threads, single queries);
``draw`` spreads over what lies between.
"""
import dataclasses
import math

import numpy as np
import torch

LAYERS = 4               # of each decoder: one period of every family's pattern
STEPS = 2                # decode steps per pass: the second one reads the state that the first one wrote
PASS_ROWS = 16384        # prompt rows of one pass, the engine's default
DECODERS = ("mistral-7b", "vofosun-7b", "zisapel-7b", "pemolorn-7b", "tadolix-7b")
EXACT_FLOPS = 4e14       # 64-bit results that cost more than this are not computed


def listed():
    return [
        # a topic search embeds one short query
        dict(name="embed-query", kind="embed", model="minilm-l6", seqs=1, tokens=12, ragged=0.0),
        # the chunks of a batch of threads, up to the model's 256 tokens each
        dict(name="embed-chunks", kind="embed", model="minilm-l6", seqs=640, tokens=256, ragged=0.6),
        # the reporting service's topic search: best 150 of a resident index of a million chunks
        dict(name="search", kind="search", queries=1, rows=1_000_000, dim=384, k=150, distance="cosine"),
        # prompts of the headline batch: one full prefill pass
        dict(name="mistral-prefill", kind="prefill", model="mistral-7b", seqs=6, tokens=2730, past=0, ragged=0.1),
        # a single short thread at light load
        dict(name="mistral-prefill-one", kind="prefill", model="mistral-7b", seqs=1, tokens=420, past=0, ragged=0.0),
        # the headline batch's decode
        dict(name="mistral-decode", kind="decode", model="mistral-7b", seqs=128, past=2617, ragged=0.2),
        # one thread at light load
        dict(name="mistral-decode-one", kind="decode", model="mistral-7b", seqs=1, past=2617, ragged=0.0),
        # the comparison's shapes, one or two per family
        dict(name="vofosun-decode", kind="decode", model="vofosun-7b", seqs=24, past=2800, ragged=0.0),
        dict(name="zisapel-prefill", kind="prefill", model="zisapel-7b", seqs=23, tokens=700, past=0, ragged=0.0),
        dict(name="pemolorn-decode", kind="decode", model="pemolorn-7b", seqs=32, past=1024, ragged=0.0),
        dict(name="tadolix-prefill", kind="prefill", model="tadolix-7b", seqs=5, tokens=2800, past=0, ragged=0.0),
        # a handful of requests being served, one more than the single-stream kernels take
        dict(name="tadolix-decode", kind="decode", model="tadolix-7b", seqs=5, past=700, ragged=0.5),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choices(("embed", "search", "prefill", "decode"), (2, 1, 4, 5))[0]
    if kind == "embed":
        model = rng.choice(("minilm-l6", "minilm-l6", "bge-small"))
        tokens = spread(4, 256)
        return dict(kind=kind, model=model, seqs=spread(1, 80_000 // tokens if tokens > 100 else 800), tokens=tokens,
                    ragged=round(rng.uniform(0.0, 0.8), 2))
    if kind == "search":
        return dict(kind=kind, queries=spread(1, 16), rows=spread(20_000, 1_000_000), dim=rng.choice((384, 384, 768)),
                    k=spread(5, 200), distance=rng.choice(("cosine", "cosine", "l2")))
    model = rng.choice(("mistral-7b",) + DECODERS)
    if kind == "prefill":
        rows = spread(24, 12_000)
        seqs = min(spread(1, 64), max(1, rows // 16))
        return dict(kind=kind, model=model, seqs=seqs, tokens=max(2, rows // seqs), past=rng.choice((0, 0, 0, spread(16, 2000))),
                    ragged=round(rng.uniform(0.0, 0.6), 2))
    seqs = spread(1, 128)
    return dict(kind=kind, model=model, seqs=seqs, past=min(spread(32, 6000), 200_000 // seqs), ragged=round(rng.uniform(0.0, 0.6), 2))


# ------------------------------------------------------------------------------------------------ inputs
def lengths(case, key):
    """Sequence lengths from (1 - ragged) to 1 of the case's, unevenly spread, whatever the seed."""
    n = case[key]
    return [max(1, round(n * (1.0 - case["ragged"] * (i * 0.6180339887 % 1.0)))) for i in range(case["seqs"])]


def generator(seed, salt, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed * 1_000_003 + salt)
    return g


def token_lists(seed, lens, vocab):
    r = np.random.default_rng([seed, 5])
    return [r.integers(3, vocab, n).tolist() for n in lens]


def configuration(model):
    from copilot_for_consensus_amd.models import registry
    c = registry.get_config(model)
    return dataclasses.replace(c, specs=c.specs[:LAYERS]) if hasattr(c, "specs") else dataclasses.replace(c, layers=LAYERS)


def family(cfg):
    return type(cfg).__name__.removesuffix("Config").lower()


def tensor_shapes(cfg):
    from copilot_for_consensus_amd.models import registry
    if family(cfg) != "decoder":
        return registry.family_of(cfg).weights.tensor_shapes(cfg)
    h, f, d = cfg.hidden, cfg.ffn, cfg.head_dim
    out = {"embed": (cfg.vocab_size, h), "head": (cfg.vocab_size, h), "final.norm": (h,)}
    for i in range(cfg.layers):
        p = f"l{i}."
        out |= {p + "norm1": (h,), p + "qkv": ((cfg.heads + 2 * cfg.kv_heads) * d, h), p + "o": (h, cfg.heads * d),
                p + "norm2": (h,), p + "gate": (f, h), p + "up": (f, h), p + "down": (h, f)}
    return out


def preferences(n, top, groups, gen):
    """[n tokens, choices]: what a token's embedding tells a trained router, clear choices spread evenly over the experts
    (and, with ``groups`` (size, kept), over that many groups)."""
    def best(x, k):
        return torch.zeros_like(x).scatter_(-1, x.topk(k, -1).indices, 1.0)
    count, size, keep = groups
    r = torch.rand(n, count, size, device="cuda", generator=gen)
    chosen = best(r, top // keep)
    if keep < count:
        chosen = chosen * best(torch.rand(n, count, device="cuda", generator=gen), keep)[..., None]
    level = 5.0 + torch.rand(n, count, size, device="cuda", generator=gen)
    rest = 0.4 * torch.randn(n, count, size, device="cuda", generator=gen).clamp(-2.5, 2.5)
    return torch.where(chosen > 0, level, rest).view(n, count * size)


def routing(cfg):
    """(choices, chosen, (groups, size, kept)) of a family with experts, else None."""
    for s in getattr(cfg, "specs", ()):
        f = getattr(s, "mlp", None)
        if hasattr(f, "identity"):
            n = f.experts + f.identity
            return n, f.top, (1, n, 1)
        if hasattr(f, "experts"):
            return f.experts, f.top, (f.groups, f.experts // f.groups, f.keep)
    return None


def tensors(cfg, seed):
    """Every tensor of the model from the seed: matrices bf16, vectors fp32."""
    fam, gen, std = family(cfg), generator(seed, 99), 0.02
    w = {}

    def normal(shape, mean, sd):
        return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, sd, generator=gen)

    def uniform(shape, a, b):
        return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(a, b, generator=gen)

    for name, shape in tensor_shapes(cfg).items():
        kind = name.rsplit(".", 1)[-1]
        if kind.startswith("norm") or name.endswith(("left.out", "right.out")):
            # around what the norm multiplies with: weights counted from zero or from one, branches of a third
            mean = 0.0 if fam == "tadolix" or fam == "vofosun" and "mix." not in name else \
                0.3 if fam == "zisapel" and kind != "norm" or fam == "pemolorn" and kind.endswith("b") else 1.0
            w[name] = normal(shape, mean, 0.05)
        elif kind == "shift" or ".mu." in name:
            w[name] = uniform(shape, 0.0, 1.0)
        elif kind == "w0":
            w[name] = uniform(shape, -6.0, 0.0)
        elif kind == "lam":
            w[name] = uniform(shape, -5.0, -1.0)
        elif kind == "dwa":
            w[name] = normal(shape, 0.0, 0.02)
            w[name][-1] += 1.0
        elif kind == "in":
            w[name] = normal(shape, 1.0 / cfg.streams, 0.02)
        elif kind == "out":
            w[name] = normal(shape, 1.0, 0.05)
        elif kind == "mix":
            w[name] = 0.9 * torch.eye(cfg.streams, device="cuda") + normal(shape, 0.1 / cfg.streams, 0.01)
        elif kind == "router":
            w[name] = normal(shape, 0.0, 0.002)
            w[name][:, :shape[0]] += (0.5 if fam == "zisapel" else 1.0) * torch.eye(shape[0], device="cuda")
            w[name] = w[name].to(torch.bfloat16)
        elif kind == "correction":
            w[name] = normal(shape, 0.0, 0.005)
        elif kind in ("b", "u", "sink", "conv", "rel") and fam != "vofosun":
            w[name] = normal(shape, 0.0, 0.5)
        elif kind.startswith("canon"):
            w[name] = normal(shape, 0.0, 0.2).to(torch.bfloat16).float()
        elif name == "embed":
            t = normal(shape, 0.0, shape[1] ** -0.5 if fam == "tadolix" else 1.0)
            if r := routing(cfg):
                t[:, :r[0]] = preferences(shape[0], r[1], r[2], gen)
            w[name] = t.to(torch.bfloat16)
        else:
            sd = shape[2] ** -0.5 if kind in ("ra", "ri") else std
            if fam in ("decoder", "vofosun") and kind in ("o", "down"):
                sd /= math.sqrt(2 * cfg.layers)
            w[name] = normal(shape, 0.0, sd).to(torch.bfloat16)
    if fam == "decoder":
        w = {k: v.to(torch.bfloat16) for k, v in w.items()}
    return w


def decoder_model(cfg, w):
    from copilot_for_consensus_amd.models import registry
    if family(cfg) != "decoder":
        return registry.build_model(registry.family_of(cfg).weights._build(cfg, w.__getitem__, "cuda:0", 0, 1, torch.bfloat16))
    from copilot_for_consensus_amd.models.decoder import DecoderWeights
    dw = DecoderWeights(cfg, "cuda:0")
    for i in range(cfg.layers):
        p = f"l{i}."
        dw.layers.append({"attn_norm": w[p + "norm1"], "qkv": w[p + "qkv"], "o": w[p + "o"], "mlp_norm": w[p + "norm2"],
                          "gate_up": torch.cat([w[p + "gate"], w[p + "up"]]), "down": w[p + "down"]})
    dw.embed, dw.final_norm, dw.lm_head = w["embed"], w["final.norm"], w["head"]
    return registry.build_model(dw.finalize())


def encoder_shapes(c):
    h, f = c.hidden, c.ffn
    out = {"word": (c.vocab_size, h), "pos": (c.max_positions, h), "type": (2, h), "emb_g": (h,), "emb_b": (h,)}
    for i in range(c.layers):
        out |= {f"{i}.{k}": s for k, s in dict(qkv=(3 * h, h), qkv_b=(3 * h,), o=(h, h), o_b=(h,), ln1_g=(h,), ln1_b=(h,),
                                               up=(f, h), up_b=(f,), down=(h, f), down_b=(h,), ln2_g=(h,), ln2_b=(h,)).items()}
    return out


def encoder_tensors(c, seed):
    gen = generator(seed, 31)
    return {k: torch.empty(s, dtype=torch.float32, device="cuda").normal_(
        1.0 if k.endswith("_g") else 0.0, 0.1 if k.endswith("_g") else 0.05 if len(s) == 2 else 0.02, generator=gen).to(torch.bfloat16)
        for k, s in encoder_shapes(c).items()}


def vectors(case, seed):
    """Rows and queries like encoders give them: a common direction, threads of alike chunks, a query near some rows."""
    gen, n, d = generator(seed, 17), case["rows"], case["dim"]

    def rnd(*s):
        return torch.empty(s, dtype=torch.float32, device="cuda").normal_(0.0, 1.0, generator=gen)
    topics = rnd(max(1, n // 40), d) + 0.7 * rnd(1, d)
    x = topics[torch.randint(0, topics.shape[0], (n,), device="cuda", generator=gen)] + 0.8 * rnd(n, d)
    q = x[torch.randint(0, n, (case["queries"],), device="cuda", generator=gen)] + 0.8 * rnd(case["queries"], d)
    return (torch.nn.functional.normalize(t, dim=1) for t in (x, q))


# ------------------------------------------------------------------------------------------------ the calls
@torch.inference_mode()
def prepare(case, seed):
    return {"embed": prepare_embed, "search": prepare_search, "prefill": prepare_prefill, "decode": prepare_decode}[case["kind"]](case, seed)


def run(state):
    return state["call"]()


def prepare_embed(case, seed):
    from copilot_for_consensus_amd.models.encoder import EncoderModel, get_encoder_config
    c = get_encoder_config(case["model"])
    w, enc = encoder_tensors(c, seed), EncoderModel(c, "cuda:0")
    enc.p = {k: w[k] for k in ("word", "pos", "type", "emb_g", "emb_b")}
    enc.layers = [{k.split(".")[1]: v for k, v in w.items() if k.startswith(f"{i}.")} for i in range(c.layers)]
    texts = token_lists(seed, lengths(case, "tokens"), c.vocab_size)
    return {"call": lambda: enc.encode_ids(texts)}


def prepare_search(case, seed):
    from copilot_for_consensus_amd.vectorstore import HipFlatIndex
    x, q = vectors(case, seed)
    index = HipFlatIndex(case["dim"], case["distance"], capacity=case["rows"], device="cuda:0")
    index.add_bulk([f"chunk-{i}" for i in range(case["rows"])], x)
    return {"call": lambda: index.search(q, case["k"])}


def serving(case, seed, lens):
    """An engine over a cache with room for the sequences' ``lens`` tokens, each one's block table and state slot."""
    from copilot_for_consensus_amd.runtime.engine import LLMEngine
    from copilot_for_consensus_amd.runtime.kv_cache import blocks_needed
    cfg = configuration(case["model"])
    model = decoder_model(cfg, tensors(cfg, seed))
    kv = model.new_cache(sum(blocks_needed(n) for n in lens) + 8, sequences=len(lens))
    eng = LLMEngine(model, kv, max_prefill_tokens=PASS_ROWS, prefix_cache=False)
    tables = [kv.pool.alloc(blocks_needed(n)) for n in lens]
    return eng, tables, kv.states.alloc(len(lens)) if kv.states is not None else [None] * len(lens)


def read_prompts(eng, prompts, tables, slots):
    """The prompts into the cache, in passes of at most PASS_ROWS rows."""
    entries, room = [], PASS_ROWS
    for p, table, slot in zip(prompts, tables, slots):
        at = 0
        while at < len(p):
            n = min(len(p) - at, room)
            entries.append((p[at:at + n], at, table, [], slot))
            at, room = at + n, room - n
            if room == 0:
                eng.forward_step(entries)
                entries, room = [], PASS_ROWS
    if entries:
        eng.forward_step(entries)


def prepare_prefill(case, seed):
    lens = lengths(case, "tokens")
    past = case["past"]
    eng, tables, slots = serving(case, seed, [n + past for n in lens])
    prompts = token_lists(seed, [n + past for n in lens], eng.cfg.vocab_size)
    if past:
        read_prompts(eng, [p[:past] for p in prompts], tables, slots)
    # the logits that the first generated token is chosen by
    entries = [(p[past:], past, t, [len(p) - past - 1], s) for p, t, s in zip(prompts, tables, slots)]
    return {"call": lambda: eng.forward_step(entries)}


def prepare_decode(case, seed):
    """STEPS decode steps over the sequences as one graph, the engines' way of decoding, on given tokens."""
    from copilot_for_consensus_amd.ops.reference import KV_BLOCK
    lens = lengths(case, "past")
    eng, tables, slots = serving(case, seed, [n + STEPS for n in lens])
    model, kv, B = eng.model, eng.kv, len(lens)
    prompts = token_lists(seed, [n + STEPS for n in lens], eng.cfg.vocab_size)
    read_prompts(eng, [p[:n] for p, n in zip(prompts, lens)], tables, slots)

    def i32(x):
        return torch.tensor(x, dtype=torch.int32, device="cuda:0")
    maxb = 8 * math.ceil(max(len(t) for t in tables) / 8)
    bt = i32([t + [0] * (maxb - len(t)) for t in tables])
    P = model.decode_partitions(B, maxb)
    ws = torch.empty(max(1, model.decode_workspace(B, P)), dtype=torch.float32, device="cuda:0")
    states = None if kv.states is None else i32([kv.states.scratch] * B)
    steps = []
    for s in range(STEPS):
        pos = [n + s for n in lens]
        steps.append((i32([p[n] for p, n in zip(prompts, pos)]), i32(pos),
                      i32([t[n // KV_BLOCK] * KV_BLOCK + n % KV_BLOCK for t, n in zip(tables, pos)]), i32([n + 1 for n in pos])))

    def decode():
        out = []
        for ids, pos, at, ctx in steps:
            kw = {} if states is None else {"states": states}
            hidden = model.forward_decode(ids, pos, at, ctx, bt, kv, attn_workspace=ws, part_blocks=-P, **kw)
            out.append(model.logits(hidden))
        return out
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):      # the warm-up runs on the scratch state
        decode()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = decode()
    if states is not None:
        states.copy_(i32(slots))

    def call():
        graph.replay()
        return out
    return {"call": call, "keep": (eng, steps, bt, ws, states, stream)}


# ------------------------------------------------------------------------------------------------ floors
def touched(cfg, rows):
    """Parameters of the layers that ``rows`` tokens cannot do without (of the experts those expected to be chosen)."""
    n = 0
    for k, s in tensor_shapes(cfg).items():
        if k in ("embed", "head"):
            continue
        share = 1.0
        if r := routing(cfg):
            if ".mlp.e" in k:
                share = 1.0 - (1.0 - r[1] / r[0]) ** rows
        n += share * math.prod(s)
    return n


def kept(cfg, ctx):
    """(bytes of a token's cache rows, bytes of the rows a token with ``ctx`` before it reads, bytes of per-sequence state)."""
    if family(cfg) == "decoder":
        row = cfg.layers * 4 * cfg.kv_heads * cfg.head_dim
        return row, row * ctx, 0
    row = read = state = 0
    for s in cfg.specs:
        m = s.mixer
        a = getattr(m, "left", m)
        if hasattr(a, "kv_rank"):
            b = 2 * (a.kv_rank + getattr(a, "rot_dim", 0))
            row, read = row + b, read + b * min(ctx, getattr(a, "window", 0) or ctx)
        elif hasattr(a, "kv_heads"):
            b = 2 * a.kv_heads * (a.dim + a.vdim)
            row += b if getattr(a, "kv_from", None) is None else 0
            read += b * (a.mask.visible(ctx) if hasattr(a, "mask") else (ctx % a.chunk if a.chunk else ctx))
        state += 4 * (m.heads * m.dim ** 2 if hasattr(m, "rank") else getattr(m, "width", 0))
    return row, read, state


def work(case):
    if case["kind"] == "embed":
        from copilot_for_consensus_amd.models.encoder import get_encoder_config
        c, lens = get_encoder_config(case["model"]), lengths(case, "tokens")
        n, mat = sum(lens), c.layers * (4 * c.hidden ** 2 + 2 * c.hidden * c.ffn)
        return {"bytes": 2 * mat + 2 * n * c.hidden + 4 * n + 4 * len(lens) * c.hidden,
                "flops": 2 * mat * n + 4 * c.layers * c.hidden * sum(x * x for x in lens)}
    if case["kind"] == "search":
        n, q, d = case["rows"], case["queries"], case["dim"]
        return {"bytes": 2 * n * d + 4 * q * d + 12 * q * case["k"], "flops": 2 * n * q * d}
    cfg = configuration(case["model"])
    V, W = cfg.vocab_size, cfg.hidden
    logit = 2 if family(cfg) == "decoder" else 4
    if case["kind"] == "decode":
        lens = lengths(case, "past")
        b = f = 0
        for n in lens:
            row, read, state = kept(cfg, n)
            b += read + row + 2 * state + 2 * W + logit * V
            f += cfg.flops_per_token(n)
        return {"bytes": STEPS * (b + 2 * touched(cfg, len(lens)) + 2 * V * W), "flops": STEPS * f}
    lens, past = lengths(case, "tokens"), case["past"]
    rows, b, f = sum(lens), 0, 0
    for n in lens:
        row, _, state = kept(cfg, 0)
        b += n * (row + 2 * W) + kept(cfg, past)[1] + (2 if past else 1) * state + logit * V
        f += n * (sum(cfg.flops_per_token(past + n * (i + 0.5) / 16) for i in range(16)) / 16 - 2 * W * V) + 2 * W * V
    return {"bytes": b + 2 * touched(cfg, rows) + 2 * V * W, "flops": f}


def tolerance(case):
    """About four times what the runs differ by from the same graph with its sums in another order."""
    if case["kind"] == "search":
        return {"rel": 2e-5, "differ": 0.005}        # fp32 sums of the same bf16 products; scores that lie that close change places
    if case["kind"] == "embed":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 2e-2, "max": 0.3}


# ------------------------------------------------------------------------------------------------ 64 bits
def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def layer_norm(x, w, eps, b=0.0):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b


def silu(z):
    return z * torch.sigmoid(z)


def gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def clamped_glu(g, u, limit):
    g = g.clamp(max=limit)
    return g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1.0)


def causal_conv(u, w):
    """u [B, T, C], w [C, taps], zeros before the first token."""
    T, taps = u.shape[1], w.shape[1]
    ext = torch.cat([u.new_zeros(u.shape[0], taps - 1, u.shape[2]), u], 1)
    return sum(w[:, j] * ext[:, j:j + T] for j in range(taps))


def attend(q, k, v, scale, see, sink=None, shape=lambda s, i, j: s):
    """q [B, T, H, D], k and v [B, J, G, .], see(i, j) for index columns and rows; heads side by side [B, T, H V]."""
    B, T, H, _ = q.shape
    J, G = k.shape[1:3]
    out = q.new_empty(B, T, H, v.shape[-1])
    j = torch.arange(J, device=q.device)[None]
    for b in range(B):
        kb, vb = k[b].permute(1, 2, 0), v[b].permute(1, 0, 2)
        for a in range(0, T, 512):
            i = torch.arange(a, min(a + 512, T), device=q.device)[:, None]
            n = i.shape[0]
            s = (q[b, a:a + n].view(n, G, H // G, -1).permute(1, 2, 0, 3).reshape(G, H // G * n, -1) @ kb * scale).view(H, n, J)
            s = shape(s, i, j).masked_fill(~see(i, j), -math.inf)
            if sink is not None:
                s = torch.cat([s, sink.view(H, 1, 1).expand(H, n, 1)], 2)
            p = torch.softmax(s, -1)[..., :J].reshape(G, H // G * n, J) @ vb
            out[b, a:a + n] = p.view(H, n, -1).transpose(0, 1)
    return out.flatten(2)


def turn(x, angle, magnitude=1.0):
    """x [B, T, H, D]: the neighbours (2i, 2i + 1) turned by angle [T, D / 2]."""
    c, s = angle.cos()[:, None] * magnitude, angle.sin()[:, None] * magnitude
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def positions(T):
    return torch.arange(T, dtype=torch.float64, device="cuda")


def frequencies(dims, base):
    return base ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device="cuda") / dims)


def linear_scan(a, b):
    """S_t = a_t S_(t - 1) + b_t from zero, [B, T, C]."""
    out, S = torch.empty_like(b), torch.zeros_like(b[:, 0])
    for t in range(b.shape[1]):
        S = torch.addcmul(b[:, t], a[:, t], S, out=out[:, t])
    return out


def min_gru(z, u):
    g = torch.sigmoid(z)
    return linear_scan(1.0 - g, g * torch.where(u >= 0, u + 0.5, torch.sigmoid(u)))


def gated_gru(h, p):
    return min_gru(h @ p["z"].T + p["z.b"], h @ p["x"].T + p["x.b"]) * silu(h @ p["g"].T)


def section(w, prefix):
    return {k[len(prefix):]: v for k, v in w.items() if k.startswith(prefix)}


def routed(h, weight, expert, E):
    """sum_e weight[..., e] expert(e, h) over the rows that chose e."""
    rows, wt = h.flatten(0, 1), weight.flatten(0, 1)
    out = torch.zeros_like(rows)
    for e in range(E):
        at = wt[:, e].nonzero()[:, 0]
        out[at] += wt[at, e, None] * expert(e, rows[at])
    return out.view_as(h)


def decoder_64(cfg, w, x):
    T, D = x.shape[1], cfg.head_dim
    angle = torch.outer(positions(T), frequencies(D, cfg.rope_theta))
    c, s = angle.cos()[:, None], angle.sin()[:, None]

    def rotate(t):
        a, b = t[..., :D // 2], t[..., D // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    for i in range(cfg.layers):
        p = section(w, f"l{i}.")
        q, k, v = ((rms(x, cfg.rms_eps) * p["norm1"]) @ p["qkv"].T).view(*x.shape[:2], -1, D).split(
            [cfg.heads, cfg.kv_heads, cfg.kv_heads], 2)
        x = x + attend(rotate(q), rotate(k), v, D ** -0.5, lambda i, j: j <= i) @ p["o"].T
        h = rms(x, cfg.rms_eps) * p["norm2"]
        x = x + (silu(h @ p["gate"].T) * (h @ p["up"].T)) @ p["down"].T
    return rms(x, cfg.rms_eps) * w["final.norm"], lambda z: z


def vofosun_64(cfg, w, x):
    eps, xs = cfg.norm_eps, [x]
    for i, spec in enumerate(cfg.specs):
        p, m = section(w, f"l{i}."), spec.mixer
        h = rms(x, eps) * (1.0 + p["norm1"])
        a = h + causal_conv(h, p["canon1"])
        q = (rms(a @ p["mix.dq"].T, eps) * p["mix.dq.norm"]) @ p["mix.uq"].T
        c = rms(a @ p["mix.dkv"].T, eps) * p["mix.dkv.norm"]
        q, k, v = (t.unflatten(-1, (m.heads, -1)) for t in (q, c @ p["mix.uk"].T, c @ p["mix.uv"].T))
        y = attend(q, k, v, m.scale, lambda i, j: j <= i) @ p["mix.o"].T
        b = h + causal_conv(h, p["canon2"])
        y = y + clamped_glu(b @ p["mlp.gate"].T + p["mlp.gate.b"], b @ p["mlp.up"].T + p["mlp.up.b"], spec.mlp.limit) @ p["mlp.down"].T
        y = y + p["mlp.down.b"]
        xs.append(x + y)
        x = sum(c * t for c, t in zip(p["dwa"], xs))
    return rms(x, eps) * (1.0 + w["final.norm"]), lambda z: cfg.logit_softcap * torch.tanh(z / cfg.logit_softcap)


def zisapel_64(cfg, w, x):
    eps, T = cfg.norm_eps, x.shape[1]

    def before(h):
        return torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1)

    def mix(h, mu):
        return h + (before(h) - h) * mu

    def yarn(m):
        n, f, sc = m.rot_dim, frequencies(m.rot_dim, m.base), dict(m.scaling or ())
        if not sc:
            return f, 1.0
        def dim(t):
            return n * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(m.base))
        lo, hi = max(math.floor(dim(sc["fast"])), 0), min(math.ceil(dim(sc["slow"])), n - 1)
        ramp = ((positions(n // 2) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0

    def latent(h, p, m):
        q = (h @ p["q"].T).unflatten(-1, (m.heads, -1))
        down, (f, mag) = h @ p["dkv"].T, yarn(m)
        c, angle = rms(down[..., :m.kv_rank], eps) * p["dkv.norm"], torch.outer(positions(T), f)
        k, v = ((c @ p[n].T).unflatten(-1, (m.heads, -1)) for n in ("uk", "uv"))
        k = torch.cat([k, turn(down[..., None, m.kv_rank:], angle, mag).expand(-1, -1, m.heads, -1)], -1)
        q = torch.cat([q[..., :m.dim], turn(q[..., m.dim:], angle, mag)], -1)
        o = attend(q, k, v, m.scale, lambda i, j: (j <= i) & (i - j < (m.window or T)), p["sink"])
        return (o * torch.sigmoid(h @ p["g"].T)) @ p["o"].T

    def wkv(h, p, m):
        r, k, v = ((mix(h, p["mu." + s]) @ p[s].T).unflatten(-1, (m.heads, m.dim)) for s in "rkv")
        d = torch.exp(-torch.exp(torch.tanh(mix(h, p["mu.w"]) @ p["w1"].T) @ p["w2"].T + p["w0"])).unflatten(-1, (m.heads, m.dim))
        S, out, u = h.new_zeros(h.shape[0], m.heads, m.dim, m.dim), torch.empty_like(v), p["u"][..., None]
        for t in range(T):
            kv = k[:, t, :, :, None] * v[:, t, :, None]
            out[:, t] = (r[:, t, :, None] @ torch.addcmul(S, u, kv))[:, :, 0]
            S = torch.addcmul(kv, d[:, t, :, :, None], S)
        return (rms(out, eps).flatten(2) * p["norm"] * silu(mix(h, p["mu.g"]) @ p["g"].T)) @ p["o"].T

    def glu(h, p, at):
        return (silu(h @ p[at + "gate"].T) * (h @ p[at + "up"].T)) @ p[at + "down"].T

    def experts(h, p, f):
        score = torch.sigmoid(h @ p["router"].T)
        choice = score + p["correction"]
        best = choice.unflatten(-1, (f.groups, -1)).topk(2, -1).values.sum(-1).topk(f.keep, -1).indices
        can = torch.zeros_like(choice).unflatten(-1, (f.groups, -1)).scatter(2, best[..., None].expand(-1, -1, -1, f.experts // f.groups), 1.0)
        at = choice.masked_fill(can.flatten(2) == 0, -math.inf).topk(f.top, -1).indices
        s = score.gather(-1, at)
        weight = torch.zeros_like(score).scatter(-1, at, s / (s.sum(-1, keepdim=True) + 1e-20) * f.scale)
        return routed(h, weight, lambda e, r: glu(r, p, f"e{e}."), f.experts) + (glu(h, p, "shared.") if f.shared else 0.0)

    for i, spec in enumerate(cfg.specs):
        p, m, f = section(w, f"l{i}."), spec.mixer, spec.mlp
        y = (wkv if hasattr(m, "rank") else latent)(mix(x, p["shift"]), section(p, "mix."), m)
        x = x + layer_norm(y * torch.sigmoid(x @ p["rg1"].T + p["rg1.b"]), p["norm1"], eps)
        q = section(p, "mlp.")
        y = experts(x, q, f) if hasattr(f, "experts") else clamped_glu(x @ q["gate"].T, x @ q["up"].T, f.limit) @ q["down"].T
        x = x + layer_norm(y * torch.sigmoid(x @ p["rg2"].T + p["rg2.b"]), p["norm2"], eps)
    return layer_norm(x, w["final.norm"], eps), lambda z: z * cfg.logit_scale


def pemolorn_64(cfg, w, x):
    eps, T, kvs = cfg.norm_eps, x.shape[1], {}

    def attention(h, p, a, i):
        q = rms((h @ p["q"].T).unflatten(-1, (a.heads, -1)), eps) * p["q.norm"]
        if a.kv_from is None:
            kvs[i] = (rms((h @ p["k"].T).unflatten(-1, (a.kv_heads, -1)), eps) * p["k.norm"],
                      (h @ p["v"].T).unflatten(-1, (a.kv_heads, -1)))
        k, v = kvs[i if a.kv_from is None else a.kv_from]
        see = lambda i, j: (j <= i) & ((i - j < (a.mask.size or T)) | (j < a.mask.keep))  # noqa: E731
        return attend(q, k, v, a.scale, see, p["sink"]) @ p["o"].T

    def pooled(h, p, a):
        q, k, v = (causal_conv(h @ p[n].T, p[n + ".conv"]) for n in "qkv")
        q, k = ((rms(t, eps) * p[n + ".norm"]).unflatten(-1, (g, -1)) for t, n, g in ((q, "q", a.heads), (k, "k", a.kv_heads)))
        v, angle = v.unflatten(-1, (a.kv_heads, -1)), torch.outer(positions(T), frequencies(a.rot, a.base))
        q, k = (torch.cat([turn(t[..., :a.rot], angle), t[..., a.rot:]], -1) for t in (q, k))
        n, pool, size = T // a.mask.pool, a.mask.pool, a.mask.size
        k, v = (torch.cat([t, t[:, :n * pool].unflatten(1, (n, pool)).mean(2)], 1) for t in (k, v))
        def see(i, j):
            last = (j - T) * pool + pool - 1
            return torch.where(j < T, (j <= i) & (i - j < size), last <= i - size)
        return attend(q, k, v, a.scale, see, p["sink"]) @ p["o"].T

    def experts(h, p, f):
        score = torch.softmax(h @ p["router"].T, -1)
        at = (score + p["correction"]).topk(f.top, -1).indices
        weight = torch.zeros_like(score).scatter(-1, at, score.gather(-1, at))
        y = routed(h, weight, lambda e, r: clamped_glu(r @ p[f"e{e}.gate"].T, r @ p[f"e{e}.up"].T, f.limit) @ p[f"e{e}.down"].T, f.experts)
        return y + weight[..., f.experts:].sum(-1, keepdim=True) * h

    for i, spec in enumerate(cfg.specs):
        p, m, f = section(w, f"l{i}."), spec.mixer, spec.mlp
        h, mx = rms(x, eps) * p["norm1"], section(p, "mix.")
        if hasattr(m, "left"):
            right = section(mx, "right.")
            y = (rms(pooled(h, section(mx, "left."), m.left), eps) * mx["left.out"] + rms(gated_gru(h, right) @ right["o"].T, eps) * mx["right.out"]) / 2
        else:
            y = attention(h, mx, m, i)
        x = x + rms(y, eps) * p["norm1b"]
        h, q = rms(x, eps) * p["norm2"], section(p, "mlp.")
        y = experts(h, q, f) if hasattr(f, "experts") else (h @ q["up"].T).clamp(min=0.0) ** 2 @ q["down"].T
        x = x + rms(y, eps) * p["norm2b"]
    return rms(x, eps) * w["final.norm"], lambda z: z


def distance_rows(T, rows, far):
    """The bias table's row for each distance: its own below half the rows, then logarithmic up to the last at ``far``."""
    half = rows // 2
    steps, out = rows - half, []
    for n in range(T):
        k = 0
        if n >= half:
            k = min(steps - 1, int(math.log(n / half) / math.log(far / half) * steps + 1e-9))
        out.append(n if n < half else half + k)
    return torch.tensor(out, device="cuda")


def tadolix_64(cfg, w, x):
    eps, T, W, n = cfg.norm_eps, x.shape[1], cfg.hidden, cfg.streams
    e = torch.arange(W, device="cuda")
    angle = positions(T)[:, None] * 10000.0 ** (-2.0 * (e // 2).double() / W)
    xs = [x * cfg.embed_scale + torch.where(e % 2 == 0, angle.sin(), angle.cos())] * n

    def norm(t, g):
        return rms(t, eps) * (1.0 + g)

    def read(q):
        return sum(a * t for a, t in zip(q, xs))

    def write(y, p):
        return [sum(p["mix"][s, t] * xs[s] for s in range(n)) + p["out"][t] * y for t in range(n)]

    def attention(h, p, a):
        q, k, v = ((h @ p[s].T).unflatten(-1, (g, -1)) for s, g in (("q", a.heads), ("k", a.kv_heads), ("v", a.kv_heads)))
        row = distance_rows(T, a.buckets, a.bias_max)
        shape = lambda s, i, j: a.softcap * torch.tanh(s / a.softcap) + p["rel"][row[(i - j).clamp(min=0)]].permute(2, 0, 1)  # noqa: E731
        o = attend(rms(q, eps), rms(k, eps), v, a.scale, lambda i, j: (j <= i) & (i // a.chunk == j // a.chunk), None, shape)
        return (o * torch.sigmoid(h @ p["g"].T)) @ p["o"].T

    def recurrent(h, p, m):
        u = causal_conv(h @ p["x"].T + p["x.b"], p["conv"]) + p["conv.b"]
        r, i = (torch.sigmoid(torch.einsum("btki,koi->btko", u.unflatten(-1, (m.blocks, -1)), p[s]) + p[s + ".b"]).flatten(2) for s in ("ra", "ri"))
        log_a = -8.0 * r * torch.nn.functional.softplus(p["lam"])
        S = linear_scan(torch.exp(log_a), torch.sqrt(-torch.expm1(2 * log_a)) * i * u)
        return (S * gelu_tanh(h @ p["y"].T + p["y.b"])) @ p["o"].T

    for i in cfg.runs:
        spec = cfg.specs[i]
        p, m = section(w, f"l{i}."), spec.mixer
        mx, c = section(p, "mix."), section(p, "hc1.")
        h = norm(read(c["in"]), p["norm1"])
        h = h + causal_conv(h, p["canon1"])
        if hasattr(m, "left"):
            right = section(mx, "right.")
            y = m.left_scale * attention(h, section(mx, "left."), m.left) + m.right_scale * gated_gru(h, right) @ right["o"].T
        else:
            y = recurrent(h, mx, m)
        xs = write(y, c)
        if spec.ff is not None:
            c = section(p, "hc2.")
            h = norm(read(c["in"]), p["norm2"])
            xs = write((gelu_tanh(h @ p["mlp.gate"].T) * (h @ p["mlp.up"].T)) @ p["mlp.down"].T, c)
    return norm(sum(xs), w["final.norm"]), lambda z: z


def encoder_64(case, seed):
    from copilot_for_consensus_amd.models.encoder import get_encoder_config
    c = get_encoder_config(case["model"])
    w = {k: v.double() for k, v in encoder_tensors(c, seed).items()}
    out = []
    for ids in token_lists(seed, lengths(case, "tokens"), c.vocab_size):
        ids = torch.tensor(ids[:c.max_seq_length], device="cuda")
        x = layer_norm(w["word"][ids] + w["pos"][:len(ids)] + w["type"][0], w["emb_g"], c.ln_eps, w["emb_b"])
        for i in range(c.layers):
            p = section(w, f"{i}.")
            q, k, v = (t.view(len(ids), c.heads, -1).transpose(0, 1) for t in (x @ p["qkv"].T + p["qkv_b"]).chunk(3, 1))
            a = (torch.softmax(q @ k.transpose(1, 2) * c.head_dim ** -0.5, -1) @ v).transpose(0, 1).reshape(len(ids), -1)
            x = layer_norm(x + a @ p["o"].T + p["o_b"], p["ln1_g"], c.ln_eps, p["ln1_b"])
            h = torch.nn.functional.gelu(x @ p["up"].T + p["up_b"])
            x = layer_norm(x + h @ p["down"].T + p["down_b"], p["ln2_g"], c.ln_eps, p["ln2_b"])
        e = x[0] if c.pooling == "cls" else x.mean(0)
        out.append(e / e.norm() if c.normalize else e)
    return torch.stack(out)


def search_64(case, seed):
    """Scores over the rows as the index holds them, in bf16: rounding them is no part of the search."""
    x, q = (t.to(torch.bfloat16) for t in vectors(case, seed))
    if case["distance"] == "cosine":
        x, q = (torch.nn.functional.normalize(t.float(), dim=1).to(torch.bfloat16) for t in (x, q))
    q, best = q.double(), []
    for part in x.split(1 << 18):
        part = part.double()
        s = q @ part.T
        if case["distance"] == "l2":
            s = 2 * s - (q * q).sum(1, keepdim=True) - (part * part).sum(1)
        best.append(s.topk(min(case["k"], part.shape[0]), 1).values)
    return torch.cat(best, 1).topk(case["k"], 1).values, None


@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "embed":
        return encoder_64(case, seed)
    if case["kind"] == "search":
        return search_64(case, seed)
    cfg = configuration(case["model"])
    decode = case["kind"] == "decode"
    lens = [n + STEPS for n in lengths(case, "past")] if decode else [n + case["past"] for n in lengths(case, "tokens")]
    if sum(n * cfg.flops_per_token(n // 2) for n in lens) > EXACT_FLOPS:
        return None
    forward = {"decoder": decoder_64, "vofosun": vofosun_64, "zisapel": zisapel_64, "pemolorn": pemolorn_64, "tadolix": tadolix_64}[family(cfg)]
    w = {k: v.double() for k, v in tensors(cfg, seed).items()}
    last = STEPS if decode else 1
    prompts, rows, at = token_lists(seed, lens, cfg.vocab_size), [], 0
    while at < len(lens):
        n = at + 1
        while n < len(lens) and (n + 1 - at) * max(lens[at:n + 1]) <= 16384:
            n += 1
        part, T = prompts[at:n], max(lens[at:n])
        ids = torch.tensor([p + [0] * (T - len(p)) for p in part], device="cuda")     # nothing looks ahead into the padding
        h, cap = forward(cfg, w, w["embed"][ids])
        rows += [cap(h[b, len(p) - last:len(p)] @ w["head"].T) for b, p in enumerate(part)]
        at = n
    return [torch.stack([r[s] for r in rows]) for s in range(STEPS)] if decode else torch.cat(rows)
