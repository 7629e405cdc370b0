"""Performance cases: the model steps that serving consists of.

One pass is one forward of a batch the way LLMEngine runs it: hidden states
of all rows, logits of the rows that are sampled, keys and values appended to
the paged caches.  Llama and Mixtral decode steps run as a captured graph, as
the engine captures them; prompt steps, mixed steps and the per-layer designs
run eagerly, as in the engine.  The sampler has a case of its own: its input
is the logits of a decode step.

Models have the layer sizes of the repository's presets.  All layers of a
Llama or Mixtral cost the same, so a few stand for the whole stack, as in the
comparison benchmarks.  Bivatar (windowed attention over paged keys, latent
attention, a gated feed-forward, an fp32 residual) stands for the per-layer
designs: their attention layers are the same kernels.

A step has `prompts` prompt portions and `decodes` decoded tokens.  Every
portion has `rows` new tokens behind `prefix` cached ones; every decoded token
has `context` tokens up to and with itself.  `ragged` (percent) is how much
shorter the shortest of them is than the longest.
"""
from __future__ import annotations

import dataclasses
import math
import random
import zlib

import torch
import torch.nn.functional as F

from inference_gateway_amd import ops
from inference_gateway_amd.engine.config import MODEL_PRESETS, EngineConfig
from inference_gateway_amd.engine.engine import LLMEngine
from inference_gateway_amd.engine.models.batch import ForwardBatch

PAGE = 16
DEVICE = "cuda"
BIVATAR = "bivatar-4k"
MIXTRAL = "mixtral-8x7b"
LLAMAS = ("llama-3-8b", "llama-3.1-8b", "phi-3-medium")


def _step(name, model, layers, prompts=0, rows=0, prefix=0, decodes=0,
          context=0, ragged=0):
    case = dict(kind="step", model=model, layers=layers, prompts=prompts,
                rows=rows, prefix=prefix, decodes=decodes, context=context,
                ragged=ragged)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one user waiting for the next token of an answer
        _step("decode-1", "llama-3-8b", 4, decodes=1, context=700),
        # a server under ordinary load: chats of all lengths, an odd batch
        _step("decode-61-ragged", "llama-3-8b", 4, decodes=61, context=4000,
              ragged=95),
        # the serving benchmark's steady state: 1024 streams, 512 token
        # prompts, some tokens into the answer
        _step("decode-1024", "llama-3-8b", 4, decodes=1024, context=590,
              ragged=6),
        # a short question: time to first token
        _step("prefill-43", "llama-3-8b", 4, prompts=1, rows=43),
        # the serving benchmark's burst: one full prefill round
        _step("prefill-16x512", "llama-3-8b", 4, prompts=16, rows=512),
        # a long document
        _step("prefill-16000", "llama-3.1-8b", 4, prompts=1, rows=16000),
        # chunked prefill beside running answers (mixed batches)
        _step("chunk-and-decode", "llama-3.1-8b", 4, prompts=1, rows=2000,
              prefix=6000, decodes=33, context=3000, ragged=90),
        # a few users of a mixture-of-experts model
        _step("moe-decode-5", MIXTRAL, 1, decodes=5, context=1500,
              ragged=50),
        # its prompts
        _step("moe-prefill-3x700", MIXTRAL, 1, prompts=3, rows=700,
              ragged=20),
        # per-layer design: prompts beyond its window
        _step("layered-prefill-2x3000", BIVATAR, 4, prompts=2, rows=3000,
              ragged=7),
        # and a decode batch
        _step("layered-decode-48", BIVATAR, 4, decodes=48, context=3500,
              ragged=80),
        # picking 1024 tokens out of Llama-3's vocabulary
        dict(kind="sample", name="sample-1024", batch=1024, vocab=128256),
    ]


def _spread(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, round(math.exp(
        rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    what = rng.choice(["decode"] * 4 + ["prefill"] * 4 + [
        "mixed", "layered", "layered", "sample"])
    if what == "sample":
        return dict(kind="sample", batch=_spread(rng, 16, 1024),
                    vocab=rng.choice([32000, 32064, 128256]))
    if what == "layered":
        if rng.random() < 0.5:
            n = _spread(rng, 1, 8)
            return _step(None, BIVATAR, 4, prompts=n,
                         rows=_spread(rng, 30, 8000 // n),
                         ragged=rng.randint(0, 50))
        return _step(None, BIVATAR, 4, decodes=_spread(rng, 1, 128),
                     context=_spread(rng, 100, 4000),
                     ragged=rng.randint(0, 95))
    model, layers = ((MIXTRAL, 1) if rng.random() < 0.2
                     else (rng.choice(LLAMAS), 4))
    longest = min(16000, MODEL_PRESETS[model].max_position)
    if what == "decode":
        n = _spread(rng, 1, 1024 if layers == 4 else 256)
        return _step(None, model, layers, decodes=n, context=_spread(
            rng, 60, min(longest, max(80, 400000 // n))),
            ragged=rng.randint(0, 95))
    n = _spread(rng, 1, 16)
    rows = _spread(rng, 12, min(longest, 12000 // n))
    if what == "prefill":
        return _step(None, model, layers, prompts=n, rows=rows,
                     ragged=rng.randint(0, 60))
    rows = min(rows, 2048)
    return _step(None, model, layers, prompts=min(n, 4), rows=rows,
                 prefix=PAGE * _spread(rng, 1, max(2, (longest - rows) // 32)),
                 decodes=_spread(rng, 1, 64), context=_spread(rng, 60, 4000),
                 ragged=rng.randint(0, 90))


def _lengths(n, longest, ragged):
    """n whole numbers from `longest` down to (100 - ragged) % of it."""
    low = longest * (100 - ragged) // 100
    got = [max(1, longest - (longest - low) * i // max(1, n - 1))
           for i in range(n)]
    random.Random(n).shuffle(got)
    return got


def _sequences(case):
    """(cached tokens, new tokens) of every sequence, portions first."""
    portions = [(case["prefix"], r) for r in _lengths(
        case["prompts"], case["rows"], case["ragged"])]
    return portions + [(c - 1, 1) for c in _lengths(
        case["decodes"], case["context"], case["ragged"])]


def _config(case):
    cfg = MODEL_PRESETS[case["model"]]
    if case["model"] == BIVATAR:
        return cfg
    return dataclasses.replace(cfg, num_layers=case["layers"])


def _pages(case):
    return [-(-(p + n) // PAGE) for p, n in _sequences(case)]


def _inputs(case, seed):
    """Tokens, the page table (pages in the scattered order that a pool has
    after some hours) and a generator for the cached keys and values."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    seqs, pages = _sequences(case), _pages(case)
    order = torch.randperm(sum(pages), generator=g, device=DEVICE) + 1
    table = torch.zeros((len(seqs), max(pages)), dtype=torch.int32,
                        device=DEVICE)
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n].to(torch.int32)
        at += n
    tokens = torch.randint(0, _config(case).vocab_size,
                           (sum(n for _, n in seqs),), generator=g,
                           device=DEVICE)
    return tokens, table, g


def _fill(t, g):
    """Cached keys, values or latents: normed inputs through random weights
    come out with about unit variance."""
    t.normal_(0.0, 1.0, generator=g)


def _tensors(buffers):
    for b in buffers:
        if isinstance(b, torch.Tensor):
            yield b
        else:
            yield from _tensors(b)


def _rows(case, table):
    """positions, slots and sequence of every row, and cu_seqlens."""
    seqs = _sequences(case)
    dev = dict(device=DEVICE)
    lens = torch.tensor([n for _, n in seqs], **dev)
    start = torch.tensor([p for p, _ in seqs], **dev)
    cu = F.pad(lens.cumsum(0), (1, 0))
    row_seq = torch.repeat_interleave(torch.arange(len(seqs), **dev), lens)
    pos = torch.arange(int(cu[-1]), **dev) - cu[row_seq] + start[row_seq]
    slots = table[row_seq, pos // PAGE].long() * PAGE + pos % PAGE
    return pos, slots, row_seq, cu, start


def _batch(case, tokens, table, with_sequences):
    """The ForwardBatch that LLMEngine assembles for such a step."""
    def i32(t):
        return t.to(torch.int32).contiguous()

    seqs = _sequences(case)
    P, D = case["prompts"], case["decodes"]
    pos, slots, row_seq, cu, start = _rows(case, table)
    pages = _pages(case)
    last = (cu[1:] - 1).contiguous()
    fb = ForwardBatch(token_ids=tokens, positions=i32(pos),
                      slot_mapping=i32(slots), is_prefill=P > 0,
                      last_token_indices=last)
    if P:
        fb.cu_seqlens = i32(cu[:P + 1])
        fb.seq_lens = [n for _, n in seqs[:P]]
        if D:
            fb.num_prefill_tokens = int(cu[P])
            fb.decode_block_table = i32(table[P:, :max(pages[P:])])
            fb.decode_ctx_lens = i32(start[P:] + 1)
        if case["prefix"]:
            fb.block_table = i32(table[:P, :max(pages[:P])])
            fb.prefix_lens = i32(start[:P])
    else:
        fb.block_table, fb.ctx_lens = table, i32(start + 1)
    if with_sequences:
        fb.seq_cu, fb.seq_start, fb.row_seq = i32(cu), i32(start), \
            i32(row_seq)
        fb.seq_slots = torch.arange(len(seqs), dtype=torch.int32,
                                    device=DEVICE)
        fb.seq_block_table = table
        fb.seq_rows = [n for _, n in seqs]
        fb.num_chunk_rows = int(cu[P])
        fb.max_context = max(p + n for p, n in seqs)
    return fb


def _preferring(embed, router):
    """Embedding and router of a model whose tokens prefer their experts.
    Random weights leave a mixture-of-experts model without a preference:
    router logits lie so close that rounding picks the experts, and one bf16
    step before the router would be compared as another expert's output.
    Here a token's row of about unit width points to its two experts, which
    get about 0.7 and 0.3 of it, as in a trained model."""
    token = torch.arange(embed.shape[0], device=embed.device)
    E = router.shape[0]
    first = token % E
    second = (first + 1 + token // E % (E - 1)) % E
    to = F.normalize(router.float(), dim=1)
    embed = 50.0 * embed.float() + 60.0 * to[first] + 48.0 * to[second]
    return embed.to(torch.bfloat16), (0.1 * router.float()).to(torch.bfloat16)


def prepare(case, seed):
    if case["kind"] == "sample":
        return _prepare_sample(case, seed)
    tokens, table, g = _inputs(case, seed)
    seqs = _sequences(case)
    engine = LLMEngine(EngineConfig(
        model=_config(case), block_size=PAGE, num_gpu_blocks=1 + sum(
            _pages(case)), max_num_seqs=len(seqs),
        max_model_len=max(p + n for p, n in seqs) + PAGE,
        use_hip_graphs=False, enforce_eager=True), device="cuda:0")
    model, caches = engine.model, engine.kv_caches
    if case["model"] == MIXTRAL:
        named = dict(model.named_parameters())
        router = [n for n in named if n.endswith("router.weight")]
        for n, w in zip(["embed"] + router, _preferring(
                named["embed"], *(named[n] for n in router))):
            named[n].copy_(w)
    for t in _tensors(caches):
        _fill(t, g)
    fb = _batch(case, tokens, table, getattr(model, "needs_seq_meta", False))
    state = dict(kind="step", model=model, caches=caches, batch=fb)
    if not case["prompts"] and getattr(model, "supports_decode_graph", True):
        _capture(state)
    return state


def _forward(state):
    model, fb = state["model"], state["batch"]
    with torch.inference_mode():
        hidden = model(fb, state["caches"])
        rows = hidden[fb.last_token_indices] if fb.is_prefill else hidden
        return dict(hidden=hidden, logits=model.compute_logits(rows),
                    caches=list(_tensors(state["caches"])))


def _capture(state):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            _forward(state)
    torch.cuda.current_stream().wait_stream(side)
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        state["out"] = _forward(state)


def _prepare_sample(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    B, V = case["batch"], case["vocab"]
    logits = torch.randn((B, V), generator=g, device=DEVICE,
                         dtype=torch.float32)
    # a bell of unlikely tokens and a few likely ones, as a trained model's
    logits = (2.0 * logits).index_add_(
        1, torch.randint(0, V, (40,), generator=g, device=DEVICE),
        8.0 * torch.rand((B, 40), generator=g, device=DEVICE))
    # most requests take the usual settings, some are greedy, some set only
    # one of the limits, some none
    kinds = [(0.8, 50, 0.95)] * 7 + [(0.0, 0, 1.0), (1.0, 0, 0.9),
                                     (0.7, 40, 1.0), (1.0, 0, 1.0)]
    rng = random.Random(seed)
    rows = [rng.choice(kinds) for _ in range(B)]
    cols = [torch.tensor(c, dtype=dt, device=DEVICE) for c, dt in zip(
        zip(*rows), (torch.float32, torch.int32, torch.float32))]
    return dict(kind="sample", logits=logits.to(torch.bfloat16),
                temperature=cols[0], top_k=cols[1], top_p=cols[2],
                uniforms=torch.rand((B,), generator=g,
                                    device=DEVICE).clamp_(1e-6, 1 - 1e-6))


def run(state):
    if state["kind"] == "sample":
        return ops.sample(state["logits"], state["temperature"],
                          state["top_k"], state["top_p"], state["uniforms"])
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _forward(state)


# ---- what a pass cannot do without ---------------------------------------
def _visible(case, window=0, keep=0):
    """(keys read per sequence, summed; score entries, summed)."""
    keys = scores = 0
    for p, n in _sequences(case):
        if not window:
            keys += p + n
            scores += n * p + n * (n + 1) // 2
            continue
        keys += min(p + n, window + n - 1 + keep)
        for i in ((p,) if n == 1 else range(p, p + n)):
            scores += min(i + 1, window + min(keep, max(0, i + 1 - window)))
    return keys, scores


def work(case):
    if case["kind"] == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 2 * n + 20 * case["batch"], "flops": 4 * n}
    cfg = _config(case)
    D, V = cfg.hidden_size, cfg.vocab_size
    T = sum(n for _, n in _sequences(case))
    S = len(_sequences(case))
    weights, per_row, kv, flops = 0, 0, 0, 0
    for i in range(case["layers"]):
        if case["model"] == BIVATAR:
            m, ff = cfg.layers[i].mixer, 3 * D * cfg.layers[i].mlp.ff
            H = m.heads
            if cfg.layers[i].type == "attention":
                w = D * (H * m.dim + m.kv_heads * (m.dim + m.vdim) + H) \
                    + H * m.vdim * D
                width, new = m.kv_heads * (m.dim + m.vdim), True
                keys, scores = _visible(case, m.window, m.keep_first)
                flops += 2 * scores * H * (m.dim + m.vdim)
            else:
                R = m.kv_rank
                own = m.kv_from < 0
                w = D * (m.q_rank + H + (R + m.rot_dim) * own) \
                    + m.q_rank * H * (m.dim + m.rot_dim) \
                    + H * R * (m.dim + m.vdim) + H * m.vdim * D
                width, new = R + m.rot_dim, own
                keys, scores = _visible(case)
                # the cheaper of absorbed (per score) and expanded (per key)
                flops += min(
                    2 * scores * H * (2 * R + m.rot_dim),
                    2 * scores * H * (m.dim + m.vdim + m.rot_dim)
                    + 2 * keys * H * R * (m.dim + m.vdim))
            weights += w + ff
            per_row += w + ff
        else:
            H, G, hd = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
            w = D * hd * (2 * H + 2 * G)
            ff = 3 * D * cfg.intermediate_size
            E = cfg.num_experts
            if E:
                K = cfg.num_experts_per_tok
                # experts that T rows with K choices each reach on average
                weights += w + ff * E * (1 - (1 - K / E) ** T)
                per_row += w + K * ff
            else:
                weights += w + ff
                per_row += w + ff
            width, new = 2 * G * hd, True
            keys, scores = _visible(case)
            flops += 4 * scores * H * hd
        kv += width * (keys - (T if new else 0))   # read from the cache
        kv += width * T if new else 0              # and written to it
    weights += V * D
    flops += 2 * T * per_row + 2 * S * V * D
    moved = 2 * (weights + kv + 2 * T * D) + S * V * (
        4 if case["model"] == BIVATAR else 2)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        # sums of weights in another order move a threshold or a draw that
        # lies on an edge
        return {"differ": 0.01}
    # bf16 activations: measured 0.015 to 0.020 against 64 bits after four
    # Llama layers, 0.006 after four of the layers with an fp32 residual;
    # two correct implementations lie as far apart
    if case["model"] == BIVATAR:
        return {"rel": 0.02, "max": 0.5}
    return {"rel": 0.03, "max": 0.9}


# ---- the same steps in 64 bits --------------------------------------------
def _weight(shape, name, scale=1.0, dtype=torch.bfloat16, plus=0.0):
    """The synthetic initialisation: normal, 0.02 wide, seeded by the
    parameter's name; rounded to the type it is held in."""
    g = torch.Generator(device=DEVICE).manual_seed(
        zlib.crc32(name.encode()) & 0x7FFFFFFF)
    w = torch.randn(shape, generator=g, device=DEVICE) * 0.02
    return (w * scale + plus).to(dtype).double()


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, pos, inv_freq, mag=1.0):
    """x [T, heads, 2n]: pairs (i, i + n) turned by pos * inv_freq."""
    a = pos.double()[:, None, None] * inv_freq
    c, s = a.cos() * mag, a.sin() * mag
    u, v = x.chunk(2, -1)
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _softmax_attention(q, k, v, pos, scale, slopes=None, window=0, keep=0):
    """q [n, H, dk] at positions pos over k [m, G, dk], v [m, G, dv]; key j
    sits at position j."""
    n, H, _ = q.shape
    m, G, dv = v.shape
    qg = q.view(n, G, H // G, -1).permute(1, 2, 0, 3)      # [G, r, n, dk]
    kg, vg = k.permute(1, 2, 0), v.permute(1, 0, 2)        # [G, dk, m]
    out = torch.empty((n, H, dv), dtype=torch.float64, device=q.device)
    step = max(1, int(4e8) // (H * m))
    j = torch.arange(m, device=q.device)
    for a in range(0, n, step):
        p = pos[a:a + step, None]
        s = torch.matmul(qg[:, :, a:a + step], kg[:, None]) * scale
        if slopes is not None:
            s -= slopes.view(G, H // G, 1, 1) * (p - j)
        hidden = j > p
        if window:
            hidden |= (j <= p - window) & (j >= keep)
        s = s.masked_fill_(hidden, -math.inf).softmax(-1)
        out[a:a + step] = torch.matmul(s, vg[:, None]).permute(
            2, 0, 1, 3).reshape(-1, H, dv)
    return out


def _attend(case, table, pos, cu, q, caches, fn):
    """fn(q rows, keys..., positions) for every sequence, its keys gathered
    from the paged caches [pages, heads or nothing, PAGE, width]."""
    out = []
    for i, (p, n) in enumerate(_sequences(case)):
        a, b = int(cu[i]), int(cu[i + 1])
        ids = table[i, :-(-(p + n) // PAGE)].long()
        kv = [c[ids].transpose(1, 2).flatten(0, 1)[:p + n] if c.dim() == 4
              else c[ids].flatten(0, 1)[:p + n] for c in caches]
        out.append(fn(q[a:b], *kv, pos[a:b]))
    return torch.cat(out)


def _store(cache, slots, rows):
    if cache.dim() == 4:
        cache.transpose(1, 2)[slots // PAGE, slots % PAGE] = rows
    else:
        cache[slots // PAGE, slots % PAGE] = rows


def exact(case, seed):
    if case["kind"] == "sample":
        return None
    torch.cuda.empty_cache()
    tokens, table, g = _inputs(case, seed)
    fn = _exact_bivatar if case["model"] == BIVATAR else _exact_llama
    hidden, last, head, caches = fn(_config(case), case, tokens, table, g)
    return dict(hidden=hidden, logits=hidden[last] @ head.t(), caches=caches)


def _new_cache(case, g, *shape):
    t = torch.empty((1 + sum(_pages(case)),) + shape, dtype=torch.bfloat16,
                    device=DEVICE)
    _fill(t, g)
    return t.double()


def _llama_frequencies(cfg):
    f = cfg.rope_base ** (-torch.arange(
        cfg.head_dim // 2, dtype=torch.float64, device=DEVICE)
        / (cfg.head_dim // 2))
    s = cfg.rope_scaling
    if s is None:
        return f
    # Llama 3.1: long wavelengths divided by the factor, short ones kept,
    # a ramp between
    turns = s["original_max_position_embeddings"] * f / (2 * math.pi)
    ramp = ((turns - s["low_freq_factor"])
            / (s["high_freq_factor"] - s["low_freq_factor"])).clamp(0, 1)
    return f * (ramp + (1 - ramp) / s["factor"])


def _exact_llama(cfg, case, tokens, table, g):
    D, hd, H, G = (cfg.hidden_size, cfg.head_dim, cfg.num_heads,
                   cfg.num_kv_heads)
    pos, slots, _, cu, _ = _rows(case, table)
    inv = _llama_frequencies(cfg)
    x = _weight((cfg.vocab_size, D), "embed")
    if cfg.num_experts:
        x, router = (w.double() for w in _preferring(
            x, _weight((cfg.num_experts, D), "l0.router")))
    x = x[tokens]
    caches = []
    for i in range(cfg.num_layers):
        caches += [_new_cache(case, g, G, PAGE, hd),
                   _new_cache(case, g, G, PAGE, hd)]
    for i in range(cfg.num_layers):
        kc, vc = caches[2 * i:2 * i + 2]
        h = _rms(x, cfg.norm_eps)
        q, k, v = ((h @ _weight((n * hd, D), f"l{i}.{c}").t()).view(-1, n, hd)
                   for c, n in (("q", H), ("k", G), ("v", G)))
        _store(kc, slots, _turn(k, pos, inv))
        _store(vc, slots, v)
        o = _attend(case, table, pos, cu, _turn(q, pos, inv), (kc, vc),
                    lambda q, k, v, p: _softmax_attention(q, k, v, p,
                                                          hd ** -0.5))
        del q, k, v
        x = x + o.flatten(1) @ _weight((D, H * hd), f"l{i}.o").t()
        h = _rms(x, cfg.norm_eps)
        shapes = (("gate", (cfg.intermediate_size, D)),
                  ("up", (cfg.intermediate_size, D)),
                  ("down", (D, cfg.intermediate_size)))

        def swiglu(h, at):
            gate, up, down = (_weight(s, f"{at}.{n}") for n, s in shapes)
            return (F.silu(h @ gate.t()) * (h @ up.t())) @ down.t()

        if not cfg.num_experts:
            x = x + swiglu(h, f"l{i}")
            continue
        w, chosen = (h @ router.t()).topk(cfg.num_experts_per_tok, -1)
        w = w.softmax(-1)
        for e in range(cfg.num_experts):
            t, slot = (chosen == e).nonzero(as_tuple=True)
            if t.numel():
                x = x.index_add(0, t, swiglu(h[t], f"l{i}.e{e}")
                                * w[t, slot, None])
    head = _weight((cfg.vocab_size, D), "lm_head")
    return _rms(x, cfg.norm_eps), cu[1:] - 1, head, caches


def _yarn(rot):
    """(angular steps, factor on cos and sin) of YaRN interpolation."""
    def where(turns):
        return rot.dims * math.log(rot.original / (2 * math.pi * turns)) / (
            2 * math.log(rot.base))

    lo = max(math.floor(where(rot.fast)), 0)
    hi = min(math.ceil(where(rot.slow)), rot.dims - 1)
    i = torch.arange(rot.dims // 2, dtype=torch.float64, device=DEVICE)
    f = rot.base ** (-2 * i / rot.dims)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    f = f / rot.factor * ramp + f * (1 - ramp)
    return f.float().double(), 0.1 * math.log(rot.factor) + 1


def _exact_bivatar(cfg, case, tokens, table, g):
    D, eps, f32 = cfg.hidden_size, cfg.norm_eps, torch.float32
    pos, slots, _, cu, _ = _rows(case, table)

    def w(shape, name, fan_in, norm=False):
        if norm:
            return _weight(shape, name, fan_in, f32, 1.0)
        return _weight(shape, name, fan_in ** -0.5 / 0.02)

    held = {}
    for i, layer in enumerate(cfg.layers):
        m = layer.mixer
        if layer.type == "attention":
            held[i] = (_new_cache(case, g, m.kv_heads, PAGE, m.dim),
                       _new_cache(case, g, m.kv_heads, PAGE, m.vdim))
        elif m.kv_from < 0:
            held[i] = (_new_cache(case, g, PAGE, m.kv_rank + m.rot_dim),)
    x = _weight((cfg.vocab_size, D), "embed", 50.0 / cfg.embed_scale)[
        tokens] * cfg.embed_scale
    for i, layer in enumerate(cfg.layers):
        m, at = layer.mixer, f"l{i}.mix"
        H = m.heads
        if layer.type == "attention":
            G, N, P = m.kv_heads, m.dim, m.vdim
            z = x @ w((H * N + G * N + G * P + H, D), at + ".qkvg", D).t()
            q, k, v, gate = z.split([H * N, G * N, G * P, H], -1)
            q = _rms(q.unflatten(1, (H, N)), eps) * w((N,), at + ".q.norm",
                                                      5.0, True)
            k = _rms(k.unflatten(1, (G, N)), eps) * w((N,), at + ".k.norm",
                                                      5.0, True)
            _store(held[i][0], slots, k)
            _store(held[i][1], slots, v.unflatten(1, (G, P)))
            slopes = 2.0 ** (-8.0 * torch.arange(
                1, H + 1, dtype=torch.float64, device=DEVICE) / H) \
                if m.distance_bias else None
            o = _attend(case, table, pos, cu, q, held[i],
                        lambda q, k, v, p: _softmax_attention(
                            q, k, v, p, m.scale, slopes, m.window,
                            m.keep_first))
            o = o * gate.sigmoid()[..., None]
            y = o.flatten(1) @ w((D, H * P), at + ".o", H * P).t()
        else:
            R, rd, dn, qr = m.kv_rank, m.rot_dim, m.dim, m.q_rank
            own = m.kv_from < 0
            inv, mag = _yarn(m.rot)
            rows = qr + H + (R + rd if own else 0)
            z = x @ w((rows, D), at + ".down", D).t()
            cq = _rms(z[:, :qr], eps) * w((qr,), at + ".qn", 2.0, True)
            if own:
                c = _rms(z[:, qr:qr + R], eps) * w((R,), at + ".kvn", 2.0,
                                                   True)
                kr = _turn(z[:, None, qr + R:qr + R + rd], pos, inv, mag)
                _store(held[i][0], slots, torch.cat([c, kr[:, 0]], -1))
            gate = z[:, -H:].sigmoid()
            q = (cq @ w((H * (dn + rd), qr), at + ".uq", qr).t()).unflatten(
                1, (H, dn + rd))
            q_lat = torch.einsum("thd,hdr->thr", q[..., :dn],
                                 w((H, dn, R), at + ".uk", R))
            q = torch.cat([q_lat, _turn(q[..., dn:], pos, inv, mag)], -1)
            o = _attend(case, table, pos, cu, q, held[i if own else
                                                      m.kv_from],
                        lambda q, c, p: _softmax_attention(
                            q, c[:, None], c[:, None, :R], p, m.scale))
            o = torch.einsum("thr,hrv->thv", o * gate[..., None],
                             w((H, R, m.vdim), at + ".uv", R))
            y = o.flatten(1) @ w((D, H * m.vdim), at + ".o", H * m.vdim).t()
        x = x + cfg.residual_mult * _rms(y, eps) * w(
            (D,), f"l{i}.norm1", 5.0, True)
        ff = layer.mlp.ff
        gate, up = (x @ w((2 * ff, D), f"l{i}.mlp.gate_up", D).t()).chunk(
            2, -1)
        y = (F.gelu(gate, approximate="tanh") * up) @ w(
            (D, ff), f"l{i}.mlp.down", ff).t()
        x = x + cfg.residual_mult * _rms(y, eps) * w(
            (D,), f"l{i}.norm2", 5.0, True)
    hidden = _rms(x, eps) * w((D,), "final.norm", 5.0, True)
    head = w((cfg.vocab_size, D), "head", D)
    return hidden, cu[1:] - 1, head, [t for i in sorted(held)
                                      for t in held[i]]
