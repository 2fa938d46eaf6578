"""The forward passes that serving spends its time in, with random weights and tokens.

Every case is one engine step of one model: a step that brings prompt tokens (``step`` "prompt": whole prompts, portions
behind a part that is cached already, several prompts of unequal length in one batch, running decodes riding along) or a
step of single tokens (``step`` "decode": replayed from a captured graph, as the engine's decode loop does).  Models: the
Llama of the decision service at the 70B's layer shapes, and three of the designs with an fp32 residual stream at the
layer sizes of ``bench.py --model-bench`` -- between them recurrent, linear, latent and windowed attention, dense
feed-forwards and experts.  A pass returns the wanted rows' logits, the paged caches and the recurrent states.

Fields of a case: ``model``, ``width`` (2048 / 4096; Llama: 8192), ``dtype``, ``step``, ``prompts`` (sequences that bring
prompt tokens), ``tokens`` (prompt tokens brought by all of them), ``past`` (tokens of each that are cached already),
``rows`` (sequences that bring one token), ``context`` (the longest of those sequences, that token included)."""

from __future__ import annotations

import gc
import math

import torch

from k8s_llm_scheduler_amd.models import favizen, katidra, putulorn
from k8s_llm_scheduler_amd.models.config import get_config
from k8s_llm_scheduler_amd.models.llama import LlamaModel

F64 = torch.float64
PAGE = 16                  # tokens of a cache page (the engine's block size)
MAX_LEN = 4096             # engine.max_model_len of the benchmark
MAX_PREFILL = 8192         # engine.max_prefill_tokens
VOCAB = 32768
LLAMA = "llama-3.3-70b@L4"     # the 70B's layer and vocabulary shapes, 4 of its 80 layers
# width: (layer pairs, feed-forward, heads, expert feed-forward, experts), as bench.py --model-bench
SIZES = {2048: (4, 8192, 16, 2048, 8), 4096: (2, 14336, 32, 3584, 8)}


def _case(name, model, width, step, *, tokens=0, prompts=0, past=0, rows=0, context=0, dtype="bfloat16"):
    c = dict(model=model, width=width, dtype=dtype, step=step, prompts=prompts, tokens=tokens, past=past, rows=rows,
             context=context)
    return {"name": name, **c} if name else c


def listed():
    return [
        # the decision service's single-pod loop: the 3-node prompt's tokens behind the cached system prompt ...
        _case("llama-decision-prompt", "llama", 8192, "prompt", tokens=241, prompts=1, past=224),
        # ... and every token of the answer
        _case("llama-decode-1", "llama", 8192, "decode", rows=1, context=497),
        # the prompt of a 64-node cluster
        _case("llama-prompt-64-nodes", "llama", 8192, "prompt", tokens=3413, prompts=1),
        # model-bench prefill and decoding of the recurrent / latent-attention design
        _case("putulorn-prompt", "putulorn", 2048, "prompt", tokens=2048, prompts=1),
        _case("putulorn-decode-8", "putulorn", 2048, "decode", rows=8, context=529),
        # the same design in true fp32 (--dtype float32)
        _case("putulorn-prompt-fp32", "putulorn", 2048, "prompt", tokens=333, prompts=1, dtype="float32"),
        # the linear / latent-attention design: a long prompt, a prompt at the wide size, one stream decoding
        _case("katidra-prompt", "katidra", 2048, "prompt", tokens=2048, prompts=1),
        _case("katidra-prompt-wide", "katidra", 4096, "prompt", tokens=512, prompts=1),
        _case("katidra-decode-1", "katidra", 2048, "decode", rows=1, context=529),
        # windowed attention and experts: a mixed step (five unequal prompts, three decodes riding along), a full batch
        # decoding, a short portion behind a long cached one
        _case("favizen-mixed-step", "favizen", 2048, "prompt", tokens=1531, prompts=5, rows=3, context=700),
        _case("favizen-decode-32", "favizen", 2048, "decode", rows=32, context=545),
        _case("favizen-portion", "favizen", 2048, "prompt", tokens=97, prompts=1, past=1000),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(("llama", "putulorn", "katidra", "favizen"))
    width = 8192 if model == "llama" else rng.choice((2048, 2048, 4096))
    if rng.random() < 0.4:
        rows = _log_uniform(rng, 1, 32)
        return _case(None, model, width, "decode", rows=rows, context=_log_uniform(rng, 48, 1500))
    fp32 = model != "llama" and rng.random() < 0.2
    tokens = _log_uniform(rng, 24, 3400 if model == "llama" else 512 if fp32 else 2048)
    prompts = 1 if rng.random() < 0.5 else rng.randint(2, max(2, min(8, tokens // 8)))
    past = PAGE * rng.randint(1, 64) if rng.random() < 0.3 else 0
    rows = rng.randint(1, 8) if rng.random() < 0.3 else 0
    return _case(None, model, width, "prompt", tokens=tokens, prompts=prompts, past=past, rows=rows,
                 context=_log_uniform(rng, 48, 1500) if rows else 0, dtype="float32" if fp32 else "bfloat16")


# ----------------------------------------------------------------------------- what a case consists of
def _sequences(case):
    """[(tokens cached already, tokens brought)] of the step's sequences, unequal lengths."""
    n = case["prompts"]
    weight = [2 + (3 * i) % 5 for i in range(n)]
    new = [max(1, case["tokens"] * w // sum(weight)) for w in weight]
    if n:
        new[-1] += case["tokens"] - sum(new)
    seqs = [(case["past"], k) for k in new]
    c = case["context"]
    return seqs + [(max(0, c - 1 - (i * 29) % (c // 2 + 1)), 1) for i in range(case["rows"])]


def _config(case):
    w = case["width"]
    if case["model"] == "llama":
        return get_config(LLAMA)
    pairs, ff, heads, eff, experts = SIZES[w]
    if case["model"] == "putulorn":
        return putulorn.preset("putulorn", w, VOCAB, pairs, heads=heads, wkv_dim=64, dim=128, rot_dim=64, vdim=128,
                               kv_rank=512, window=1024, ff=ff)
    if case["model"] == "katidra":
        return katidra.preset("katidra", w, VOCAB, ("lightning", "latent_attention") * pairs, heads=heads, dim=128,
                              rot_dim=64, vdim=128, kv_rank=512, q_rank=w * 3 // 4, window=1024, scan_heads=w // 128,
                              scan_dim=128, scan_vdim=128, ff=ff)
    return favizen.preset("favizen", w, VOCAB, ("attention", "attention_2", "attention", "shared") * (pairs // 2),
                          heads=heads, kv_heads=heads // 4, dim=128, window=1024, rot_dims=64, side_heads=heads,
                          side_kv_heads=heads // 4, side_dim=128, chunk=1024, ff=ff, experts=experts, top=2,
                          expert_ff=eff, shared_ff=eff, mlps=("moe",))


DESIGNS = {"putulorn": (putulorn, putulorn.PutulornModel), "katidra": (katidra, katidra.KatidraModel),
           "favizen": (favizen, favizen.FavizenModel)}


def _weights(case, seed):
    """The checkpoint tensors of a stream design (random, from the seed)."""
    return DESIGNS[case["model"]][0].random_tensors(_config(case), seed, "cuda")


def _llama(case, seed):
    return LlamaModel(_config(case), device="cuda", seed=seed, max_model_len=MAX_LEN)


def _layout(case, seed):
    """Tokens, cache pages and cache slots of the step's sequences (the pages of a sequence lie scattered)."""
    g = torch.Generator().manual_seed(seed)
    seqs = _sequences(case)
    vocab = get_config(LLAMA).vocab if case["model"] == "llama" else VOCAB
    toks = [torch.randint(0, vocab - 512, (a + n,), generator=g) for a, n in seqs]
    need = [-(-len(t) // PAGE) for t in toks]
    order = torch.randperm(sum(need), generator=g)
    pages, at = [], 0
    for k in need:
        pages.append(order[at:at + k])
        at += k
    slots = [(p[:, None] * PAGE + torch.arange(PAGE)).reshape(-1)[:len(t)] for p, t in zip(pages, toks)]
    return seqs, toks, pages, slots, sum(need)


# ----------------------------------------------------------------------------- the framework's side
def _varlen(model, pick, toks, pages, slots, spans):
    """Arguments of ``forward_prefill`` for the spans [(first, end)] of the sequences ``pick``."""
    i32 = lambda x: x.to(torch.int32).cuda()
    ids = torch.cat([toks[i][a:b] for i, (a, b) in zip(pick, spans)])
    pos = torch.cat([torch.arange(a, b) for a, b in spans])
    slot = torch.cat([slots[i][a:b] for i, (a, b) in zip(pick, spans)])
    cu = torch.tensor([0] + [b - a for a, b in spans]).cumsum(0)
    tables = torch.zeros(len(pick), MAX_LEN // PAGE, dtype=torch.int32)
    for r, i in enumerate(pick):
        tables[r, :len(pages[i])] = pages[i].to(torch.int32)
    args = (i32(ids), i32(pos), i32(slot), i32(cu), i32(torch.tensor([b for _, b in spans])), tables.cuda(),
            max(b - a for a, b in spans), i32(cu[1:] - 1))
    kw = {"seq_slots": i32(torch.tensor(pick))} if getattr(model, "stateful", False) else {}
    return args, kw


def prepare(case, seed):
    seqs, toks, pages, slots, n_pages = _layout(case, seed)
    if case["model"] == "llama":
        model = _llama(case, seed)
    else:
        dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
        model = DESIGNS[case["model"]][1](_config(case), device="cuda", dtype=dtype, tensors=_weights(case, seed),
                                          max_model_len=MAX_LEN)
    model.allocate_kv(n_pages, PAGE)
    stateful = getattr(model, "stateful", False)
    if stateful:
        model.allocate_state(len(seqs))
    state = {"model": model}
    if case["step"] == "decode":
        n = len(seqs)
        tokens = torch.stack([t[-1] for t in toks]).to(torch.int32).cuda()
        tables = torch.zeros(n, MAX_LEN // PAGE, dtype=torch.int32)
        for r in range(n):
            tables[r, :len(pages[r])] = pages[r].to(torch.int32)
        ctx = torch.zeros(n, dtype=torch.int32, device="cuda")      # idle rows while the graph is captured
        args = (tokens, ctx, tables.cuda(), 1024 if case["context"] <= 1024 else MAX_LEN)
        collecting = gc.isenabled()
        gc.collect()
        gc.disable()
        try:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                model.forward_decode(*args)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                logits = model.forward_decode(*args)
        finally:
            if collecting:
                gc.enable()
        state.update(graph=graph, logits=logits, inputs=args)
        ctx.copy_(torch.tensor([len(t) for t in toks], dtype=torch.int32))
    else:
        state["args"], state["kw"] = _varlen(model, range(len(seqs)), toks, pages, slots, [(a, a + n) for a, n in seqs])
    # what is cached already: brought in earlier steps of at most MAX_PREFILL tokens
    pick, held = [], 0
    for i, (past, _) in enumerate(seqs):
        if past and held + past > MAX_PREFILL:
            args, kw = _varlen(model, pick, toks, pages, slots, [(0, seqs[j][0]) for j in pick])
            model.forward_prefill(*args, **kw)
            pick, held = [], 0
        if past:
            pick, held = pick + [i], held + past
    if pick:
        args, kw = _varlen(model, pick, toks, pages, slots, [(0, seqs[j][0]) for j in pick])
        model.forward_prefill(*args, **kw)
    return state


def run(state):
    m = state["model"]
    if "graph" in state:
        state["graph"].replay()
        logits = state["logits"]
    else:
        logits = m.forward_prefill(*state["args"], **state["kw"])
    return {"logits": logits, "cache": m.kv_cache, "states": getattr(m, "states", [])}


# ----------------------------------------------------------------------------- work and tolerance
def _visible(seqs, window, chunk):
    """Query-key pairs of the step's tokens."""
    n = 0
    for past, new in seqs:
        for p in range(past, past + new):
            n += p % chunk + 1 if chunk else min(p + 1, window) if window else p + 1
    return n


def work(case):
    """Products with every weight matrix once per token, attention over the visible keys at the heads' own sizes; every
    weight, every visible cache row and every state read once, new cache rows, states and logits written once."""
    cfg, seqs, w = _config(case), _sequences(case), case["width"]
    T, S = sum(n for _, n in seqs), len(seqs)
    eb = 4 if case["dtype"] == "float32" else 2
    per_token = weights = flops = other = 0.0       # multiply-adds of the matrices, their values; the rest

    def matrix(*values):
        nonlocal per_token, weights
        per_token += sum(values)
        weights += sum(values)

    def attention(heads, dk, dv, row, window=0, chunk=0, writes=True):
        nonlocal flops, other
        flops += 2.0 * heads * (dk + dv) * _visible(seqs, window, chunk)
        seen = sum(min(a + n, (window or a + n) + n - 1, (a + n if not chunk else (a % chunk) + n)) for a, n in seqs)
        other += eb * row * (seen + (T if writes else 0))

    if case["model"] == "llama":
        D, H, G, I = cfg.head_dim, cfg.num_heads, cfg.num_kv_heads, cfg.intermediate
        for _ in range(cfg.num_layers):
            matrix(w * (H + 2 * G) * D, H * D * w, 3 * w * I)
            attention(H, D, D, 2 * G * D)
    for L in [] if case["model"] == "llama" else cfg.layers:
        m = L.mixer
        kind = getattr(L, "type", "") or m.type
        if kind == "wkv":
            hd = m.heads * m.dim
            matrix(5 * w * hd, 2 * hd * max(8, hd // 16))
            flops += 8.0 * T * hd * m.dim
            other += 8.0 * S * hd * m.dim
        elif kind == "lightning":
            matrix(w * m.heads * (2 * m.dim + 2 * m.vdim), w * m.heads * m.vdim)
            flops += 6.0 * T * m.heads * m.dim * m.vdim
            other += 8.0 * S * m.heads * m.dim * m.vdim
        elif kind == "latent_attention":
            q_rank = getattr(m, "q_rank", 0)
            q = m.heads * (m.dim + m.rot_dim)
            matrix(*((w * q_rank, q_rank * q, w * m.heads) if q_rank else (w * q,)), w * (m.kv_rank + m.rot_dim),
                   m.heads * m.kv_rank * (m.dim + m.vdim), w * m.heads * m.vdim)
            attention(m.heads, m.dim + m.rot_dim, m.vdim, m.kv_rank + m.rot_dim, m.window)
        else:
            own = m.kv_from is None
            matrix(w * m.heads * (m.dim + 1), w * m.heads * m.vdim)
            if own:
                matrix(w * m.kv_heads * (m.dim if m.tied_values else m.dim + m.vdim))
            attention(m.heads, m.dim, m.vdim, m.kv_heads * (m.dim + m.vdim), m.window, m.chunk, own)
        if case["model"] == "putulorn":
            matrix(3 * w * L.mlp.ff)
        elif case["model"] == "katidra":
            matrix(2 * w * L.ff)
        else:
            f = L.mlp
            matrix(3 * w * f.shared_ff + w)
            per_token += 3 * w * f.ff * f.top
            weights += 3 * w * f.ff * f.experts * (1.0 - (1.0 - f.top / f.experts) ** T)
    head = w * cfg.vocab
    return {"bytes": eb * (weights + head + T * w) + other + 4.0 * S * cfg.vocab,
            "flops": 2.0 * (T * per_token + S * head) + flops}


def tolerance(case):
    """Four times what the outputs of one prompt brought whole and in two portions differ by (other tiles, splits and
    batches in every product): 3.5e-6 in fp32, 6e-3 to 1.6e-2 in bf16, whose bound is rounded down to 3e-2."""
    return {"rel": 1.5e-5 if case["dtype"] == "float32" else 3e-2}


# ----------------------------------------------------------------------------- the same in 64 bits
def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _angles(dims, base, T, kind=None, sc=None):
    """cos, sin [T, dims / 2] of the rotary positions; ``kind`` "llama3" or "yarn" with the constants ``sc``."""
    freq, mag = [], 1.0
    if kind == "yarn":
        turn = lambda t: dims * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
        lo, hi = max(math.floor(turn(sc["fast"])), 0), min(math.ceil(turn(sc["slow"])), dims - 1)
        mag = 0.1 * math.log(sc["factor"]) + 1.0
    for i in range(dims // 2):
        f = base ** (-2.0 * i / dims)
        if kind == "llama3":
            wave = 2.0 * math.pi / f
            if wave > sc["original"] / sc["low"]:
                f /= sc["factor"]
            elif wave >= sc["original"] / sc["high"]:
                s = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
                f = (1.0 - s) * f / sc["factor"] + s * f
        elif kind == "yarn":
            r = min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0)
            f = f / sc["factor"] * r + f * (1.0 - r)
        freq.append(f)
    a = torch.arange(T, dtype=F64, device="cuda")[:, None] * torch.tensor(freq, dtype=F64, device="cuda")
    return mag * torch.cos(a), mag * torch.sin(a)


def _turn(x, cs, interleaved=False):
    """x [T, heads, D]: the first dims dimensions turned, as halves or as interleaved pairs."""
    c, s = (t[:x.shape[0], None, :] for t in cs)
    n = 2 * c.shape[2]
    a, b = (x[..., 0:n:2], x[..., 1:n:2]) if interleaved else (x[..., :n // 2], x[..., n // 2:n])
    u, v = a * c - b * s, b * c + a * s
    turned = torch.stack([u, v], -1).flatten(-2) if interleaved else torch.cat([u, v], -1)
    return torch.cat([turned, x[..., n:]], -1)


def _attend(q, k, v, scale, window=0, chunk=0, sinks=None, slopes=None):
    """q [T, H, D] over k [T, G, D], v [T, G, V]: softmax over the visible earlier tokens; a key head at a time."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    i = torch.arange(T, device="cuda")
    age = i[:, None] - i[None, :]
    hide = age < 0
    if window:
        hide |= age >= window
    if chunk:
        hide |= (i[:, None] // chunk) != (i[None, :] // chunk)
    out = []
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h] @ k[:, g].T) * scale
        if slopes is not None:
            s -= slopes[h] * age
        s.masked_fill_(hide, -math.inf)
        if sinks is not None:
            s = torch.cat([s, sinks[h].expand(T, 1)], 1)
        out.append(torch.softmax(s, -1)[:, :T] @ v[:, g])
    return torch.stack(out, 1)


def _latent(P, p, m, eps, h, q, cs, interleaved):
    """(heads' attended values [T, H, V], the cached rows) of a latent attention with the queries q [T, H, D + R]."""
    C, T = m.kv_rank, h.shape[0]
    q = torch.cat([q[..., :m.dim], _turn(q[..., m.dim:], cs, interleaved)], -1)
    down = h @ P(p + "dkv").T
    c = _unit(down[:, :C], eps) * P(p + "dkv.norm")
    kr = _turn(down[:, None, C:], cs, interleaved)
    k = torch.cat([(c @ P(p + "uk").T).view(T, m.heads, m.dim), kr.expand(T, m.heads, m.rot_dim)], -1)
    v = (c @ P(p + "uv").T).view(T, m.heads, m.vdim)
    return _attend(q, k, v, m.scale, m.window), torch.cat([c, kr[:, 0]], 1)


def _putulorn(P, cfg, ids):
    eps, x, caches, states = cfg.rms_eps, P("embed")[ids], [], []
    T = len(ids)
    norm = lambda y, n: _unit(y, eps) * (1.0 + P(n))
    for i, L in enumerate(cfg.layers):
        p, m = f"l{i}.mix.", L.mixer
        h = norm(x, f"l{i}.norm1")
        if m.type == "wkv":
            before = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
            mix = lambda s: h + (before - h) * P(p + "mu." + s)
            r, k, v, g = ((mix(s) @ P(p + s).T).view(T, m.heads, m.dim) for s in ("r", "k", "v", "g"))
            z = torch.tanh(mix("w") @ P(p + "w1").T) @ P(p + "w2").T + P(p + "w0")
            decay = torch.exp(-torch.exp(z)).view(T, m.heads, m.dim, 1)
            u = P(p + "u").view(m.heads, m.dim, 1)
            S, o = torch.zeros(m.heads, m.dim, m.dim, dtype=F64, device="cuda"), []
            for t in range(T):
                kv = k[t, :, :, None] * v[t, :, None, :]
                o.append(((S + u * kv) * r[t, :, :, None]).sum(1))
                S = decay[t] * S + kv
            y = _unit(torch.stack(o), eps).reshape(T, -1) * P(p + "norm") * torch.nn.functional.silu(g).reshape(T, -1)
            states.append((S, h[-1]))
        else:
            q = (h @ P(p + "q").T).view(T, m.heads, m.dim + m.rot_dim)
            y, row = _latent(P, p, m, eps, h, q, _angles(m.rot_dims, m.rot_base, T), False)
            caches.append(row)
        x = x + y.reshape(T, -1) @ P(p + "o").T
        h, f = norm(x, f"l{i}.norm2"), f"l{i}.mlp."
        x = x + (torch.nn.functional.gelu(h @ P(f + "gate").T, approximate="tanh") * (h @ P(f + "up").T)) @ P(f + "down").T
    return norm(x[-1], "final.norm") @ P("head").T, caches, states


def _katidra(P, cfg, ids):
    eps, x, caches, states = cfg.rms_eps, P("embed")[ids] * cfg.embed_scale, [], []
    T = len(ids)
    silu = torch.nn.functional.silu
    norm = lambda y, n: _unit(y, eps) * P(n)
    for i, L in enumerate(cfg.layers):
        p, m = f"l{i}.mix.", L.mixer
        if L.type == "lightning":
            q, k, v = (silu(x @ P(p + s).T).view(T, m.heads, -1) for s in ("q", "k", "v"))
            age = torch.arange(T, dtype=F64, device="cuda")
            age = age[:, None] - age[None, :]
            y, S = [], []
            for h, a in enumerate(m.decay):
                fade = torch.where(age >= 0, a ** age.clamp(min=0.0), 0.0)
                y.append((fade * (q[:, h] @ k[:, h].T)) @ v[:, h])
                S.append((k[:, h] * fade[-1][:, None]).T @ v[:, h])
            y = norm(torch.stack(y, 1).reshape(T, -1), p + "norm") * torch.sigmoid(x @ P(p + "g").T)
            states.append(torch.stack(S).reshape(m.heads, -1))
        else:
            q = (norm(x @ P(p + "dq").T, p + "dq.norm") @ P(p + "uq").T).view(T, m.heads, m.dim + m.rot_dim)
            cs = _angles(m.rot_dims, m.rot_base, T, "yarn" if m.yarn else None, m.yarn)
            y, row = _latent(P, p, m, eps, x, q, cs, True)
            y = y * torch.sigmoid(x @ P(p + "g").T)[:, :, None]
            caches.append(row)
        x = x + norm(y.reshape(T, -1) @ P(p + "o").T, f"l{i}.norm1")
        f = torch.clamp(x @ P(f"l{i}.mlp.up").T, min=0.0) ** 2 @ P(f"l{i}.mlp.down").T
        x = x + norm(f, f"l{i}.norm2")
    return norm(x[-1], "final.norm") @ P("head").T, caches, states


def _favizen(P, cfg, ids):
    eps, x, caches, states, kv = cfg.rms_eps, P("embed")[ids] * cfg.embed_scale, [], [], {}
    T = len(ids)
    norm = lambda y, n: _unit(y, eps) * P(n)

    def glu(h, f, limit):
        g, u = (h @ P(f + "gate").T).clamp(max=limit), (h @ P(f + "up").T).clamp(-limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ P(f + "down").T

    for i, L in enumerate(cfg.layers):
        p, m, f = f"l{i}.mix.", L.mixer, L.mlp
        h = norm(x, f"l{i}.norm1")
        names = ["q"] + ([] if m.kv_from is not None else ["k"] if m.tied_values else ["k", "v"])
        parts = [h @ P(p + n).T for n in names]
        if m.conv:
            parts = [y + P(f"{p}{n}.b") for n, y in zip(names, parts)]
            full = torch.nn.functional.pad(torch.cat(parts, 1), (0, 0, m.conv - 1, 0))
            states.append(full[T:])
            taps = torch.cat([P(f"{p}{n}.conv") for n in names])
            y = sum(full[j:j + T] * taps[:, j] for j in range(m.conv))
            parts = list(y.split([t.shape[1] for t in parts], 1))
        q = parts[0].view(T, m.heads, m.dim)
        if m.kv_from is None:
            k, v = parts[1].view(T, m.kv_heads, -1), parts[-1].view(T, m.kv_heads, -1)
        slopes = torch.exp2(-8.0 * torch.arange(1, m.heads + 1, dtype=F64, device="cuda") / m.heads) if m.distance else None
        if m.rot_dims:
            cs = _angles(m.rot_dims, m.rot_base, T, "llama3" if m.rot_scaling else None, m.rot_scaling)
            q, k = _turn(q, cs), _turn(k, cs)
        if m.kv_from is None:
            kv[i] = (k, v)
            caches.append((k, v))
        k, v = kv[i if m.kv_from is None else m.kv_from]
        y = _attend(q, k, v, m.scale, m.window, m.chunk, P(p + "sink"), slopes)
        y = y * torch.sigmoid(h @ P(p + "g").T)[:, :, None]
        x = x + norm(y.reshape(T, -1) @ P(p + "o").T, f"l{i}.norm1b")
        h, q = norm(x, f"l{i}.norm2"), f"l{i}.mlp."
        y = glu(h, q + "shared.", f.shared_limit) * torch.sigmoid(h @ P(q + "shared.sg").T)
        table = P(q + "table", torch.long)[ids]
        for e in range(f.experts):
            rows = (table == e).any(1).nonzero()[:, 0]
            if len(rows):
                y[rows] += glu(h[rows], f"{q}e{e}.", f.limit) / f.top
        x = x + norm(y, f"l{i}.norm2b")
    return norm(x[-1], "final.norm") @ P("head").T * cfg.logit_scale, caches, states


def _llama64(model, cfg, ids):
    D, H, G, I = cfg.head_dim, cfg.num_heads, cfg.num_kv_heads, cfg.intermediate
    T, caches = len(ids), []
    s = cfg.rope_scaling
    sc = {"factor": s["factor"], "low": s["low_freq_factor"], "high": s["high_freq_factor"],
          "original": s["original_max_position_embeddings"]}
    cs = _angles(D, cfg.rope_theta, T, "llama3", sc)
    x = model.embed[ids].to(F64)
    for w in model.layers:                    # the norms' weights are folded into the projections behind them
        y = (_unit(x, cfg.rms_eps) @ w.wqkv.to(F64).T).view(T, H + 2 * G, D)
        q, k, v = _turn(y[:, :H], cs), _turn(y[:, H:H + G], cs), y[:, H + G:]
        caches.append(torch.stack([k, v]))
        x = x + _attend(q, k, v, 1.0 / math.sqrt(D)).reshape(T, -1) @ w.wo.to(F64).T
        y = _unit(x, cfg.rms_eps) @ w.wgu.to(F64).T
        x = x + (torch.nn.functional.silu(y[:, :I]) * y[:, I:]) @ w.wdown.to(F64).T
    return _unit(x[-1], cfg.rms_eps) @ model.lm_head.to(F64).T, torch.stack(caches), []


def exact(case, seed):
    cfg = _config(case)
    seqs, toks, _, slots, n_pages = _layout(case, seed)
    if case["model"] == "llama":
        model = _llama(case, seed)
        forward = lambda ids: _llama64(model, cfg, ids)
    else:
        tensors = _weights(case, seed)
        P = lambda name, dtype=F64: tensors[name].to(dtype)
        f = {"putulorn": _putulorn, "katidra": _katidra, "favizen": _favizen}[case["model"]]
        forward = lambda ids: f(P, cfg, ids)
    logits, cache, states = [], None, None
    n = n_pages * PAGE
    new = lambda first, *shape: torch.zeros(first, *shape, dtype=F64, device="cuda")
    for i, t in enumerate(toks):
        z, c, s = forward(t.cuda())
        logits.append(z)
        at = slots[i].cuda()
        if case["model"] == "llama":                      # [layers, 2, tokens, heads, dim]
            if cache is None:
                cache = torch.zeros(*c.shape[:2], n, *c.shape[3:], dtype=F64, device="cuda")
            cache[:, :, at] = c
            states = []
            continue
        if cache is None:
            pair = isinstance(c[0], tuple)
            cache = [tuple(new(n, *y.shape[1:]) for y in x) if pair else new(n, *x.shape[1:]) for x in c]
            states = [tuple(new(len(toks), *y.shape) for y in x) if isinstance(x, tuple) else new(len(toks), *x.shape)
                      for x in s]
        for dst, src in zip(cache, c):
            for d, r in zip(dst, src) if isinstance(dst, tuple) else ((dst, src),):
                d[at] = r
        for dst, src in zip(states, s):
            for d, r in zip(dst, src) if isinstance(dst, tuple) else ((dst, src),):
                d[i] = r
    return {"logits": torch.stack(logits)[None], "cache": cache, "states": states}
