"""Kernels of the fp32-stream designs at the edges of their tiles and dispatch rules, against the fp32 reference ops or 64
bits."""

import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture
def entries(monkeypatch):
    """Names of the extension's entry points in the order of their calls."""
    nat, calls = ops.native(), []

    class Spy:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Spy)
    return calls


def sum_bound(a, w):
    """Elementwise bound on |fp32 product - exact| for any order of the K products: K 2^-24 sum |a| |w| (twice that)."""
    return 2.0 * a.shape[-1] * 2.0 ** -24 * (a.double().abs() @ w.double().abs().transpose(-1, -2)) + 1e-30


@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (31, 33, 60), (32, 32, 64), (33, 65, 68), (64, 64, 256), (97, 130, 260),
                                   (40, 16388, 8), (1031, 576, 132), (256, 2048, 320)])
def test_fp32_products(M, N, K):
    """Both tile shapes of gemm_f32_kernel (every depth here is below 512), remainders in every dimension, an odd row stride, a
    batch."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K + 4, generator=g)[:, :K], torch.randn(N, K, generator=g)
    a[:, 0] *= 1e4
    ag = torch.randn(M, K + 4, generator=g).to(DEV)[:, :K].copy_(a)
    exact = a.double() @ w.double().T
    assert ((sm.gemm(ag, w.to(DEV)).cpu().double() - exact).abs() <= sum_bound(a, w)).all()
    b = torch.stack([a, 2.0 * a])
    got = sm.gemm(b.to(DEV), torch.stack([w, w]).to(DEV)).cpu()
    assert torch.equal(got[1], 2.0 * got[0])
    assert torch.equal(got[0], sm.gemm(ag, w.to(DEV)).cpu())      # within this kernel the order of the sums depends on K alone
    assert torch.equal(got[0][M // 2:], sm.gemm(ag[M // 2:], w.to(DEV)).cpu())


@pytest.mark.parametrize("tokens,top,E", [(5, 2, 3), (150, 2, 3), (400, 1, 2)])
def test_fp32_grouped_products(tokens, top, E):
    g = torch.Generator().manual_seed(tokens)
    N, K = 72, 132
    idx = torch.rand(tokens, E, generator=g).argsort(1)[:, :top].to(torch.int32)
    rows, pos, seg, tiles = sm.moe_align(idx.to(DEV), E)
    h, w = torch.randn(tokens, K, generator=g), torch.randn(E, N, K, generator=g)
    got = sm.gemm(h.to(DEV), w.to(DEV), a_rows=rows, tiles=tiles, rows=tokens * top).cpu().double()[pos.cpu().long()]
    for t in range(tokens):
        for c in range(top):
            e = int(idx[t, c])
            y = got.view(tokens, top, N)[t, c]
            assert ((y - h[t].double() @ w[e].double().T).abs() <= sum_bound(h[t:t + 1], w[e])[0]).all()


# ----------------------------------------------------------------------------- latent attention of prompts
# (tokens cached already, tokens brought) of every sequence; window.  Portions at the edges of the 64- and 128-token tiles,
# windows cutting inside a step, a window of one, sequences without tokens, single tokens riding along behind long contexts,
# many heads (the two tile heights of the bf16 kernel)
LATENT = [([(0, 200)], 0, 3), ([(0, 64), (0, 449)], 100, 2), ([(37, 191), (0, 0), (5, 129)], 64, 2),
          ([(700, 1), (0, 640), (333, 1), (16, 2)], 300, 16), ([(0, 513)], 1, 1), ([(0, 1153)], 513, 32),
          ([(48, 400), (2, 300)], 0, 8)]


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("seqs,window,H", LATENT)
@pytest.mark.parametrize("extra", ["", "gate", "sinks"])
def test_latent_prompt(dt, tol, seqs, window, H, extra, monkeypatch):
    """Written-out keys and values against 64 bits and against the absorbed form.  Tolerance: the type's rounding of keys,
    values, weights and result, as for the absorbed kernels."""
    C, R, Dn, V, bs = 512, 64, 128, 128, 16
    g = torch.Generator().manual_seed(len(seqs) + window + H)
    ends = [a + n for a, n in seqs]
    pages = -(-max(ends) // bs)
    bt = torch.randperm(len(seqs) * pages, generator=g).view(len(seqs), pages).to(torch.int32)
    cache = torch.randn(len(seqs) * pages * bs, C + R, generator=g).to(dt)
    T = sum(n for _, n in seqs)
    q = torch.randn(T, H * (Dn + R), generator=g).to(dt)
    uk, uv = ((torch.randn(H * d, C, generator=g) / C ** 0.5).to(dt) for d in (Dn, V))
    gate = torch.randn(T, H + 3, generator=g).to(dt)[:, 1:H + 1] if extra == "gate" else None
    sinks = torch.randn(H, generator=g) * 3.0 if extra == "sinks" else None
    cu = torch.tensor([0] + [n for _, n in seqs]).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(a, a + n) for a, n in seqs]).to(torch.int32)
    tok_seq = torch.repeat_interleave(torch.arange(len(seqs)), torch.tensor([n for _, n in seqs])).to(torch.int32)
    d = lambda t: None if t is None else t.to(DEV)
    b = {"positions": d(pos), "cu_q": d(cu), "tok_seq": d(tok_seq), "block_tables": d(bt), "max_qlen": max(n for _, n in seqs)}
    ukv = sm.latent_expand(d(uk), d(uv), H, R)
    args = (d(uk.view(H, Dn, C).transpose(1, 2).contiguous()), d(uv.view(H, V, C)), ukv, b, C, R, H, Dn, V, window, 0.07, bs)
    gd = torch.randn(T, H + 3, generator=g).to(dt).to(DEV)[:, 1:H + 1].copy_(gate) if gate is not None else None
    monkeypatch.setattr(sm, "LATENT_EXPAND_MIN", 1)
    got = sm.latent_mix(d(q), d(cache), *args, sinks=d(sinks), gate=gd)
    assert "latent_keys" in b
    monkeypatch.setattr(sm, "LATENT_EXPAND_MIN", 0)
    absorbed = sm.latent_mix(d(q), d(cache), *args, sinks=d(sinks), gate=gd)
    want = torch.zeros(T, H, V, dtype=torch.float64, device=DEV)
    for s, (a, n) in enumerate(seqs):
        if not n:
            continue
        key = torch.arange(a + n)
        rows = d(cache)[(bt[s].long()[key // bs] * bs + key % bs).to(DEV)].double()
        k = torch.cat([(rows[:, :C] @ d(uk).double().T).view(-1, H, Dn), rows[:, None, C:].expand(-1, H, R)], 2)
        v = (rows[:, :C] @ d(uv).double().T).view(-1, H, V)
        r = slice(int(cu[s]), int(cu[s + 1]))
        sc = torch.einsum("thd,khd->htk", d(q).double().view(T, H, -1)[r], k) * 0.07
        age = (torch.arange(a, a + n)[:, None] - key[None, :]).to(DEV)
        sc = sc.masked_fill((age < 0) | ((age >= window) if window else (age < 0)), -float("inf"))
        if sinks is not None:
            sc = torch.cat([sc, d(sinks).double()[:, None, None].expand(H, n, 1)], 2)
        y = torch.einsum("htk,khv->thv", torch.softmax(sc, -1)[..., :a + n], v)
        want[r] = y * (torch.sigmoid(gd[r].double())[:, :, None] if gate is not None else 1.0)
    want = want.view(T, H * V)
    scale = want.abs().max()
    assert (got.double() - want).abs().max() <= tol * scale
    err = lambda y: float((y.double() - want).norm() / want.norm())
    assert err(got) <= 1.1 * err(absorbed) + 1e-7      # no less exact than the absorbed form


def attend64(q, k, v, first, scale, window=0, chunk=0, sinks=None, slopes=None, softcap=0.0):
    """q [n, H, D] of the tokens from position ``first`` on over k, v [first + n, G, ..]: softmax in 64 bits, [n, H, V]."""
    n, H, R = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    at, key = torch.arange(first, first + n, device=q.device)[:, None], torch.arange(first + n, device=q.device)[None]
    hide = (key > at) | ((at - key >= window) if window else key > at) | ((at // chunk != key // chunk) if chunk else key > at)
    out = []
    for h in range(H):
        s = (q[:, h].double() @ k[:, h // R].double().T) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        if slopes is not None:
            s = s - slopes[h].double() * (at - key)
        s = s.masked_fill(hide, -float("inf"))
        if sinks is not None:
            s = torch.cat([s, sinks[h].double().expand(n, 1)], 1)
        out.append(torch.softmax(s, 1)[:, :first + n] @ v[:, h // R].double())
    return torch.stack(out, 1)


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("window", [0, 100])
def test_latent_prompt_idle_rows_and_non_finite_scores(dt, tol, window, monkeypatch):
    """An idle row between two portions is zero and changes nothing; a NaN query head and a key whose rotated part makes
    infinite scores: NaN exactly where 64 bits give NaN, the tolerance of finite keys elsewhere."""
    C, R, D, H, bs = 512, 64, 128, 3, 16
    g = torch.Generator().manual_seed(window)
    r = lambda *s: torch.randn(*s, generator=g)
    seqs, pages = [(0, 200), (-1, 1), (30, 170)], 13
    T = sum(n for _, n in seqs)
    q, cache = r(T, H, D + R), r(3 * pages * bs, C + R)
    q[50, 1, D + 5] = float("nan")
    cache[2 * pages * bs + 60, C + 9] = float("inf")
    q, cache = q.to(dt).to(DEV), cache.to(dt).to(DEV)
    uk, uv = ((r(H * D, C) / C ** 0.5).to(dt).to(DEV) for _ in range(2))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    b = {"positions": i32([a + i for a, n in seqs for i in range(n)]), "cu_q": i32([0, 200, 201, 371]),
         "tok_seq": i32([s for s, (_, n) in enumerate(seqs) for _ in range(n)]), "max_qlen": 200,
         "block_tables": torch.arange(3 * pages, dtype=torch.int32, device=DEV).view(3, pages)}
    monkeypatch.setattr(sm, "LATENT_EXPAND_MIN", 1)
    got = sm.latent_mix(q.view(T, -1), cache, uk.view(H, D, C).transpose(1, 2).contiguous(), uv.view(H, D, C),
                        sm.latent_expand(uk, uv, H, R), b, C, R, H, D, D, window, 0.07, bs).view(T, H, D)
    assert "latent_keys" in b and (got[200] == 0).all()
    for s, at in ((0, 0), (2, 201)):
        first, n = seqs[s]
        rows = cache.view(3, pages * bs, -1)[s, :first + n].double()
        k = torch.cat([(rows[:, :C] @ uk.double().T).view(-1, H, D), rows[:, None, C:].expand(-1, H, R)], 2)
        want = attend64(q[at:at + n], k, (rows[:, :C] @ uv.double().T).view(-1, H, D), first, 0.07, window)
        bad, y = torch.isnan(want), got[at:at + n]
        assert bad.any() and not bad.all() and torch.equal(bad, torch.isnan(y))
        assert (y.double() - want)[~bad].abs().max() <= tol * want[~bad].abs().max()


# contexts of the rows (0: idle), window: around one 64-key step, one split per step and several steps per split, windows that
# start inside a page, one row, more rows than a group of four
@pytest.mark.parametrize("ctx,window,H", [([1, 63, 64, 65, 0, 129], 0, 3), ([530], 1024, 16), ([700, 2, 333], 100, 32),
                                          ([0], 0, 16), ([1025] * 18, 0, 16), ([600, 17, 0, 900, 64], 513, 20)])
@pytest.mark.parametrize("extra", ["", "gate", "sinks"])
def test_latent_token(ctx, window, H, extra):
    """Decoding in the latent space against 64 bits; tolerance as for the kernels it replaces, and no less exact than them."""
    C, R, Dn, V, bs, dt = 512, 64, 128, 128, 16, torch.bfloat16
    g = torch.Generator().manual_seed(sum(ctx) + window + H)
    T, pages = len(ctx), -(-max(max(ctx), 1) // bs) + 2
    bt = torch.randperm(T * pages, generator=g).view(T, pages).to(torch.int32)
    r = lambda *s: torch.randn(*s, generator=g)
    cache, q = r(T * pages * bs, C + R).to(dt).to(DEV), r(T, H * (Dn + R)).to(dt).to(DEV)
    uk, uv = ((r(H * d, C) / C ** 0.5).to(dt).to(DEV) for d in (Dn, V))
    gate = r(T, H + 3).to(dt).to(DEV)[:, 1:H + 1] if extra == "gate" else None
    sinks = (r(H) * 3.0).to(DEV) if extra == "sinks" else None
    pos = torch.tensor(ctx, dtype=torch.int32) - 1
    ar = torch.arange(T + 1, dtype=torch.int32, device=DEV)
    b = {"positions": pos.to(DEV), "cu_q": ar, "tok_seq": ar[:T], "block_tables": bt.to(DEV), "max_keys": pages * bs}
    uk_t, uv3 = uk.view(H, Dn, C).transpose(1, 2).contiguous(), uv.view(H, V, C)
    got = sm.latent_mix(q, cache, uk_t, uv3, None, b, C, R, H, Dn, V, window, 0.07, bs, sinks=sinks, gate=gate)
    qa = torch.empty(T, H, C, dtype=dt, device=DEV)
    sm.gemm(q.view(T, H, Dn + R)[:, :, :Dn].permute(1, 0, 2), uk_t, out=qa.permute(1, 0, 2))
    lat = sm.latent_attention(qa, q, cache, b["block_tables"], b["tok_seq"], b["positions"], C, R, H, Dn, window, 0.07, bs,
                              sinks=sinks, gate=gate)
    old = torch.empty(T, H, V, dtype=dt, device=DEV)
    sm.gemm(lat.permute(1, 0, 2), uv3, out=old.permute(1, 0, 2))
    want = torch.zeros(T, H, V, dtype=torch.float64, device=DEV)
    for t, n in enumerate(ctx):
        if not n:
            continue
        key = torch.arange(max(0, n - window) if window else 0, n)
        rows = cache[(bt[t].long()[key // bs] * bs + key % bs).to(DEV)].double()
        k = torch.cat([(rows[:, :C] @ uk.double().T).view(-1, H, Dn), rows[:, None, C:].expand(-1, H, R)], 2)
        sc = torch.einsum("hd,khd->hk", q[t].double().view(H, -1), k) * 0.07
        if sinks is not None:
            sc = torch.cat([sc, sinks.double()[:, None]], 1)
        y = torch.einsum("hk,khv->hv", torch.softmax(sc, -1)[:, :len(key)], (rows[:, :C] @ uv.double().T).view(-1, H, V))
        want[t] = y * (torch.sigmoid(gate[t].double())[:, None] if gate is not None else 1.0)
    want = want.view(T, H * V)
    assert (got.double() - want).abs().max() <= 2e-2 * want.abs().max()
    err = lambda y: float((y.double() - want).norm() / want.norm().clamp(min=1e-30))
    assert err(got) <= 1.1 * err(old.view(T, H * V)) + 1e-7


@pytest.mark.parametrize("keys", [40, 700])
@pytest.mark.parametrize("sink", [False, True])
def test_latent_token_lets_non_finite_scores_through(keys, sink):
    """A NaN query head and a key of infinite score, in one split and in many: NaN where 64 bits give NaN (score +inf, or all
    scores NaN), finite where the infinite score is -inf (weight 0), idle rows zero."""
    C, R, Dn, V, H, bs, dt = 512, 64, 128, 128, 16, 16, torch.bfloat16
    g = torch.Generator().manual_seed(keys)
    r = lambda *s: torch.randn(*s, generator=g)
    pages = -(-keys // bs)
    q, cache = r(3, H, Dn + R), r(3 * pages * bs, C + R)
    q[0, 5, Dn + 3] = float("nan")
    cache[pages * bs + keys // 2, C + 7] = float("inf")      # (a rotated part: no value)
    q, cache = q.to(dt).to(DEV), cache.to(dt).to(DEV)
    uk, uv = ((r(H * d, C) / C ** 0.5).to(dt).to(DEV) for d in (Dn, V))
    sinks = torch.zeros(H, device=DEV) if sink else None
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    b = {"positions": i32([keys - 1, keys - 1, -1]), "cu_q": i32([0, 1, 2, 3]), "tok_seq": i32([0, 1, 2]),
         "block_tables": torch.arange(3 * pages, dtype=torch.int32, device=DEV).view(3, pages), "max_keys": pages * bs}
    got = sm.latent_mix(q.view(3, -1), cache, uk.view(H, Dn, C).transpose(1, 2).contiguous(), uv.view(H, V, C), None, b, C, R, H,
                        Dn, V, 0, 0.07, bs, sinks=sinks).view(3, H, V)
    assert (got[2] == 0).all()
    for t in range(2):
        rows = cache.view(3, pages * bs, -1)[t, :keys].double()
        k = torch.cat([(rows[:, :C] @ uk.double().T).view(-1, H, Dn), rows[:, None, C:].expand(-1, H, R)], 2)
        sc = (q[t].double()[None] * k).sum(2) * 0.07                                  # [keys, H]
        p = torch.softmax(sc if sinks is None else torch.cat([sc, sinks.double()[None]]), 0)[:keys]
        want = torch.einsum("kh,khv->hv", p, (rows[:, :C] @ uv.double().T).view(-1, H, V))
        bad = torch.isnan(want)
        assert bad.any() and not bad.all() and torch.equal(bad, torch.isnan(got[t]))
        assert (got[t].double() - want)[~bad].abs().max() <= 2e-2 * want[~bad].abs().max()


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-6), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("W", [4, 1023, 1024, 1028, 2052, 8192, 8196])
def test_row_norm_and_token_shift_widths(dt, tol, W):
    """Widths around the vector forms' register counts and the scalar forms beyond them, every optional operand, idle rows."""
    from k8s_llm_scheduler_amd.ops import reference as ref
    g = torch.Generator().manual_seed(W)
    r = lambda *s: torch.randn(*s, generator=g)
    T = 7
    x, b1, b2, rv, w = r(T, W), r(T, W).to(dt), r(T, W).to(dt), r(W).to(dt), r(W).to(dt)
    for branch, branch2, rowvec in ((b1, b2, rv), (b1, None, None), (None, None, rv), (None, None, None)):
        xg, xc = x.to(DEV), x.clone()
        d = lambda t: None if t is None else t.to(DEV)
        got = sm.resnorm(xg, d(w), 1e-6, branch=d(branch), branch2=d(branch2), mult=0.3, rowvec=d(rowvec), offset=1.0, out_dtype=dt)
        want = sm.resnorm(xc, w, 1e-6, branch=branch, branch2=branch2, mult=0.3, rowvec=rowvec, offset=1.0, out_dtype=dt)
        assert (got.cpu().float() - want.float()).abs().max() <= tol * want.float().abs().max()
        assert (xg.cpu() - xc).abs().max() <= 1e-6 * xc.abs().max()
    cu = torch.tensor([0, 3, 3, 4, 5, 7], dtype=torch.int32)
    pos = torch.tensor([0, 1, 2, -1, 9, 4, 5], dtype=torch.int32)
    slots, tok_seq = torch.tensor([4, 0, 1, 2, 3], dtype=torch.int32), torch.tensor([0, 0, 0, 2, 3, 4, 4], dtype=torch.int32)
    h, mu, st = r(T, W).to(dt), torch.rand(5, W, generator=g).to(dt), r(5, W).to(dt)
    sg, sc = st.to(DEV), st.clone()
    got = sm.token_shift(h.to(DEV), mu.to(DEV), sg, *(t.to(DEV) for t in (cu, tok_seq, slots, pos)), save=True).cpu()
    want = ref.token_shift(h, mu, sc, cu, slots, pos)
    ref.shift_save(sc, h, cu, slots, pos)
    live = pos >= 0
    assert (got[:, live].float() - want[:, live].float()).abs().max() <= tol * want.float().abs().max()
    assert (got[:, ~live] == 0).all() and torch.equal(sg.cpu(), sc)


# ----------------------------------------------------------------------------- grouped products on big tiles, activations in the epilogue
KINDS = [sm.ACT_GELU_TANH, sm.ACT_SWISH_CLAMP, sm.ACT_RELU]
ELEMENTWISE = [sm.ACT_TANH, sm.ACT_SILU, sm.ACT_GELU_ERF, sm.ACT_RELU2, sm.ACT_SOFTCAP]


def act64(z, kind, limit, alpha):
    if kind in KINDS:
        g, u = z.chunk(2, -1)
        if kind == sm.ACT_GELU_TANH:
            return torch.nn.functional.gelu(g, approximate="tanh") * u
        if kind == sm.ACT_RELU:
            return g.clamp(min=0) * u
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(alpha * g) * (u + 1.0)
    return {sm.ACT_TANH: torch.tanh, sm.ACT_SILU: torch.nn.functional.silu, sm.ACT_GELU_ERF: torch.nn.functional.gelu,
            sm.ACT_RELU2: lambda v: v.clamp(min=0) ** 2, sm.ACT_SOFTCAP: lambda v: limit * torch.tanh(v / limit)}[kind](z)


@pytest.fixture
def grouped_tile(monkeypatch):
    """Forces the tile configuration of grouped products: set ``cfg``; ``ran`` lists those that were launched."""
    class Force:
        cfg, ran = None, []

    nat, force = ops.native(), Force()
    force.ran = []

    class Spy:
        def __getattr__(self, name):
            if name != "pgemm4_grouped":
                return getattr(nat, name)
            return lambda *args: (force.ran.append(args[11]), nat.pgemm4_grouped(*args))[1]

    monkeypatch.setattr(ops, "native", Spy)
    monkeypatch.setattr(sm, "_grouped_tile", lambda *args: force.cfg)
    return force


GROUPED_TILES = [1, 2, 3, 4, 5, 6]      # 256 x 128, 128 x 256, 128 x 128, 256 x 256, 128 x 64, 64 x 64 (weight rows x tokens)


@pytest.mark.parametrize("sizes", [(1, 127, 0, 128, 129), (40, 40, 40), (0, 0, 300), (257,), tuple([17] * 63 + [1]), (63, 65, 0, 64, 255, 256)])
@pytest.mark.parametrize("N,K", [(128, 64), (392, 192), (1024, 256)])
@pytest.mark.parametrize("kind", [None] + KINDS)
def test_grouped_big_tiles(sizes, N, K, kind, grouped_tile):
    """Every tile with groups at the edges of its 64, 128 or 256 tokens, empty ones, more than fit a wave; gathered rows with a row
    stride."""
    g = torch.Generator().manual_seed(sum(sizes) + N + K)
    E, P = len(sizes), sum(sizes)
    seg = torch.tensor((0,) + sizes).cumsum(0).to(torch.int32)
    if P < sm.GROUP_BIG_MIN * E:
        pytest.skip("too few rows for this path")
    x = torch.randn(90, K + 8, generator=g).to(torch.bfloat16).to(DEV)[:, :K]
    rows = torch.randint(0, 90, (P,), generator=g).to(torch.int32).to(DEV)
    w = (torch.randn(E, N * (1 if kind is None else 2), K, generator=g) * 2 / K ** 0.5).to(torch.bfloat16).to(DEV)
    tiles = torch.full((1, 3), -1, dtype=torch.int32, device=DEV)      # the big tiles come from seg
    assert sm._grouped_big(x, w, seg.to(DEV), P, N)
    kw = dict(a_rows=rows, tiles=tiles, rows=P, seg=seg.to(DEV))
    want = []
    for e in range(E):
        z = x[rows[int(seg[e]):int(seg[e + 1])].long()].double() @ w[e].double().T
        want.append(z if kind is None else act64(z, kind, 1.5, 1.702))
    want = torch.cat(want)
    for cfg in GROUPED_TILES:
        grouped_tile.cfg = cfg
        got = sm.gemm(x, w, **kw) if kind is None else sm.gemm_act(x, w, kind, 1.5, 1.702, **kw)
        # one rounding to bf16, and the fp32 sums'
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all(), cfg
    assert grouped_tile.ran == GROUPED_TILES


@pytest.mark.parametrize("M", [1, 63, 65, 128, 257])
@pytest.mark.parametrize("N,K", [(128, 64), (392, 192)])
def test_several_inputs_on_every_big_tile(M, N, K, grouped_tile):
    """Groups of one size, without a list of their offsets: rows at the edges of every tile."""
    g = torch.Generator().manual_seed(M + N)
    a, w = (torch.randn(3, n, K, generator=g).to(torch.bfloat16).to(DEV) for n in (M, N))
    for cfg in GROUPED_TILES:
        grouped_tile.cfg = cfg
        got = sm._pgemm4_grouped(a.view(3 * M, K), w, None, 3 * M, None, N).view(3, M, N)
        for i in range(3):
            exact = a[i].double() @ w[i].double().T
            bound = sum_bound(a[i].cpu(), w[i].cpu()).to(DEV) + 2.0 ** -8 * exact.abs()
            assert ((got[i].double() - exact).abs() <= bound).all(), (cfg, i)
    assert grouped_tile.ran == GROUPED_TILES


@pytest.mark.parametrize("M,N,K", [(129, 1024, 512), (200, 520, 1024), (1031, 2048, 256), (2048, 2064, 320), (160, 512, 4096)])
@pytest.mark.parametrize("kind", KINDS + ELEMENTWISE)
@pytest.mark.parametrize("bias", [False, True])
def test_linear_act(M, N, K, kind, bias, entries):
    """The activation in the epilogue, every tile configuration's edges, against 64 bits: one rounding.  Two launches and two
    roundings only where the product's plan splits k (160 rows of depth 4096), and for the elementwise kinds without an epilogue of the
    big tiles (200 x 520 is few tiles, which have one for all but the cap)."""
    if bias and kind not in KINDS:
        pytest.skip("elementwise kinds take no bias")
    g = torch.Generator().manual_seed(M + N + K + kind)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(2 * N if kind in KINDS else N, K, generator=g) * 2 / K ** 0.5).to(torch.bfloat16).to(DEV)
    b = torch.randn(2 * N, generator=g).to(torch.bfloat16).to(DEV) if bias else None
    z = x.double() @ w.double().T + (b.double() if bias else 0.0)
    want = act64(z, kind, 1.5, 1.702)
    nat = sm._native()
    for cfg in (1, 2, 3, 4) if kind in KINDS + [sm.ACT_RELU2] else ():
        out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
        nat.pgemm4_act(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, cfg, 4, kind, 1.5, 1.702,
                       b.data_ptr() if bias else 0, -1)
        assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all(), cfg
    entries.clear()
    got = sm.linear_act(x, w, kind, 1.5, 1.702, bias=b)
    few = M == 200 and kind not in KINDS + [sm.ACT_SOFTCAP]
    kern, plan = ops.gemm_route(M, w.shape[0], K, ops.EPI_BF16, False)
    assert kern == "pgemm4" and (plan[1] > 1) == (K == 4096)
    fused = few or (plan[1] == 1 and kind in KINDS + [sm.ACT_RELU2])
    assert ("act" in entries) != fused and ("gemm_few_act" if few else "pgemm4_act" if fused else "act") in entries
    if fused:
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()
    else:
        assert ((got.double() - want).abs() <= 2.0 ** -6 * want.abs() + 4e-2).all()


@pytest.mark.parametrize("tokens,top,E,N,K", [(1, 1, 3, 130, 64), (5, 2, 3, 15, 128), (48, 2, 8, 72, 320), (100, 1, 2, 33, 2048)])
@pytest.mark.parametrize("kind", KINDS)
def test_few_rows_gated(tokens, top, E, N, K, kind, entries):
    """Tiles of at most 16 and of up to 64 rows, columns that do not fill 16, gathered rows with a stride: one rounding."""
    g = torch.Generator().manual_seed(tokens + N + K)
    idx = torch.rand(tokens, E, generator=g).argsort(1)[:, :top].to(torch.int32)
    rows, pos, seg, tiles = sm.moe_align(idx.to(DEV), E)
    h = torch.randn(tokens, K + 8, generator=g).to(torch.bfloat16).to(DEV)[:, :K]
    w = (torch.randn(E, 2 * N, K, generator=g) * 2 / K ** 0.5).to(torch.bfloat16).to(DEV)
    got = sm.gemm_act(h, w, kind, 1.5, 1.702, a_rows=rows, tiles=tiles, rows=tokens * top).double()[pos.long()]
    assert entries[-1] == "gemm_few_act"
    for c in range(top):
        z = (h.double().unsqueeze(1) @ w.double()[idx[:, c].long().to(DEV)].transpose(1, 2)).squeeze(1)
        want = act64(z, kind, 1.5, 1.702)
        assert ((got.view(tokens, top, N)[:, c] - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (16, 130, 128), (17, 100, 64), (200, 33, 320)])
@pytest.mark.parametrize("kind", [k for k in ELEMENTWISE if k != sm.ACT_SOFTCAP])
def test_few_tiles_elementwise(M, N, K, kind, entries):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g).to(torch.bfloat16).to(DEV)[:, 8:]
    w = (torch.randn(N, K, generator=g) * 2 / K ** 0.5).to(torch.bfloat16).to(DEV)
    want = act64(x.double() @ w.double().T, kind, 0.0, 1.0)
    assert ((sm.linear_act(x, w, kind).double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()
    assert entries == ["gemm_few_act"]


@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (16, 130, 128), (17, 100, 64), (64, 15, 1024), (65, 128, 2048), (200, 33, 320),
                                   (2048, 128, 192)])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_narrow_products(M, N, K, out):
    """Few tiles: k shared by a workgroup's waves; rows and columns at the 16s and 64s, a row stride, a batch."""
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(2, M, K + 8, generator=g).to(torch.bfloat16).to(DEV)[:, :, 8:]
    w = torch.randn(2, N, K, generator=g).to(torch.bfloat16).to(DEV)
    bound = lambda a, w, y: sum_bound(a.cpu(), w.cpu()) + (2.0 ** -8 * y.abs().cpu() if out == torch.bfloat16 else 0.0)
    got, exact = sm.gemm(a, w, out).cpu().double(), a.double() @ w.double().transpose(1, 2)
    assert ((got - exact.cpu()).abs() <= bound(a, w, exact)).all()
    one = sm.gemm(a[0], w[0], out).cpu().double()
    assert ((one - exact[0].cpu()).abs() <= bound(a[0], w[0], exact[0])).all()


def test_recurrence_prefix_over_many_chunks():
    """More chunks than the prefix keeps in flight, head sizes that do not fill its workgroups, a resumed sequence beside a
    new one: chunked against one workgroup per sequence."""
    g = torch.Generator().manual_seed(5)
    for H, D, lens, first in ((2, 64, (700, 129), (0, 33)), (1, 40, (1, 900), (7, 0)), (1, 128, (65, 300), (9, 1)),
                              (3, 17, (64, 128), (2, 0))):
        T = sum(lens)
        r, k, v, gate = (torch.randn(T, H * D, generator=g).to(DEV) for _ in range(4))
        z, w0, u, lnw = (torch.randn(T, H * D, generator=g).to(DEV), *(torch.randn(H * D, generator=g).to(DEV) for _ in range(3)))
        st = torch.randn(2, H, D, D, generator=g).to(DEV)
        cu = torch.tensor([0, lens[0], T], dtype=torch.int32, device=DEV)
        pos = torch.cat([torch.arange(p, p + n) for p, n in zip(first, lens)]).to(torch.int32).to(DEV)
        slots = torch.tensor([1, 0], dtype=torch.int32, device=DEV)
        outs = []
        for chunk in (0, 16, 64, 67, 150):
            s = st.clone()
            y = sm.wkv_scan(r, k, v, gate, z, w0, u, lnw, s, cu, slots, pos, H, D, 1e-6, chunk=chunk)
            outs.append((y, s))
        for y, s in outs[1:]:
            assert (y - outs[0][0]).abs().max() <= 1e-4 * outs[0][0].abs().max()
            assert (s - outs[0][1]).abs().max() <= 1e-5 * outs[0][1].abs().max()


@pytest.mark.parametrize("records", [1, 7, 8, 9, 15, 16, 17, 33])
@pytest.mark.parametrize("empty", [0, 10])
def test_recurrence_prefix_at_the_ends_of_its_groups(records, empty):
    """Chunks whose records fill the prefix's groups, one more and one less, against 64 bits: 16 loads in flight, and 8
    where the states are many (empty sequences beside the long one) and have few chunks on average."""
    H, D, chunk = 2, 64, 16
    T, n = chunk * (records + 1), 1 + empty
    gen = torch.Generator().manual_seed(records)
    r, k, v, g = (torch.randn(T, H, D, generator=gen) for _ in range(4))
    z, w0, u, lnw = torch.randn(T, H, D, generator=gen) - 4.0, *(torch.randn(H, D, generator=gen) for _ in range(3))
    S0 = torch.randn(n, H, D, D, generator=gen)
    S, i32 = S0.to(DEV).clone(), lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    got = sm.wkv_scan(*(x.reshape(T, -1).to(DEV) for x in (r, k, v, g, z)), *(x.reshape(-1).to(DEV) for x in (w0, u, lnw)), S,
                      i32([0] + [T] * n), i32(range(n)), i32(range(7, 7 + T)), H, D, 1e-6, chunk=chunk).view(T, H, D).double().cpu()
    want, end = wkv64(*(x.double() for x in (r, k, v, g, z, w0, u, lnw, S0[0])), 1e-6)
    # fp32 sums of at most 64 terms a product, the chunks' of at most their number: as the outputs by 16 tokens below
    assert (got - want).abs().max() <= 2.0 ** -15 * (1 + want.abs().max())
    assert (S[0].double().cpu() - end).abs().max() <= 2.0 ** -17 * (1 + end.abs().max())
    assert torch.equal(S[1:].cpu(), S0[1:])


@pytest.mark.parametrize("bs", [1, 16])
@pytest.mark.parametrize("B", [1, 5, 255, 256, 300])
def test_decode_meta(B, bs):
    """Against the reference ops: idle rows, first and last position of a page, of the table; beyond it a row idles."""
    nb = 7
    ctx = torch.tensor([(0, 1, bs, bs + 1, nb * bs, nb * bs - 1, 3)[i % 7] for i in range(B)], dtype=torch.int32)
    bt = torch.randperm(B * nb).int().view(B, nb)
    want, got = sm.decode_meta(ctx, bt, bs), sm.decode_meta(ctx.to(DEV), bt.to(DEV), bs)
    for w, g in zip(want, got):
        assert torch.equal(w, g.cpu())
    pos, slots, _ = sm.decode_meta(torch.full((B,), nb * bs + 1, dtype=torch.int32, device=DEV), bt.to(DEV), bs)
    assert (pos == -1).all() and (slots == -1).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_embedding_copy(dt):
    ids, table = torch.tensor([3, 0, 6, 3], dtype=torch.int32), torch.randn(7, 1030).to(dt)
    want, got = sm.embed_rows(ids, table, 1.7, copy=True), sm.embed_rows(ids.to(DEV), table.to(DEV), 1.7, copy=True)
    assert all(torch.equal(w, g.cpu()) for w, g in zip(want, got))
    assert torch.equal(got[0], sm.embed_rows(ids.to(DEV), table.to(DEV), 1.7))


@pytest.mark.parametrize("H,G,D,kw", [
    (16, 4, 128, dict(window=0)), (8, 2, 64, dict(window=150, slopes=True)), (6, 6, 96, dict(chunk=200, softcap=3.0)),
    (4, 2, 96, dict(window=1)), (8, 4, 128, dict(chunk=96, slopes=True, gate=False)),
])
@pytest.mark.parametrize("ns", [2, 3, 16])
def test_prompt_attention_key_splits(H, G, D, kw, ns, monkeypatch):
    """Splits of several steps, of one, without any (short sequences, windows) and the sink in split 0 only, against one
    workgroup per tile: the same fp32 sums in another order, rounded once to bf16 (2^-9 of a value, both sides), and the
    weights' second bf16 term (2^-16) of every key."""
    torch.manual_seed(3)
    bs, dt = 16, torch.bfloat16
    lens = [(0, 133), (290, 70), (40, 1), (-1, 1), (500, 35)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    cu = i32([0] + [n for _, n in lens]).cumsum(0).int()
    pos = i32([p for a, n in lens for p in (range(a, a + n) if a >= 0 else [-1])])
    tok_seq = i32([s for s, (_, n) in enumerate(lens) for _ in range(n)])
    bt = torch.randperm(5 * 36, device=DEV).int().view(5, 36)
    kc, vc = (torch.randn(5 * 36 * bs, G, D, device=DEV).to(dt) for _ in range(2))
    q = torch.randn(pos.shape[0], H * D + 16, device=DEV).to(dt)
    gate = torch.randn(pos.shape[0], H * D, device=DEV).to(dt) if kw.get("gate", True) else None
    slopes = torch.linspace(0.003, 1.0, H, device=DEV) if kw.get("slopes") else None
    outs = []
    for n in (1, ns):
        monkeypatch.setattr(sm, "prompt_splits", lambda groups, keys: n)
        outs.append(sm.window_attention(q, gate, kc, vc, None, None, bt, tok_seq, pos, H, kw.get("window", 0), 0, D ** -0.5,
                                        True, bs, cu, 133, chunk=kw.get("chunk", 0), softcap=kw.get("softcap", 0.0),
                                        sinks=torch.linspace(-3, 3, H, device=DEV), slopes=slopes).float())
    assert (outs[1][pos < 0] == 0).all()
    assert ((outs[1] - outs[0]).abs() <= 2.0 ** -7 * outs[0].abs() + 2.0 ** -13 * outs[0].abs().max()).all()
    for s, (a, n) in enumerate(lens):
        if a < 0:
            continue
        r, rows = slice(int(cu[s]), int(cu[s + 1])), torch.arange(a + n, device=DEV)
        rows = bt[s].long()[rows // bs] * bs + rows % bs
        want = attend64(q[r, :H * D].reshape(n, H, D), kc[rows], vc[rows], a, D ** -0.5, kw.get("window", 0), kw.get("chunk", 0),
                        torch.linspace(-3, 3, H, device=DEV), slopes, kw.get("softcap", 0.0)).view(n, H * D)
        want = want * torch.sigmoid(gate[r].double()) if gate is not None else want
        for y in outs:      # one rounding to bf16; weights of two bf16 terms and fp32 scores: 2^-13 of the largest value
            assert ((y[r].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * want.abs().max()).all()


@pytest.mark.parametrize("ns", [1, 2, 6])
@pytest.mark.parametrize("sink", [False, True])
def test_prompt_attention_lets_non_finite_scores_through(ns, sink, monkeypatch):
    """A NaN query and a key that makes infinite scores, in one piece and in key splits: NaN where 64 bits give NaN."""
    g = torch.Generator().manual_seed(ns)
    H, G, D, bs, first, n = 8, 4, 128, 16, 400, 70
    q, kc, vc = (torch.randn(*s, generator=g) for s in ((n, H, D), (512, G, D), (512, G, D)))
    q[20, 3, 7] = float("nan")
    kc[430, 1, 5] = float("inf")
    q, kc, vc = (t.to(torch.bfloat16).to(DEV) for t in (q, kc, vc))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    sinks = torch.linspace(-1, 1, H, device=DEV) if sink else None
    monkeypatch.setattr(sm, "prompt_splits", lambda groups, keys: ns)
    got = sm.window_attention(q.view(n, -1), None, kc, vc, None, None, torch.arange(32, dtype=torch.int32, device=DEV).view(1, 32),
                              i32([0] * n), i32(list(range(first, first + n))), H, 0, 0, D ** -0.5, sink, bs, i32([0, n]), n,
                              sinks=sinks).view(n, H, D)
    want = attend64(q, kc[:first + n], vc[:first + n], first, D ** -0.5, sinks=sinks)
    bad = torch.isnan(want)
    assert bad.any() and not bad.all() and torch.equal(bad, torch.isnan(got))
    assert (got.double() - want)[~bad].abs().max() <= 2.0 ** -7 * want[~bad].abs().max()


@pytest.mark.parametrize("M", [1, 32, 33, 64, 127, 129, 1031, 2048, 2049])
@pytest.mark.parametrize("N,K", [(2048, 256), (1040, 512), (4096, 192)])
def test_products_of_several_inputs(M, N, K, entries):
    """Every way a launch is shared: few tiles (up to 32, 64 and no rows of these widths), even groups of the big tiles with
    remainders, one launch per input."""
    g = torch.Generator().manual_seed(M + N)
    a, w = (torch.randn(3, n, K, generator=g).to(torch.bfloat16) for n in (M, N))
    a_dev, w_dev = a.to(DEV), w.to(DEV)
    entries.clear()
    got = sm.linear_each(a_dev, w_dev)
    if M <= {2048: 32, 1040: 64, 4096: 0}[N]:
        assert entries == ["gemm_any"]
    elif M <= 2048:
        assert entries == ["pgemm4_grouped"]
    else:
        assert len(entries) >= 3 and not {"gemm_any", "pgemm4_grouped"} & set(entries)
    assert len({t.stride(0) for t in got}) == 1
    for x, y, z in zip(a, w, got):
        exact = x.double() @ y.double().T
        assert ((z.cpu().double() - exact).abs() <= sum_bound(x, y) + 2.0 ** -8 * exact.abs()).all()


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("N,K", [(16, 256), (1028, 512), (2592, 2048), (4096, 3072), (8192, 512), (16400, 256), (40000, 256),
                                 (520, 8192), (2048, 8192)])
@pytest.mark.parametrize("epi", [0, 1])
def test_untuned_products_of_17_to_128_rows(M, N, K, epi):
    """Every tile and split that the one-round rule picks, columns and rows that do not fill the tile, both outputs."""
    from k8s_llm_scheduler_amd import ops

    g = torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16), torch.randn(N, K, generator=g).to(torch.bfloat16)
    cfg, split = ops.mgemm_heuristic(M, N, K, epi, False)
    got = ops.mgemm(x.to(DEV), w.to(DEV), epi, cfg=cfg, grid=split)
    a, b = x.to(DEV).double(), w.to(DEV).double()
    exact, bound = a @ b.T, 2.0 * K * 2.0 ** -24 * (a.abs() @ b.abs().T) + 1e-30
    assert ((got.double() - exact).abs() <= bound + (2.0 ** -8 * exact.abs() if epi == 0 else 0.0)).all()


def wkv64(r, k, v, g, z, w0, u, lnw, S, eps):
    """The recurrence of one sequence in 64 bits, token by token: r .. z [T, H, D], S [H, D, D]; outputs and end state."""
    w, out = torch.exp(-torch.exp(z + w0)), []
    for t in range(r.shape[0]):
        kv = k[t][:, :, None] * v[t][:, None, :]
        out.append((r[t][:, :, None] * (S + u[:, :, None] * kv)).sum(1))
        S = w[t][:, :, None] * S + kv
    o = torch.stack(out)
    return o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * lnw * g * torch.sigmoid(g), S


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D", [(3, 64), (2, 20), (5, 48)])
@pytest.mark.parametrize("T,chunk", [(15, 64), (16, 64), (17, 16), (64, 64), (65, 64), (129, 48), (200, 25)])
@pytest.mark.parametrize("value", [None, float("inf"), float("nan")])
def test_wkv_outputs_by_16_tokens(dt, H, D, T, chunk, value):
    """Ends of 16 tokens and of chunks, decays from none to all of the state within a token, and a value that is not finite:
    it reaches its column from its own token on and nothing before it."""
    gen = torch.Generator().manual_seed(T + D)
    rnd = lambda *s: torch.randn(*s, generator=gen)
    r, k, v, g = (rnd(T, H, D).to(dt) for _ in range(4))
    z, w0, u, lnw = 3.0 * rnd(T, H, D), rnd(H, D).to(dt), (0.5 * rnd(H, D)).to(dt), (1 + 0.1 * rnd(H, D)).to(dt)
    at = T - T // 3
    if value is not None:
        v[at, 1, 3] = value
    S0 = rnd(1, H, D, D)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    S = S0.to(DEV).clone()
    got = sm.wkv_scan(*(x.reshape(T, -1).to(DEV) for x in (r, k, v, g, z)), *(x.reshape(-1).to(DEV) for x in (w0, u, lnw)), S,
                      i32([0, T]), i32([0]), i32(range(7, 7 + T)), H, D, 1e-6, chunk=chunk).view(T, H, D).double().cpu()
    want, end = wkv64(*(x.double() for x in (r, k, v, g, z, w0, u, lnw, S0[0])), 1e-6)
    head = torch.ones(T, H, dtype=torch.bool)
    if value is not None:
        head[at:, 1] = False
        assert not torch.isfinite(got[at, 1]).all()
    # chains of at most 64 + 16 + 64 fp32 terms and the decays' products: 2^-24 times their number at most, then the norm
    # (outputs are of the order of one) and one rounding
    ulp = 2.0 ** -24 if dt == torch.float32 else 2.0 ** -8
    assert ((got - want)[head].abs() <= ulp * want[head].abs() + 2.0 ** -15 * (1 + want[head].abs())).all()
    if value is None:
        assert ((S[0].double().cpu() - end).abs() <= 2.0 ** -17 * (1 + end.abs().max())).all()


@pytest.mark.parametrize("H,G,D,kw", [(16, 4, 128, dict(window=0)), (8, 4, 64, dict(window=150)), (6, 3, 96, dict(chunk=100))])
@pytest.mark.parametrize("T,max_keys", [(1, 1024), (3, 4096), (32, 1024), (43, 0), (172, 1024)])
def test_token_attention_by_waves(H, G, D, kw, T, max_keys):
    """8 waves with and without key splits and 4 waves (more than 512 tokens x key heads), waves with two tiles, one and none."""
    gen = torch.Generator().manual_seed(T)
    bs, n, i32 = 16, 40, lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ctx = [(1, 32, 33, 600, 257, 513)[i % 6] + (i // 6) % 7 for i in range(T)]
    kc, vc, q = (torch.randn(*s, generator=gen).to(torch.bfloat16).to(DEV) for s in ((T * n * bs, G, D),) * 2 + ((T, H * D),))
    bt = torch.randperm(T * n, generator=gen).int().view(T, n).to(DEV)
    got = sm.window_attention(q, None, kc, vc, None, None, bt, i32(range(T)), i32([c - 1 for c in ctx]), H, kw.get("window", 0), 0,
                              D ** -0.5, False, bs, max_keys=max_keys, chunk=kw.get("chunk", 0))
    for t, c in enumerate(ctx):
        rows = torch.arange(c, device=DEV)
        rows = bt[t].long()[rows // bs] * bs + rows % bs
        want = attend64(q[t:t + 1].view(1, H, D), kc[rows], vc[rows], c - 1, D ** -0.5, kw.get("window", 0), kw.get("chunk", 0)).view(-1)
        assert ((got[t].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * want.abs().max()).all(), t


@pytest.mark.parametrize("H,G,D", [(16, 4, 128), (8, 4, 96), (4, 2, 64)])
@pytest.mark.parametrize("groups,context", [(256, 40), (260, 90), (260, 1100), (320, 1100), (512, 33), (516, 65)])
def test_token_attention_where_the_waves_change(H, G, D, groups, context):
    """8 waves up to the workgroups that run at once, 4 beyond (256 tokens x key heads, at 64 dimensions 512), with and without key
    splits: against 64 bits."""
    T, bs, i32 = groups // G, 16, lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    n = -(-context // bs)
    gen = torch.Generator().manual_seed(groups + context)
    ctx = [1 + (i * 37) % context for i in range(T)]
    kc, vc = (torch.randn(n * bs + 16 * bs, G, D, generator=gen).to(torch.bfloat16).to(DEV) for _ in range(2))
    q = torch.randn(T, H * D, generator=gen).to(torch.bfloat16).to(DEV)
    bt = torch.stack([(torch.arange(n) + i % 16) for i in range(T)]).int().to(DEV)      # (pages may be shared: nothing is written)
    got = sm.window_attention(q, None, kc, vc, None, None, bt, i32(range(T)), i32([c - 1 for c in ctx]), H, 0, 0, D ** -0.5, False, bs,
                              max_keys=max(context, 2100 if context > 1000 else 0))
    for t, c in enumerate(ctx):
        rows = torch.arange(c, device=DEV)
        rows = bt[t].long()[rows // bs] * bs + rows % bs
        want = attend64(q[t:t + 1].view(1, H, D), kc[rows], vc[rows], c - 1, D ** -0.5, 0, 0).view(-1)
        assert ((got[t].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * want.abs().max()).all(), t
