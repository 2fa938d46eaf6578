"""Kernels of the fp32-stream designs at the edges of their tiles and dispatch rules, against the fp32 reference ops or 64
bits."""

import pytest
import torch

from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda"


def sum_bound(a, w):
    """Elementwise bound on |fp32 product - exact| for any order of the K products: K 2^-24 sum |a| |w| (twice that)."""
    return 2.0 * a.shape[-1] * 2.0 ** -24 * (a.double().abs() @ w.double().abs().transpose(-1, -2)) + 1e-30


@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (31, 33, 60), (32, 32, 64), (33, 65, 68), (64, 64, 256), (97, 130, 260),
                                   (40, 16388, 8), (1031, 576, 132), (256, 2048, 320)])
def test_fp32_products(M, N, K):
    """Both tile shapes of the fp32 matrix-core product, remainders in every dimension, an odd row stride, a batch."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K + 4, generator=g)[:, :K], torch.randn(N, K, generator=g)
    a[:, 0] *= 1e4
    ag = torch.randn(M, K + 4, generator=g).to(DEV)[:, :K].copy_(a)
    exact = a.double() @ w.double().T
    assert ((sm.gemm(ag, w.to(DEV)).cpu().double() - exact).abs() <= sum_bound(a, w)).all()
    b = torch.stack([a, 2.0 * a])
    got = sm.gemm(b.to(DEV), torch.stack([w, w]).to(DEV)).cpu()
    assert torch.equal(got[1], 2.0 * got[0])
    assert torch.equal(got[0], sm.gemm(ag, w.to(DEV)).cpu())      # the order of the sums depends on K alone
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
