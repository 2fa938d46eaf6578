"""Rows of an fp32 stream between the product that adds to it and the product that reads its norm, against 64 bits: widths and depths at
the ends of a wave's steps and in several k-groups, output counts at the ends of a band, every output form, both parts of a split; and the
norm with the token shift behind it, bit for bit as the two launches."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV, EPS, BF, F32 = "cuda", 1e-5, torch.bfloat16, torch.float32


@pytest.fixture
def entries(monkeypatch):
    nat, seen = ops.native(), []

    class Spy:
        def __getattr__(self, name):
            seen.append(name)
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Spy)
    return seen


def data(seed):
    g = torch.Generator().manual_seed(seed)
    return lambda *s, dt=BF, m=1.0: (torch.randn(*s, generator=g) * m).to(dt).to(DEV)


def stream(r, M, K, N):
    """Inputs of linear_rows, its stream in 64 bits and a bound of that: fp32 sums of K products in any order, one addition."""
    x, a, w, nw = r(M, N, dt=F32, m=3.0), r(M, K), r(N, K, m=K ** -0.5), r(N, m=0.3)
    b = a.double() @ w.double().T
    mass = a.double().abs() @ w.double().abs().T
    y = x.double() + 0.6 * b
    return x, a, w, nw, y, 0.6 * 2.0 * K * 2.0 ** -24 * mass + 2.0 ** -23 * (y.abs() + b.abs())


def read(y, nw):
    return y * (1.0 + nw.double()) * (y.square().mean(-1, keepdim=True) + EPS).rsqrt()


def close(got, y, ey, nw, w, out_dtype, act=None):
    """The product of the normed rows: those rounded to bf16 once (2^-9 of a row, and y's own error), its sums in fp32, its output."""
    K = y.shape[1]
    h, W = read(y, nw), w.double()
    slack = (ey / y.abs().clamp(min=1e-30) * h.abs()).clamp(max=1e3) + ey.square().mean(-1, keepdim=True).sqrt() * h.abs()
    z, mass = h @ W.T, h.abs() @ W.abs().T
    e = (2.0 ** -8 + 2.0 * K * 2.0 ** -24) * mass + slack @ W.abs().T
    if act is None:
        assert ((got.double() - z).abs() <= e + (2.0 ** -8 * z.abs() if out_dtype != F32 else 0) + 1e-30).all()
        return
    g, u = z.chunk(2, -1)
    eg, eu = e.chunk(2, -1)
    if act == sm.ACT_GELU_TANH:
        want, slope = torch.nn.functional.gelu(g, approximate="tanh") * u, 1.13
    elif act == sm.ACT_RELU:
        want, slope = g.clamp(min=0) * u, 1.0
    else:
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5) + 1.0
        want, slope = g * torch.sigmoid(1.702 * g) * u, 1.1
    assert ((got.double() - want).abs() <= slope * eg * u.abs() + slope * (g.abs() * eu + eg * eu) + 2.0 ** -7 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("M", [1, 2, 3, 8, 9, 16])
@pytest.mark.parametrize("K,N", [(128, 128), (1152, 2048), (2048, 2048), (8192, 2048), (14336, 4096), (2176, 1280), (4096, 3968)])
def test_stream_and_rows(M, K, N, entries):
    r = data(M + K + N)
    x, a, w, nw, y, ey = stream(r, M, K, N)
    x0 = x.clone()
    rows = sm.linear_rows(a, w, x, nw, EPS, mult=0.6, offset=1.0)
    assert rows.sums is not None and "resnorm" not in entries and torch.equal(x, x0)
    assert ((rows.x.double() - y).abs() <= ey).all()
    want = rows.x.double() * (1.0 + nw.double())
    assert ((rows.h.double() - want).abs() <= 2.0 ** -8 * want.abs()).all()
    ss = rows.sums.view(-1)[:M * rows.count].view(M, rows.count).double().sum(-1)
    assert ((ss - rows.x.double().square().sum(-1)).abs() <= 2.0 ** -17 * ss).all()     # bands of at most 64 squares, in fp32
    for n in (1, 5, 2050):
        v = r(n, N, m=N ** -0.5)
        close(sm.rows_linear(rows, v, EPS), y, ey, nw, v, BF)
        close(sm.rows_linear(rows, v, EPS, out_dtype=F32), y, ey, nw, v, F32)
    assert entries.count("rows_in") == 6 and "resnorm" not in entries


@pytest.mark.parametrize("act", [sm.ACT_GELU_TANH, sm.ACT_SWISH_CLAMP, sm.ACT_RELU])
@pytest.mark.parametrize("M,W", [(1, 2048), (3, 128), (8, 2048), (16, 2048), (8, 4096), (13, 4096)])
@pytest.mark.parametrize("N", [1, 63, 2050, 14336])
def test_gated(act, M, W, N, entries):
    r = data(M + W + N)
    x, a, w, nw, y, ey = stream(r, M, 256, W)
    rows = sm.linear_rows(a, w, x, nw, EPS, mult=0.6, offset=1.0)
    v = r(2 * N, W, m=W ** -0.5)
    got = sm.rows_linear(rows, v, EPS, act_kind=act, limit=1.5, alpha=1.702)
    assert "rows_in" in entries and "resnorm" not in entries
    close(got, y, ey, nw, v, BF, act)


@pytest.mark.parametrize("M,W", [(1, 2048), (8, 2048), (16, 2048), (5, 4096), (17, 2048), (3, 192)])
@pytest.mark.parametrize("n1,n2", [(1, 1), (3072, 576), (2045, 13), (7, 4096)])
def test_split_and_other_sizes(M, W, n1, n2, entries):
    r = data(M + n1)
    x, a, w, nw, y, ey = stream(r, M, 256, W)
    rows = sm.linear_rows(a, w, x, nw, EPS, mult=0.6, offset=1.0)
    v = r(n1 + n2, W, m=W ** -0.5)
    first, rest = sm.rows_linear(rows, v, EPS, split=n1)
    assert first.shape == (M, n1) and rest.shape == (M, n2)
    if M > 16 or W % 128:
        assert rows.sums is None and "resnorm" in entries        # the product and the norm: the branch is rounded on its way
        ey = ey + 0.6 * 2.0 ** -8 * (a.double() @ w.double().T).abs()
    close(torch.cat([first, rest], 1), y, ey, nw, v, BF)


@pytest.mark.parametrize("dt", [BF, F32])
@pytest.mark.parametrize("W", [4, 1024, 1028, 2048, 4096])
@pytest.mark.parametrize("T,n,branch,rowvec", [(1, 5, True, False), (8, 5, False, False), (33, 4, True, True), (3, 1, False, True)])
def test_norm_shift(dt, W, T, n, branch, rowvec, entries):
    r = data(W + T)
    x, w, mu, state = r(T, W, dt=F32, m=2.0), r(W, dt=dt), r(n, W, dt=dt), r(T + 2, W, dt=dt)
    kw = dict(branch=r(T, W, dt=dt) if branch else None, mult=0.6, rowvec=r(W, dt=dt) if rowvec else None, offset=1.0)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    b = {"seq_slots": i32([T + 1 - i for i in range(T)]), "cu_q": i32(list(range(T + 1))),
         "tok_seq": i32(list(range(T))), "positions": i32([(0, 7, -1, 3)[i % 4] for i in range(T)])}
    x2, s2 = x.clone(), state.clone()
    got = sm.norm_shift(x, w, EPS, mu, state, b, single=True, **kw)
    assert entries == ["norm_shift"]
    want = sm.norm_shift(x2, w, EPS, mu, s2, b, **kw)
    assert torch.equal(got, want) and torch.equal(x, x2) and torch.equal(state, s2)


@pytest.mark.parametrize("M", [1, 3, 8, 9, 16, 17])
@pytest.mark.parametrize("N,L,K", [(2048, 128, 2048), (8, 8, 128), (24, 1, 1152), (4096, 256, 4096), (2040, 127, 1024), (20, 4, 256),
                                   (8, 9, 128), (8, 24, 128), (64, 300, 256), (16, 2048, 1024)])
def test_several_inputs(M, N, L, K, entries):
    r = data(M + N + L)
    a, w = r(5, M, K), r(4 * N + L, K, m=K ** -0.5)
    outs, last = sm.linear_each_tanh(a, w, N)
    assert ("rows_each" in entries) == (M <= (16 if K <= 2048 else 8) and N % 8 == 0)
    bound = lambda x, v, slope=1.0: slope * 2.0 * K * 2.0 ** -24 * (x.double().abs() @ v.double().abs().T)    # fp32 sums in any order
    for i in range(4):
        z = a[i].double() @ w[i * N:(i + 1) * N].double().T
        assert ((outs[i].double() - z).abs() <= bound(a[i], w[i * N:(i + 1) * N]) + 2.0 ** -8 * z.abs()).all()
    z = a[4].double() @ w[4 * N:].double().T
    twice = 0.0 if "rows_each" in entries else 2.0 ** -8 * z.abs()     # (other routes may round the product first)
    assert ((last.double() - z.tanh()).abs() <= bound(a[4], w[4 * N:]) + twice + 2.0 ** -8 * z.tanh().abs() + 1e-7).all()


@pytest.mark.parametrize("dt", [BF, F32])
@pytest.mark.parametrize("H,D,L", [(32, 64, 128), (2, 20, 24), (3, 128, 256), (1, 16, 4), (2, 48, 8)])
@pytest.mark.parametrize("T", [1, 8, 33])
def test_wkv_step(dt, H, D, L, T, entries):
    r = data(H + D + L + T)
    rkvg = r(4, T, H * D, dt=dt)
    lo, w2 = r(T, L, dt=dt).tanh(), r(H * D, L, dt=dt, m=L ** -0.5)
    w0, u, lnw, state = r(H * D, dt=dt), r(H * D, dt=dt), r(H * D, dt=dt), r(T + 1, H, D, D, dt=F32)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    b = {"seq_slots": i32([T - i for i in range(T)]), "cu_q": i32(list(range(T + 1))), "positions": i32([(9, 0, -1)[i % 3] for i in range(T)])}
    s2 = state.clone()
    got = sm.wkv_step(*rkvg, lo, w2, w0, u, lnw, state, b, H, D, 1e-6, True)
    groups = -(-D // 16)
    assert ("wkv_step" in entries) and ("wkv_scan" in entries) == (L % (4 * groups) != 0)
    z = lo.double() @ w2.double().T
    want = sm.wkv_scan(*rkvg, z.float(), w0, u, lnw, s2, b["cu_q"], b["seq_slots"], b["positions"], H, D, 1e-6)
    live = b["positions"] >= 0
    assert torch.equal(got[live], want[live])                        # a token's output reads the state before its own decay
    # |d exp(-exp(z)) / dz| <= 1 / e, z in fp32 sums
    dz = (L + 8) * 2.0 ** -24 * (lo.double().abs() @ w2.double().abs().T) + 2.0 ** -22 * (z.abs() + w0.double().abs() + 1)
    bound = torch.zeros_like(s2, dtype=torch.float64)
    bound[b["seq_slots"].long()] = dz.view(T, H, D, 1).expand(T, H, D, D) / 2.7
    assert ((state.double() - s2.double()).abs() <= bound * (8.0 + s2.double().abs()) + 1e-6).all()


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("C,R,H,Dn,dims", [(512, 64, 16, 128, 64), (512, 64, 16, 128, 32), (16, 8, 3, 64, 8), (1024, 64, 2, 64, 64), (64, 24, 5, 128, 16),
                                           (512, 64, 33, 64, 0)])
@pytest.mark.parametrize("T", [1, 16, 17, 64, 65])
def test_latent_begin(C, R, H, Dn, dims, interleaved, T, entries):
    """The cache rows and the queries against 64 bits, and the one launch bit for bit as the two."""
    r = data(C + H + T)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    wide, nw, q, uk, cache = r(T, C + R + 8, m=2.0), r(C), r(T, H * (Dn + R)), r(H, C, Dn, m=Dn ** -0.5), r(T + 3, C + R)
    dkv, cs = wide[:, 8:], r(40, max(dims, 1), dt=F32)[:, :dims].contiguous()
    pos, slots = [(i * 7) % 40 if i % 5 != 3 else -1 for i in range(T)], [T + 2 - i if i % 4 != 2 else -1 for i in range(T)]
    run = lambda c, qq, absorb: sm.latent_kv_write(c, dkv, nw, qq, cs, i32(pos), i32(slots), C, R, H, Dn, dims, 1e-6, interleaved, absorb)
    c2, q2, c1, q1 = cache.clone(), q.clone(), cache.clone(), q.clone()
    got = run(c1, q1, uk)
    assert ("latent_begin" in entries) == (T <= 64) and (got is not None) == (T <= 64)
    assert run(c2, q2, None) is None
    assert torch.equal(c1, c2) and torch.equal(q1, q2)
    if got is not None:
        want = torch.empty(T, H, C, dtype=BF, device=DEV)
        sm.gemm(q.view(T, H, Dn + R)[:, :, :Dn].permute(1, 0, 2), uk, out=want.permute(1, 0, 2))
        z = torch.matmul(q.view(T, H, Dn + R)[:, :, :Dn].permute(1, 0, 2).double(), uk.double().transpose(1, 2).contiguous()).permute(1, 0, 2)
        assert ((got.double() - z).abs() <= 2.0 ** -8 * z.abs() + 2.0 * Dn * 2.0 ** -24 * 8 * Dn ** 0.5).all()

    def rotated(v, p):
        v, half = v.double().clone(), dims // 2
        c, s = cs[p, :half].double(), cs[p, half:].double()
        ia, ib = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, half), slice(half, dims))
        a, b = v[..., ia].clone(), v[..., ib].clone()
        v[..., ia], v[..., ib] = a * c - b * s, b * c + a * s
        return v
    for t in range(T):
        qt, qo = q1[t].view(H, Dn + R), q[t].view(H, Dn + R)
        if pos[t] < 0:
            assert torch.equal(qt, qo)
            continue
        want = torch.cat([qo[:, :Dn].double(), rotated(qo[:, Dn:], pos[t])], 1)
        assert ((qt.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()
        if slots[t] >= 0:
            d = dkv[t].double()
            row = torch.cat([d[:C] * (d[:C].square().mean() + 1e-6).rsqrt() * nw.double(), rotated(dkv[t, C:], pos[t])])
            assert ((c1[slots[t]].double() - row).abs() <= 2.0 ** -8 * row.abs() + 1e-5).all()
    untouched = [i for i in range(T + 3) if i not in [s for s, p in zip(slots, pos) if s >= 0 and p >= 0]]
    assert torch.equal(c1[untouched], cache[untouched])


@pytest.mark.parametrize("dt", [BF, F32])
@pytest.mark.parametrize("B,W,copy", [(1, 2048, True), (8, 48, False), (255, 64, True), (256, 4096, False), (600, 8, True)])
def test_embed_step(dt, B, W, copy, entries):
    r = data(B + W)
    table, ids = r(90, W, dt=dt), torch.randint(-1, 91, (B,), dtype=torch.int32).to(DEV)
    ctx = torch.randint(0, 70, (B,), dtype=torch.int32).to(DEV)              # (beyond the tables' 4 pages of 16: idle)
    tables = torch.randint(0, 999, (B + 1, 4), dtype=torch.int32).to(DEV)
    got, meta = sm.embed_step(ids, table, ctx, tables, 16, 1.7, copy)
    assert entries == ["embed_step"]
    want = sm.embed_rows(ids, table, 1.7, copy)
    for a, b in zip(got if copy else (got,), want if copy else (want,)):
        assert torch.equal(a, b)
    for a, b in zip(meta, sm.decode_meta(ctx, tables, 16)):
        assert torch.equal(a, b) and a.data_ptr() % 16 == 0


@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("T,H", [(1, 16), (5, 3), (28, 16), (32, 16), (9, 40), (13, 40), (1, 130)])
@pytest.mark.parametrize("ctx", [40, 700, 2200])
def test_single_tokens_value_columns(T, H, ctx, gate):
    """A quarter of a head's value columns a workgroup, and all of them, on both sides of the change; up to 32 splits."""
    r = data(T + H + ctx)
    C, R, Dn, V, bs = 512, 64, 128, 128, 16
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    pages = -(-ctx // bs)
    cache, q, q_abs, uv = r(T * pages * bs, C + R), r(T, H * (Dn + R)), r(T, H, C), r(H, V, C, m=C ** -0.5)
    g = r(T, H) if gate else None
    pos = [ctx - 1 - (7 * i) % 30 for i in range(T)]
    b = {"cu_q": i32(list(range(T + 1))), "tok_seq": i32(list(range(T))), "positions": i32(pos), "max_keys": ctx,
         "block_tables": torch.randperm(T * pages).to(torch.int32).to(DEV).view(T, pages)}
    got = sm.latent_mix(q, cache, r(H, C, Dn), uv, None, b, C, R, H, Dn, V, 0, 0.05, bs, gate=g, q_abs=q_abs).view(T, H, V)
    for t in {0, T // 2, T - 1}:
        rows = (b["block_tables"][t].long()[:, None] * bs + torch.arange(bs, device=DEV)).reshape(-1)[:pos[t] + 1]
        k = cache[rows].double()
        qq = torch.cat([q_abs[t], q[t].view(H, Dn + R)[:, Dn:]], 1).double()
        p = torch.softmax(0.05 * qq @ k.T, -1)
        lat = p @ k[:, :C]
        mass = p @ k[:, :C].abs()
        if gate:
            s = torch.sigmoid(g[t].double())[:, None]
            lat, mass = lat * s, mass * s
        want = torch.matmul(uv.double(), lat.unsqueeze(-1)).squeeze(-1)
        # weights and the latent sum in bf16 (2^-9 each, and a score's fp32 error), sums in fp32, the output in bf16
        bound = torch.matmul(uv.double().abs(), (2.0 ** -7 * mass).unsqueeze(-1)).squeeze(-1) + 2.0 ** -8 * want.abs()
        assert ((got[t].double() - want).abs() <= bound).all()
