"""Windowed attention of portions in true fp32 on the matrix cores (window_f32.hip) against 64 bits, and beside the plain-FMA kernel."""
import pytest
import torch

from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


def exact(q, gate, kc, vc, bt, seq, pos, H, window, scale, sink, bs, chunk, softcap, sinks, per_head, slopes):
    T, G, D = len(pos), kc.shape[1], kc.shape[2]
    out = torch.zeros(T, H, D, dtype=torch.float64)
    qd = q[:, :H * D].double().reshape(T, H, D)
    for t, p in enumerate(pos.tolist()):
        if p < 0:
            continue
        j = torch.arange(p - p % chunk if chunk else max(0, p - window + 1) if window else 0, p + 1)
        slot = bt[int(seq[t])].long()[j // bs] * bs + j % bs
        k, v = (x[slot].double().repeat_interleave(H // G, 1) for x in (kc, vc))
        s = torch.einsum("jhd,hd->hj", k, qd[t]) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        if slopes is not None:
            s = s - slopes.double()[:, None] * (p - j)
        if sink:
            s = torch.cat([s, (sinks.double() if sinks is not None else torch.zeros(H, dtype=torch.float64))[:, None]], 1)
        out[t] = torch.einsum("hj,jhd->hd", torch.softmax(s, -1)[:, :len(j)], v)
    if gate is not None:
        out *= torch.sigmoid(gate.double()).view(T, H, -1)
    return out.view(T, H * D)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,G,window,chunk,bs,extra", [(16, 4, 0, 0, 16, ""), (4, 4, 70, 0, 8, "sink slopes"), (8, 4, 0, 32, 24, "gate"),
                                                       (16, 2, 5, 0, 16, "sinks softcap"), (16, 1, 33, 0, 16, "head")])
def test_against_64_bits(D, H, G, window, chunk, bs, extra, monkeypatch):
    """One token, a workgroup's tokens and one more, a chunk's and a window's edge among them, fewer tiles than waves; an idle sequence."""
    g = torch.Generator().manual_seed(D + H + G)
    lens, past = [1, 17, 40, 3, 130], [0, 60, 25, 0, 300]
    T, nb = sum(lens), -(-430 // bs)
    pos = torch.cat([torch.arange(a, a + n) for a, n in zip(past, lens)]).int()
    seq = torch.cat([torch.full((n,), (2 * i) % 5) for i, n in enumerate(lens)]).int()     # the block table's rows, as they are named
    pos[seq == 1] = -1
    cu = torch.tensor([0, *lens]).cumsum(0).int()
    bt = torch.randperm(5 * nb, generator=g).view(5, nb).int()
    kc, vc = (torch.randn(5 * nb * bs, G, D, generator=g) for _ in range(2))
    q = torch.randn(T, H * D + 4, generator=g)
    gate = torch.randn(T, (H if extra == "head" else H * D) + 4, generator=g)[:, :-4] if extra in ("gate", "head") else None
    sinks = torch.randn(H, generator=g) if "sinks" in extra else None
    slopes = torch.rand(H, generator=g) * 0.1 if "slopes" in extra else None
    softcap = 5.0 if "softcap" in extra else 0.0
    kw = dict(chunk=chunk, softcap=softcap, gate_per_head=extra == "head")
    want = exact(q, gate, kc, vc, bt, seq, pos, H, window, D**-0.5, "sink" in extra, bs, chunk, softcap, sinks, extra == "head", slopes)

    def run(mfma, v):
        monkeypatch.setattr(sm, "WINDOW_MFMA", mfma)
        monkeypatch.setattr(sm, "window_f32_plain", lambda *sizes: False)
        c = lambda x: x.cuda() if x is not None else None
        full = None
        if gate is not None:                       # the rows' own stride
            full = torch.zeros(T, gate.shape[1] + 4).cuda()[:, :-4]
            full.copy_(gate)
        return sm.window_attention(c(q), full, c(kc), c(v), None, None, c(bt), c(seq), c(pos), H, window, 0, D**-0.5, "sink" in extra, bs,
                                   c(cu), max(lens), sinks=c(sinks), slopes=c(slopes), **kw).cpu()

    err = [float((run(m, vc).double() - want).norm() / want.norm()) for m in (True, False)]
    assert err[0] <= 1e-6 and err[0] <= 1.25 * err[1], err        # 2^-24 times the few units of a score, no more than plain FMAs give
    assert (run(True, vc)[pos < 0] == 0).all()
    # a value reaches the tokens that see it and no other, whatever it is
    bad = vc.clone()
    for p, v in ((302, float("nan")), (331, float("inf")), (50, float("inf"))):
        bad[int(bt[3, p // bs]) * bs + p % bs] = v
    a, b = run(True, bad), run(False, bad)
    assert torch.equal(a.isfinite(), b.isfinite()) and torch.equal(a.isnan(), b.isnan())


def test_rows_behind_the_last_sequence(monkeypatch):
    """Idle rows that no sequence has (a batch filled up to its size) are zeros."""
    g = torch.Generator().manual_seed(5)
    T, H, G, D, bs = 40, 8, 2, 64, 16
    pos, seq = torch.cat([torch.arange(29), torch.full((11,), -1)]).int().cuda(), torch.zeros(T, dtype=torch.int32, device="cuda")
    kc, vc, q = (torch.randn(*n, generator=g).cuda() for n in ((32, G, D), (32, G, D), (T, H * D)))
    bt, cu = torch.tensor([[1, 0]], dtype=torch.int32).cuda(), torch.tensor([0, 29], dtype=torch.int32).cuda()
    monkeypatch.setattr(sm, "window_f32_plain", lambda *sizes: False)
    stale = torch.full((T, H * D), float("nan"), device="cuda")
    del stale
    y = sm.window_attention(q, None, kc, vc, None, None, bt, seq, pos, H, 0, 0, D**-0.5, False, bs, cu, 29)
    assert (y[29:] == 0).all() and y[:29].isfinite().all()
