"""Latent attention over cached rows against 64 bits: true fp32 on the matrix cores (latent_f32.hip) beside the plain-FMA kernel, and the
key splits of portions of prompts in bf16."""
import pytest
import torch

from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


def exact(qa, q, cache, bt, seq, pos, C, R, H, Dn, window, scale, bs, sinks, gate):
    out = torch.zeros(len(pos), H, C, dtype=torch.float64)
    qr = q.double().view(len(pos), H, Dn + R)[..., Dn:]
    for t, p in enumerate(pos.tolist()):
        if p < 0:
            continue
        j = torch.arange(max(0, p - window + 1) if window else 0, p + 1)
        rows = cache[bt[int(seq[t])].long()[j // bs] * bs + j % bs].double()
        s = torch.cat([qa[t].double(), qr[t]], -1) @ rows.T * scale
        if sinks is not None:
            s = torch.cat([s, sinks.double()[:, None]], 1)
        out[t] = torch.softmax(s, -1)[:, :len(j)] @ rows[:, :C]
        if gate is not None:
            out[t] *= torch.sigmoid(gate[t].double())[:, None]
    return out


@pytest.mark.parametrize("C,R", [(512, 64), (256, 64), (128, 64), (128, 32), (64, 32)])
@pytest.mark.parametrize("H,window,bs,extra", [(16, 0, 16, ""), (4, 70, 8, "sinks"), (21, 0, 24, "gate"), (32, 33, 16, "both")])
def test_against_64_bits(C, R, H, window, bs, extra, monkeypatch):
    """One key, a tile's last and the next one's first, fewer tiles than waves, one more round of them; idle rows; heads beyond a block."""
    g = torch.Generator().manual_seed(C + R + H)
    pos = torch.tensor([0, 15, 16, -1, 47, 48, 63, 64, 129, 400, -1], dtype=torch.int32)
    T, Dn, nb = len(pos), 12, -(-401 // bs)
    seq = torch.tensor([0, 1, 2, 0, 1, 2, 0, 1, 2, 1, 2], dtype=torch.int32)
    bt = torch.randperm(3 * nb, generator=g).view(3, nb).int()
    cache = torch.randn(3 * nb * bs, C + R, generator=g)
    qa, q = torch.randn(T, H, C, generator=g), torch.randn(T, H * (Dn + R), generator=g)
    sinks = torch.randn(H, generator=g) * 3 if extra in ("sinks", "both") else None
    gate = torch.randn(T, H + 3, generator=g) if extra in ("gate", "both") else None
    if gate is not None:
        gate = gate[:, :H]
    scale = 2.0 * (C + R)**-0.5
    want = exact(qa, q, cache, bt, seq, pos, C, R, H, Dn, window, scale, bs, sinks, gate)
    err = []
    for mfma in (True, False):
        monkeypatch.setattr(sm, "LATENT_MFMA", mfma)
        gp = torch.randn(T, H + 3).cuda()[:, :H].copy_(gate) if gate is not None else None
        y = sm.latent_attention(qa.cuda(), q.cuda(), cache.cuda(), bt.cuda(), seq.cuda(), pos.cuda(), C, R, H, Dn, window, scale, bs,
                                sinks=sinks.cuda() if sinks is not None else None, gate=gp).cpu().double()
        assert (y[pos < 0] == 0).all()
        err.append(float((y - want).norm() / want.norm()))
    assert err[0] <= 2e-6 and err[0] <= 1.25 * err[1], err        # scores of up to 10: a part in 2^22 of them, and no more than plain FMAs give


@pytest.mark.parametrize("first,last", [(0, 16), (16, 32), (0, 64), (48, 101)])
def test_scores_of_minus_infinity(first, last):
    """Keys whose scores overflow to -infinity weigh nothing, wherever a wave meets them."""
    C, R, H, Dn, bs, p = 64, 32, 4, 8, 16, 100
    g = torch.Generator().manual_seed(first + last)
    cache = torch.randn(7 * bs, C + R, generator=g)
    cache[:, C] = 0.0
    cache[first:last, C] = -1e20
    qa, q = torch.randn(1, H, C, generator=g), torch.randn(1, H * (Dn + R), generator=g)
    q.view(H, Dn + R)[:, Dn] = 1e20
    bt, seq, pos = torch.arange(7, dtype=torch.int32)[None], torch.zeros(1, dtype=torch.int32), torch.tensor([p], dtype=torch.int32)
    want = exact(qa, q, cache, bt, seq, pos, C, R, H, Dn, 0, 0.1, bs, None, None)
    y = sm.latent_attention(qa.cuda(), q.cuda(), cache.cuda(), bt.cuda(), seq.cuda(), pos.cuda(), C, R, H, Dn, 0, 0.1, bs).cpu().double()
    assert float((y - want).norm()) <= 2e-6 * float(want.norm())


@pytest.mark.parametrize("first,last", [(0, 32), (128, 160), (256, 512)])
def test_scores_of_minus_infinity_in_bf16_splits(first, last):
    """The same for four tokens a workgroup, where those keys are the first of a split, or a whole one."""
    C, R, H, Dn, bs, T, past = 512, 64, 16, 16, 16, 200, 400
    g = torch.Generator().manual_seed(first)
    pos, seq = torch.arange(past, past + T, dtype=torch.int32), torch.zeros(T, dtype=torch.int32)
    nb = (past + T) // bs + 1
    bt, cu = torch.arange(nb, dtype=torch.int32)[None], torch.tensor([0, T], dtype=torch.int32)
    cache = torch.randn(nb * bs, C + R, generator=g).bfloat16()
    cache[:, C] = 0.0
    cache[first:last, C] = -1e30
    qa, q = torch.randn(T, H, C, generator=g).bfloat16(), torch.randn(T, H * (Dn + R), generator=g).bfloat16()
    q.view(T, H, Dn + R)[:, :, Dn] = 1e30
    assert sm.latent_quad_splits(T, 1, H, nb * bs) > 1
    want = exact(qa, q, cache, bt, seq, pos, C, R, H, Dn, 0, 0.04, bs, None, None)
    y = sm.latent_attention(qa.cuda(), q.cuda(), cache.cuda(), bt.cuda(), seq.cuda(), pos.cuda(), C, R, H, Dn, 0, 0.04, bs, 0, cu.cuda(),
                            T).cpu().double()
    assert float((y - want).norm()) <= 2.0**-7 * float(want.norm())          # (weights and result rounded to bf16)


@pytest.mark.parametrize("H,lens,past,window", [(16, (4, 9), 600, 0), (16, (97, 1, 1), 300, 1024), (20, (30, 3), 1000, 70), (32, (60, 5), 130, 0),
                                                (16, (5, 2), 189, 0), (3, (8,), 2000, 0)])
def test_key_splits_of_portions_in_bf16(H, lens, past, window):
    """Four tokens a workgroup, their keys split: fewer keys than a split, around the fewest that are split, splits that stay empty; an
    idle sequence at the batch's end, whose workgroups leave no records; sinks and gates through the kernel that joins and through the
    one that has nothing to join."""
    C, R, Dn, bs, idle = 512, 64, 16, 16, 5
    g = torch.Generator().manual_seed(past + H)
    n, lens = len(lens) + 1, (*lens, idle)
    T = sum(lens)
    pos = torch.cat([torch.arange(k) + (past if i != 1 else 0) for i, k in enumerate(lens)]).int()
    pos[-idle:] = -1
    seq = torch.cat([torch.full((k,), n - 1 - i) for i, k in enumerate(lens)]).int()      # the block table's rows, as they are named
    nb = (past + max(lens)) // bs + 1
    bt = torch.randperm(n * nb, generator=g).view(n, nb).int()
    cu = torch.tensor([0, *lens]).cumsum(0).int()
    cache = torch.randn(n * nb * bs, C + R, generator=g).bfloat16()
    qa, q = torch.randn(T, H, C, generator=g).bfloat16(), torch.randn(T, H * (Dn + R), generator=g).bfloat16()
    sinks, gate = torch.randn(H, generator=g), torch.randn(T, H, generator=g).bfloat16()
    scale = (C + R)**-0.5
    ns = sm.latent_quad_splits(T, n, H, min(window or nb * bs, nb * bs))
    assert ns > 1
    want = exact(qa, q, cache, bt, seq, pos, C, R, H, Dn, window, scale, bs, sinks, gate)
    args = [x.cuda() for x in (qa, q, cache, bt, seq, pos)]
    kw = dict(sinks=sinks.cuda(), gate=gate.cuda())
    cu = cu.cuda()
    HP = (H + 15) // 16 * 16
    stale = [torch.full((k,), float("nan"), device="cuda") for k in (T * HP * ns * C, T * HP * ns * 2, (T * H * C + 1) // 2)]
    del stale                  # what the result and the records are given: one that is read without being written shows
    y = sm.latent_attention(*args, C, R, H, Dn, window, scale, bs, 0, cu, max(lens), **kw).cpu().double()
    assert (y[-idle:] == 0).all()
    T -= idle
    for t in range(T):          # weights and result rounded to bf16: 2^-9 of each, 2-norm below 2^-8 a row
        assert float((y[t] - want[t]).norm()) <= 2.0**-7 * float(want[t].norm()), t
