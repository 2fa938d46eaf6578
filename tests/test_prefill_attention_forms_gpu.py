"""Paged prefill attention in each of its workgroup forms against 64 bits: contexts at the ends of a tile and of a pair of tiles, pages that
do not divide a tile, every head grouping in every form, rows whose weights outgrow the first tile's maximum late, a negative scale, keys and
queries that are not finite."""
import math

import pytest
import torch

from k8s_llm_scheduler_amd import ops

pytestmark = pytest.mark.gpu
DEV, D, BF = "cuda", 128, torch.bfloat16


def run(nq, nkv, qlens, cached, bs=16, scale=1 / math.sqrt(D), spikes=0, seed=0, poison=None):
    g = torch.Generator().manual_seed(seed + sum(qlens) + nq)
    r = lambda *s: torch.randn(*s, generator=g).to(BF).to(DEV)
    ctx = [a + b for a, b in zip(qlens, cached)]
    pages = [-(-c // bs) for c in ctx]
    n = sum(pages) + 2
    kc, vc, q = r(n, bs, nkv, D), r(n, bs, nkv, D), r(sum(qlens), nq, D)
    order = torch.randperm(n, generator=g).to(torch.int32)
    bt, at, slots = torch.zeros(len(qlens), max(pages), dtype=torch.int32), 0, []
    for i, p in enumerate(pages):
        bt[i, :p] = order[at:at + p]
        slots.append((order[at:at + p].long()[:, None] * bs + torch.arange(bs)).reshape(-1)[:ctx[i]].to(DEV))
        at += p
    unused = torch.ones(n * bs, dtype=torch.bool, device=DEV)
    unused[torch.cat(slots)] = False
    kc.view(n * bs, nkv, D)[unused] = float("nan")          # behind a context's last key, and pages of nobody
    vc.view(n * bs, nkv, D)[unused] = float("nan")
    for j in range(spikes):                                  # keys that outdo all before them, ever larger, for ever later rows
        key = ctx[0] * (j + 1) // (spikes + 1)
        row = min(qlens[0] - 1, max(0, key - cached[0] + 3))
        kc.view(n * bs, nkv, D)[slots[0][key]] = (q[row, ::nq // nkv].float() * (2.0 + 2 * j)).to(BF)
    if poison is not None:
        poison(q, kc.view(n * bs, nkv, D), slots[0])
    cu = torch.tensor([0] + qlens).cumsum(0).to(torch.int32).to(DEV)
    got = ops.paged_prefill_attention(q, kc, vc, cu, torch.tensor(ctx, dtype=torch.int32, device=DEV), bt.to(DEV), scale, bs, max(qlens))
    assert poison is not None or got.isfinite().all()
    base, odd = 0, 0
    for i, (ql, c) in enumerate(zip(qlens, cached)):
        k, v = (t.view(n * bs, nkv, D)[slots[i]].double() for t in (kc, vc))
        rows = sorted({0, 1, ql // 3, ql // 2, ql - 2, ql - 1, *range(0, ql, max(1, ql // 9))} & set(range(ql)))
        pos = torch.tensor(rows, device=DEV) + c
        hidden = torch.arange(ctx[i], device=DEV)[None] > pos[:, None]
        for h in range(nq):
            kh, vh, qh = k[:, h * nkv // nq], v[:, h * nkv // nq], q[base:base + ql][rows, h].double()
            s = (scale * qh @ kh.T).masked_fill(hidden, -math.inf)
            p = torch.softmax(s, -1)
            want, mass = p @ vh, p @ vh.abs()
            # weights in bf16 (2^-9), scores in fp32 sums of 128 products (2^-9 of a weight up to scores of 100), the output in bf16
            out = got[base:base + ql][rows, h].double()
            err = (out - want).abs()
            assert ((err <= 2.0 ** -8 * mass + 2.0 ** -8 * want.abs() + 1e-30) | (want.isnan() & out.isnan())).all(), (i, h, err.max())
            odd += int(want.isnan().any(-1).sum())
        base += ql
    return odd


# heads, kv heads, tokens brought and tokens cached of a batch that takes the form by itself
FORMS = {5: (16, 2, [97], [0]), 4: (64, 8, [250, 30], [0, 9]), 8: (32, 8, [1100], [3]), 16: (64, 8, [1100], [0])}


def forced(monkeypatch, form):
    monkeypatch.setattr(ops, "_prefill_form", lambda *a: form)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("spikes,scale", [(0, 1 / math.sqrt(D)), (5, 1 / math.sqrt(D)), (3, -0.07), (0, 0.0)])
def test_forms(form, spikes, scale):
    nq, nkv, qlens, _ = FORMS[form]
    assert ops._prefill_form(sum(qlens), max(qlens), len(qlens), nq, nkv) == form
    run(*FORMS[form], scale=scale, spikes=spikes)


@pytest.mark.parametrize("nq,nkv", [(2, 2), (4, 2), (8, 2), (8, 1), (16, 1)])
@pytest.mark.parametrize("qlens,cached", [([1], [0]), ([1, 2, 40], [63, 64, 88]), ([65], [63]), ([300], [0]), ([2200, 1], [0, 700])])
def test_head_groups_and_tile_ends(nq, nkv, qlens, cached):
    run(nq, nkv, qlens, cached, spikes=2)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("nq,nkv", [(2, 2), (4, 2), (8, 2), (8, 1), (16, 1)])
def test_head_groups_in_every_form(form, nq, nkv, monkeypatch):
    forced(monkeypatch, form)
    run(nq, nkv, [1, 2, 40], [63, 64, 88], spikes=2)
    run(nq, nkv, [300, 7], [5, 130], spikes=3, scale=-0.07, bs=24)
    run(nq, nkv, [129], [0], bs=8)


@pytest.mark.parametrize("bs", [1, 8, 24, 64, 96, 160])
@pytest.mark.parametrize("nq,nkv,qlens,cached", [(16, 2, [130, 7], [0, 250]), (64, 8, [1100], [77])])
def test_page_sizes(bs, nq, nkv, qlens, cached):
    run(nq, nkv, qlens, cached, bs=bs)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("what", ["nan key", "infinite key", "nan query", "infinite query"])
def test_values_that_are_not_finite(form, what, monkeypatch):
    """A key spoils the rows that see it (infinite: those of a positive product, the others leave it out), a query its own row."""
    forced(monkeypatch, form)

    def poison(q, k, slots):
        if what == "nan key":
            k[slots[150], 0, 7] = math.nan
        elif what == "infinite key":
            k[slots[150], :, 7] = math.inf
            k[slots[3], 1, 9] = -math.inf
        else:
            q[66, 3, 11] = math.nan if what == "nan query" else math.inf

    odd = run(16, 2, [200, 30], [20, 1], poison=poison)
    assert odd > (0 if "query" in what else 10)
