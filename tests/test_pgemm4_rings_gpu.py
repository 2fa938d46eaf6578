"""The 4-wave big-tile products with deeper rings, 224- and 192-wide tiles and the XCDs spread over k: whole numbers, so that every
sum is exact in any order, and bf16 results where they are; rows that do not fill the tile, one stage to more than the ring holds."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
TILES = {0: (256, 256), 1: (256, 128), 2: (128, 256), 3: (128, 128), 5: (128, 64), 6: (64, 64), 7: (224, 256), 8: (256, 192), 9: (128, 96),
         10: (192, 96), 11: (192, 128), 12: (128, 192), 13: (192, 192), 14: (224, 192), 15: (192, 224), 16: (224, 224), 17: (256, 224)}


def whole(n, K, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randint(-3, 4, (n, K), generator=g) * (torch.rand(n, K, generator=g) < 0.15)).to(torch.bfloat16).cuda()


def out_of(M, N, shift=0):
    buf = torch.full((M * N + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    return buf, buf[shift:shift + M * N].view(M, N)


def untouched(buf, M, N, shift=0):
    return bool((buf[:shift] == 7).all() and (buf[shift + M * N:] == 7).all())


@pytest.mark.parametrize("cfg", sorted(TILES))
@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 6, 7, 9, 13])
def test_stages_of_every_ring(cfg, stages):
    """One row tile (every XCD begins at its own stage and wraps) and two (all begin at the first)."""
    bp, bq = TILES[cfg]
    K = 64 * stages
    for M, N, shift in ((1, 8, 0), (bq - 3, bp + 4, 0), (bq, 9 * bp - 8, 0), (bq + 1, bp + 16, 0), (bq - 1, 2 * bp - 4, 4)):
        x, w = whole(M, K, M + K), whole(N, K, N)
        want = x.float() @ w.float().T
        assert want.abs().max() <= 256
        buf, out = out_of(M, N, shift)
        ops.native().pgemm4(out.data_ptr(), 0, x.data_ptr(), w.data_ptr(), M, N, K, ops.EPI_BF16, cfg, 1, 4, 0, 0, 0.0, -1)
        assert torch.equal(out.float(), want) and untouched(buf, M, N, shift), (M, N, shift)
        assert torch.equal(ops.pgemm4(x, w, ops.EPI_F32, cfg=cfg), want), (M, N)
        if stages >= 3:
            assert torch.equal(ops.pgemm4(x, w, ops.EPI_BF16, cfg=cfg, splits=3).float(), want), (M, N, "split")


@pytest.mark.parametrize("cfg", [6, 7, 8, 9, 10, 13, 14, 16, 17])
@pytest.mark.parametrize("K", [64, 448])
def test_pairs_and_activations(cfg, K):
    """Gate and up rows of a feature in one fragment (224 rows) or in two; columns that do not fill the tile, a bias, split k."""
    bp, bq = TILES[cfg]
    for M, N, shift in ((bq - 1, bp // 2 + 8, 0), (bq + 5, bp // 2 - 4, 0), (17, bp + 12, 4), (3, 4, 0)):
        x, w = whole(M, K, M), whole(2 * N, K, N + 1)
        b = torch.randint(-2, 3, (2 * N,), generator=torch.Generator().manual_seed(N)).to(torch.bfloat16).cuda()
        y = x.float() @ w.float().T
        for bias in (None, b):
            z = y if bias is None else y + b.float()
            buf, out = out_of(M, N, shift)
            ops.native().pgemm4_act(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, cfg, 4, sm.ACT_RELU, 0.0, 1.0,
                                    0 if bias is None else b.data_ptr(), -1)
            assert torch.equal(out, (z[:, :N].clamp(min=0) * z[:, N:]).to(torch.bfloat16)) and untouched(buf, M, N, shift), (M, N)
        x = x + 1
        y = (x.double() @ w.double().T) * (x.double().square().mean(1, keepdim=True) + 1e-5).rsqrt()
        want = torch.nn.functional.silu(y[:, :N]) * y[:, N:]
        for splits in (1, 2) if K > 64 else (1,):
            got = ops.pgemm4(x, w, ops.EPI_SWIGLU, cfg=cfg, splits=splits, rms_eps=1e-5).double()
            # a rounding to bf16; the gate's exponential and division, |y| <= 60: its argument's error 60 x 2^-22
            assert ((got - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -14) + 1e-6).all(), (M, N, splits)


@pytest.mark.parametrize("sizes", [(1, 0, 3, 2, 7, 0, 5, 2), (64, 65, 0, 63, 1, 128, 200, 10), tuple([40] * 7 + [0, 3])])
@pytest.mark.parametrize("cfg", [1, 6, 7, 8, 10, 11, 12, 13, 15, 16, 17])
@pytest.mark.parametrize("kind", [None, sm.ACT_RELU])
def test_groups_spread_over_k(sizes, cfg, kind, monkeypatch):
    """8 and more groups of few rows: every XCD at its own stage; gathered rows."""
    monkeypatch.setattr(sm, "_grouped_tile", lambda *a: cfg)
    E, P, N, K = len(sizes), sum(sizes), 264, 576
    seg = torch.tensor((0,) + sizes).cumsum(0).to(torch.int32).cuda()
    x, w = whole(70, K, P), whole(E * N * (1 if kind is None else 2), K, cfg).view(E, -1, K)
    rows = torch.randint(0, 70, (P,), generator=torch.Generator().manual_seed(P)).to(torch.int32).cuda()
    tiles = torch.full((1, 3), -1, dtype=torch.int32, device="cuda")
    kw = dict(a_rows=rows, tiles=tiles, rows=P, seg=seg)
    assert sm._grouped_big(x, w, seg, P, N)
    got = sm.gemm(x, w, **kw) if kind is None else sm.gemm_act(x, w, kind, 0.0, 1.0, **kw)
    y = torch.cat([x[rows[int(seg[e]):int(seg[e + 1])].long()].float() @ w[e].float().T for e in range(E)])
    want = y if kind is None else y[:, :N].clamp(min=0) * y[:, N:]
    assert torch.equal(got, want.to(torch.bfloat16))


@pytest.mark.parametrize("cfg,bp", [(18, 64), (19, 96), (20, 128), (21, 160)])
@pytest.mark.parametrize("stages", [1, 2, 3, 5, 7, 32, 33])
@pytest.mark.parametrize("kind", [None, sm.ACT_RELU])
def test_groups_of_few_rows(cfg, bp, stages, kind):
    """The tiles of 32 tokens: groups at their edges, empty ones, columns that do not fill the last tile, one stage to more than the ring
    holds, k walked from every column's own stage (up to 32) and in step or an XCD's; rows stored whole and piecewise."""
    K = 64 * stages
    for sizes, N, shift in (((1, 0, 31, 32, 33, 0, 65, 2), bp + 16, 0), ((3, 32), 2 * bp, 0), ((0, 7, 64), bp - 4, 4), ((1, 2, 0, 1, 5, 0, 0, 2, 9), 3 * bp + 4, 0)):
        E, P = len(sizes), sum(sizes)
        seg = torch.tensor((0,) + sizes).cumsum(0).to(torch.int32).cuda()
        x, w = whole(70, K, P + stages), whole(E * N * (1 if kind is None else 2), K, cfg + N).view(E, -1, K)
        rows = torch.randint(0, 70, (P,), generator=torch.Generator().manual_seed(P)).to(torch.int32).cuda()
        y = torch.cat([x[rows[int(seg[e]):int(seg[e + 1])].long()].float() @ w[e].float().T for e in range(E)])
        want = y if kind is None else y[:, :N].clamp(min=0) * y[:, N:]
        buf, out = out_of(P, N, shift)
        ops.native().pgemm4_grouped(out.data_ptr(), x.data_ptr(), w.data_ptr(), 70, P, N, K, E, seg.data_ptr(), rows.data_ptr(),
                                    K, cfg, 4, -1 if kind is None else kind, 0.0, 1.0, 0.0, -1)
        assert torch.equal(out, want.to(torch.bfloat16)) and untouched(buf, P, N, shift), (sizes, N)


@pytest.mark.parametrize("cfg", [0, 1, 3, 5, 6, 8, 9, 10, 14])
@pytest.mark.parametrize("K", [2048, 2112, 16384])
def test_walks_over_k(cfg, K):
    """Columns of tiles that start apart (up to 2048), XCDs of deep rows with several row tiles (from 16384): whole, split and gated."""
    bp, bq = TILES[cfg]
    M, N = 2 * bq + 5, 3 * bp + 8
    x, w = whole(M, K, K), whole(N, K, N)
    y = x.float() @ w.float().T                       # whole numbers below 2^24
    assert torch.equal(ops.pgemm4(x, w, ops.EPI_F32, cfg=cfg), y)
    assert torch.equal(ops.pgemm4(x, w, ops.EPI_F32, cfg=cfg, splits=4), y)
    out = torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda")
    ops.native().pgemm4_act(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N // 2, K, cfg, 4, sm.ACT_RELU, 0.0, 1.0, 0, -1)
    assert torch.equal(out, (y[:, :N // 2].clamp(min=0) * y[:, N // 2:]).to(torch.bfloat16))


@pytest.mark.parametrize("cfg", [3, 8, 13])
@pytest.mark.parametrize("tiles", [5, 8, 9])
@pytest.mark.parametrize("group_m", [1, 4])
def test_deep_weights_in_one_group_of_row_tiles(cfg, tiles, group_m):
    """From 16384 columns on up to 8 row tiles follow each other whatever group they are asked for in; 9 do not."""
    bp, bq = TILES[cfg]
    M, N, K = tiles * bq - 3, 2 * bp + 8, 16384
    x, w = whole(M, K, tiles), whole(N, K, cfg)
    y = x.float() @ w.float().T                       # whole numbers below 2^24
    assert torch.equal(ops.pgemm4(x, w, ops.EPI_F32, cfg=cfg, group_m=group_m), y)
    assert torch.equal(ops.pgemm4(x, w, ops.EPI_F32, cfg=cfg, group_m=group_m, splits=3), y)
