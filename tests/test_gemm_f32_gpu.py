"""The fp32 products of many tiles (gemm_f32.hip) against 64 bits: every tile height at the edges of tiles, stages and chains."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix

pytestmark = pytest.mark.gpu


def bound(a, w, K):
    """Worst case of chains of at most 128 terms and then of at most K / 32: (terms) 2^-24 sum |a w|, and the product's own."""
    return (128 + K // 32 + 2) * 2.0**-24 * (a.abs().double() @ w.abs().double().T) + 1e-30


def tiles_call(a, w, fq, out_dtype=torch.float32, ldc=None):
    M, K = a.shape
    N = w.shape[0]
    out = torch.full((M + 1, ldc or N), 7.0, dtype=out_dtype, device="cuda")
    ops.native().gemm_f32_tiles(out.data_ptr(), a.data_ptr(), w.data_ptr(), M, N, K, a.stride(0), w.stride(0), out.stride(0), 1,
                                0, 0, 0, 0, 0, 0, int(out_dtype == torch.float32), fq, -1)
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()
    return out[:M, :N]


@pytest.mark.parametrize("fq", range(1, 9))
@pytest.mark.parametrize("rows,N,K", [(0, 64, 32), (1, 130, 64), (-1, 67, 160), (5, 200, 1056), (0, 63, 2208)])
def test_every_tile_height(fq, rows, N, K):
    """16 fq rows, one more, one less, two tiles and a tail; columns past a tile and not a multiple of 4; whole numbers exactly."""
    M = 16 * fq * (2 if rows == 5 else 1) + rows
    g = torch.Generator().manual_seed(fq * 1000 + N)
    a, w = (torch.randint(-8, 9, (n, K), generator=g).float().cuda() for n in (M, N))
    assert torch.equal(tiles_call(a, w, fq).double(), a.double() @ w.double().T)      # |sums| < 2^24
    a = torch.randn(M, K + 4, generator=g).cuda()[:, :K]                              # rows 16 bytes apart from K
    w = torch.randn(N, K, generator=g).cuda()
    ref = a.double() @ w.double().T
    assert ((tiles_call(a, w, fq, ldc=N + 1).double() - ref).abs() <= bound(a, w, K)).all()
    y = tiles_call(a, w, fq, torch.bfloat16).double()
    assert ((y - ref).abs() <= bound(a, w, K) + 2.0**-8 * ref.abs()).all()


@pytest.mark.parametrize("M,N,K", [(333, 2048, 2048), (200, 16384, 512), (96, 2048, 8192), (40, 3000, 1024)])
def test_products_of_the_rule(M, N, K):
    """Through the public entry point, whichever kernel the rule takes; infinities and NaN reach exactly their row or column."""
    g = torch.Generator().manual_seed(M)
    a, w = (torch.randn(n, K, generator=g).cuda() for n in (M, N))
    ref = a.double() @ w.double().T
    assert ((seqmix.gemm(a, w).double() - ref).abs() <= bound(a, w, K)).all()
    a[M // 2, K - 1], w[N // 3, 0] = float("inf"), float("nan")
    y = seqmix.gemm(a, w)
    bad = ~y.isfinite()
    assert bad[M // 2].all() and bad[:, N // 3].all() and int(bad.sum()) == M + N - 1


def test_batched_and_grouped():
    g = torch.Generator().manual_seed(3)
    a, w = torch.randn(4, 333, 2048, generator=g).cuda(), torch.randn(4, 2048, 2048, generator=g).cuda()
    y = seqmix.gemm(a, w)
    for i in range(4):
        assert ((y[i].double() - a[i].double() @ w[i].double().T).abs() <= bound(a[i], w[i], 2048)).all(), i
    counts = [70, 0, 64, 1, 130]                       # tiles: full, partial, an empty group; one listed beyond the end
    seg = torch.tensor([0] + counts).cumsum(0).int()
    rows, listed = int(seg[-1]), []
    for e, n in enumerate(counts):
        listed += [(e, int(seg[e]) + r, min(64, n - r)) for r in range(0, n, 64)]
    listed += [(-1, 0, 0)] * 3
    tiles = torch.tensor(listed, dtype=torch.int32).cuda()
    a, w = torch.randn(50, 1024, generator=g).cuda(), torch.randn(5, 1030, 1024, generator=g).cuda()
    pick = torch.randint(0, 50, (rows,), generator=g).int().cuda()
    for fq in (0, 1, 2, 4):
        out = torch.empty(rows, 1030, device="cuda")
        args = (out.data_ptr(), a.data_ptr(), w.data_ptr(), rows, 1030, 1024, 1024, 1024, 1030, 1, 0, 1030 * 1024, 0,
                pick.data_ptr(), tiles.data_ptr(), len(listed))
        if fq:
            ops.native().gemm_f32_tiles(*args, 1, fq, -1)
        else:
            ops.native().gemm_any(*args, 1, 1, -1)
        for e in range(5):
            x = a[pick[seg[e]:seg[e + 1]].long()]
            d = (out[seg[e]:seg[e + 1]].double() - x.double() @ w[e].double().T).abs()
            assert (d <= bound(x, w[e], 1024)).all(), (fq, e)


@pytest.mark.parametrize("fq", range(1, 5))
@pytest.mark.parametrize("rows,N,K", [(0, 64, 64), (1, 130, 96), (-1, 67, 160), (5, 200, 1056), (0, 63, 2208), (1, 64, 544)])
def test_k_shared_by_the_waves(fq, rows, N, K):
    """As above for the tiles whose waves share k: one stage a wave and more, uneven shares, an odd number of them, and infinities
    and NaN in the last and the first k."""
    M = 16 * fq * (2 if rows == 5 else 1) + rows
    g = torch.Generator().manual_seed(fq * 1000 + N)
    a, w = (torch.randint(-8, 9, (n, K), generator=g).float().cuda() for n in (M, N))
    assert torch.equal(tiles_call(a, w, 16 + fq).double(), a.double() @ w.double().T)      # |sums| < 2^24
    a = torch.randn(M, K + 4, generator=g).cuda()[:, :K]
    w = torch.randn(N, K, generator=g).cuda()
    ref = a.double() @ w.double().T
    assert ((tiles_call(a, w, 16 + fq, ldc=N + 1).double() - ref).abs() <= bound(a, w, K)).all()
    assert ((tiles_call(a, w, 16 + fq, torch.bfloat16).double() - ref).abs() <= bound(a, w, K) + 2.0**-8 * ref.abs()).all()
    a[M // 2, K - 1], w[N // 3, 0] = float("inf"), float("nan")
    bad = ~tiles_call(a, w, 16 + fq).isfinite()
    assert bad[M // 2].all() and bad[:, N // 3].all() and int(bad.sum()) == M + N - 1


@pytest.mark.parametrize("fq", [1, 2, 4])
def test_listed_tiles_with_k_shared(fq):
    g = torch.Generator().manual_seed(fq)
    counts = [70, 0, 64, 1]
    seg = torch.tensor([0] + counts).cumsum(0).int()
    listed = [(e, int(seg[e]) + r, min(64, n - r)) for e, n in enumerate(counts) for r in range(0, n, 64)] + [(-1, 0, 0)]
    tiles = torch.tensor(listed, dtype=torch.int32).cuda()
    a, w = torch.randn(50, 576, generator=g).cuda(), torch.randn(4, 130, 576, generator=g).cuda()
    pick = torch.randint(0, 50, (int(seg[-1]),), generator=g).int().cuda()
    out = torch.empty(int(seg[-1]), 130, device="cuda")
    ops.native().gemm_f32_tiles(out.data_ptr(), a.data_ptr(), w.data_ptr(), out.shape[0], 130, 576, 576, 576, 130, 1, 0, 130 * 576, 0,
                                pick.data_ptr(), tiles.data_ptr(), len(listed), 1, 16 + fq, -1)
    for e in range(4):
        x = a[pick[seg[e]:seg[e + 1]].long()]
        assert ((out[seg[e]:seg[e + 1]].double() - x.double() @ w[e].double().T).abs() <= bound(x, w[e], 576)).all(), e
