"""The fp32 products on the bf16 matrix cores (gemm_f32_parts.hip) against 64 bits: every tile at the edges of rows, columns and steps."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix

pytestmark = pytest.mark.gpu

MENU = [111, 112, 121, 122, 222, 223, 224, 225, 226, 423, 424, 425, 426, 427, 826, 827, 828]
NORM = 2.0**-22      # of the error, 2-norm, normal inputs: what the fp32 pipes' kernels show at K = 2048 and more


def call(a, w, tile, ldc=None):
    (M, K), N = a.shape, w.shape[0]
    out = torch.full((M + 1, ldc or N), 7.0, device="cuda")
    ops.native().gemm_f32_parts(out.data_ptr(), a.data_ptr(), w.data_ptr(), M, N, K, a.stride(0), w.stride(0), out.stride(0), 1, 0, 0, 0,
                                0, 0, 0, tile, -1)
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()
    return out[:M, :N]


@pytest.mark.parametrize("tile", MENU)
@pytest.mark.parametrize("rows,cols,K", [(0, 0, 32), (1, 2, 96), (-1, -1, 288), (5, 70, 1056), (0, 3, 2208)])
def test_every_tile(tile, rows, cols, K):
    """A tile's rows and columns, one more, one less, two of them and a rest; steps that not every share of k has."""
    wc, cw, fq = tile // 100, tile // 10 % 10, tile % 10
    M, N = 16 * fq * (2 if rows == 5 else 1) + rows, 16 * cw * wc + cols
    g = torch.Generator().manual_seed(tile + K)
    a, w = (torch.randint(-4000, 4001, (n, K), generator=g).float().cuda() for n in (M, N))
    a *= torch.rand(M, K, generator=g).cuda() < 0.0004                               # |sums| < 2^24 where at most one of a row is left
    keep = (a != 0).sum(1) <= 1
    assert torch.equal(call(a, w, tile)[keep].double(), (a.double() @ w.double().T)[keep])
    a, w = (torch.randint(-8, 9, (n, K), generator=g).float().cuda() for n in (M, N))
    assert torch.equal(call(a, w, tile).double(), a.double() @ w.double().T)
    a = torch.randn(M, K + 4, generator=g).cuda()[:, :K]                             # rows 16 bytes apart from K
    w = torch.randn(N, K, generator=g).cuda()
    ref = a.double() @ w.double().T
    assert (call(a, w, tile, ldc=N + 1).double() - ref).norm() <= NORM * ref.norm()


@pytest.mark.parametrize("tile", [111, 224, 826])
def test_values_without_parts(tile):
    """Infinities, NaN and values that round to infinity give what fp32 products give; rows too small for their low parts keep them."""
    M, N, K = 70, 100, 544
    g = torch.Generator().manual_seed(tile)
    a, w = torch.randn(M, K, generator=g).cuda(), torch.randn(N, K, generator=g).cuda()
    a[3, K - 1], a[5, 0], w[7, 2], a[9, 4], a[11, :] = float("inf"), -float("inf"), float("nan"), 3.4028234e38, 0.0
    w[:, 4] *= 1e-3
    y, ref = call(a, w, tile), (a.double() @ w.double().T).float()
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    assert torch.equal(y[y.isinf()], ref[ref.isinf()])
    fine = ref.isfinite()
    assert ((y - ref).abs()[fine] <= 1e-5 * (a.nan_to_num(0, 0, 0).abs() @ w.nan_to_num(0).abs().T)[fine]).all()
    a, w = torch.randn(M, K, generator=g).cuda() * 2.0**-112, torch.randn(N, K, generator=g).cuda()
    ref = a.double() @ w.double().T
    assert ((call(a, w, tile).double() - ref).norm()) <= NORM * ref.norm()


@pytest.mark.parametrize("tile", MENU)
@pytest.mark.parametrize("small,large", [(-116, 60), (-120, 100), (-125, 60), (-136, 100), (-140, 120)])
def test_small_values_against_large_ones(tile, small, large):
    """Operands that lose parts to their size, or all of them, where the other side's size makes ordinary outputs of theirs."""
    M, N, K = 40, 70, 544
    g = torch.Generator().manual_seed(tile - small)
    a, w = torch.randn(M, K, generator=g) * 2.0**small, torch.randn(N, K, generator=g) * 2.0**large
    a[7] = 0.0
    for x, y in ((a.cuda(), w.cuda()), (w.cuda(), a.cuda())):
        ref = x.double() @ y.double().T
        got = call(x, y, tile).double()
        assert (got - ref).norm() <= NORM * ref.norm()
        assert (got[ref == 0] == 0).all()


@pytest.mark.parametrize("tile", MENU)
def test_rows_and_columns_of_every_size(tile):
    """Each output by the sizes of its own row and column, whatever lies beside them; rows and columns that do not fill the tiles."""
    M, N, K = 16 * (tile % 10) + 5, 16 * (tile // 10 % 10) * (tile // 100) + 6, 288
    g = torch.Generator().manual_seed(tile)
    a = torch.randn(M, K, generator=g) * 2.0**torch.tensor([-120.0, 0.0, 20.0, -60.0])[torch.arange(M) % 4, None]
    w = torch.randn(N, K, generator=g) * 2.0**torch.tensor([100.0, -20.0, 0.0])[torch.arange(N) % 3, None]
    a, w = a.cuda(), w.cuda()
    ref, most = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    assert ((call(a, w, tile).double() - ref).abs() <= 2.0**-20 * most + 2.0**-120).all()


@pytest.mark.parametrize("tile", MENU)
@pytest.mark.parametrize("K", [32, 288, 2208])
def test_outputs_that_are_computed_again(tile, K):
    """Sums that cancel to zero beside others, in every place of a tile, and k that does not fill the wave."""
    M, N = 16 * (tile % 10) + 3, 16 * (tile // 10 % 10) * (tile // 100) + 5
    g = torch.Generator().manual_seed(tile + K)
    a, w = torch.randint(-9, 10, (M, K), generator=g).float(), torch.randint(-9, 10, (N, K), generator=g).float()
    a[::3, 2:], w[::5, 2:] = 0.0, 0.0
    a[::3, :2], w[::5, 0], w[::5, 1] = 1.0, 7.0, -7.0
    a[1, 5] = 2.0**-130                                 # a row of small values with an ordinary one
    a, w = a.cuda(), w.cuda()
    ref = a.double() @ w.double().T
    assert (ref[::3, ::5] == 0).all() and torch.equal(call(a, w, tile).double(), ref.float().double())


@pytest.mark.parametrize("tile", [111, 224, 826])
def test_results_next_to_the_largest(tile):
    """High parts whose product rounds to infinity where the values' own does not; sums that are infinite stay so."""
    M, N, K = 20, 40, 96
    a, w = torch.zeros(M, K, device="cuda"), torch.ones(N, K, device="cuda")
    most = 2.0 - 2.0**-23
    a[:, 5], w[:, 5] = most * 2.0**63, most * 2.0**63
    a[3, 5] = -a[3, 5]
    a[4, 6] = 3e38
    y, ref = call(a, w, tile), (a.double() @ w.double().T).float()
    assert torch.equal(y, ref) and ref[4].isinf().all() and ref[:3].isfinite().all()


@pytest.mark.parametrize("fq,tile", [(1, 111), (2, 222), (4, 224), (4, 424)])
def test_listed_tiles(fq, tile):
    g = torch.Generator().manual_seed(tile)
    counts = [70, 0, 64, 1, 130]                       # tiles: full, partial, an empty group; one listed beyond the end
    seg = torch.tensor([0] + counts).cumsum(0).int()
    listed = [(e, int(seg[e]) + r, min(64, n - r)) for e, n in enumerate(counts) for r in range(0, n, 64)] + [(-1, 0, 0)] * 2
    tiles = torch.tensor(listed, dtype=torch.int32).cuda()
    a, w = torch.randn(50, 1024, generator=g).cuda(), torch.randn(5, 1030, 1024, generator=g).cuda()
    pick = torch.randint(0, 50, (int(seg[-1]),), generator=g).int().cuda()
    out = torch.empty(int(seg[-1]), 1030, device="cuda")
    ops.native().gemm_f32_parts(out.data_ptr(), a.data_ptr(), w.data_ptr(), out.shape[0], 1030, 1024, 1024, 1024, 1030, 1, 0, 1030 * 1024,
                                0, pick.data_ptr(), tiles.data_ptr(), len(listed), tile, -1)
    for e in range(5):
        x = a[pick[seg[e]:seg[e + 1]].long()]
        ref = x.double() @ w[e].double().T
        assert (out[seg[e]:seg[e + 1]].double() - ref).norm() <= NORM * ref.norm(), e


@pytest.mark.parametrize("G,M,N,K", [(1, 1, 2048, 2048), (1, 16, 2048, 8192), (1, 333, 3072, 2048), (4, 130, 512, 512), (1, 457, 4096, 14336)])
def test_products_of_the_rule(G, M, N, K):
    """Through the public entry point, batched ones with strides of their own, captured and replayed."""
    g = torch.Generator().manual_seed(M)
    a = torch.randn(M, G, K, generator=g).cuda().transpose(0, 1)
    w = torch.randn(G, N, K, generator=g).cuda() * K**-0.5
    assert ops.native().gemm_f32_parts_rule(M, N, K, G, 0) > 0
    ref = a.double() @ w.double().transpose(1, 2).contiguous()
    y = seqmix.gemm(a, w)
    assert (y.double() - ref).norm() <= NORM * ref.norm()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = seqmix.gemm(a, w)
    for _ in range(3):
        z.fill_(3.0)
        graph.replay()
        assert torch.equal(z, y)
