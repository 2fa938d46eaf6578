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
