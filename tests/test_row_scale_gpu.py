"""1 / rms of the rows in a pass of its own ahead of a big-tile product: against 64 bits, on every tile that takes it."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [0, 1, 2, 4, 7, 8])
@pytest.mark.parametrize("M,N,K,splits", [(1, 8, 64, 1), (257, 264, 192, 1), (300, 520, 2112, 2), (33, 100, 320, 3)])
def test_scaled_products(cfg, M, N, K, splits, monkeypatch):
    g = torch.Generator().manual_seed(M + N)
    x = (torch.randn(M, K, generator=g) * torch.logspace(-2, 2, M)[:, None]).to(torch.bfloat16).cuda()
    w = (torch.randn(2 * N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    monkeypatch.setattr(ops, "P4_SCALE_FLOPS", 0.0)
    assert ops.native().pgemm4_scaled_ok(cfg) and not any(map(ops.native().pgemm4_scaled_ok, (3, 5, 6, -1, 99)))
    xd = x.double()
    s = (xd.square().mean(1, keepdim=True) + 1e-5).rsqrt()
    y, mag = xd @ w.double().T * s, xd.abs() @ w.double().abs().T * s
    sums = 2.0 * K * 2.0 ** -24 * mag                  # the fp32 sums, and the scale's own, an order smaller
    got = ops.pgemm4(x, w, ops.EPI_BF16, cfg=cfg, splits=splits, rms_eps=1e-5).double()
    assert ((got - y).abs() <= sums + 2.0 ** -8 * y.abs() + 1e-30).all()
    got = ops.pgemm4(x, w, ops.EPI_SWIGLU, cfg=cfg, splits=splits, rms_eps=1e-5).double()
    a, b = y[:, :N], y[:, N:]
    want = torch.nn.functional.silu(a) * b
    # |d silu| <= 1.1; a product's error is each factor's times the other
    slack = 1.1 * sums[:, :N] * b.abs() + a.abs() * sums[:, N:] + 1.1 * sums[:, :N] * sums[:, N:]
    assert ((got - want).abs() <= slack + (2.0 ** -8 + 2.0 ** -14) * want.abs() + 1e-30).all()


def test_long_products_take_their_scales_ahead(monkeypatch):
    """By the operations and the tile, no more for an fp32 output; both forms within the sums' order of each other."""
    calls = []
    nat = ops.native()

    class Spy:
        def __getattr__(self, name):
            if name in ("pgemm4", "pgemm4_scaled"):
                calls.append(name)
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Spy)
    x, w = torch.randn(256, 1024).to(torch.bfloat16).cuda(), torch.randn(512, 1024).to(torch.bfloat16).cuda()
    for limit, epi, cfg, want in ((2.0 * 256 * 512 * 1024, ops.EPI_BF16, 0, "pgemm4_scaled"), (2.1 * 256 * 512 * 1024, ops.EPI_BF16, 0, "pgemm4"),
                                  (0.0, ops.EPI_F32, 0, "pgemm4"), (0.0, ops.EPI_BF16, 3, "pgemm4")):
        monkeypatch.setattr(ops, "P4_SCALE_FLOPS", limit)
        calls.clear()
        ops.pgemm4(x, w, epi, cfg=cfg, rms_eps=1e-5)
        assert calls == [want]
