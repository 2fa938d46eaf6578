"""The 4-wave big-tile products at one to five 64-deep stages, with rows stored through LDS (N a multiple of 8, aligned) and piece
by piece: whole numbers, so every sum and every bf16 result is exact."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
TILES = {0: (256, 256), 1: (256, 128), 2: (128, 256), 3: (128, 128), 4: (256, 256), 5: (128, 64), 6: (64, 64)}


def whole(n, K, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randint(-3, 4, (n, K), generator=g) * (torch.rand(n, K, generator=g) < 0.2)).to(torch.bfloat16).cuda()


def out_of(M, N, shift=0):
    buf = torch.full((M * N + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    return buf, buf[shift:shift + M * N].view(M, N)


def untouched(buf, M, N, shift=0):
    return bool((buf[:shift] == 7).all() and (buf[shift + M * N:] == 7).all())


@pytest.mark.parametrize("cfg", range(7))
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320])
def test_stages_and_row_stores(cfg, K):
    bp, bq = TILES[cfg]
    for M, N, shift in ((1, 8, 0), (bq - 1, bp + 4, 0), (bq + 3, bp - 8, 0), (2 * bq, 2 * bp + 24, 0), (bq + 1, bp + 16, 4)):
        x, w = whole(M, K, M + K), whole(N, K, N)
        want = x.float() @ w.float().T
        assert want.abs().max() <= 256                    # exact in bf16
        buf, out = out_of(M, N, shift)
        ops.native().pgemm4(out.data_ptr(), 0, x.data_ptr(), w.data_ptr(), M, N, K, ops.EPI_BF16, cfg, 1, 4, 0, 0, 0.0, -1)
        assert torch.equal(out.float(), want) and untouched(buf, M, N, shift), (M, N, shift)
        assert torch.equal(ops.pgemm4(x, w, ops.EPI_F32, cfg=cfg), want), (M, N)
        if K >= 128:
            assert torch.equal(ops.pgemm4(x, w, ops.EPI_BF16, cfg=cfg, splits=2).float(), want), (M, N, "split")


@pytest.mark.parametrize("cfg", range(7))
@pytest.mark.parametrize("K", [64, 192])
def test_activations_and_rms(cfg, K):
    bp, bq = TILES[cfg]
    for M, N, shift in ((bq - 1, bp // 2 + 8, 0), (bq + 5, bp // 2 - 4, 0), (17, bp + 8, 4)):
        x, w = whole(M, K, M), whole(2 * N, K, N + 1)
        y = x.float() @ w.float().T
        buf, out = out_of(M, N, shift)                    # relu(g) u: exact up to the last rounding
        ops.native().pgemm4_act(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, cfg, 4, sm.ACT_RELU, 0.0, 1.0, 0, -1)
        assert torch.equal(out, (y[:, :N].clamp(min=0) * y[:, N:]).to(torch.bfloat16)) and untouched(buf, M, N, shift), (M, N)
        buf, out = out_of(M, 2 * N, shift)
        ops.native().pgemm4_act(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, 2 * N, K, cfg, 4, sm.ACT_RELU2, 0.0, 1.0, 0, -1)
        assert torch.equal(out, y.clamp(min=0).square().to(torch.bfloat16)) and untouched(buf, M, 2 * N, shift), (M, N)
        x += 1                                            # rows of a root mean square that is not zero
        y = (x.double() @ w.double().T) * (x.double().square().mean(1, keepdim=True) + 1e-5).rsqrt()
        got = ops.pgemm4(x, w, ops.EPI_BF16, cfg=cfg, rms_eps=1e-5).double()
        # the scale's relative error (a square root and a division, 4 units) and the result's rounding
        assert ((got - y).abs() <= y.abs() * (2.0**-8 + 2.0**-21) + 1e-30).all(), (M, N)
        got = ops.pgemm4(x, w, ops.EPI_SWIGLU, cfg=cfg, rms_eps=1e-5).double()
        ref = torch.nn.functional.silu(y[:, :N]) * y[:, N:]
        # silu on the hardware's exponential: (|g| + 4) units of 2^-24 of its value
        assert ((got - ref).abs() <= ref.abs() * (2.0**-8 + (y[:, :N].abs() + 16) * 2.0**-23) + 1e-30).all(), (M, N)


@pytest.mark.parametrize("cfg", range(7))
def test_grouped(cfg):
    counts, N, K = [130, 0, 1, 257], 264, 192
    seg = torch.tensor([0] + counts).cumsum(0).int().cuda()
    rows = sum(counts)
    x, w = whole(40, K + 8, 5), whole(4 * N, K, 6).view(4, N, K)
    pick = torch.randint(0, 40, (rows,), generator=torch.Generator().manual_seed(1)).int().cuda()
    buf, out = out_of(rows, N)
    ops.native().pgemm4_grouped(out.data_ptr(), x.data_ptr(), w.data_ptr(), 40, rows, N, K, 4, seg.data_ptr(), pick.data_ptr(),
                                K + 8, cfg, 4, -1, 0.0, 1.0, -1)
    e = torch.repeat_interleave(torch.arange(4), torch.tensor(counts)).cuda()
    want = torch.bmm(x[pick.long(), :K].float().unsqueeze(1), w.float()[e].transpose(1, 2).contiguous())[:, 0]
    assert torch.equal(out.float(), want) and untouched(buf, rows, N)
