"""Products of 256 - 512 Ki weights on the tuned kernels against 64 bits, at both ends of their range of rows and behind tanh."""
import pytest
import torch

from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [33, 129, 200, 512, 777, 2048])
@pytest.mark.parametrize("N,K", [(2048, 128), (1024, 256), (512, 512), (256, 1024), (128, 2048), (144, 2048), (128, 3584)])
def test_against_64_bits(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    z, mass = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    sums = 2.0 * K * 2.0 ** -24 * mass + 1e-30                                  # fp32, in any order
    assert ((sm.linear(a, w, torch.float32).double() - z).abs() <= sums).all()
    assert ((sm.linear(a, w).double() - z).abs() <= sums + 2.0 ** -8 * z.abs()).all()
    # an activation takes the sums as they are wherever its product has few tiles (others may round them first)
    twice = 0.0 if -(-M // 64) * -(-N // 64) <= 128 else 2.0 ** -8 * z.abs()
    for kind, t, slope in ((sm.ACT_TANH, z.tanh(), 1.0), (sm.ACT_SILU, z * z.sigmoid(), 1.1), (sm.ACT_RELU2, z.clamp(min=0).square(), 2 * z.abs())):
        assert ((sm.linear_act(a, w, kind).double() - t).abs() <= slope * (sums + twice) + 2.0 ** -8 * t.abs() + 1e-6).all(), kind
