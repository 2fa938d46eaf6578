"""Products of 1 - 128 rows with the activation in the epilogue, against 64 bits and beside the product and the activation as two
launches: every kernel's row edges, k slices, widths that leave a remainder."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda"


def act64(z, kind, limit, alpha):
    if kind == sm.ACT_RELU2:
        return z.clamp(min=0.0) ** 2
    g, u = z.chunk(2, dim=-1)
    if kind == sm.ACT_GELU_TANH:
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    if kind == sm.ACT_RELU:
        return g.clamp(min=0.0) * u
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(alpha * g) * (u + 1.0)


@pytest.mark.parametrize("M", [1, 2, 3, 8, 9, 16, 17, 32, 33, 64, 65, 127, 128])
@pytest.mark.parametrize("N,K", [(136, 4096), (1032, 576), (512, 8192), (4104, 1024), (2048, 14336)])
@pytest.mark.parametrize("kind", [sm.ACT_GELU_TANH, sm.ACT_SWISH_CLAMP, sm.ACT_RELU, sm.ACT_RELU2])
def test_activation_in_the_epilogue(M, N, K, kind, monkeypatch):
    pair = kind != sm.ACT_RELU2
    rows = 2 * N if pair else -(-N // 16) * 16
    g = torch.Generator(device=DEV).manual_seed(M * 7 + N + K + kind)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(rows, K, generator=g, device=DEV) * 2 / K ** 0.5).to(torch.bfloat16)
    want = act64(x.double() @ w.double().T, kind, 1.5, 1.702)
    got = sm.linear_act(x, w, kind, 1.5, 1.702)
    two = sm.act(sm.linear(x, w), kind, 1.5, 1.702)          # a rounding of the product ahead of it
    fused = ops.linear_act_rows(x, w, pair, kind, 1.5, 1.702)
    if fused is None:       # 3 - 16 rows of a depth that is no multiple of 128: two launches
        assert 3 <= M <= 16 and K % 128 and torch.equal(got, two)
    else:                   # one rounding to bf16, and the fp32 sums' and the sigmoid's error
        assert torch.equal(got, fused) and got.shape == want.shape
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()
        assert (got.double() - want).norm() <= (two.double() - want).norm() * 1.01
    monkeypatch.setattr(ops, "GEMM_BACKEND", "mgemm")        # a forced kernel family keeps its own two launches
    assert ops.linear_act_rows(x, w, pair, kind, 1.5, 1.702) is None


def test_replays_equal_the_eager_result():
    x = torch.randn(5, 4096, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * 1024, 4096, device=DEV) / 64).to(torch.bfloat16)
    xs = [x[:m].contiguous() for m in (1, 5)] + [torch.randn(40, 4096, device=DEV).to(torch.bfloat16)]
    run = lambda: [sm.linear_act(t, w, sm.ACT_SWISH_CLAMP, 7.0, 1.702) for t in xs]  # noqa: E731
    want = run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(4):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        again = run()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(again, want))


@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("kind", [sm.ACT_SWISH_CLAMP, sm.ACT_RELU2])
def test_row_sets_in_a_loop(M, kind):
    """One or two rows with the GEMV's row-set loop off and at 1 - 3 workgroups a CU, row sets that do not divide among the waves."""
    pair, N, K = kind != sm.ACT_RELU2, 4104 if kind != sm.ACT_RELU2 else 8224, 1024
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * N if pair else N, K, generator=g, device=DEV) * 2 / K ** 0.5).to(torch.bfloat16)
    want = act64(x.double() @ w.double().T, kind, 1.5, 1.702)
    before = ops.native().gemv_set_loop(-2)
    try:
        for loop in (0, 1, 2, 3):
            ops.native().gemv_set_loop(loop)
            got = ops.linear_act_rows(x, w, pair, kind, 1.5, 1.702)
            assert ops.native().gemv_act_plan(M, N, K, pair)[2] == (1 if loop == 0 else -(-(1026 if pair else 1028) // (256 * loop)))
            assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all(), loop
    finally:
        ops.native().gemv_set_loop(before)
