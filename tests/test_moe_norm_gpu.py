"""The experts' combine inside the norm that follows it: the same bits as the two kernels, whatever the width, the type, the shared
expert's place and gate; sizes that its kernel does not take fall back on the two."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda"


def inputs(T, W, top, dt, joint, seed=0):
    g = torch.Generator().manual_seed(seed + T + W + top)
    r = lambda *s, d=dt: torch.randn(*s, generator=g).to(d).to(DEV)
    cols = top + joint
    D, pos = r(cols * T, W), torch.randperm(cols * T, generator=g).to(torch.int32).to(DEV)
    return r(T, W, d=torch.float32), D, pos, r(W), r(W), r(W), r(T, W), r(T, 1, d=torch.float32)


@pytest.fixture
def entries(monkeypatch):
    nat, seen = ops.native(), []

    class Spy:
        def __getattr__(self, name):
            seen.append(name)
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Spy)
    return seen


@pytest.mark.parametrize("W", [4, 100, 1024, 1028, 2048, 2052, 4096, 8192])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,top", [(1, 1), (5, 2), (37, 3)])
def test_same_bits_as_combine_and_norm(W, dt, T, top, entries):
    for where in ("none", "beside", "beside ungated", "joint", "joint ungated"):
        x, D, pos, w, nw, dw, shared, gate = inputs(T, W, top, dt, where.startswith("joint"))
        b = sm.MoeBranch(D, pos, top, 1.0 / top, shared if where.startswith("beside") else None,
                         None if where == "none" or "ungated" in where else gate, T)
        z = b.combined()
        for kw in (dict(), dict(out_dtype=dt), dict(out_dtype=dt, next_w=nw, gain=0.5), dict(out_dtype=dt, next_w=nw, dot_w=dw)):
            x1, x2 = x.clone(), x.clone()
            want = sm.branchnorm(x1, z, w, 1e-5, **kw)
            entries.clear()
            got = sm.branchnorm(x2, b, w, 1e-5, **kw)
            assert entries == ["branchnorm_moe"] and torch.equal(x1, x2), (where, kw)
            for a, c in zip(want if isinstance(want, tuple) else (want,), got if isinstance(got, tuple) else (got,)):
                assert a is c is None or torch.equal(a, c), (where, kw)


@pytest.mark.parametrize("W", [6, 8196])
def test_widths_that_the_kernel_does_not_take(W, entries):
    x, D, pos, w, nw, _, shared, gate = inputs(5, W, 2, torch.bfloat16, 1)
    b = sm.MoeBranch(D, pos, 2, 0.5, None, gate, 5)
    x1 = x.clone()
    want = sm.branchnorm(x1, b.combined(), w, 1e-5, out_dtype=torch.bfloat16, next_w=nw)
    entries.clear()
    got = sm.branchnorm(x, b, w, 1e-5, out_dtype=torch.bfloat16, next_w=nw)
    assert entries == ["branchnorm_moe", "moe_combine", "branchnorm"] and torch.equal(got, want) and torch.equal(x, x1)


@pytest.mark.parametrize("joint", [0, 1])
def test_chosen_tokens(joint):
    x, D, pos, w, _, _, shared, gate = inputs(9, 64, 2, torch.bfloat16, joint)
    b, rows = sm.MoeBranch(D, pos, 2, 0.5, None if joint else shared, gate, 9), torch.tensor([8, 0, 3], device=DEV)
    assert torch.equal(b.select(rows).combined(), b.combined().index_select(0, rows))
    x1, x2 = x.index_select(0, rows), x.clone()
    got = sm.branchnorm(x1, b.select(rows), w, 1e-5, out_dtype=torch.bfloat16)
    assert torch.equal(got, sm.branchnorm(x2, b, w, 1e-5, out_dtype=torch.bfloat16).index_select(0, rows))
