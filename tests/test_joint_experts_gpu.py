"""A shared expert as the last group of the experts' products: its own limit in every kernel that can run them, and a layer against
the two products apart."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.models import favizen
from k8s_llm_scheduler_amd.ops import seqmix as sm

DEV = "cuda"


def glu64(z, limit):
    g, u = z.chunk(2, -1)
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("T,path", [(1, "few"), (5, "few"), (6, "big"), (97, "big"), (300, "big"), (6, "plain"), (97, "plain")])
@pytest.mark.parametrize("limits", [(1.5, 0.5), (0.0, 0.7), (0.6, 0.0), (1.0, 1.0)])
@pytest.mark.parametrize("E,top", [(8, 2), (3, 1)])
def test_limit_of_the_last_group(T, path, limits, E, top, monkeypatch):
    """One rounding in the epilogues; the sums rounded ahead of the activation too where it is a launch of its own."""
    W, F = 256, 128 + 8
    g = torch.Generator().manual_seed(T + E)
    h = torch.randn(T, W, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(E + 1, 2 * F, W, generator=g) * 2 / W ** 0.5).to(torch.bfloat16).to(DEV)
    idx = torch.cat([torch.rand(T, E, generator=g).argsort(1)[:, :top], torch.full((T, 1), E)], 1).to(torch.int32).to(DEV)
    tok, pos, seg, tiles = sm.moe_align(idx, E + 1)
    if path == "plain":
        monkeypatch.setattr(sm, "_grouped_big", lambda *a: False)
        monkeypatch.setattr(sm, "_few_fits", lambda *a: False)
    elif path == "few":
        monkeypatch.setattr(sm, "_grouped_big", lambda *a: False)
    names = []
    nat = ops.native()

    class Spy:
        def __getattr__(self, name):
            names.append(name)
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Spy)
    got = sm.gemm_act(h, w, sm.ACT_SWISH_CLAMP, limits[0], 1.702, a_rows=tok, tiles=tiles, rows=T * (top + 1), seg=seg, common=T,
                      common_limit=limits[1])
    if path != "plain":
        assert names == ["pgemm4_grouped" if path == "big" else "gemm_few_act"]
    slack = 2.0 ** -8 if path != "plain" else 2.0 ** -6
    got = got.double()[pos.long()].view(T, top + 1, F)
    for c in range(top + 1):
        z = (h.double().unsqueeze(1) @ w.double()[idx[:, c].long()].transpose(1, 2)).squeeze(1)
        want = glu64(z, limits[1] if c == top else limits[0])
        assert ((got[:, c] - want).abs() <= slack * want.abs() + (1e-4 if slack < 2.0 ** -7 else 4e-2)).all(), c


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 5])
@pytest.mark.parametrize("limits", [(1.0, 1.0), (0.0, 0.7)])
def test_large_weights_of_few_tokens(T, limits, monkeypatch):
    """More than 4 Mi values an expert and fewer rows than the big tiles take: one launch, the sums not rounded ahead of the activation."""
    W, F, E, top = 1536, 1408, 8, 2
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, W, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(E + 1, 2 * F, W, generator=g) * 2 / W ** 0.5).to(torch.bfloat16).to(DEV)
    idx = torch.cat([torch.rand(T, E, generator=g).argsort(1)[:, :top], torch.full((T, 1), E)], 1).to(torch.int32).to(DEV)
    tok, pos, seg, tiles = sm.moe_align(idx, E + 1)
    names, nat = [], ops.native()

    class Spy:
        def __getattr__(self, name):
            names.append(name)
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Spy)
    got = sm.gemm_act(h, w, sm.ACT_SWISH_CLAMP, limits[0], 1.702, a_rows=tok, tiles=tiles, rows=T * (top + 1), seg=seg, common=T,
                      common_limit=limits[1])
    assert names == ["gemm_few_act"]
    got = got.double()[pos.long()].view(T, top + 1, F)
    for c in range(top + 1):
        z = torch.stack([h[t].double() @ w[int(idx[t, c])].double().T for t in range(T)])
        want = glu64(z, limits[1] if c == top else limits[0])
        assert ((got[:, c] - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all(), c


def model(dev, dtype, shared_ff, tokens=None):
    cfg = favizen.preset("favizen", 128, 96, ("attention", "shared"), heads=4, kv_heads=2, dim=32, window=16, rot_dims=16, side_heads=4,
                         side_kv_heads=2, side_dim=32, chunk=16, ff=64, experts=5, top=2, expert_ff=128, shared_ff=shared_ff,
                         mlps=("moe",))
    t = favizen.random_tensors(cfg, 3, dev)
    return cfg, t, favizen.FavizenModel(cfg, device=dev, dtype=dtype, tensors=t, max_model_len=64)


def test_stacks_hold_every_weight_once():
    """Of one size in bf16: one stack, counted once; of another, or in fp32: apart."""
    for dtype, ff, joint in ((torch.bfloat16, 128, True), (torch.bfloat16, 64, False), (torch.float32, 128, False)):
        cfg, t, m = model("cpu", dtype, ff)
        e = 2 if dtype == torch.bfloat16 else 4
        for L in m.layers:
            f = L.mlp
            assert (f.joint is not None) == joint and f.route[0] == ((6, 3) if joint else (5, 2))
            if joint:
                assert f.experts.w_gu.data_ptr() == f.joint.w_gu.data_ptr()
                assert f.shared.w_down.data_ptr() == f.joint.w_down.data_ptr() + e * 5 * f.shared.w_down.numel()
        p = "l0.mlp."
        assert torch.equal(m.layers[0].mlp.shared.w_down, t[p + "shared.down"].to(dtype))
        assert torch.equal(m.layers[0].mlp.experts.w_gu[4, 128:], t[p + "e4.up"].to(dtype))
        moe = sum(v.numel() for k, v in t.items() if ".mlp." in k and "table" not in k and not k.endswith(".sg"))
        own = {x.data_ptr(): x.numel() for L in m.layers for g in (L.mlp.experts, L.mlp.shared) for x in (g.w_gu, g.w_down)}
        assert sum(own.values()) == moe and m.weight_bytes() >= e * moe


@pytest.mark.parametrize("dev", ["cpu", pytest.param(DEV, marks=pytest.mark.gpu)])
@pytest.mark.parametrize("T", [1, 7, 40])
def test_layer_with_the_shared_expert_joined_and_apart(T, dev):
    """The same layer by one product of six experts and by five and one: sums of another order, a rounding of each output."""
    _, _, m = model(dev, torch.bfloat16, 128)
    L = m.layers[0].mlp
    ids = torch.randint(0, 96, (T,), generator=torch.Generator().manual_seed(T)).to(torch.int32).to(dev)
    h = torch.randn(T, 128, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).to(dev)
    sg = torch.randn(T, 1, generator=torch.Generator().manual_seed(T)).to(dev)
    table = m._tables[(6, 3)]
    joined = m._moe(L, h, sg, {"routes": {(6, 3): sm.moe_table_align(ids, table, 6)}}).combined().double()
    apart = type(L)(L.cfg, L.experts, L.shared, L.sg, ((5, 2), 0))
    two = table[:, :, :2].contiguous()
    want = m._moe(apart, h, sg, {"routes": {(5, 2): sm.moe_table_align(ids, two, 5)}}).combined().double()
    assert ((joined - want).norm() / want.norm()) < 2.0 ** -7
