"""Which kernel and which plan a product takes, without a GPU: the launches are noted instead of made, every size question goes
to the extension."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

BF16 = torch.bfloat16


class Launches:
    """The extension, its launches noted as (name, arguments)."""

    LAUNCH = ("gemv_act", "sgemv_act", "mgemm_act", "gemv", "gemv_w", "sgemv", "mgemm", "pgemm", "pgemm4", "pgemm4_act",
              "pgemm4_grouped", "gemm_any", "gemm_few_act", "act")

    def __init__(self, real):
        self.real, self.made = real, []

    def __getattr__(self, name):
        if name not in self.LAUNCH:
            return getattr(self.real, name)
        return lambda *args: self.made.append((name, args))

    def names(self):
        return [n for n, _ in self.made]


@pytest.fixture
def launches(monkeypatch):
    nat = Launches(ops.native())
    monkeypatch.setattr(sm, "_gpu", lambda *ts: True)
    monkeypatch.setattr(ops, "_gpu", lambda *ts: True)
    monkeypatch.setattr(ops, "native", lambda: nat)
    monkeypatch.setattr(ops, "_chk", lambda t, *a: t.data_ptr())
    monkeypatch.setattr(sm, "_p", lambda t, *a: 0 if t is None else t.data_ptr())
    monkeypatch.setattr(ops, "_zeroed_scratch", lambda *a: 0)
    return nat


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("rows,K", [(16384, 2048), (28672, 4096), (4096, 2048), (2080, 1024), (4096, 14336), (272, 4096)])
def test_gated_products_of_17_to_128_rows_take_the_plan_of_their_weight_rows(M, rows, K, launches):
    """Gate and up share a tile, so [gate; up] is tiled and split as the plain product of the same weight rows is (up to
    the configurations that have no pairs of fragments): the activation in the epilogue costs no slower product."""
    a, w = torch.zeros(M, K, dtype=BF16), torch.zeros(rows, K, dtype=BF16)
    sm.linear_act(a, w, sm.ACT_GELU_TANH)
    (name, args), = launches.made
    cfg, nwg = args[8], args[9]
    plain, split = ops.mgemm_plan(M, rows, K, ops.EPI_BF16, False)
    assert name == "mgemm_act"
    if ops.mgemm_configs()[plain][4]:      # gate / up pairs
        assert (cfg, nwg) == (plain, ops.mgemm_nwg(plain, M, rows, K, ops.EPI_BF16, False, split))
    assert nwg <= 256 or ops.mgemm_configs()[cfg][1] >= 64       # small tiles only where one round holds them
