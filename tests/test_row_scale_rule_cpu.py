"""Which normed big-tile products take their rows' 1 / rms from a pass ahead, without a GPU: long ones whose rows that pass can read in
whole vectors; the others, as they always did, from the product's own prologue."""
import pytest
import torch

from k8s_llm_scheduler_amd import ops


@pytest.mark.parametrize("offset,flops,epi,cfg,want", [(0, 0.0, ops.EPI_BF16, 0, "pgemm4_scaled"), (8, 0.0, ops.EPI_SWIGLU, 1, "pgemm4_scaled"),
                                                       (4, 0.0, ops.EPI_BF16, 0, "pgemm4"), (1, 0.0, ops.EPI_SWIGLU, 0, "pgemm4"),
                                                       (0, 1e12, ops.EPI_BF16, 0, "pgemm4"), (0, 0.0, ops.EPI_F32, 0, "pgemm4")])
def test_rule(offset, flops, epi, cfg, want, monkeypatch):
    called = []

    class Native:
        pgemm4_plan = staticmethod(lambda *a: (1, 0))
        pgemm4_scaled_ok = staticmethod(lambda cfg: True)

        def __getattr__(self, name):
            return lambda *a: called.append(name)

    M, N, K = 6, 64, 128
    store = torch.empty(M * K + 16, dtype=torch.bfloat16)
    first = (-store.data_ptr() // 2) % 8 + offset          # elements to a 16-byte boundary, and past it
    x, w = store[first:first + M * K].view(M, K), torch.empty(N, K, dtype=torch.bfloat16)
    monkeypatch.setattr(ops, "native", Native)
    monkeypatch.setattr(ops, "P4_SCALE_FLOPS", flops)
    ops.pgemm4(x, w, epi, cfg=cfg, rms_eps=1e-5)
    assert called == [want]
