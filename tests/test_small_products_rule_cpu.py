"""Which bf16 products go to the tuned kernels: from 512 Ki weights on all, of half that size those of many rows or great depth."""
import pytest
import torch

from k8s_llm_scheduler_amd.ops import seqmix as sm


@pytest.mark.parametrize("M,N,K,fast", [
    (1, 1024, 512, True), (1, 512, 1008, False), (511, 2048, 128, False), (512, 2048, 128, True), (512, 2032, 128, False),
    (512, 512, 512, True), (511, 512, 512, False), (128, 256, 1024, False), (129, 256, 1024, True), (32, 128, 2048, False),
    (33, 128, 2048, True), (33, 112, 4096, False), (4096, 128, 1984, False), (33, 136, 2048, False), (512, 4096, 64, False)])
def test_rule(M, N, K, fast):
    a, w = torch.empty(M, K, dtype=torch.bfloat16), torch.empty(N, K, dtype=torch.bfloat16)
    assert sm._route_fast(a, w, torch.bfloat16) == fast and sm._route_fast(a, w, torch.float32) == fast
    assert not sm._route_fast(a.float(), w.float(), torch.float32)


@pytest.mark.parametrize("rows,N,pair,even,want", [(27, 2048, False, False, 6), (6, 2048, True, False, 6), (6, 2052, True, False, 5),
                                                   (27, 4100, False, False, 5), (28, 2048, False, False, 5), (27, 2048, False, True, 5)])
def test_grouped_tiles_of_few_rows(rows, N, pair, even, want):
    assert sm._grouped_tile(rows, 9, N, 2048, pair, even, rows // 3) == want
