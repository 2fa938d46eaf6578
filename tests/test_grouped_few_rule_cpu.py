"""Which grouped products take the tiles of 32 tokens: uneven groups of few rows and 2 - 16 Mi weights each."""
import pytest

from k8s_llm_scheduler_amd.ops import seqmix as sm


@pytest.mark.parametrize("rows,E,N,K,pair,even,common,few", [
    (96, 9, 2048, 2048, True, False, 32, True), (1, 9, 2048, 2048, False, False, 0, True), (241, 9, 2048, 2048, False, False, 80, False),
    (240, 9, 2048, 2048, False, False, 80, True), (96, 9, 1023, 2048, False, False, 32, False), (96, 9, 1024, 2048, False, False, 32, True),
    (96, 9, 4096, 4096, False, False, 32, True), (96, 9, 4096, 4096, True, False, 32, False), (96, 8, 2048, 2048, False, True, 0, False),
    (64, 1, 2048, 2048, False, False, 0, False), (64, 2, 2048, 2048, False, False, 64, False)])
def test_rule(rows, E, N, K, pair, even, common, few):
    got = sm._grouped_plan(rows, E, N, K, pair, even, common)
    if few:
        assert got in sm._GROUP_FEW_TILE and got == sm._grouped_few(rows, E - (common > 0), N, K, pair, common)
    else:
        assert got == sm._grouped_tile(rows, E, N, K, pair, even, common)
