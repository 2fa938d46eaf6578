"""The tiles between the others: a plan changes to one of them where it is cheaper, split if it was; tuned plans at their own row count stay."""
import pytest

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm


@pytest.mark.parametrize("M,N,K,plan,want", [
    (1536, 2048, 2048, (3, 1), (9, 1)), (2048, 3072, 1536, (2, 1), (11, 1)), (1300, 10240, 8192, (0, 1), (17, 1)), (160, 2048, 2048, (3, 1), (3, 1)),
    (2048, 2048, 2048, (3, 1), (3, 1)), (2048, 8192, 2048, (0, 1), (0, 1))])
def test_picks(M, N, K, plan, want):
    assert ops._pgemm_more(M, N, K, *plan) == want


@pytest.mark.parametrize("N,K", [(576, 2048), (2048, 192), (16384, 4096), (1024, 4096), (2048, 8192)])
def test_plans_run_and_keep_their_split(N, K, monkeypatch):
    monkeypatch.setattr(ops, "_PG_TABLE", {})
    for M in (129, 161, 192, 257, 448, 1000, 2048, 4097, 70000):
        kern, cfg, splits, _ = ops.pgemm_heuristic(M, N, K, ops.EPI_BF16, False)
        assert kern == "pgemm4" and ops.native().pgemm4_plan(M, N, K, ops.EPI_BF16, cfg, splits)[0] > 0
        assert (splits > 1) == (ops._pgemm_cheapest(-(-M // 64) * 64, N, K, 256)[2] > 1)


def test_tuned_plans_stay_at_their_row_count(monkeypatch):
    monkeypatch.setattr(ops, "_PG_TABLE", {(10240, 8192, 0, 0): [(1024, "pgemm4", 8, 1, 4, 137.0), (1536, "pgemm4", 0, 1, 8, 175.0)],
                                           (28672, 8192, 2, 0): [(1024, "pgemm4", 7, 1, 4, 689.0)], (8192, 512, 0, 0): [(1024, "pgemm", 0, 1, 4, 9.0)]})
    assert ops.gemm_route(1024, 10240, 8192, 0, False) == ("pgemm4", (8, 1, 4))
    assert ops.gemm_route(1300, 10240, 8192, 0, False) == ("pgemm4", (17, 1, 8))
    assert ops.gemm_route(850, 28672, 8192, 2, False) == ("pgemm4", (16, 1, 4))
    assert ops.gemm_route(4000, 28672, 8192, 2, False) == ("pgemm4", (7, 1, 4))      # past the largest: its plan
    assert ops.gemm_route(850, 8192, 512, 0, False) == ("pgemm", (0, 1, 4))


def test_plans_of_a_table_that_is_named_stand(monkeypatch):
    monkeypatch.setattr(ops, "_PG_TABLE", {(10240, 8192, 0, 0): [(1024, "pgemm4", 8, 1, 4, 137.0), (1536, "pgemm4", 0, 1, 8, 175.0)]})
    monkeypatch.setattr(ops, "PG_TABLE_NAMED", True)
    assert ops.gemm_route(1300, 10240, 8192, 0, False) == ("pgemm4", (0, 1, 8)) == ops.gemm_route(1536, 10240, 8192, 0, False)


@pytest.mark.parametrize("rows,E,N,K,pair,even,common,want", [
    (4602, 9, 2048, 2048, True, False, 1534, 15), (2800, 4, 2048, 2048, False, True, 0, 12), (8192, 4, 2048, 2048, False, True, 0, 4),
    (2800, 4, 512, 2048, False, True, 0, None), (249, 9, 2048, 2048, True, False, 83, None), (288, 9, 2048, 2048, True, False, 96, None),
    (291, 9, 2048, 2048, True, False, 97, 10), (243, 9, 4096, 3584, False, False, 81, 10), (288, 9, 4096, 3584, False, False, 96, 10),
    (243, 9, 2560, 2048, True, False, 81, 10), (288, 9, 2560, 2048, True, False, 96, 10), (396, 6, 2560, 2048, True, False, 132, 10)])
def test_grouped_picks(rows, E, N, K, pair, even, common, want):
    got = sm._grouped_plan(rows, E, N, K, pair, even, common)
    assert got == (want if want is not None else sm._grouped_tile(rows, E, N, K, pair, even, common))


def test_rules_of_grouped_products_take_every_tile_that_is_built():
    """... and no other: 128 x 96 (9) and 224 x 192 (14) are not."""
    assert set(sm._GROUP_MORE_COST) | set(sm._GROUP_FEW_TILE) | {4} == set(range(1, len(ops.pgemm4_configs()) + 4)) - {9, 14}
