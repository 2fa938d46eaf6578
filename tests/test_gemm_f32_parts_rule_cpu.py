"""Which fp32 products run on the bf16 matrix cores (gemm_f32_parts.hip): by sizes alone, over the forms that the rule is asked about."""
import pytest

from k8s_llm_scheduler_amd import ops

MENU = {0, 111, 112, 121, 122, 222, 223, 224, 225, 226, 423, 424, 425, 426, 427, 826, 827, 828}


def test_tiles_are_of_the_menu():
    rule = ops.native().gemm_f32_parts_rule
    for K in (512, 1536, 2048, 14336):
        for N in (1, 65, 576, 2048, 16384, 32769):
            assert {rule(M, N, K, G, 0) for M in (1, 16, 17, 47, 64, 333, 2048, 9000) for G in (1, 3, 32)} <= MENU, (N, K)


def test_other_depths_are_not_asked():
    rule = ops.native().gemm_f32_parts_rule
    assert [rule(333, 2048, K, 1, 0) for K in (0, 32, 480, 500, 2056)] == [0] * 5
    assert rule(0, 2048, 2048, 1, 0) == rule(333, 0, 2048, 1, 0) == rule(333, 2048, 2048, 0, 0) == 0


@pytest.mark.parametrize("M,N,K", [(333, 16384, 2048), (333, 2048, 8192), (333, 3072, 2048), (512, 4096, 14336), (8, 2048, 2048), (1, 2048, 8192),
                                   (150, 8192, 2048), (64, 16384, 2048)])
def test_large_products_and_few_rows_of_deep_weights_take_it(M, N, K):
    assert ops.native().gemm_f32_parts_rule(M, N, K, 1, 0) > 0


@pytest.mark.parametrize("M,N,K", [(48, 3072, 2048), (40, 4096, 14336), (96, 2048, 8192), (24, 1024, 512), (3, 32768, 2048), (128, 576, 2048)])
def test_where_the_fp32_pipes_are_as_fast_they_stay(M, N, K):
    assert ops.native().gemm_f32_parts_rule(M, N, K, 1, 0) == 0


@pytest.mark.parametrize("E,N,K", [(8, 2048, 2048), (8, 4096, 2048), (8, 7168, 4096), (16, 1024, 2048)])
def test_listed_tiles_go_by_the_groups_rows(E, N, K):
    rule = ops.native().gemm_f32_parts_rule
    listed = lambda rows: (rows + 63) // 64 + E
    assert [rule(per * E, N, K, 1, listed(per * E)) for per in (1, 8, 24, 31)] == [0] * 4
    assert all(rule(per * E, N, K, 1, listed(per * E)) in (222, 224, 424) for per in (32, 48, 64, 130, 500))
    assert rule(64 * E, N, 512, 1, listed(64 * E)) == 0 and rule(64 * E, 256, K, 1, listed(64 * E)) == 0
