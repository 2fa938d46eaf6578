"""Which bf16 products of 17 - 128 rows go to the 4-wave tiles, without a GPU."""
import pytest

from k8s_llm_scheduler_amd import ops


@pytest.mark.parametrize("M,rows,K,takes", [(17, 16384, 2048, True), (32, 14336, 4096, True), (17, 8192, 8192, False), (33, 8192, 8192, True),
                                            (64, 8192, 2048, True), (64, 4096, 2048, False), (65, 1280, 8192, True), (128, 4096, 2048, False),
                                            (128, 8192, 28672, True), (16, 57344, 8192, False), (129, 57344, 8192, False),
                                            (64, 8192, 2080, False), (64, 8196, 8192, False)])
def test_products_of_few_rows_by_their_weights(M, rows, K, takes):
    assert (ops._few_rows_tile(M, rows, K, ops.EPI_BF16) is not None) == takes


def test_plans_of_few_rows_run():
    """The kernel's own planner accepts every pick, splits included; SwiGLU only from 33 rows on."""
    for M in (17, 32, 33, 48, 64, 65, 97, 128):
        for rows, K in ((16384, 2048), (57344, 8192), (8192, 28672), (10240, 8192), (12296, 4096), (32768, 1024), (1280, 64 * 128)):
            for epi in (ops.EPI_BF16, ops.EPI_F32, ops.EPI_SWIGLU):
                pick = ops._few_rows_tile(M, rows, K, epi)
                if pick is None:
                    continue
                assert epi != ops.EPI_SWIGLU or M > 32
                cfg, splits = pick
                n = rows // 2 if epi == ops.EPI_SWIGLU else rows
                assert ops.native().pgemm4_plan(M, n, K, epi, cfg, splits)[0] > 0
