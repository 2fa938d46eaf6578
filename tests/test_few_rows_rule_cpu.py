"""Which bf16 products of 17 - 128 rows go to the 4-wave tiles, without a GPU."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

from k8s_llm_scheduler_amd import ops

ROOT = Path(__file__).resolve().parents[1]


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


@pytest.mark.parametrize("M,rows,K,takes", [(33, 8192, 28672, False), (64, 8192, 28672, False), (65, 8192, 28672, True), (64, 8192, 14336, True),
                                            (64, 4096, 14336, True)])
def test_deep_products_with_a_tuned_plan_keep_it(M, rows, K, takes):
    """(4096 x 14336: as deep, not in the table)"""
    assert (ops._few_rows_tile(M, rows, K, ops.EPI_BF16) is not None) == takes


def test_a_plan_named_by_the_environment_is_taken():
    """K8S_MGEMM_OVERRIDE, at the rows of its bucket, as for any other product of mgemm's."""
    code = ("from k8s_llm_scheduler_amd import ops\n"
            "t = [ops._few_rows_tile(M, 10240, 8192, ops.EPI_BF16) is None for M in (48, 49, 64, 65)]\n"
            "s = [ops._few_rows_tile(M, 57344, 8192, ops.EPI_SWIGLU) is None for M in (33, 49, 128)]\n"
            "print(t == [False, True, True, False], s == [False, False, True], ops.mgemm_plan(64, 10240, 8192, 0, False))")
    env = {**os.environ, "K8S_MGEMM_OVERRIDE": "64,10240,8192,0,0=11:1; 128,28672,8192,2,0=12:1"}
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, cwd=ROOT)
    assert r.stdout.split("\n")[0] == "True True (11, 1)", r.stdout + r.stderr
