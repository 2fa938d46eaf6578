"""Which kernel and which plan a product takes, without a GPU: the launches are noted instead of made, every size question goes
to the extension."""
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.ops import seqmix as sm

BF16 = torch.bfloat16
ROOT = Path(__file__).resolve().parent.parent


class Launches:
    """The extension, its launches noted as (name, arguments)."""

    LAUNCH = ("gemv_act", "sgemv_act", "mgemm_act", "gemv", "gemv_w", "sgemv", "mgemm", "pgemm", "pgemm4", "pgemm4_act",
              "pgemm4_grouped", "gemm_any", "gemm_few_act", "act")

    def __init__(self, real):
        self.real, self.made = real, []

    def __getattr__(self, name):
        if name not in self.LAUNCH:
            return getattr(self.real, name)
        return lambda *args: self.made.append((name, args)) or 0

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


@pytest.mark.parametrize("N,K", [(64, 2048), (576, 2048), (2048, 2048), (8192, 2048), (4096, 4096), (1024, 8192), (4096, 14336)])
def test_fp32_products_of_few_rows_keep_the_tiles_that_fill_the_chip(N, K):
    """Up to 32 rows in one round of 32 x 32 tiles: those, but for up to 4 rows of very narrow weights and 17 - 24 of narrow ones,
    where k is shared by the waves; with more rows or rounds one of the wider tiles."""
    rule = ops.native().gemm_f32_rule
    for M in (5, 8, 16, 25, 32):
        assert rule(M, N, K, 1, 0) == 0, M
    for M in (1, 2, 4):
        assert rule(M, N, K, 1, 0) == (17 if N <= 256 else 0), M
    for M in (17, 24):
        assert rule(M, N, K, 1, 0) == (17 if N <= 2048 else 0), M
    assert rule(33, N, K, 1, 0) > 0
    for M in (1, 16, 32):
        assert rule(M, 16384, 2048, 1, 0) > 0 and rule(M, 2048, 2048, 8, 0) > 0, M


@pytest.mark.parametrize("M,N,K", [(350, 4096, 4096), (512, 4096, 4096), (384, 4096, 14336), (512, 4096, 14336), (80, 6144, 3072), (300, 6144, 4096),
                                   (190, 7168, 4096), (128, 14336, 4096), (24, 28672, 4096), (64, 28672, 4096), (48, 32768, 4096)])
def test_fp32_products_of_shared_k_keep_it(M, N, K):
    """Whether k is shared decides the error (2.15e-7 against 2.29e-7 at K = 4096, 2.3e-7 against 2.8e-7 at 14336): by one fit alone."""
    assert ops.native().gemm_f32_rule(M, N, K, 1, 0) > 16


@pytest.mark.parametrize("M,N,K,fq", [(401, 6144, 4096, 2), (352, 7168, 4096, 2), (320, 14336, 4096, 2), (160, 28672, 4096, 2), (441, 3072, 1536, 3),
                                      (457, 6720, 4096, 8), (393, 14336, 4096, 5), (333, 16384, 2048, 7), (333, 3072, 2048, 1)])
def test_fp32_tiles_of_columns_by_their_rounds(M, N, K, fq):
    assert ops.native().gemm_f32_rule(M, N, K, 1, 0) == fq


def test_fp32_products_of_other_depths_are_not_asked():
    rule = ops.native().gemm_f32_rule
    assert [rule(333, 2048, K, 1, 0) for K in (480, 500, 2056)] == [0, 0, 0]


@pytest.mark.parametrize("E,N,K", [(8, 2048, 2048), (8, 4096, 2048), (8, 7168, 4096), (16, 1024, 2048)])
def test_fp32_products_of_listed_tiles_go_by_the_groups_rows(E, N, K):
    """The list holds a tile a group more than the rows fill: groups of fewer than 32 rows keep the 32 x 32 tiles, as products do that
    64-row tiles would not spread over the chip; the rest takes tiles of 32 rows, or of 64 where there are many."""
    rule = ops.native().gemm_f32_rule
    listed = lambda rows: (rows + 63) // 64 + E
    for per in (1, 4, 16, 24, 31):
        assert rule(per * E, N, K, 1, listed(per * E)) == 0, per
    for per in (40, 63):
        assert rule(per * E, N, K, 1, listed(per * E)) == 2, per
    assert rule(500 * E, N, K, 1, listed(500 * E)) == 4 and rule(96 * E, 1024, K, 1, listed(96 * E)) in (0, 2)
    assert rule(40 * E, 64, K, 1, listed(40 * E)) == 0 and rule(40 * 4, 2048, K, 1, 3 + 4) == 0
    assert rule(500 * E, N, 480, 1, listed(500 * E)) == 0


def test_key_splits_of_single_tokens():
    """No splits where two tiles a wave cost less than the merge, nor where they would only add a round of workgroups; long contexts
    of 65 - 512 tokens x key heads are split where that fills a round."""
    s = sm.token_splits
    assert [s(T, 4, 1024, 128) for T in (1, 8, 16, 31, 32, 64, 65, 80, 128, 200)] == [4, 4, 4, 2, 1, 1, 1, 1, 1, 1]
    assert [s(T, 4, 4096, 128) for T in (1, 4, 16, 40, 48, 56, 64, 80, 128)] == [16, 16, 4, 3, 4, 1, 1, 3, 1]
    assert [s(T, 4, 4096, 64) for T in (40, 48, 64, 128)] == [3, 2, 2, 1]
    assert [s(T, 4, 4096, 96) for T in (64, 80, 96)] == [1, 2, 2] and [s(T, 4, 1024, 96) for T in (64, 80, 112)] == [1, 2, 1]
    for D in (64, 96, 128):
        assert all(1 <= s(T, G, keys, D) <= 16 for T in (1, 7, 33, 65, 300, 5000) for G in (1, 4, 8) for keys in (0, 1, 31, 2049, 8192))
        assert s(300, 8, 40, D) == 1 and s(160, 4, 4096, D) == 1
        assert [s(T, 4, 8192, D, False) for T in (8, 32, 40, 97, 400)] == [8, 2, 1, 1, 1]      # how many keys there are is not known


def test_key_splits_of_prompts():
    """Windows keep to 256 workgroups; where more than 2048 keys may be visible, 65 - 170 workgroups are split up to the 512 that run
    at once."""
    s = sm.prompt_splits
    assert [s(g, 1040) for g in (1, 28, 52, 76, 128, 129, 512)] == [6, 6, 4, 3, 2, 1, 1]
    assert [s(g, 8192) for g in (28, 52, 64, 65, 76, 100, 128, 152, 170, 171, 256, 512)] == [6, 4, 4, 6, 6, 5, 4, 3, 3, 1, 1, 1]
    assert s(76, 100) == 1 and s(3, 300) == 3


@pytest.mark.parametrize("M,N,K,kind", [(200, 1040, 1024, sm.ACT_RELU), (129, 1040, 1024, sm.ACT_RELU2), (333, 2048, 2048, sm.ACT_GELU_TANH),
                                        (160, 1024, 4096, sm.ACT_GELU_TANH), (200, 1536, 4096, sm.ACT_RELU2)])
def test_activations_join_every_unsplit_product_of_big_tiles(M, N, K, kind, launches):
    """However few its tiles; products whose k is split get the activation as a launch of its own."""
    kern, plan = ops.gemm_route(M, N, K, ops.EPI_BF16, False)
    assert kern == "pgemm4"
    sm.linear_act(torch.zeros(M, K, dtype=BF16), torch.zeros(N, K, dtype=BF16), kind)
    assert launches.names() == (["pgemm4_act"] if plan[1] == 1 else ["pgemm4", "act"]) and (plan[1] > 1) == (K == 4096)


@pytest.mark.parametrize("M,N,K,joins", [(192, 14336, 4096, True), (130, 16384, 4096, True), (900, 5120, 5120, True), (256, 7168, 4096, True),
                                         (333, 6720, 4096, True), (384, 5120, 5120, False), (448, 2048, 8192, False)])
def test_activations_keep_split_products_from_rounding_ahead_of_them(M, N, K, joins, launches):
    """A product whose split plan is a little cheaper takes the unsplit one with its activation, one rounding; the product alone does not."""
    assert ops.gemm_route(M, N, K, ops.EPI_BF16, False)[1][1] > 1
    sm.linear_act(torch.zeros(M, K, dtype=BF16), torch.zeros(N, K, dtype=BF16), sm.ACT_GELU_TANH)
    assert launches.names() == (["pgemm4_act"] if joins else ["pgemm4", "act"])


def test_activations_follow_the_switches_of_the_gemv(launches, monkeypatch):
    """K8S_GEMV_MAX_M moves 3 - 8 rows to the GEMV, whose form with an activation takes two: then the product and the activation."""
    for rows, kind in ((4096, sm.ACT_GELU_TANH), (2048, sm.ACT_RELU2)):
        w = torch.zeros(rows, 2048, dtype=BF16)
        for limit, M, want in ((2, 1, "gemv_act"), (2, 3, "sgemv_act"), (8, 2, "gemv_act"), (8, 3, "act"), (8, 8, "act"), (8, 9, "sgemv_act"),
                               (1, 1, "gemv_act")):
            monkeypatch.setattr(ops, "GEMV_MAX_M", limit)
            launches.made.clear()
            sm.linear_act(torch.zeros(M, 2048, dtype=BF16), w, kind)
            assert launches.names()[-1] == want and len(launches.made) == (2 if want == "act" else 1), (limit, M)
            assert want != "act" or launches.names()[0].startswith("gemv")


@pytest.mark.parametrize("env,want", [
    ({}, [(1, 342, 3), (1, 512, 2), (1, 3584, 1), (1, 1024, 1)]), ({"K8S_GEMV_LOOP": "0"}, [(1, 1026, 1), (1, 1024, 1), (1, 3584, 1), (1, 1024, 1)]),
    ({"K8S_GEMV_LOOP": "1"}, [(1, 206, 5), (1, 256, 4), (1, 256, 14), (1, 256, 4)]), ({"K8S_GEMV_LOOP": "3"}, [(1, 513, 2), (1, 512, 2), (1, 717, 5), (1, 512, 2)]),
    ({"K8S_GEMV_LOOP_SWIGLU_MAX": "1000"}, [(1, 1026, 1), (1, 1024, 1), (1, 3584, 1), (1, 1024, 1)]), ({"K8S_GEMV_KW": "2"}, [None] * 4),
    ({"K8S_GEMV_RPW1": "2"}, [(1, 257, 2), (1, 512, 1), (1, 448, 4), (1, 1024, 1)])])
def test_launches_with_an_activation_follow_the_gemv_switches(env, want):
    """(k splits, workgroups, row sets a wave) of 2 x 4104 x 1024, 2 x 4096 x 2048, 2 x 14336 x 4096 and, elementwise, 8192 x 2048."""
    code = ("from k8s_llm_scheduler_amd import ops\n"
            "print([ops.native().gemv_act_plan(1, n, k, p) for n, k, p in ((4104, 1024, 1), (4096, 2048, 1), (14336, 4096, 1), (8192, 2048, 0))])")
    clean = {k: v for k, v in os.environ.items() if not k.startswith("K8S_GEMV")}
    out = subprocess.run([sys.executable, "-c", code], env={**clean, **env}, cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert out.stdout.strip() == str(want), out.stderr


@pytest.mark.parametrize("G,N,K,any_to,grouped_from", [(4, 2048, 2048, 32, 33), (2, 2048, 2048, 64, 65), (4, 512, 2048, 128, 129), (4, 1024, 4096, 64, 65),
                                                       (4, 4096, 4096, 0, 16), (8, 2048, 2048, 0, 1), (3, 6144, 2048, 0, 16)])
def test_products_of_several_inputs_share_a_launch_where_that_is_faster(G, N, K, any_to, grouped_from, launches):
    """Up to which rows the any-shape kernel takes them, from which the grouped big tiles do; else one launch each."""
    w = torch.zeros(G, N, K, dtype=BF16)
    for M in (1, 8, 15, 16, 32, 33, 64, 65, 128, 129, 512, 2048, 2049):
        launches.made.clear()
        sm.linear_each(torch.zeros(G, M, K, dtype=BF16), w)
        want = ["gemm_any"] if M <= any_to else ["pgemm4_grouped"] if grouped_from <= M <= 2048 else None
        assert launches.names() == want if want else len(launches.made) >= G, M
