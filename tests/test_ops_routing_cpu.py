"""GEMM routing without a GPU: the mgemm / pgemm plan tables' row buckets and nearest-bucket lookups, the auto policy
(hand-written kernels always; the library only as the K8S_GEMM=library oracle), and the GEMV row threshold."""

import json
import math
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from k8s_llm_scheduler_amd import ops
from k8s_llm_scheduler_amd.models.stream import StreamModel
from k8s_llm_scheduler_amd.ops import seqmix as sm

ROOT = Path(__file__).resolve().parent.parent


def test_row_buckets():
    assert [ops._mg_bucket(m) for m in (1, 2, 3, 4, 5, 8, 9, 16, 17, 1000, 1025, 2000, 5000, 8192)] == \
        [2, 2, 4, 4, 8, 8, 16, 16, 32, 1024, 2048, 2048, 8192, 8192]


def test_mgemm_table_lookup_stays_inside_the_tuned_range():
    table = ops._mg_load_table()
    assert table, "engine/assets/mgemm_gfx950.json is missing or empty"
    fp8_keys = [k for k in table if k[3] == 1]
    assert fp8_keys
    n, k, epi, _ = fp8_keys[0]
    top = max(r[0] for r in table[fp8_keys[0]])
    assert ops._mg_table_row(top, n, k, epi, True) is not None
    assert ops._mg_table_row(4 * top + 1, n, k, epi, True) is None


def test_mgemm_override_replaces_a_table_row(monkeypatch):
    monkeypatch.setenv("K8S_MGEMM_OVERRIDE", "64,10240,8192,0,0=11:1;64,8192,8192,0,0=12:2")
    monkeypatch.setattr(ops, "_MG_TABLE", None)
    try:
        assert ops._mg_table_row(64, 10240, 8192, ops.EPI_BF16, False)[1:3] == (11, 1)
        assert ops._mg_table_row(64, 8192, 8192, ops.EPI_BF16, False)[1:3] == (12, 2)
    finally:
        monkeypatch.delenv("K8S_MGEMM_OVERRIDE")
        ops._MG_TABLE = None   # the next lookup reloads the bundled table


LLAMA_TP1 = [(10240, 8192, ops.EPI_BF16), (8192, 8192, ops.EPI_BF16), (28672, 8192, ops.EPI_SWIGLU),
             (8192, 28672, ops.EPI_BF16)]


@pytest.mark.parametrize("backend", ["auto", "pgemm"])
@pytest.mark.parametrize("fp8", [False, True])
def test_auto_never_routes_to_the_library(monkeypatch, backend, fp8):
    monkeypatch.setattr(ops, "GEMM_BACKEND", backend)
    for M in (3, 8, 64, 128, 129, 245, 256, 1000, 2048, 8192, 20000):
        for N, K, epi in LLAMA_TP1:
            kern, plan = ops.gemm_route(M, N, K, epi, fp8)
            assert kern in ("mgemm", "pgemm", "pgemm4"), (M, N, K, kern)
            if fp8:
                assert kern != "pgemm4"           # the 4-wave kernel is bf16 only
            if backend == "auto" and M < ops.PG_MIN_M:
                assert kern == "mgemm"
            if kern.startswith("pgemm"):
                cfg, sp, gm = plan
                cfgs = ops.pgemm_configs() if kern == "pgemm" else ops.pgemm4_configs()
                assert 0 <= cfg < len(cfgs) and sp >= 1 and gm >= 1


def test_pgemm_table_picks_nearest_bucket_at_or_above(monkeypatch):
    monkeypatch.setattr(ops, "_PG_TABLE", {(100, 256, 0, 0): [(256, "pgemm4", 3, 2, 4, 10.0),
                                                               (2048, "pgemm", 0, 1, 8, 50.0)]})
    assert ops.pgemm_plan_for(200, 100, 256, 0, False) == (("pgemm4", 3, 2, 4), 10.0)
    assert ops.pgemm_plan_for(257, 100, 256, 0, False) == (("pgemm", 0, 1, 8), 50.0)
    assert ops.pgemm_plan_for(9000, 100, 256, 0, False) == (("pgemm", 0, 1, 8), None)   # past the top: its plan
    # fp8 has no 4-wave kernel: a bf16-only plan is not used for it
    monkeypatch.setattr(ops, "_PG_TABLE", {(100, 256, 0, 1): [(256, "pgemm4", 3, 2, 4, 10.0)]})
    assert ops.pgemm_plan_for(200, 100, 256, 0, True)[0][0] == "pgemm"


def test_untuned_shapes_take_a_plan_that_runs(monkeypatch):
    """Row counts around the tile heights and odd ones, weights of any aligned size: the cost rule's plan is one that the
    kernel's own planner accepts, and it depends on the row count rounded up to 64 only."""
    monkeypatch.setattr(ops, "_PG_TABLE", {})
    for M in (129, 191, 192, 257, 333, 1000, 2048, 4097, 70000):
        for N, K in ((16, 128), (100, 64), (576, 2048), (2048, 192), (16384, 4096), (128, 28672)):
            for epi in (ops.EPI_BF16, ops.EPI_F32):
                kern, cfg, sp, gm = ops.pgemm_heuristic(M, N, K, epi, False)
                assert kern in ("pgemm", "pgemm4") and sp <= max(1, K // 64 // 4)
                plan = ops.native().pgemm4_plan(M, N, K, epi, cfg, sp) if kern == "pgemm4" else \
                    ops.native().pgemm_plan(M, N, K, epi, 0, cfg, sp)
                assert plan[0] > 0
                assert ops.pgemm_heuristic(-(-M // 64) * 64, N, K, epi, False) == (kern, cfg, sp, gm)
    assert ops.pgemm_heuristic(2048, 2048, 2048, ops.EPI_BF16, True)[0] == "pgemm"
    assert ops.pgemm_heuristic(2048, 2048, 2048, ops.EPI_SWIGLU, False)[0] == "pgemm"


def test_auto_follows_the_tuned_winner(monkeypatch):
    monkeypatch.setattr(ops, "GEMM_BACKEND", "auto")
    monkeypatch.setattr(ops, "_PG_TABLE", {(1024, 1024, 0, 0): [(256, "mgemm", 0, 0, 0, 25.0),
                                                                 (512, "pgemm", 0, 2, 4, 30.0)]})
    assert ops.gemm_route(256, 1024, 1024, 0, False)[0] == "mgemm"
    assert ops.gemm_route(300, 1024, 1024, 0, False) == ("pgemm", (0, 2, 4))
    monkeypatch.setattr(ops, "GEMM_BACKEND", "pgemm")
    assert ops.gemm_route(256, 1024, 1024, 0, False)[0] == "pgemm"
    monkeypatch.setattr(ops, "GEMM_BACKEND", "library")
    assert ops.gemm_route(256, 1024, 1024, 0, False) == ("library", None)


def test_shipped_pgemm_table_is_consistent():
    if not __import__("os").path.isfile(ops.PG_TABLE_PATH):
        pytest.skip("no tuned pgemm table")
    with open(ops.PG_TABLE_PATH) as f:
        plans = json.load(f)["plans"]
    assert plans
    for key, v in plans.items():
        m, n, k, epi, fp8 = (int(t) for t in key.split(","))
        kern, cfg, sp, gm = v[:4]
        assert kern in ("mgemm", "pgemm", "pgemm4") and not (fp8 and kern == "pgemm4")
        assert ops.pgemm_plan_for(m, n, k, epi, bool(fp8))[0] == (kern, cfg, sp, gm)


def test_gemv_threshold_and_kernel_limit():
    assert 1 <= ops.GEMV_MAX_M <= ops.GEMV_KERNEL_MAX_M == 8


if __name__ == "__main__":
    pytest.main([__file__])


@pytest.mark.parametrize("backend", ["auto", "mgemm", "pgemm"])
def test_unroutable_shape_raises_instead_of_calling_the_library(monkeypatch, backend):
    """a shape no hand-written kernel accepts (N % 4 != 0 here) raises under every hand-written
    route -- linear and linear_swiglu never fall through to hipBLASLt / _scaled_mm silently."""
    import torch

    monkeypatch.setattr(ops, "GEMM_BACKEND", backend)
    monkeypatch.setattr(ops, "_gpu", lambda *a: True)           # route as on the GPU, compute nothing
    called = []
    monkeypatch.setattr(ops, "_lib_linear", lambda x, w: called.append("lib") or x @ w.t())
    x = torch.randn(300, 256, dtype=torch.bfloat16)
    w = torch.randn(130, 256, dtype=torch.bfloat16)              # N = 130: no 4-column output groups
    assert ops.gemm_route(300, 130, 256, ops.EPI_BF16, False)[0] == "library"
    with pytest.raises(ops.NoKernelForShape, match="K8S_GEMM=library"):
        ops.linear(x, w)
    with pytest.raises(ops.NoKernelForShape):
        ops.linear_swiglu(x, torch.randn(2 * 130, 256, dtype=torch.bfloat16))
    assert not called


def test_library_route_only_under_k8s_gemm_library(monkeypatch):
    import torch

    monkeypatch.setattr(ops, "GEMM_BACKEND", "library")
    monkeypatch.setattr(ops, "_gpu", lambda *a: True)
    called = []
    monkeypatch.setattr(ops, "_lib_linear", lambda x, w: called.append("lib") or (x.float() @ w.float().t()).to(x.dtype))
    y = ops.linear(torch.randn(300, 256, dtype=torch.bfloat16), torch.randn(128, 256, dtype=torch.bfloat16))
    assert called == ["lib"] and y.shape == (300, 128)


def _llama70b_decode_shapes(tp):
    hidden, inter, nq, nkv, d = 8192, 28672, 64, 8, 128
    return [((nq + 2 * nkv) * d // tp, hidden, ops.EPI_BF16), (hidden, nq * d // tp, ops.EPI_BF16),
            (inter // tp, hidden, ops.EPI_SWIGLU), (hidden, inter // tp, ops.EPI_BF16)]


@pytest.mark.parametrize("tp", [1, 2, 4, 8])
def test_every_batched_decode_shape_has_a_valid_tuned_plan(tp):
    """The 17-128-row bf16 plans (re-tuned in situ) and the MX plans (keys 3 / 4) cover every projection of a Llama-70B
    decode layer at TP = 1 / 2 / 4 / 8, and each tuned plan is valid for every row count of its bucket -- a shape that
    fell off the table would silently run the heuristic plan."""
    for i, (N, K, epi) in enumerate(_llama70b_decode_shapes(tp)):
        for M in (17, 24, 32, 33, 48, 64, 65, 100, 128):
            row = ops._mg_table_row(M, N, K, epi, False)
            assert row is not None, (tp, M, N, K, epi)
            assert ops.mgemm_valid(row[1], M, N, K, epi, 0, row[2]), (tp, M, N, K, epi, row)
            if K % 128 == 0:
                mx_out = i > 0   # O / down: the residual epilogue's MX copy; gate/up: MX SwiGLU output
                assert ops.mgemm_mx_plan(M, N, K, epi, True, mx_out) is not None, (tp, M, N, K, epi)


def test_mx_plans_are_tuned_for_every_tp_shard():
    """fp8 batched decode at TP = 1 / 2 / 4 / 8: every projection has TUNED MX plans (table keys 3 / 4) for 32-256 rows,
    not only a heuristic one."""
    table = ops._mg_load_table()
    for tp in (1, 2, 4, 8):
        for N, K, epi in _llama70b_decode_shapes(tp):
            key = (N, K, epi, 4 if epi == ops.EPI_SWIGLU else 3)
            assert sorted(r[0] for r in table.get(key, [])) == [32, 64, 128, 256], (tp, key)


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 97, 128])
def test_untuned_batched_decode_plans_run(M):
    """The one-round plans of 17 - 128 rows over sizes and k: valid, at most one round of small tiles, split k only with steps
    left; other k keep the general rule."""
    for N in (16, 100, 576, 1024, 2048, 3104, 4096, 8192, 16384, 32768, 151936):
        for K in (64, 128, 192, 256, 768, 1024, 1408, 2048, 3584, 4096, 8192, 14336):
            for epi in (ops.EPI_BF16, ops.EPI_F32):
                cfg, split = ops.mgemm_heuristic(M, N, K, epi, False)
                assert ops.mgemm_valid(cfg, M, N, K, epi, False, split), (M, N, K, cfg, split)
                one = ops._mgemm_one_round(M, N, K, epi, 256)
                assert (one is None) == (K % 256 != 0)
                if one is not None:
                    assert one == (cfg, split)
                    tiles = ops._mg_tiles(cfg, M, N, epi) * split
                    assert tiles <= 256 or cfg in (22, 31), (M, N, K, cfg, split)
                    assert split == 1 or K * 2 // ops.mgemm_configs()[cfg][5] // split >= 8


# ----------------------------------------------------------------------------- stream designs: routing without a GPU
class Recorder:
    """Stands for the extension: notes the entry points that a call reaches, answers every size question with yes."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def entry(*args):
            self.calls.append(name)
            return True

        return entry


@pytest.fixture
def recorder(monkeypatch):
    nat = Recorder()
    monkeypatch.setattr(sm, "_gpu", lambda *ts: True)
    monkeypatch.setattr(ops, "_gpu", lambda *ts: True)
    monkeypatch.setattr(ops, "native", lambda: nat)
    return nat


@pytest.mark.parametrize("M", [1, 8, 40, 200, 1024])
def test_products_refuse_operands_of_unequal_k(M, recorder):
    """Sizes of the tuned kernels, which take k from one operand: an error ahead of any launch, also for more inputs than
    weights."""
    a, w = torch.zeros(M, 1024, dtype=torch.bfloat16), torch.zeros(2048, 512, dtype=torch.bfloat16)
    for call in (lambda: sm.linear(a, w), lambda: sm.linear_act(a, w, sm.ACT_RELU2), lambda: sm.linear_act(a, w, sm.ACT_RELU),
                 lambda: sm.linear_each(a.expand(2, M, 1024), w.expand(2, 2048, 512)),
                 lambda: sm.linear_each(a.expand(3, M, 1024), torch.zeros(2, 2048, 1024, dtype=torch.bfloat16))):
        with pytest.raises(ValueError):
            call()
    assert recorder.calls == []


def test_grouped_products_on_big_tiles_take_what_the_kernel_reads(recorder, monkeypatch):
    """Row offsets of another length, type or layout, gathered rows that share memory or are strided in k: the route that goes
    by the tiles alone, or its refusal."""
    monkeypatch.setattr(ops, "LEAN", False)
    E, N, K, rows = 4, 256, 128, 300
    w, tiles = torch.zeros(E, 2 * N, K, dtype=torch.bfloat16), torch.zeros(9, 3, dtype=torch.int32)
    a = torch.zeros(rows, K, dtype=torch.bfloat16)

    class Seg(torch.Tensor):
        is_cuda = True

    seg = lambda n=E + 1, dt=torch.int32, step=1: torch.zeros(n * step, dtype=dt)[::step].as_subclass(Seg)

    def reached(a, seg, kind=None):
        recorder.calls.clear()
        try:
            if kind is None:
                sm.gemm(a, w, tiles=tiles, rows=rows, seg=seg)
            else:
                sm.gemm_act(a, w, kind, tiles=tiles, rows=rows, seg=seg)
        except ValueError:
            return "refused"
        return recorder.calls[0]

    for kind in (None, sm.ACT_RELU):
        assert reached(a, seg(), kind) == "pgemm4_grouped"
        for s in (None, seg(E), seg(E + 2), seg(dt=torch.int64), seg(step=2), torch.zeros(E + 1, dtype=torch.int32)):
            assert reached(a, s, kind) in ("gemm_any", "gemm_few_act")
        assert reached(a[:1].expand(rows, K), seg(), kind) in ("gemm_any", "gemm_few_act")       # one row for all: stride 0
        assert reached(a.T.contiguous().T, seg(), kind) == "refused"


def latent_calls(recorder, T, *, seqs=1, decode=False, dt=torch.bfloat16, q=None, cache=None, uv=None, blocks=64, H=4, keep=None):
    """Entry points that latent_mix reaches for a batch of T tokens of ``seqs`` sequences, sizes of the matrix-core kernels."""
    C, R, D, bs = 512, 64, 128, 16
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32)
    z = lambda *s: torch.zeros(*s, dtype=dt)
    b = {"positions": i32(T), "cu_q": i32(seqs + 1), "tok_seq": i32(T), "block_tables": i32(seqs, blocks),
         "max_qlen": 0 if decode else T, **(keep or {})}
    recorder.calls.clear()
    pick = lambda t, *s: z(*s) if t is None else t
    sm.latent_mix(pick(q, T, H * (D + R)), pick(cache, 2 * bs, C + R), z(H, C, D), pick(uv, H, D, C), z(2 * H * D, C), b, C, R, H,
                  D, D, 0, 0.1, bs)
    if keep is not None:
        keep.update(b)
    return [c for c in recorder.calls if c.startswith("latent") and not c.endswith("_ok")]


def test_latent_attention_on_plain_fmas_when_told_so(recorder, monkeypatch):
    for dt in (torch.bfloat16, torch.float32):
        assert latent_calls(recorder, 200, dt=dt) == ["latent_keys", "latent_prompt"]
        assert latent_calls(recorder, 2, seqs=2, decode=True, dt=dt) == [
            "latent_token" if dt == torch.bfloat16 else "latent_attention"]
        monkeypatch.setattr(sm, "LATENT_MFMA", False)
        assert latent_calls(recorder, 200, dt=dt) == ["latent_attention"]
        assert latent_calls(recorder, 2, seqs=2, decode=True, dt=dt) == ["latent_attention"]
        monkeypatch.setattr(sm, "LATENT_MFMA", True)


def test_latent_attention_of_unaligned_operands_is_absorbed(recorder):
    """Queries (both forms) or value weights (single tokens) that do not start at a whole vector: the kernels without that
    demand, as ever."""
    odd = lambda *s: torch.zeros(1 + math.prod(s), dtype=torch.bfloat16)[1:].view(*s)
    attend = ["latent_attention_mfma"]
    assert latent_calls(recorder, 200, q=odd(200, 4 * 192)) == attend
    assert latent_calls(recorder, 200, uv=odd(4, 128, 512)) == ["latent_keys", "latent_prompt"]      # (not read)
    assert latent_calls(recorder, 2, seqs=2, decode=True, q=odd(2, 4 * 192)) == attend
    assert latent_calls(recorder, 2, seqs=2, decode=True, uv=odd(4, 128, 512)) == attend


@pytest.mark.parametrize("T,decode", [(200, False), (2, True)])
def test_latent_attention_refuses_operands_of_other_sizes(recorder, T, decode):
    """Queries, cache rows and value weights of other sizes than the heads': an error ahead of the attention, on every route."""
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    for kw in ({"q": z(T, 4 * 128)}, {"cache": z(32, 512)}, {"uv": z(4, 64, 512)}, {"uv": z(3, 128, 512)}):
        with pytest.raises((ValueError, RuntimeError)):
            latent_calls(recorder, T, seqs=1 if not decode else T, decode=decode, **kw)
        assert not [c for c in recorder.calls if c in ("latent_prompt", "latent_token", "latent_attention_mfma")], kw


def test_latent_attention_without_room_for_keys_and_values(recorder, monkeypatch):
    """The written-out keys and values are bounded by LATENT_EXPAND_BYTES; where the device has no room for them the batch
    runs absorbed, and its other layers do not ask again."""
    attend = ["latent_attention_mfma"]
    bs, per_row = 16, 4 * 256 * 2
    assert latent_calls(recorder, 200, blocks=sm.LATENT_EXPAND_BYTES // per_row // bs) == ["latent_keys", "latent_prompt"]
    assert latent_calls(recorder, 200, blocks=sm.LATENT_EXPAND_BYTES // per_row // bs + 1) == attend
    gemm, asked = sm.gemm, []

    def full(a, w, *args, rows=None, **kw):
        if rows is None:
            return gemm(a, w, *args, **kw)
        asked.append(rows)
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(sm, "gemm", full)
    batch = {}
    assert latent_calls(recorder, 200, keep=batch) == ["latent_keys"] + attend
    assert latent_calls(recorder, 200, keep=batch) == attend
    assert asked == [64 * bs]


@pytest.mark.parametrize("env,want", [
    ({}, [0, 0, 32, 32, 64, 32]), ({"K8S_WKV_CHUNK": "0"}, [0] * 6), ({"K8S_WKV_CHUNK": "48"}, [0, 0, 48, 48, 48, 48]),
    ({"K8S_WKV_CHUNK_MIN": "0"}, [32, 32, 32, 32, 64, 32]), ({"K8S_WKV_CHUNK_MIN": "300"}, [0, 0, 0, 0, 64, 32]),
    ({"K8S_WKV_CHUNK": "16", "K8S_WKV_CHUNK_MIN": "1"}, [16] * 6)])
def test_recurrence_chunks_follow_their_switches(env, want):
    """(tokens, sequences, heads): decoding, below and at 32 tokens a sequence, from 256 tokens on, chunks that fill the CUs,
    a batch of many rows.  0 in K8S_WKV_CHUNK turns the chunks off, in K8S_WKV_CHUNK_MIN always on."""
    code = ("from k8s_llm_scheduler_amd.ops import seqmix as sm\n"
            "print([sm.wkv_chunk(*a) for a in ((8, 8, 32), (63, 2, 32), (64, 2, 4), (255, 3, 2), (2048, 1, 32), (300, 300, 1))])")
    clean = {k: v for k, v in os.environ.items() if not k.startswith("K8S_WKV")}
    out = subprocess.run([sys.executable, "-c", code], env={**clean, **env}, cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert out.stdout.strip() == str(want), out.stderr


@pytest.mark.parametrize("dt", [torch.int32, torch.int64])
def test_decode_steps_take_block_tables_of_both_integer_types(recorder, dt):
    """A design without attention reads its block table for the step's slots alone; layers that attend get it as it came."""
    class Model(StreamModel):
        block_size = 16

        def __init__(self):
            pass

        def _check_ready(self):
            pass

        def _forward(self, ids, b, rows):
            return b

    tables = torch.zeros(3, 4, dtype=dt)
    b = Model().forward_decode(torch.zeros(3, dtype=torch.int32), torch.ones(3, dtype=torch.int64), tables, 64)
    assert recorder.calls == ["decode_meta"] and b["block_tables"].dtype == dt


def test_plans_are_worked_out_once_and_in_bounded_time(monkeypatch):
    """Plans stand on every product's way to the device: a shape's second call looks its plan up, and the expected tiles of
    large groups are not summed term by term (the same number: the terms left out are 0 or 1 to 1e-9)."""
    valid, calls = ops.mgemm_valid, []
    monkeypatch.setattr(ops, "mgemm_valid", lambda *a: calls.append(a) or valid(*a))
    first = ops.mgemm_heuristic(71, 3104, 2048, ops.EPI_BF16, False)
    asked = len(calls)
    assert ops.mgemm_heuristic(71, 3104, 2048, ops.EPI_BF16, False) == first and len(calls) == asked
    erf, terms = math.erf, []
    monkeypatch.setattr(sm.math, "erf", lambda x: terms.append(x) or erf(x))
    for rows, E, N, K, pair in ((131072, 1, 4096, 512, False), (131072, 2, 2048, 2048, True), (3068, 8, 2048, 2048, True),
                                (194, 8, 2048, 2048, False), (90000, 8, 128, 64, False)):
        r = rows / E
        terms.clear()
        got = sm._grouped_tile.__wrapped__(rows, E, N, K, pair)
        assert len(terms) <= sum(2 + 12.0 * r ** 0.5 / bq for _, bq in sm._GROUP_TILE.values())
        cost = {}
        for cfg, (bp, bq) in sm._GROUP_TILE.items():
            start, tile, per_round, step, wmb, omb, act = sm._GROUP_COST[cfg]
            more = sum(0.5 + 0.5 * erf((r - bq * k) / (2.0 * r) ** 0.5) for k in range(1, int((r + 6.0 * r ** 0.5) / bq) + 2))
            tiles, spare = (E + E * more, 0.02) if E > 1 else (-(-rows // bq), 0.0)
            per, kt = (2 if pair else 1) * N, K / 64
            rounds = max(1, math.ceil(tiles * -(-per // bp) / 256 - spare))
            cost[cfg] = start + rounds * (tile * kt + per_round + (act * bp * bq / 65536 if pair else 0.0)) + step * kt + \
                2e-6 * (wmb * E * per * K + omb * rows * N)
        assert got == min(cost, key=cost.get)


@pytest.mark.parametrize("rows,E,N,K,pair,want", [(600, 8, 2048, 2048, True, 3), (1700, 8, 2048, 2048, False, 3), (1700, 16, 2048, 4096, True, 1),
                                                  (160, 8, 2048, 2048, False, 6)])
def test_grouped_products_take_the_cheapest_tile_of_all(rows, E, N, K, pair, want):
    """Where one tile was left out of the choice, or a few expected tiles past a whole round priced the better one out of it."""
    assert sm._grouped_tile(rows, E, N, K, pair) == want
