"""Ops of models with an fp32 residual stream, recurrent / windowed- or latent-attention mixers and mixtures of experts.

Same dispatch rule as the rest of :mod:`..ops`: CUDA (= HIP) tensors always run the gfx950 kernels
(``stream32.hip``, ``mixers.hip``, ``latent_prompt.hip``,
``latent_token.hip``, ``window_attn.hip``, ``gated_scan.hip``, ``decay_scan.hip``, ``delta_scan.hip``, ``moe.hip``) and raise when the extension is missing; CPU tensors run the fp32
reference in :mod:`.reference` (the CPU test-suite).  Every op takes bf16 or true-fp32 activations / weights (the
``f32`` flag of the kernels); what a design computes in fp32 regardless (residual sum, recurrent state, decays, router,
attention scores) is fp32 in both.
"""

from __future__ import annotations

import functools
import math
import os
import sys
from typing import NamedTuple, Optional

import torch

from . import reference as ref
from .reference import ACT_GELU_ERF, ACT_GELU_TANH, ACT_RELU, ACT_RELU2, ACT_SILU, ACT_SOFTCAP, ACT_SWISH_CLAMP  # noqa: F401
from .reference import ACT_TANH  # noqa: F401
from .reference import CONV_NONE, CONV_SILU  # noqa: F401
from .reference import GATE_SIGMOID, GATE_SILU  # noqa: F401
from .reference import SCAN_DECAY, SCAN_HGRN2, SCAN_MLSTM, SCAN_SSD  # noqa: F401

BF16, F32, I32 = torch.bfloat16, torch.float32, torch.int32
GROUP_BM = 64   # row-tile height of the grouped GEMM (gemm_any_kernel's BM)


# Short prompts are bound by their launches' preparation here: an import statement in a function costs about 1 us of every
# call (97 tokens, 118 launches: 1475 us of preparation with them, 1396 us).
_ops = sys.modules[__package__]


def _native():
    return _ops.native()


def _gpu(*ts) -> bool:
    cuda = None
    for t in ts:
        if t is not None and t.is_cuda is not cuda:
            if cuda is not None:
                raise ValueError("mixed CPU/GPU tensors")
            cuda = t.is_cuda
    return bool(cuda)


def _p(t: Optional[torch.Tensor], dtype=None, name: str = "tensor") -> int:
    if t is None:
        return 0
    if dtype is not None and t.dtype != dtype:
        raise TypeError(f"{name}: expected {dtype}, got {t.dtype}")
    if not t.is_contiguous():
        raise ValueError(f"{name}: must be contiguous")
    return t.data_ptr()


def _f32(dtype) -> int:
    if dtype == F32:
        return 1
    if dtype == BF16:
        return 0
    raise TypeError(f"activations must be bfloat16 or float32, got {dtype}")


# ----------------------------------------------------------------------------- residual stream
def embed_rows(ids: torch.Tensor, table: torch.Tensor, scale: float = 1.0, copy: bool = False):
    """fp32 [T, W] rows of ``table`` (bf16 or fp32) times ``scale``; ``copy``: (rows, the same in the table's type)."""
    if not _gpu(ids, table):
        x = ref.embed_rows(ids, table, scale)
        return (x, x.to(table.dtype, copy=True)) if copy else x
    T, W = ids.shape[0], table.shape[1]
    out = torch.empty(T, W, dtype=F32, device=table.device)
    same = torch.empty(T, W, dtype=table.dtype, device=table.device) if copy else None
    _native().embed_rows(out.data_ptr(), _p(same), _p(ids, I32, "ids"), _p(table), T, W, table.shape[0], float(scale),
                         _f32(table.dtype), -1)
    return (out, same) if copy else out


def _step_meta(context_lens: torch.Tensor, block_tables: torch.Tensor):
    B = context_lens.shape[0]
    if block_tables.dim() != 2 or block_tables.shape[0] < B:
        raise ValueError("decode_meta: a row of the block table for every context length")
    n = (B + 4) // 4 * 4
    meta = torch.empty(3, n, dtype=I32, device=context_lens.device)      # rows 16 bytes aligned
    return meta[0, :B], meta[1, :B], meta[2, :B + 1]


def decode_meta(context_lens: torch.Tensor, block_tables: torch.Tensor, block_size: int):
    """Of a step of single tokens, row i = state slot i with ``context_lens[i]`` tokens (0: idle): int32 (positions,
    cache slots (-1: idle), 0 .. B)."""
    if not _gpu(context_lens, block_tables):
        return ref.decode_meta(context_lens, block_tables, block_size)
    pos, slots, ar = _step_meta(context_lens, block_tables)
    _native().decode_meta(pos.data_ptr(), slots.data_ptr(), ar.data_ptr(), _p(context_lens, I32, "context_lens"),
                          _p(block_tables, I32, "block_tables"), block_tables.shape[1], context_lens.shape[0], int(block_size), -1)
    return pos, slots, ar


def embed_step(ids: torch.Tensor, table: torch.Tensor, context_lens: torch.Tensor, block_tables: torch.Tensor, block_size: int,
               scale: float = 1.0, copy: bool = False):
    """(:func:`embed_rows`, :func:`decode_meta`) of a step of single tokens in one launch."""
    B, W = ids.shape[0], table.shape[1]
    if B == 0 or context_lens.shape[0] != B or not _gpu(ids, table, context_lens, block_tables):
        return embed_rows(ids, table, scale, copy), decode_meta(context_lens, block_tables, block_size)
    pos, slots, ar = _step_meta(context_lens, block_tables)
    out = torch.empty(B, W, dtype=F32, device=table.device)
    same = torch.empty(B, W, dtype=table.dtype, device=table.device) if copy else None
    _native().embed_step(out.data_ptr(), _p(same), _p(ids, I32, "ids"), _p(table), W, table.shape[0], float(scale), _f32(table.dtype),
                         pos.data_ptr(), slots.data_ptr(), ar.data_ptr(), _p(context_lens, I32, "context_lens"),
                         _p(block_tables, I32, "block_tables"), block_tables.shape[1], B, int(block_size), -1)
    return ((out, same) if copy else out), (pos, slots, ar)


def resnorm(x: torch.Tensor, w: Optional[torch.Tensor], eps: float, *, branch: Optional[torch.Tensor] = None,
            mult: float = 1.0, rowvec: Optional[torch.Tensor] = None, offset: float = 0.0,
            out_dtype=BF16, groups: int = 1, branch2: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``x`` (fp32 [T, W], updated in place) += mult * (branch + branch2) + rowvec (two sublayers that read one norm
    leave two branches); returns rms-norm(x) * (offset + w) in
    ``out_dtype``, or None when ``w`` is None (add only).  ``groups`` > 1: every one of that many equal consecutive
    parts of a row is divided by its own root mean square."""
    if x.dtype != F32:
        raise TypeError("the residual stream is fp32")
    T, W = x.shape
    if groups < 1 or W % groups:
        raise ValueError(f"resnorm: {groups} groups do not divide the width {W}")
    if branch is None and branch2 is not None:
        branch, branch2 = branch2, None
    if not _gpu(x, w, branch, rowvec, branch2):
        return ref.resnorm(x, branch, mult, rowvec, w, offset, eps, out_dtype, groups, branch2)
    out = torch.empty(T, W, dtype=out_dtype, device=x.device) if w is not None else None
    f32 = _f32(out_dtype)
    for t, n in ((branch, "branch"), (branch2, "branch2"), (rowvec, "rowvec"), (w, "w")):
        if t is not None and t.dtype != out_dtype:
            raise TypeError(f"{n}: expected {out_dtype}, got {t.dtype}")
    _native().resnorm(_p(x), _p(branch), _p(branch2), float(mult), _p(rowvec), _p(w), float(offset), float(eps),
                      _p(out), T, W, int(groups), f32, -1)
    return out


def norm_mix(a: torch.Tensor, wa: torch.Tensor, b: Optional[torch.Tensor], wb: Optional[torch.Tensor], eps: float,
             ca: float = 1.0, cb: float = 1.0, out_dtype=None, groups: int = 1, gate: Optional[torch.Tensor] = None,
             gate_kind: int = GATE_SIGMOID) -> torch.Tensor:
    """ca * rms-norm(a) * wa + cb * rms-norm(b) * wb over rows [T, W] (norms in fp32; ``b`` None: the first term
    only): the outputs of two mixers that run side by side, each normed, joined.  ``a`` may be a column slice of a
    wider tensor (row stride free).  ``groups`` > 1 (``a`` alone): every one of that many equal consecutive parts of a
    row is divided by its own root mean square.  ``gate`` [T, W] of the output type (row stride free): the result times
    sigmoid(gate) or silu(gate), element by element."""
    out_dtype = out_dtype or a.dtype
    T, W = a.shape
    if gate is not None and (gate.shape != a.shape or gate.dtype != out_dtype or gate.stride(1) != 1):
        raise ValueError("norm_mix: the gate must be [T, W] of the output type with contiguous rows")
    if groups < 1 or W % groups or (groups > 1 and b is not None):
        raise ValueError(f"norm_mix: {groups} groups must divide the width {W} and go with one input")
    if not _gpu(a, wa, b, wb, gate):
        return ref.norm_mix(a, wa, b, wb, eps, ca, cb, out_dtype, groups, gate, gate_kind)
    if a.stride(1) != 1:
        raise ValueError("norm_mix: rows must be contiguous")
    if b is not None and (b.shape != a.shape or b.dtype != a.dtype or wb is None):
        raise ValueError("norm_mix: the two inputs must agree in shape and dtype")
    out = torch.empty(T, W, dtype=out_dtype, device=a.device)
    _native().norm_mix(out.data_ptr(), a.data_ptr(), a.stride(0), _p(wa, a.dtype, "wa"), _p(b), _p(wb, a.dtype, "wb"),
                       float(eps), float(ca), float(cb), T, W, int(groups), gate.data_ptr() if gate is not None else 0,
                       gate.stride(0) if gate is not None else 0, int(gate_kind), _f32(a.dtype), _f32(out_dtype), -1)
    return out


def branchnorm(x: torch.Tensor, branch: Optional[torch.Tensor], w: Optional[torch.Tensor], eps: float, *,
               out_dtype=None, bias: Optional[torch.Tensor] = None, next_w: Optional[torch.Tensor] = None,
               gain: float = 1.0, dot_w: Optional[torch.Tensor] = None):
    """Norm of the sublayer's output only: ``x`` (fp32 [T, W], updated in place) += rms-norm(branch + ``bias``) * w.
    ``branch`` is of w's type, or fp32 (None, with ``next_w``: nothing is added), or a :class:`MoeBranch`.  With ``out_dtype`` (the weights' type)
    the new rows are also returned in that type, for a sublayer that reads the stream itself -- or, with ``next_w``, their
    norm rms-norm(x) * next_w * gain, for a sublayer that is normed on both sides.  ``dot_w`` [W] (with ``next_w``):
    returns (rows, the normed rows' products with it, fp32 [T, 1])."""
    if x.dtype != F32 or not x.is_contiguous():
        raise TypeError("the residual stream is contiguous fp32")
    if isinstance(branch, MoeBranch):
        if bias is None and w is not None and _gpu(x, branch.D, w, next_w) and branch.joins(x, w, out_dtype, next_w, dot_w):
            T, W = x.shape
            out = torch.empty(T, W, dtype=out_dtype, device=x.device) if out_dtype is not None else None
            dot = torch.empty(T, 1, dtype=F32, device=x.device) if dot_w is not None else None
            if _native().branchnorm_moe(_p(x), branch.D.data_ptr(), _p(branch.pos, I32), branch.pos.numel() // max(T, 1), branch.top,
                                        float(branch.scale), _p(branch.shared), _p(branch.gate), _p(w), _p(next_w), float(gain),
                                        _p(dot_w), _p(dot), float(eps), _p(out), T, W, _f32(w.dtype), -1):
                return (out, dot) if dot_w is not None else out
        branch = branch.combined()
    wt = (w if w is not None else next_w).dtype
    if branch is not None and (branch.shape != x.shape or branch.dtype not in (wt, F32) or w is None):
        raise TypeError("branchnorm: branch [T, W] of the weight's type or fp32, w [W]")
    if branch is None and (next_w is None or bias is not None):
        raise TypeError("branchnorm: without a branch only the norm that follows is left")
    for t, n in ((w, "w"), (bias, "bias"), (next_w, "next_w"), (dot_w, "dot_w")):
        if t is not None and (t.numel() != x.shape[1] or t.dtype != wt):
            raise TypeError(f"branchnorm: {n} is [W] of the weights' type")
    if out_dtype is not None and out_dtype != wt:
        raise TypeError("branchnorm: the returned rows take the weight's type")
    if next_w is not None and out_dtype is None or dot_w is not None and next_w is None:
        raise TypeError("branchnorm: next_w needs out_dtype, dot_w needs next_w")
    if not _gpu(x, branch, w, next_w):
        return ref.branchnorm(x, branch, w, eps, out_dtype, bias, next_w, gain, dot_w)
    T, W = x.shape
    out = torch.empty(T, W, dtype=out_dtype, device=x.device) if out_dtype is not None else None
    dot = torch.empty(T, 1, dtype=F32, device=x.device) if dot_w is not None else None
    _native().branchnorm(_p(x), _p(branch), _p(w), _p(bias), _p(next_w), float(gain), _p(dot_w), _p(dot), float(eps), _p(out),
                         T, W, int(branch is None or branch.dtype == F32), _f32(wt), -1)
    return (out, dot) if dot_w is not None else out


def postnorm(x: torch.Tensor, branch: Optional[torch.Tensor], alpha: float, gain: float, eps: float, *,
             branch2: Optional[torch.Tensor] = None, c1: float = 1.0, c2: float = 1.0,
             out_dtype=None) -> Optional[torch.Tensor]:
    """Norm after the sum: ``x`` (fp32 [T, W], updated in place) <- rms-norm(alpha x + c1 branch + c2 branch2) * gain
    with one ``gain`` for the whole row, so the stream itself stays normed.  With ``out_dtype`` the new rows are also
    returned in that type (the input of the sublayer that reads them next)."""
    if x.dtype != F32 or not x.is_contiguous():
        raise TypeError("the residual stream is contiguous fp32")
    if branch is None and branch2 is not None:
        branch, branch2, c1, c2 = branch2, None, c2, c1
    if not _gpu(x, branch, branch2):
        return ref.postnorm(x, branch, branch2, alpha, c1, c2, gain, eps, out_dtype)
    T, W = x.shape
    bt = branch.dtype if branch is not None else out_dtype
    for t, n in ((branch, "branch"), (branch2, "branch2")):
        if t is not None and (t.dtype != bt or t.shape != x.shape):
            raise TypeError(f"postnorm: {n} must be [T, W] of one activation type")
    if out_dtype is not None and bt is not None and out_dtype != bt:
        raise TypeError("postnorm: the returned rows take the branches' type")
    out = torch.empty(T, W, dtype=out_dtype, device=x.device) if out_dtype is not None else None
    _native().postnorm(_p(x), _p(branch), _p(branch2), float(alpha), float(c1), float(c2), float(gain), float(eps),
                       _p(out), T, W, _f32(bt or F32), -1)
    return out


def gate_mul(y: torch.Tensor, gate: torch.Tensor, kind: int = GATE_SIGMOID) -> torch.Tensor:
    """y * sigmoid(gate) (GATE_SIGMOID) or y * silu(gate) (GATE_SILU), element by element; ``y`` [T, F] (the gate's
    type, or fp32) and ``gate`` [T, F] may be column slices of wider tensors.  Returns [T, F] of the gate's type."""
    if y.shape != gate.shape or y.dim() != 2:
        raise ValueError("gate_mul: y and gate must be [T, F]")
    if not _gpu(y, gate):
        return ref.gate_mul(y, gate, kind)
    if y.stride(1) != 1 or gate.stride(1) != 1 or y.dtype not in (gate.dtype, F32):
        raise ValueError("gate_mul: rows must be contiguous; y is of the gate's type or fp32")
    T, F = y.shape
    out = torch.empty(T, F, dtype=gate.dtype, device=y.device)
    _native().gate_mul(out.data_ptr(), y.data_ptr(), y.stride(0), gate.data_ptr(), gate.stride(0), T, F, int(kind),
                       int(y.dtype == F32), _f32(gate.dtype), -1)
    return out


def act(x: torch.Tensor, kind: int, limit: float = 0.0, alpha: float = 1.0, *,
        row_scale: Optional[torch.Tensor] = None, row_map: Optional[torch.Tensor] = None,
        bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Gated kinds (ACT_GELU_TANH, ACT_SWISH_CLAMP, ACT_RELU = relu(g) u): [T, 2F] = [gate | up] -> [T, F], with ``bias``
    [2F] added to [gate | up] first; ACT_TANH /
    ACT_SILU / ACT_GELU_ERF (exact gelu) / ACT_RELU2 (the square of relu) / ACT_SOFTCAP (limit tanh(x / limit)): elementwise.  Elementwise kinds take an
    fp32 factor per row, ``row_scale`` [T]: logical row i is row ``row_map[i]`` (a permutation; default i) and its
    input is multiplied by ``row_scale[i]`` before the function."""
    gated = kind in (ACT_GELU_TANH, ACT_SWISH_CLAMP, ACT_RELU)
    if kind == ACT_SOFTCAP and not limit > 0:
        raise ValueError("act: a soft cap needs a positive limit")
    if gated and (row_scale is not None or row_map is not None):
        raise ValueError("act: row factors go with the elementwise kinds")
    if bias is not None and (not gated or bias.numel() != x.shape[1]):
        raise ValueError("act: the bias is [2F] and goes with the gated kinds")
    if not _gpu(x, row_scale, row_map, bias):
        return ref.act(x, kind, limit, alpha, row_scale, row_map, bias)
    T = x.shape[0]
    F = x.shape[1] // 2 if gated else x.shape[1]
    for t, n in ((row_scale, "row_scale"), (row_map, "row_map")):
        if t is not None and t.numel() != T:
            raise ValueError(f"act: {n} must have one entry per row")
    out = torch.empty(T, F, dtype=x.dtype, device=x.device)
    _native().act(out.data_ptr(), _p(x), T, F, kind, float(limit or 0.0), float(alpha), _p(row_scale, F32, "row_scale"),
                  _p(row_map, I32, "row_map"), _p(bias, x.dtype, "bias"), _f32(x.dtype), -1)
    return out


FAST_WEIGHTS = 512 * 1024        # weights from which on a bf16 product goes to the tuned kernels with any number of rows


def _route_fast(a: torch.Tensor, w: torch.Tensor, out_dtype) -> bool:
    """bf16 products of production size whose shape the framework's tuned GEMV / MFMA GEMM kernels take (128-byte
    k steps, N % 16 == 0, at least 1024 x 512 weights: the sizes their plan tables and heuristics were tuned and
    tested on).  Smaller products are launch-bound and stay on the any-shape kernel, but of half that size those with rows enough to
    fill it or with a depth that its few tiles walk alone: us, any-shape / tuned, M x N x K in bf16 and (N >= K) fp32: 512 x 2048 x 128
    5.4 / 4.4, 2048 12.9 / 7.4; 512 x 512 x 512 5.2 / 4.9, 2048 9.0 / 4.7; 2048 x 256 x 1024 12.8 / 6.2; x 128 x 2048 33 rows 7.0 /
    5.6, 64 10.0 / 5.6, 200 11.4 / 7.5, 2048 14.5 / 9.4.  200 x 1024 x 256 and x 512 x 512 in fp32 are 4 - 10 % slower there."""
    if _ops.LEAN:
        return False
    if a.dtype != BF16 or w.dtype != BF16 or out_dtype not in (BF16, F32) or a.dim() != 2 or w.dim() != 2:
        return False
    if _ops.GEMM_BACKEND == "library" or not a.is_contiguous() or not w.is_contiguous():
        return False
    N, K = w.shape
    M, size = a.shape[0], K * N
    return a.shape[1] == K and K % 64 == 0 and N % 16 == 0 and K >= 128 and N >= 128 and \
        (size >= FAST_WEIGHTS or (2 * size >= FAST_WEIGHTS and (M >= 512 or (K >= 1024 and M > 128) or (K >= 2048 and M >= 33))))


# route fitting bf16 shapes to ops.linear (K8S_SEQMIX_FAST_GEMM=0: every product on the any-shape kernel)
FAST_GEMM = os.environ.get("K8S_SEQMIX_FAST_GEMM", "1") != "0"


def linear(a: torch.Tensor, w: torch.Tensor, out_dtype=None) -> torch.Tensor:
    """a [M, K] @ w [N, K]^T for any shape, bf16 or fp32 operands (fp32: fp32 products and sums, on the matrix cores' fp32
    instruction or plain FMAs, no reduced-precision mode), fp32 accumulation.  Shapes that fit the tuned bf16 kernels go there."""
    out_dtype = out_dtype or a.dtype
    if not _gpu(a, w):
        return ref.gemm_any(a, w, out_dtype)
    if FAST_GEMM and _route_fast(a, w, out_dtype):
        try:
            return _ops.linear(a, w, out_dtype=F32 if out_dtype == F32 else None)
        except _ops.NoKernelForShape:
            pass
    return gemm(a, w, out_dtype)


def gemm(a: torch.Tensor, w: torch.Tensor, out_dtype=None, *, a_rows: Optional[torch.Tensor] = None,
         tiles: Optional[torch.Tensor] = None, rows: Optional[int] = None,
         seg: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None, common: int = 0) -> torch.Tensor:
    """The any-shape GEMM.  2-D: a [M, K] (row stride free) @ w [N, K]^T.  3-D: batched over dim 0 (a [G, M, K] with
    any strides whose last is 1, w [G, N, K]) -> [G, M, N]; ``out``: a [G, M, N] view with any batch / row strides.
    Grouped (``tiles`` [n, 3] from :func:`moe_align`, w [G, N, K]): ``rows`` compact rows, row r = a[a_rows[r]] (or
    a[r]), the rows of tile (g, r0, n) use w[g] -> [rows, N].  ``seg`` int32 [G + 1]: the groups' row offsets, the same
    rows as ``tiles`` lists; the CPU reference and the big-tile kernel (:func:`_grouped_big`) go by them.  ``common``: that many of
    the rows are the last group's (an expert that every token has), which the choice of the tile goes by.  The order of an output's
    sums depends on the kernel, and that on the sizes: in bf16, and in fp32 from a depth of 512 on, a row's result may differ in the last
    bits with the rows beside it (fp32 of less depth or of rows that are not 16-byte aligned: not)."""
    out_dtype = out_dtype or a.dtype
    if a.dtype != w.dtype:
        raise TypeError(f"gemm operands differ in dtype: {a.dtype} and {w.dtype}")
    if a.stride(-1) != 1 or w.stride(-1) != 1:
        raise ValueError("gemm: the k dimension must be contiguous")
    if tiles is not None:
        G, N, K = w.shape
        if a.shape[-1] != K:
            raise ValueError("gemm: k mismatch")
        if not _gpu(a, w):
            return ref.gemm_any(a, w, out_dtype, a_rows, tiles, seg)
        if out_dtype == BF16 and _grouped_big(a, w, seg, rows, N):
            return _pgemm4_grouped(a, w, a_rows, rows, seg, N, common=common)
        out = torch.empty(rows, N, dtype=out_dtype, device=a.device)
        _native().gemm_any(out.data_ptr(), a.data_ptr(), _p(w), rows, N, K, a.stride(0), K, N, 1, 0, N * K, 0,
                           _p(a_rows, I32, "a_rows"), _p(tiles, I32, "tiles"), tiles.shape[0], _f32(a.dtype),
                           _f32(out_dtype), -1)
        return out
    if a.shape[-1] != w.shape[-1]:
        raise ValueError(f"gemm: k mismatch {tuple(a.shape)} x {tuple(w.shape)}")
    if not _gpu(a, w):
        y = ref.gemm_any(a, w, out_dtype)
        if out is not None:
            out.copy_(y)
            return out
        return y
    if a.dim() == 2:
        M, K = a.shape
        N = w.shape[0]
        out = torch.empty(M, N, dtype=out_dtype, device=a.device)
        _native().gemm_any(out.data_ptr(), a.data_ptr(), w.data_ptr(), M, N, K, a.stride(0), w.stride(0), N, 1, 0, 0,
                           0, 0, 0, 0, _f32(a.dtype), _f32(out_dtype), -1)
        return out
    G, M, K = a.shape
    N = w.shape[1]
    if out is None:
        out = torch.empty(G, M, N, dtype=out_dtype, device=a.device)
    elif out.shape != (G, M, N) or out.stride(2) != 1 or out.dtype != out_dtype:
        raise ValueError("gemm: out must be a [G, M, N] view of the output dtype with contiguous rows")
    _native().gemm_any(out.data_ptr(), a.data_ptr(), w.data_ptr(), M, N, K, a.stride(1), w.stride(1), out.stride(1), G,
                       a.stride(0), w.stride(0), out.stride(0), 0, 0, 0, _f32(a.dtype), _f32(out_dtype), -1)
    return out


# Grouped bf16 products of at least GROUP_BIG_MIN rows per group on average (GROUP_BIG_MIN_FEW of up to 12 groups; whole rows of at
# least 64 elements) run on the big-tile kernel (pgemm4.hip); fewer stream the weights past the LDS (gemm_group_kernel), whose time
# goes with the groups that have rows.  us, weights from memory, past the LDS / big tiles: gate / up of 8 groups with the activation
# (2 x 2048 x 2048), 0.5 / 1 / 2 / 4 / 8 / 16 rows per group 17.1 / 19.0, 23.3 / 22.6, 29.8 / 26.1, 34.7 / 28.2, 33.7 / 28.4, 41.9 /
# 28.4; down (2048 x 2048) 8.8 / 10.8, 12.8 / 13.2, 16.7 / 15.1, 18.5 / 17.1, 19.0 / 17.2, 23.0 / 16.2; 8 of 4096 x 3584, 1 / 2 / 8 31.5 /
# 40.7, 42.0 / 43.0, 56.3 / 47.9; 16 of 2 x 2048 x 4096, 2 / 4 / 6 / 8 91 / 103, 105 / 111, 109 / 110, 112 / 111; 16 of 2048 x 1024, 4 / 6 / 8
# 15.6 / 17.1, 16.4 / 16.9, 17.8 / 17.1.
GROUP_BIG_MIN = 6
GROUP_BIG_MIN_FEW = 2            # of up to 12 groups
GROUP_BIG_MAX_GROUPS = 64        # every workgroup walks the groups' offsets


def _grouped_big(a: torch.Tensor, w: torch.Tensor, seg: Optional[torch.Tensor], rows: int, N: int) -> bool:
    E, _, K = w.shape
    return (not _ops.LEAN and FAST_GEMM and a.dtype == BF16 and seg is not None and seg.is_cuda and seg.dtype == I32
            and seg.is_contiguous() and seg.numel() == E + 1 and E <= GROUP_BIG_MAX_GROUPS
            and rows >= (GROUP_BIG_MIN if E > 12 else GROUP_BIG_MIN_FEW) * E and K % 64 == 0 and N % 4 == 0 and N >= 128 and a.dim() == 2 and a.stride(1) == 1
            and a.stride(0) >= K and a.stride(0) % 8 == 0 and a.data_ptr() % 16 == 0 and w.is_contiguous()
            and w.data_ptr() % 16 == 0 and w.shape[1] * K * 2 < 1 << 32 and a.shape[0] * a.stride(0) * 2 < 1 << 32)


# Time of a grouped product in us, configuration -> (fixed, per round of tiles over the CUs and 64-deep k-step, per round, per
# k-step, per MB of weights, per MB of output, per round and 65536 outputs of a gated activation).  Fitted to 10 products of 4 -
# 16 groups, 2048 x 1024 .. 2 x 3584 x 4096, 4 - 768 rows per group drawn at random, weights cold: rms error 4 - 8 % per
# configuration, the pick within 1 % of the best configuration on average, 23 % at most, and 7 % faster on average than the pick of
# the six tiles there were.  _GROUP_TILE: weight rows and tokens of a tile.
_GROUP_TILE = {1: (256, 128), 2: (128, 256), 3: (128, 128), 4: (256, 256), 5: (128, 64), 6: (64, 64), 7: (224, 256), 8: (256, 192)}
_GROUP_COST = {1: (0.0, 0.632, 2.7, 0.0, 0.0957, 0.701, 3.45), 2: (1.58, 0.488, 5.91, 0.0, 0.0921, 0.574, 8.35),
               3: (4.05, 0.397, 0.0, 0.0266, 0.0876, 0.397, 3.35), 4: (0.0, 0.897, 8.92, 0.0, 0.0896, 0.484, 5.54),
               5: (2.99, 0.317, 0.0, 0.0184, 0.103, 0.324, 4.53), 6: (0.417, 0.164, 0.608, 0.0738, 0.105, 0.636, 1.43),
               7: (0.0, 0.849, 7.16, 0.0, 0.0733, 0.465, 3.83), 8: (0.0, 0.762, 4.85, 0.0, 0.0828, 0.515, 2.92)}


@functools.lru_cache(maxsize=4096)
def _grouped_tile(rows: int, E: int, N: int, K: int, pair: bool, even: bool = False, common: int = 0) -> int:
    """Configuration of the grouped big-tile product: the cheapest of them all by _GROUP_COST, for groups of the same size (``even``)
    or of about equal size drawn at random beside ``common`` rows that are the last group's, whose tiles are expected ones: up to 5 that
    would begin another round most often are not there (1700 rows of 16 experts, 2 x 2048 x 4096: 260.5 tiles expected, 136 us in one
    round, 152 the next best).  With three rows a group or fewer there are groups without any, and what is left is a stream of weights
    that the smallest tiles, two of them on a CU, keep up best, of wide groups the next ones: us, 64 x 64 / 128 x 64 tiles, 8 groups
    beside a common one, 0.5 / 1 / 2 rows each: 2048 x 2048 12.2 / 19.1, 14.7 / 20.2, 16.3 / 20.8; 4096 x 3584 24.8 / 32.0, 42.3 / 43.1,
    47.2 / 48.1; gated 2 x 2048 x 2048 15.5 / 19.0, 25.6 / 26.0, 27.7 / 29.2; 2 x 3584 x 4096 48.4 / 48.1, 86.2 / 81.3, 89.4 / 86.9 (256 x
    128: 65.5, 82.2, 90.7)."""
    drawn = E - (common > 0)
    r, n, kt, best = (rows - common) / max(drawn, 1), (2 * N if pair else N), K / 64, None
    if rows <= 3 * E and E > 1 and not even:
        return 6 if n <= 4096 else 5
    for cfg, (t0, tile, rnd, step, wmb, omb, act_us) in _GROUP_COST.items():
        bp, bq = _GROUP_TILE[cfg]
        if even or E == 1:
            tiles, spare = E * -(-rows // E // bq), 1e-9
        else:   # a group's tiles beyond k: the chance that it has more than bq k rows, 1 up to six deviations below the mean
            d = 6.0 * math.sqrt(max(r, 1.0))
            sure = max(0, int((r - d) // bq))
            tiles = -(-common // bq) + drawn * (1 + sure + sum(0.5 + 0.5 * math.erf((r - bq * k) / math.sqrt(2.0 * max(r, 1.0)))
                                        for k in range(sure + 1, int((r + d) / bq) + 2)))
            spare = 0.02
        rounds = max(1, math.ceil(tiles * -(-n // bp) / 256 - spare))
        us = t0 + rounds * (tile * kt + rnd + (act_us * bp * bq / 65536 if pair else 0.0)) + step * kt + \
            wmb * E * n * K * 2e-6 + omb * rows * N * 2e-6
        if best is None or us < best[0]:
            best = (us, cfg)
    return best[1]


# The same for groups of GROUP_FEW_ROWS drawn rows each on average and fewer, of GROUP_FEW_WEIGHTS weights (least, most), which are a stream
# of weights at which the CUs have to be equally busy: configuration -> (fixed, per MB of the weights that are read, per 64-deep
# k-step of a CU's first tile, of its other ones, per tile, per tile and 65536 outputs of a gated activation); the stream and the
# busiest CU's tiles hide each other but for where they are about as long (the root of their fourth powers' sum).  Fitted to 312
# products of 4 - 33 groups, 2048 x 1024 .. 2 x 3584 x 4096, 1 - 160 tokens, weights cold: rms error 9 %.  8 groups and a common one of 1 - 80
# tokens, by the rule above and its tiles / here: 2 x 2048 x 2048 8 33.2 / 32.6, 32 36.7 / 33.2, 64 40.3 / 35.9; 2048 x 2048 32 22.0 / 18.5;
# 4096 x 3584 2 28.4 / 28.5, 32 59.6 / 50.3; over 60 such products 10 % less on average, 1 % more at most.  Larger weights have tiles for
# many rounds whatever their width: 2 x 3584 x 4096, 64 tokens 94.9 / 108.5.
GROUP_FEW_ROWS, GROUP_FEW_WEIGHTS = 20, (1 << 21, 1 << 24)
_GROUP_FEW_TILE = {3: (128, 128), 5: (128, 64), 6: (64, 64), 18: (64, 32), 19: (96, 32), 20: (128, 32), 21: (160, 32)}
_GROUP_FEW_COST = {3: (5.43, 0.186, 0.434, 0.537, 0.0, 8.03), 5: (4.93, 0.187, 0.346, 0.517, 0.0, 17.0),
                   6: (3.10, 0.169, 0.210, 0.293, 1.30, 5.90), 18: (3.29, 0.185, 0.170, 0.228, 1.0, 6.11),
                   19: (3.97, 0.187, 0.185, 0.356, 0.66, 15.3), 20: (4.75, 0.182, 0.203, 0.529, 0.0, 20.7),
                   21: (5.38, 0.187, 0.256, 0.552, 0.0, 40.0)}


@functools.lru_cache(maxsize=4096)
def _grouped_few(rows: int, drawn: int, N: int, K: int, pair: bool, common: int) -> int:
    """Configuration of the grouped product of ``drawn`` groups, of few rows each, and ``common`` rows of one more, by _GROUP_FEW_COST:
    the mean over the tiles that are expected and 1.2 deviations on both sides of them (the groups' sizes as Poisson's).  Below 1.5 rows a
    group too many of them have none for whole rounds to go by: the smallest tile, 0 - 7 % faster than 64 x 64 (2048 x 2048, 5 tokens 15.1 /
    14.9, on 96 x 32 16.0, on 128 x 32 17.7)."""
    r, n, kt, best = (rows - common) / drawn, (2 * N if pair else N), K / 64, None
    if r < 1.5:
        return 18
    more, p, left = [], math.exp(-r), 1.0            # the chances of more than 0, 32, 64, ... rows
    for k in range(1 + int(r + 8.0 * math.sqrt(r) + 8.0)):
        left -= p
        if k % 32 == 0:
            more.append(max(left, 0.0))
        p *= r / (k + 1)
    stream = (drawn * more[0] + (common > 0)) * n * K * 2e-6
    dist = {}                                        # tokens of a tile: tiles of the groups, the deviation of their number
    for bq in (32, 64, 128):
        m1, m2 = sum(more[::bq // 32]), sum((2 * t + 1) * c for t, c in enumerate(more[::bq // 32]))
        dist[bq] = drawn * m1 + -(-common // bq), math.sqrt(max(0.0, m2 - m1 * m1) * drawn)
    for cfg, (t0, wmb, first, other, tile, act_us) in _GROUP_FEW_COST.items():
        bp, bq = _GROUP_FEW_TILE[cfg]
        tiles, dev = dist[bq]
        us = 0.0
        for z in (-1.2, 0.0, 1.2):
            q = max(1, math.ceil(max(tiles + z * dev, 0.0) * -(-n // bp) / 256 - 0.01))
            busy = kt * (first + other * (q - 1)) + q * (tile + (act_us * bp * bq / 65536 if pair else 0.0))
            us += t0 + ((stream * wmb) ** 4 + busy ** 4) ** 0.25
        if best is None or us < best[0]:
            best = (us, cfg)
    return best[1]


# The tiles between the others, and those again, for uneven groups of more rows: configuration -> as _GROUP_COST.  Fitted to 220 products of
# 5 - 16 groups, 2048 x 1024 .. 2 x 3584 x 4096, 21 rows a group to 2100 tokens, weights cold, rms error 4 - 8 %; a tile of these is taken where it
# is 4 % cheaper than _grouped_tile's by the mean over the tiles expected and 1.2 deviations on both sides: 2.5 % less time on average over
# all 220, up to 20 % (8 groups and a common one, gated 2 x 2048 x 2048, 1300 tokens 88 -> 77 us, 1534 89 -> 85; 2048 x 2048, 640 32.3 -> 30.0).
_GROUP_MORE_TILE = {**_GROUP_TILE, 10: (192, 96), 11: (192, 128), 12: (128, 192), 13: (192, 192), 15: (192, 224), 16: (224, 224), 17: (256, 224)}
_GROUP_MORE_COST = {1: (0.0, 0.613, 3.47, 0.0, 0.104, 0.44, 5.08), 2: (0.497, 0.557, 4.55, 0.0, 0.086, 0.43, 4.74),
                    3: (3.0, 0.381, 0.0, 0.0402, 0.0978, 0.299, 5.55), 4: (0.0, 0.942, 7.91, 0.0, 0.0786, 0.34, 6.26),
                    5: (2.36, 0.331, 0.0, 0.0, 0.123, 0.0886, 0.0), 6: (1.62, 0.199, 0.0, 0.0, 0.115, 0.229, 0.0),
                    7: (0.0, 0.866, 7.28, 0.0, 0.0631, 0.39, 4.59), 8: (0.236, 0.746, 5.61, 0.0, 0.0847, 0.41, 3.8),
                    10: (0.0, 0.51, 1.02, 0.0, 0.106, 0.539, 7.29), 11: (0.0, 0.546, 1.97, 0.0, 0.0971, 0.494, 6.51),
                    12: (1.04, 0.501, 2.48, 0.0, 0.0826, 0.535, 7.01), 13: (0.0, 0.632, 4.95, 0.0, 0.0749, 0.429, 5.13),
                    15: (0.0, 0.686, 6.1, 0.0, 0.0699, 0.416, 4.79), 16: (0.0, 0.777, 6.37, 0.0, 0.0695, 0.43, 4.81),
                    17: (0.0, 0.853, 6.61, 0.0, 0.0756, 0.441, 3.83)}
# ... and per MB of weights where the common rows are one row of tiles, each of which reads weights of its own; with two of them, pairs
# share theirs.  8 groups and a common one, 96 / 97 tokens, us: on 192 x 96 gated 2 x 2048 x 2048 36.9 / 34.4 (64 x 64 35.1 / 35.0), 4096 x 3584 56.1 /
# 50.1 (56.3 / 56.5), 2048 x 2048 27.0 / 24.8; 128 / 130 on 192 x 128 38.1 / 34.9, 57.5 / 52.0, 28.8 / 26.1; none on the tiles of _GROUP_TILE that are
# picked there.  Over 936 products of 4 - 17 groups, 17 weights, 41 - 2900 tokens the picks take 2.2 % less than _grouped_tile's, 20 of them 2 %
# more and over, up to 25 % (4096 x 2048 of 4 groups, 214 tokens 20.4 -> 25.6); with twice or half the term they are the same.
_GROUP_MORE_ALONE = {10: 0.008, 11: 0.008, 12: 0.002, 13: 0.002}


@functools.lru_cache(maxsize=4096)
def _grouped_more(rows: int, E: int, N: int, K: int, pair: bool, even: bool, common: int, base: int) -> int:
    """``base``, or the tile between the others that is cheaper by _GROUP_MORE_COST."""
    drawn = E - (common > 0)
    r, n, kt, best = (rows - common) / drawn, (2 * N if pair else N), K / 64, None
    sd = math.sqrt(max(r, 1.0))
    for cfg in [base] + [c for c in _GROUP_MORE_COST if c not in _GROUP_TILE]:
        t0, tile, rnd, step, wmb, omb, act_us = _GROUP_MORE_COST[cfg]
        bp, bq = _GROUP_MORE_TILE[cfg]
        if even:
            tiles, dev = E * -(-rows // E // bq), 0.0
        else:
            sure = max(0, int((r - 6.0 * sd) // bq))       # (as _grouped_tile)
            odds = [0.5 + 0.5 * math.erf((r - bq * k) / (math.sqrt(2.0) * sd)) for k in range(sure + 1, int((r + 6.0 * sd) / bq) + 2)]
            tiles, dev = -(-common // bq) + drawn * (1 + sure + sum(odds)), math.sqrt(drawn * sum(p * (1.0 - p) for p in odds))
        rounds = sum(max(1, math.ceil((tiles + z * dev) * -(-n // bp) / 256 - 0.01)) for z in (-1.2, 0.0, 1.2)) / 3.0
        us = t0 + rounds * (tile * kt + rnd + (act_us * bp * bq / 65536 if pair else 0.0)) + step * kt + wmb * E * n * K * 2e-6 + \
            omb * rows * N * 2e-6
        if 0 < common <= bq:
            us += _GROUP_MORE_ALONE.get(cfg, 0.0) * E * n * K * 2e-6
        if best is None or us < best[0]:
            best = (us if best is not None else 0.96 * us, cfg)
    return best[1]


def _grouped_plan(rows: int, E: int, N: int, K: int, pair: bool, even: bool, common: int) -> int:
    """Configuration of the grouped big-tile product: :func:`_grouped_few`'s, :func:`_grouped_tile`'s or one between those."""
    drawn = E - (common > 0)
    least, most = GROUP_FEW_WEIGHTS
    size = (2 * N if pair else N) * K
    few = rows - common <= GROUP_FEW_ROWS * drawn
    if E == 1 or rows <= common or size < least or (few and (even or size > most)):
        return _grouped_tile(rows, E, N, K, pair, even, common)
    if few:
        return _grouped_few(rows, drawn, N, K, pair, common)
    return _grouped_more(rows, E, N, K, pair, even, common, _grouped_tile(rows, E, N, K, pair, even, common))


def _pgemm4_grouped(a, w, a_rows, rows: int, seg, N: int, kind: int = -1, limit: float = 0.0, alpha: float = 1.0, common: int = 0,
                    common_limit: Optional[float] = None):
    E, _, K = w.shape
    out = torch.empty(rows, N, dtype=BF16, device=a.device)
    _native().pgemm4_grouped(out.data_ptr(), a.data_ptr(), w.data_ptr(), a.shape[0], rows, N, K, E, _p(seg, I32, "seg"),
                             _p(a_rows, I32, "a_rows"), a.stride(0), _grouped_plan(rows, E, N, K, kind >= 0, seg is None, common), 4, kind,
                             float(limit), float(alpha), float(limit if common_limit is None else common_limit), -1)
    return out


def _few_fits(a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the few-row products (gemm_group_tile) take these operands."""
    K = w.shape[-1]
    return (_gpu(a, w) and a.dtype == BF16 and w.dtype == BF16 and K % 64 == 0 and a.shape[-1] == K and a.stride(-1) == 1
            and a.stride(-2) % 8 == 0 and w.is_contiguous() and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def linear_each(a: torch.Tensor, w: torch.Tensor):
    """[a[i] @ w[i].T]: several inputs, a weight each (a [G, M, K], w [G, N, K]) -> G tensors [M, N] of one row stride.  One
    launch where that is faster than G of :func:`linear`: the any-shape kernel (k shared by the waves while its tiles are few) up to
    32 rows, and as long as its workgroups of 16 columns run at once; else the grouped big tiles from 16 rows on, of small weights from
    the first.  us, weights from memory, any-shape / big tiles / G launches: 4 weights of 2048 x 2048, M = 8 10.9 / 17.7 / 19.9, 32 17.2 /
    17.8 / 24.2, 64 24.5 / 18.3 / 29.2, 512 51.7 / 23.8 / 60.3; of 512 x 2048, 128 13.3 / 15.6 / 23.3, 200 20.9 / 15.1 / 39.8; of 4096 x
    4096, 8 71 / 37.2 / 33.1, 16 71 / 36.8 / 39.4, 64 73.6 / 38.6 / 54.6, 2048 - / 195 / 236; 8 of 2048 x 2048, 1 36.7 / 20.4 / 34.2."""
    G, M, K = a.shape
    N = w.shape[1]
    if w.shape != (G, N, K):
        raise ValueError(f"linear_each: inputs {tuple(a.shape)} and weights {tuple(w.shape)}")
    if not (FAST_GEMM and _gpu(a, w) and _route_fast(a[0], w[0], a.dtype)):
        return gemm(a, w).unbind(0)
    if _each_once(a, w):
        rows = G * (-(-M // 64))
        if rows * (-(-N // 64)) <= 128 and (M <= 32 or rows * (-(-N // 16)) <= 256):
            return gemm(a, w).unbind(0)
        if M <= 2048 and (M >= 16 or N * K <= 1 << 23):
            return _pgemm4_grouped(a.view(G * M, K), w, None, G * M, None, N).view(G, M, N).unbind(0)
    return tuple(linear(a[i], w[i]) for i in range(G))


def each_parts(w: torch.Tensor, G: int, N: int):
    """The weights of :func:`linear_each_tanh` apart, for its ``parts``: [G, N, K] and [L, K]."""
    return w[:G * N].view(G, N, w.shape[1]), w[G * N:]


def linear_each_tanh(a: torch.Tensor, w: torch.Tensor, N: int, parts: Optional[tuple] = None):
    """(:func:`linear_each` of all inputs but the last, tanh of the last one's product): a [G + 1, M, K], w [G N + L, K] the weights one
    after the other (``parts``: views of them, :func:`each_parts`, where a caller keeps them).  A few bf16 rows in one launch (stream_gemv.hip).  us, two launches or more / one, weights from memory: 4 weights of
    2048 x 2048 and one of 128 x 2048, 1 row 15.4 / 12.0, 8 17.5 / 13.3, 16 19.1 / 17.5; of 4096 x 4096 and 256 x 4096, 1 39.2 / 37.0,
    8 42.4 / 39.6, 16 44.1 / 46.4 (x in registers: 16 rows of 4096 leave room for less of the weights under way)."""
    G, M, K = a.shape[0] - 1, a.shape[1], a.shape[2]
    L = w.shape[0] - G * N
    if G < 1 or L < 1 or w.shape[1] != K:
        raise ValueError(f"linear_each_tanh: inputs {tuple(a.shape)}, weights {tuple(w.shape)} of {N} rows each")
    if rows_join(M, K) and (M <= 8 or K <= 2048) and _gpu(a, w) and a.dtype == w.dtype == BF16 and a.is_contiguous() and w.is_contiguous() and N % 8 == 0:
        out = torch.empty(G, M, N, dtype=BF16, device=a.device)
        last = torch.empty(M, L, dtype=BF16, device=a.device)
        if _native().rows_each(out.data_ptr(), last.data_ptr(), a.data_ptr(), w.data_ptr(), G, N, L, M, K, -1):
            return out.unbind(0), last
    each, last = parts or each_parts(w, G, N)
    return linear_each(a[:G], each), linear_act(a[G], last, ACT_TANH)


def _each_once(a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether products of several inputs may share a launch: the routing is free, sizes and places fit the big tiles."""
    G, M, K = a.shape
    return (_ops.GEMM_BACKEND == "auto" and a.is_contiguous() and w.is_contiguous() and G <= GROUP_BIG_MAX_GROUPS
            and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and w.shape[1] * K * 2 < 1 << 32 and G * M * K * 2 < 1 << 32)


def gemm_act(a: torch.Tensor, w: torch.Tensor, kind: int, limit: float = 0.0, alpha: float = 1.0, *,
             a_rows: Optional[torch.Tensor] = None, tiles: Optional[torch.Tensor] = None, rows: int = 0,
             seg: Optional[torch.Tensor] = None, common: int = 0, common_limit: Optional[float] = None) -> torch.Tensor:
    """act(gemm(a, w)) of a grouped product and a gated kind, w [E, 2 N, K] = gate | up: in the product's epilogue where
    it runs on the big-tile kernel (the sums are then not rounded ahead of the activation).  ``common``, ``seg``: as in
    :func:`gemm`; the last group's limit is then ``common_limit``, if given."""
    N, E = w.shape[1] // 2, w.shape[0]
    own = common > 0 and common_limit is not None and common_limit != limit
    if a.shape[-1] == w.shape[-1] and w.shape[1] % 2 == 0 and a.dtype == w.dtype and _gpu(a, w) and \
            _grouped_big(a, w, seg, rows, N):
        return _pgemm4_grouped(a, w, a_rows, rows, seg, N, kind, limit, alpha, common, common_limit if own else None)
    if tiles is not None and w.dim() == 3 and kind in (ACT_GELU_TANH, ACT_SWISH_CLAMP, ACT_RELU) and 0 < rows <= 512 and \
            rows <= 32 * tiles.shape[0] and (rows >= 6 * E or common > 0 or w.shape[1] * w.shape[2] <= 1 << 22) and \
            w.shape[1] % 2 == 0 and a.dim() == 2 and _few_fits(a, w):
        # (16 experts of 2 x 2048 x 4096: 8 rows 53 / 56 us, 64 rows 102 / 102 us, 96 rows 109 / 105 us; with a common expert always, whose
        # product alone, linear_act of as many rows, does not round its sums either)
        out = torch.empty(rows, N, dtype=BF16, device=a.device)
        _native().gemm_few_act(out.data_ptr(), a.data_ptr(), w.data_ptr(), rows, N, w.shape[2], a.stride(0),
                               _p(a_rows, I32, "a_rows"), _p(tiles, I32, "tiles"), tiles.shape[0], kind, float(limit),
                               float(alpha), E - 1 if own else -1, float(common_limit if own else 0.0), -1)
        return out
    y = gemm(a, w, a_rows=a_rows, tiles=tiles, rows=rows, seg=seg, common=common)
    out = act(y, kind, limit, alpha)
    if own:
        mine = torch.arange(rows, device=y.device) >= seg[E - 1]
        out = torch.where(mine.unsqueeze(-1), act(y, kind, common_limit, alpha), out)
    return out


def linear_act(a: torch.Tensor, w: torch.Tensor, kind: int, limit: float = 0.0, alpha: float = 1.0, *,
               bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """act(linear(a, w), kind, bias=bias): in the product's epilogue where its plan is an unsplit big-tile one, which saves a
    pass over the product (2048 x 2 x 8192, gated: 22 us; 2048 x 8192 elementwise: 15 us; 200 x 1040 x 1024, few tiles: 9.8 -> 7.3)
    and its rounding, and up to 128 rows (a captured step of 1 row 477 -> 456 us, of 8 rows 655 -> 637, of 32 rows 1028 -> 1016)."""
    pair = kind in (ACT_GELU_TANH, ACT_SWISH_CLAMP, ACT_RELU)
    if (pair or kind == ACT_RELU2) and FAST_GEMM and _gpu(a, w, bias) and _route_fast(a, w, BF16) and a.dtype == BF16 and (not pair or w.shape[0] % 8 == 0):
        M, K = a.shape
        if M <= 128 and bias is None:
            out = _ops.linear_act_rows(a, w, pair, kind, float(limit), float(alpha))
            if out is not None:
                return out
        kern, plan = _ops.gemm_act_route(M, w.shape[0], K) if M >= 129 else ("", None)
        if kern == "pgemm4" and plan[1] == 1 and a.data_ptr() % 16 == 0 and \
                (bias is None or (pair and bias.dtype == BF16 and bias.numel() == w.shape[0] and bias.data_ptr() % 8 == 0)):
            N = w.shape[0] // 2 if pair else w.shape[0]
            out = torch.empty(M, N, dtype=BF16, device=a.device)
            _native().pgemm4_act(out.data_ptr(), _p(a), _p(w), M, N, K, plan[0], plan[2], kind, float(limit), float(alpha),
                                 _p(bias), -1)
            return out
    # few tiles: gemm() would take that kernel, or of 256 - 512 Ki weights a tuned one, whose sums an activation of its own would take
    # rounded to bf16: of these one launch and one rounding too, faster or not (us, one launch / the tuned product and tanh, M x N x K: 64 x
    # 128 x 2048 11.9 / 7.6, 333 11.9 / 10.9, 2048 15.0 / 12.1, 4096 25.2 / 12.7; 333 x 256 x 1024 7.7 / 8.8; 512 x 512 x 512 5.7 / 8.3)
    if bias is None and not pair and kind != ACT_SOFTCAP and a.dim() == w.dim() == 2 and a.shape[0] > 0 and \
            -(-a.shape[0] // 64) * (-(-w.shape[0] // 64)) <= 128 and _few_fits(a, w) and \
            (w.numel() < FAST_WEIGHTS or not (FAST_GEMM and _route_fast(a, w, BF16))):
        out = torch.empty(a.shape[0], w.shape[0], dtype=BF16, device=a.device)
        _native().gemm_few_act(out.data_ptr(), a.data_ptr(), w.data_ptr(), a.shape[0], w.shape[0], w.shape[1], a.stride(0), 0, 0,
                               0, kind, float(limit), float(alpha), -1)
        return out
    return act(linear(a, w), kind, limit, alpha, bias=bias)


# ----------------------------------------------------------------------------- recurrent mixer
NORM_GEMV_MAX_M = 1       # rows (norm_gemv.hip)


def norm_linear(x: Optional[torch.Tensor], branch: torch.Tensor, w: Optional[torch.Tensor], eps: float, weight: torch.Tensor, *,
                act_kind: Optional[int] = None, limit: float = 0.0, alpha: float = 1.0, out_dtype=None, mult: float = 1.0,
                next_w: Optional[torch.Tensor] = None, offset: float = 0.0, gain: float = 1.0, gate: Optional[torch.Tensor] = None,
                gate_kind: int = GATE_SIGMOID):
    """A product and the norms between it and the output ``branch`` of the sublayer before, (out, stream): with a stream x (fp32 [T,
    W]) first x + ``mult`` * branch (``w`` None: :func:`resnorm`) or x + rms-norm(branch) * w (:func:`branchnorm`), that row itself or,
    with ``next_w``, its rms-norm * (``offset`` + next_w) * ``gain`` -- without one rms-norm(branch) * w, times ``gate``'s sigmoid or
    silu (:func:`norm_mix`) -- times ``weight``, with :func:`linear_act`'s activation if ``act_kind`` is given.  The stream is a new
    tensor or x itself, updated: the caller goes on with what is returned.  One bf16 row runs in one launch; more, or other sizes, as
    the norm and the product."""
    T, W = branch.shape
    dt = weight.dtype
    if T <= NORM_GEMV_MAX_M and dt == BF16 and FAST_GEMM and not _ops.LEAN and _ops.GEMM_BACKEND == "auto" and _ops.GEMV_MAX_M >= T > 0 and \
            _gpu(branch, weight, x, w, next_w, gate) and weight.is_contiguous() and branch.stride(1) == 1 and weight.shape[1] == W:
        pair = act_kind in (ACT_GELU_TANH, ACT_SWISH_CLAMP, ACT_RELU)
        b32, N = branch.dtype == F32, weight.shape[0] // 2 if pair else weight.shape[0]
        ok = act_kind is None or act_kind == ACT_RELU2 or (pair and weight.shape[0] % 2 == 0)
        ok = ok and out_dtype in (None, BF16, F32) and (act_kind is None or out_dtype != F32) and branch.dtype in (BF16, F32)
        for t, d in ((w, branch.dtype), (next_w, BF16)):
            ok = ok and (t is None or (t.dtype == d and t.numel() == W and t.is_contiguous()))
        if x is not None:
            ok = ok and x.dtype == F32 and x.shape == branch.shape and x.is_contiguous() and not b32 and gate is None
        else:
            ok = ok and w is not None and next_w is None and (gate is None or (gate.dtype == BF16 and gate.shape == branch.shape
                                                                               and gate.stride(1) == 1))
        if ok:
            out = torch.empty(T, N, dtype=out_dtype or BF16, device=branch.device)
            new = torch.empty_like(x) if x is not None else None
            kind = act_kind if act_kind is not None else -2 if out_dtype == F32 else -1
            if _native().norm_gemv(out.data_ptr(), _p(new), _p(x), branch.data_ptr(), int(b32), _p(w), float(mult),
                                   gate.data_ptr() if gate is not None else 0, int(gate_kind == GATE_SILU), _p(next_w), float(offset),
                                   float(gain), float(eps), weight.data_ptr(), N, W, kind, float(limit), float(alpha), -1):
                return out, new
    if x is None:
        h = norm_mix(branch, w, None, None, eps, out_dtype=dt, gate=gate, gate_kind=gate_kind)
    elif w is not None:
        if offset:
            raise ValueError("norm_linear: branchnorm's second norm has no offset")
        h = branchnorm(x, branch, w, eps, out_dtype=dt, next_w=next_w, gain=gain)
    else:
        if next_w is None or gain != 1.0:
            raise ValueError("norm_linear: resnorm's row is normed, without a gain")
        h = resnorm(x, next_w, eps, branch=branch, mult=mult, offset=offset, out_dtype=dt)
    if act_kind is not None:
        return linear_act(h, weight, act_kind, limit, alpha), x
    return linear(h, weight, out_dtype), x


class Rows(NamedTuple):
    """A stream and its rows as the next product reads them: normed (``sums`` None), or times the norm's weight alone with what is
    missing of the norm, sums of squares."""
    x: torch.Tensor
    h: torch.Tensor
    sums: Optional[torch.Tensor]      # [T, 256] of which the first T * count are used, rows of count
    count: int
    w: torch.Tensor                   # the norm's weight and what is added to it
    offset: float


def rows_join(T: int, W: int) -> bool:
    """Whether T rows of a stream of W columns go from product to product as :class:`Rows` with sums (bf16)."""
    return FAST_GEMM and not _ops.LEAN and _ops.GEMM_BACKEND == "auto" and 1 <= T <= _ops.SGEMV_MAX_M and W % 128 == 0 and W <= 4096


def linear_rows(a: torch.Tensor, weight: torch.Tensor, x: torch.Tensor, next_w: torch.Tensor, eps: float, *, mult: float = 1.0,
                offset: float = 0.0) -> Rows:
    """x (fp32) + ``mult`` * linear(a, weight), a new tensor or x itself, updated, and its rows for :func:`rows_linear`, normed with
    (``offset`` + next_w).  Up to 16 bf16 rows in one launch (stream_gemv.hip), which rounds neither the branch nor -- the norm's factor
    being the next product's -- the rows more than once; otherwise the product and :func:`resnorm`."""
    T, K = a.shape
    N = weight.shape[0]
    if rows_join(T, N) and _gpu(a, weight, x, next_w) and a.dtype == weight.dtype == next_w.dtype == BF16 and x.dtype == F32 and \
            x.shape == (T, N) and weight.shape[1] == K and all(t.is_contiguous() for t in (a, weight, x, next_w)):
        y, h = torch.empty_like(x), torch.empty(T, N, dtype=BF16, device=x.device)
        sums = torch.empty(T, 256, dtype=F32, device=x.device)
        n = _native().rows_workspace(T, N, K, 0)
        part = torch.empty(n, dtype=F32, device=x.device) if n > 0 else None
        count = _native().rows_out(_p(y), _p(h), _p(sums), _p(x), _p(next_w), a.data_ptr(), weight.data_ptr(), _p(part), T, N, K,
                                   float(mult), float(offset), -1)
        if count:
            return Rows(y, h, sums, count, next_w, offset)
    h = resnorm(x, next_w, eps, branch=linear(a, weight), mult=mult, offset=offset, out_dtype=weight.dtype)
    return Rows(x, h, None, 0, next_w, offset)


def rows_linear(r: Rows, weight: torch.Tensor, eps: float, *, act_kind: Optional[int] = None, limit: float = 0.0, alpha: float = 1.0,
                out_dtype=None, split: int = 0):
    """linear(rms-norm(r.x) * (r.offset + r.w), weight) or, with a gated kind, :func:`linear_act`; ``split``: two tensors, of the first
    ``split`` rows of ``weight`` and of the others."""
    h = r.h
    if r.sums is not None:
        T, K = h.shape
        pair = act_kind in (ACT_GELU_TANH, ACT_SWISH_CLAMP, ACT_RELU)
        N = weight.shape[0] // 2 if pair else weight.shape[0]
        if weight.dtype == BF16 and weight.is_contiguous() and weight.shape[1] == K and out_dtype in (None, BF16, F32) and \
                (act_kind is None or (pair and weight.shape[0] % 2 == 0 and out_dtype != F32)) and \
                (not split or (act_kind is None and out_dtype != F32 and 0 < split < N)):
            out = torch.empty(T, split or N, dtype=out_dtype or BF16, device=h.device)
            rest = torch.empty(T, N - split, dtype=BF16, device=h.device) if split else None
            n = _native().rows_workspace(T, N, K, int(pair))
            part = torch.empty(n, dtype=F32, device=h.device) if n > 0 else None
            kind = act_kind if act_kind is not None else -2 if out_dtype == F32 else -1
            if _native().rows_in(out.data_ptr(), _p(rest), split or N, _p(h), _p(r.sums), r.count, weight.data_ptr(), _p(part), T, N, K,
                                 float(eps), kind, float(limit), float(alpha), -1):
                return (out, rest) if split else out
        h = resnorm(r.x, r.w, eps, offset=r.offset, out_dtype=BF16)
    if act_kind is not None:
        return linear_act(h, weight, act_kind, limit, alpha)
    if split:
        return linear(h, weight[:split], out_dtype), linear(h, weight[split:], out_dtype)
    return linear(h, weight, out_dtype)


def norm_shift(x: torch.Tensor, w: torch.Tensor, eps: float, mu: torch.Tensor, state: torch.Tensor, b: dict, *,
               branch: Optional[torch.Tensor] = None, mult: float = 1.0, rowvec: Optional[torch.Tensor] = None, offset: float = 0.0,
               single: bool = False) -> torch.Tensor:
    """:func:`token_shift`, with its save, of :func:`resnorm`'s rows in the type of ``w``, ``b`` a batch description; in one launch if
    every sequence brings a single token (``single``)."""
    T, W = x.shape
    if single and _gpu(x, w, mu, state, branch, rowvec) and W % 4 == 0 and W <= 4096 and mu.shape[0] <= 5 and x.dtype == F32 and \
            all(t is None or t.dtype == w.dtype for t in (mu, state, branch, rowvec)):
        out = torch.empty(mu.shape[0], T, W, dtype=w.dtype, device=x.device)
        if _native().norm_shift(_p(out), _p(x), _p(branch), float(mult), _p(rowvec), _p(w), float(offset), float(eps), _p(mu), _p(state),
                                _p(b["seq_slots"], I32, "seq_slots"), _p(b["positions"], I32, "positions"), mu.shape[0], T, W,
                                _f32(w.dtype), -1):
            return out
    h = resnorm(x, w, eps, branch=branch, mult=mult, rowvec=rowvec, offset=offset, out_dtype=w.dtype)
    return token_shift(h, mu, state, b["cu_q"], b["tok_seq"], b["seq_slots"], b["positions"], save=True)


def token_shift(h: torch.Tensor, mu: torch.Tensor, state: torch.Tensor, cu_q: torch.Tensor, tok_seq: torch.Tensor,
                seq_slots: torch.Tensor, positions: torch.Tensor, save: bool = False) -> torch.Tensor:
    """[n, T, W]: h + (previous token's h - h) * mu[s]; the previous token of a portion's first token is the slot's
    row of ``state`` (zeros at position 0).  ``save``: then, as :func:`shift_save`, state[slot] = the portion's last h."""
    if not _gpu(h, mu, state):
        out = ref.token_shift(h, mu, state, cu_q, seq_slots, positions)
        if save:
            ref.shift_save(state, h, cu_q, seq_slots, positions)
        return out
    T, W = h.shape
    n = mu.shape[0]
    out = torch.empty(n, T, W, dtype=h.dtype, device=h.device)
    _native().token_shift(out.data_ptr(), _p(h), _p(mu, h.dtype, "mu"), _p(state, h.dtype, "state"),
                          _p(cu_q, I32, "cu_q"), _p(tok_seq, I32, "tok_seq"), _p(seq_slots, I32, "seq_slots"),
                          _p(positions, I32, "positions"), n, T, W, int(save), _f32(h.dtype), -1)
    return out


def shift_save(state: torch.Tensor, h: torch.Tensor, cu_q: torch.Tensor, seq_slots: torch.Tensor,
               positions: torch.Tensor) -> None:
    """state[slot of s] = h[last token of sequence s]: the save of :func:`token_shift` as a launch of its own."""
    if not _gpu(h, state):
        return ref.shift_save(state, h, cu_q, seq_slots, positions)
    _native().shift_save(_p(state, h.dtype, "state"), _p(h), _p(cu_q, I32), _p(seq_slots, I32), _p(positions, I32),
                         cu_q.shape[0] - 1, h.shape[1], _f32(h.dtype), -1)


def wkv_max_dim() -> int:
    return 128


def _env_int(name: str) -> Optional[int]:
    return int(os.environ[name]) if name in os.environ else None


WKV_CHUNK = _env_int("K8S_WKV_CHUNK")            # set: chunks of that many tokens (0: none, every sequence is walked)
WKV_CHUNK_MIN = _env_int("K8S_WKV_CHUNK_MIN")    # set: chunks from that many tokens on


def wkv_chunk(T: int, nseq: int, H: int) -> int:
    """Tokens of a chunk where the recurrence runs as three passes over chunks (parallel over them), 0 where a workgroup walks
    each sequence alone.  The walk takes 1.4 us a token of the longest sequence, the passes about 20 us and more with the
    batch: (heads of 64) one sequence of 32 tokens 48 / 22 us, 8 of 32 49 / 37 us.  Chunks from 32 tokens a sequence on, the
    average standing for the longest, which is not known here, and from 256 tokens on whatever the sequences (one long one
    beside many short ones is the costly case; 16 of 32 alone would walk faster, 52 / 65 us, 16 of 64 102 / 91 us).  Below
    256 rows decoding walks.  Chunks of 64, of 32 while those would leave CUs without two workgroups (512 tokens of 32 heads:
    46 / 56 us; 2048: 109 / 78 us)."""
    if T < (min(256, 32 * nseq) if WKV_CHUNK_MIN is None else WKV_CHUNK_MIN):
        return 0
    if WKV_CHUNK is not None:
        return max(0, WKV_CHUNK)
    return 64 if (-(-T // 64) + nseq) * H >= 512 else 32


def wkv_scan(r: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor, z: torch.Tensor, w0: torch.Tensor,
             u: torch.Tensor, lnw: torch.Tensor, state: torch.Tensor, cu_q: torch.Tensor, seq_slots: torch.Tensor,
             positions: torch.Tensor, H: int, D: int, eps: float, chunk: Optional[int] = None) -> torch.Tensor:
    """The recurrence with its per-head unit norm, norm weight and silu gate; r, k, v, g [T, H D] (one row stride),
    z [T, H D] fp32 decay logits (w = exp(-exp(z + w0))), ``state`` [slots, H, D, D] fp32 updated in place."""
    T = r.shape[0]
    if z.dtype != F32 or state.dtype != F32:
        raise TypeError("decay logits and recurrent state are fp32")
    if not _gpu(r, state):
        return ref.wkv_scan(r, k, v, g, z, w0, u, lnw, state, cu_q, seq_slots, positions, H, D, eps, r.dtype)
    if D > wkv_max_dim():
        raise ValueError(f"wkv_scan: head dimension {D} exceeds the kernel's {wkv_max_dim()}")
    ld = r.stride(0)
    for t in (r, k, v, g):
        if t.stride(0) != ld or t.stride(1) != 1 or t.dtype != r.dtype:
            raise ValueError("wkv_scan: r, k, v, g must share dtype and row stride")
    out = torch.empty(T, H * D, dtype=r.dtype, device=r.device)
    nseq = cu_q.shape[0] - 1
    Lc = wkv_chunk(T, nseq, H) if chunk is None else int(chunk)
    ws = torch.empty(_native().wkv_workspace(T, nseq, H, D, Lc), dtype=F32, device=r.device) if Lc > 0 else None
    _native().wkv_scan(out.data_ptr(), r.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(), ld, _p(z),
                       _p(w0, r.dtype, "w0"), _p(u, r.dtype, "u"), _p(lnw, r.dtype, "lnw"), _p(state),
                       _p(cu_q, I32), _p(seq_slots, I32), _p(positions, I32), nseq, H, D, float(eps),
                       _f32(r.dtype), T, Lc, _p(ws), -1)
    return out


def wkv_step(r: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor, lo: torch.Tensor, w2: torch.Tensor, w0: torch.Tensor,
             u: torch.Tensor, lnw: torch.Tensor, state: torch.Tensor, b: dict, H: int, D: int, eps: float, single: bool) -> torch.Tensor:
    """:func:`wkv_scan` with the decay logits' product z = lo @ w2.T in fp32, ``b`` a batch description; the product inside the scan's
    launch if every sequence brings a single token (``single``)."""
    if single and _gpu(r, state) and 0 < D <= wkv_max_dim() and lo.dtype == w2.dtype == r.dtype and state.dtype == F32 and \
            r.shape[0] == b["cu_q"].shape[0] - 1 and all(t.stride() == r.stride() and t.dtype == r.dtype and t.stride(1) == 1 for t in (r, k, v, g)):
        T, L = lo.shape
        out = torch.empty(T, H * D, dtype=r.dtype, device=r.device)
        if _native().wkv_step(out.data_ptr(), r.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(), r.stride(0), _p(lo), _p(w2), L,
                              _p(w0, r.dtype, "w0"), _p(u, r.dtype, "u"), _p(lnw, r.dtype, "lnw"), _p(state), _p(b["cu_q"], I32),
                              _p(b["seq_slots"], I32), _p(b["positions"], I32), T, H, D, float(eps), _f32(r.dtype), -1):
            return out
    z = linear(lo, w2, out_dtype=F32)                                      # decay logits stay fp32
    return wkv_scan(r, k, v, g, z, w0, u, lnw, state, b["cu_q"], b["seq_slots"], b["positions"], H, D, eps)


# ----------------------------------------------------------------------------- latent attention
def latent_kv_write(cache: torch.Tensor, dkv: torch.Tensor, normw: torch.Tensor, q: torch.Tensor,
                    cos_sin: torch.Tensor, positions: torch.Tensor, slot_mapping: torch.Tensor, C: int, R: int, H: int,
                    Dn: int, rot_dims: int, eps: float, interleaved: bool = False,
                    absorb: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """cache[slot] = [rms-norm(dkv[:, :C]) * normw | rotated dkv[:, C:]]; rotates the last R of every head of q
    ([T, H (Dn + R)]) in place.  ``cos_sin`` [positions, rot_dims] = [cos | sin] fp32.  The rotation pairs dimension i
    with i + rot_dims / 2, or (``interleaved``) dimension 2i with 2i + 1.  ``dkv`` [T, C + R] may be a column slice of
    a wider projection.  ``absorb``: :func:`latent_mix`'s ``uk_t``, whose product with the queries is then, for up to 64 bf16 tokens,
    part of the launch and returned for ``q_abs`` there (None: not taken)."""
    if dkv.dim() != 2 or dkv.shape[1] != C + R:
        raise ValueError("latent_kv_write: dkv must be [T, C + R]")
    if not _gpu(cache, dkv, q):
        return ref.latent_kv_write(cache, dkv, normw, q, cos_sin, positions, slot_mapping, C, R, H, Dn, rot_dims, eps,
                                   interleaved)
    dt = dkv.dtype
    if dkv.stride(1) != 1:
        raise ValueError("latent_kv_write: rows must be contiguous")
    T = dkv.shape[0]
    if absorb is not None and dt == BF16 and 0 < T <= 64 and _gpu(absorb) and absorb.shape == (H, C, Dn) and absorb.dtype == dt and \
            absorb.is_contiguous():
        q_abs = torch.empty(T, H, C, dtype=dt, device=q.device)
        if _native().latent_begin(q_abs.data_ptr(), absorb.data_ptr(), _p(cache, dt, "cache"), dkv.data_ptr(), _p(normw, dt, "normw"),
                                  _p(q, dt, "q"), _p(cos_sin, F32, "cos_sin"), _p(positions, I32), _p(slot_mapping, I32), T, C, R, H, Dn,
                                  rot_dims, float(eps), dkv.stride(0), int(bool(interleaved)), -1):
            return q_abs
    _native().latent_kv_write(_p(cache, dt, "cache"), dkv.data_ptr(), _p(normw, dt, "normw"), _p(q, dt, "q"),
                              _p(cos_sin, F32, "cos_sin"), _p(positions, I32), _p(slot_mapping, I32), dkv.shape[0], C,
                              R, H, Dn, rot_dims, float(eps), _f32(dt), dkv.stride(0), int(bool(interleaved)), -1)


LATENT_MFMA = os.environ.get("K8S_LATENT_MFMA", "1") != "0"   # 0: always the plain-FMA attention kernel


def latent_splits(T: int, H: int, max_keys: int) -> int:
    """Key splits of the MFMA latent attention: one when the (token, 16-head group) grid fills the chip by itself
    (prefill), else enough splits of at least one 32-key step each for about 256 workgroups (decoding)."""
    groups = T * ((H + 15) // 16)
    if groups >= 128:
        return 1
    return max(1, min(256 // groups, (max(1, max_keys) + 31) // 32, 32))


def latent_quad_splits(T: int, nseq: int, H: int, max_keys: int) -> int:
    """Key splits of portions of ``nseq`` sequences, ``T`` tokens in all, whose workgroups are four consecutive tokens."""
    groups = min(T, T // 4 + nseq) * ((H + 15) // 16)
    return max(1, min(256 // groups, (max(1, max_keys) + 63) // 64, 32, 65535 // nseq))       # (the grid's third side)


def latent_attention(q_abs: torch.Tensor, q: torch.Tensor, cache: torch.Tensor, block_tables: torch.Tensor,
                     tok_seq: torch.Tensor, positions: torch.Tensor, C: int, R: int, H: int, Dn: int, window: int,
                     scale: float, block_size: int, max_keys: int = 0, cu_q: Optional[torch.Tensor] = None,
                     max_qlen: int = 0, sinks: Optional[torch.Tensor] = None,
                     gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Sliding-window attention in the latent space over the paged cache; returns softmax-weighted latents [T, H, C].
    ``max_keys``: an upper bound of the keys any token sees (sizes the key splits; 0: the table's capacity).
    ``cu_q`` / ``max_qlen`` (the sequences' query offsets and longest portion): portions of prompts run four
    consecutive tokens per workgroup, sharing the staged cache rows.
    ``sinks`` [H] fp32: the softmax denominator of head h holds one more term e^sinks[h] (no key, no value).
    ``gate`` [T, H] of q's type (row stride free): head h's result is multiplied by sigmoid(gate[t, h]), which commutes
    with the value up-projection that follows.
    bf16 with 16-byte-aligned parts and fp32 of the usual sizes run on the matrix cores; other sizes on the plain-FMA kernel."""
    if sinks is not None and (sinks.dtype != F32 or sinks.numel() != H):
        raise ValueError("latent_attention: sinks are fp32 [H]")
    if gate is not None and (gate.shape != (q.shape[0], H) or gate.dtype != q.dtype or gate.stride(1) != 1):
        raise ValueError("latent_attention: the gate is [T, H] of the queries' type with contiguous rows")
    if not _gpu(q_abs, q, cache, sinks, gate):
        return ref.latent_attention(q_abs, q, cache, block_tables, tok_seq, positions, C, R, H, Dn, window, scale,
                                    block_size, q.dtype, sinks, gate)
    T = q.shape[0]
    dt = q.dtype
    out = torch.empty(T, H, C, dtype=dt, device=q.device)
    nat = _native()
    args = (_p(q_abs, dt, "q_abs"), _p(q), _p(cache, dt, "cache"), _p(block_tables, I32, "block_tables"),
            block_tables.shape[1], _p(tok_seq, I32), _p(positions, I32), T, C, R, H, Dn, int(window), float(scale),
            block_size)
    gp, ldg = (gate.data_ptr(), gate.stride(0)) if gate is not None else (0, 0)
    if LATENT_MFMA and dt == BF16 and nat.latent_mfma_ok(C, R, Dn):
        cap = block_tables.shape[1] * block_size
        bound = min(max_keys or cap, window or cap, cap)
        nseq = cu_q.shape[0] - 1 if cu_q is not None else 0
        ns = latent_quad_splits(T, nseq, H, bound) if nseq and max_qlen > 1 else latent_splits(T, H, bound)
        pacc = pml = None
        if ns > 1:
            HP = (H + 15) // 16 * 16
            pacc = torch.empty(T * HP * ns * C, dtype=F32, device=q.device)
            pml = torch.empty(T * HP * ns * 2, dtype=F32, device=q.device)
        nat.latent_attention_mfma(out.data_ptr(), _p(pacc), _p(pml), *args, ns, _p(cu_q, I32, "cu_q"), nseq,
                                  int(max_qlen), _p(sinks), gp, ldg, -1)
    else:
        nat.latent_attention(out.data_ptr(), *args, 2 if LATENT_MFMA and dt == F32 else _f32(dt), _p(sinks), gp, ldg, -1)
    return out


# A batch of prompts writes its visible keys and values out (latent_prompt.hip) when its sequences bring at least
# LATENT_EXPAND_MIN tokens on average: a portion that sees K rows then spends K C (Dn + V) multiply-adds per head on them
# instead of n C (Dn + V) on its own queries and outputs, and saves n K (2 C - Dn - V) in the attention, which breaks even
# at n = 170 for C = 512, Dn = V = 128 where everything in sight is cached already, and at any n where nothing is.  The
# average, riding single tokens included, is what the host knows (a sequence's cached length is on the device): it is safe
# for long cached parts and leaves fresh short prompts and prompts with many riders absorbed, as they ran before this form.
# 2048 tokens, 16 heads, window 1024: 383 us absorbed, 85 us written out; 512 tokens, 32 heads: 139 us and 42 us; fp32, 333
# tokens, 16 heads: 1290 us and 70 us.
LATENT_EXPAND_MIN = int(os.environ.get("K8S_LATENT_EXPAND_MIN", "160"))
LATENT_EXPAND_BYTES = 1 << 30     # of keys and values


def latent_expand(uk: torch.Tensor, uv: torch.Tensor, H: int, R: int) -> Optional[torch.Tensor]:
    """W_uk [H Dn, C] and W_uv [H V, C] as one product per latent row, [H (Dn + V), C] (per head: key rows, value rows), or
    None for sizes whose keys and values are never written out."""
    C, Dn, V = uk.shape[1], uk.shape[0] // H, uv.shape[0] // H
    if not (C % 8 == 0 and Dn == 128 and R == 64 and V == 128):
        return None
    return torch.cat([uk.view(H, Dn, C), uv.view(H, V, C)], 1).reshape(H * (Dn + V), C)


def _latent_keys(b: dict, window: int, block_size: int, cap: int) -> tuple:
    """(cache slots of the rows the batch's tokens see, first row of every sequence, row tiles, (0, rows)): made once per
    batch."""
    made = b.setdefault("latent_keys", {})
    if window not in made:
        dev, nseq = b["positions"].device, b["cu_q"].shape[0] - 1
        ntiles = cap // 64 + nseq
        rows = torch.empty(cap, dtype=I32, device=dev)
        kbase = torch.empty(nseq, dtype=I32, device=dev)
        tiles = torch.empty(ntiles, 3, dtype=I32, device=dev)
        seg = torch.empty(2, dtype=I32, device=dev)
        _native().latent_keys(rows.data_ptr(), kbase.data_ptr(), tiles.data_ptr(), seg.data_ptr(), _p(b["cu_q"], I32),
                              _p(b["positions"], I32), _p(b["block_tables"], I32), b["block_tables"].shape[1], nseq, window,
                              block_size, cap, ntiles, -1)
        made[window] = (rows, kbase, tiles, seg)
    return made[window]


def latent_mix(q: torch.Tensor, cache: torch.Tensor, uk_t: torch.Tensor, uv: torch.Tensor, ukv: Optional[torch.Tensor],
               b: dict, C: int, R: int, H: int, Dn: int, V: int, window: int, scale: float, block_size: int, *,
               sinks: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None,
               q_abs: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Latent attention with its up-projections, [T, H V]: queries q [T, H (Dn + R)] (rotated) over the batch ``b``'s cached
    rows, ``uk_t`` [H, C, Dn], ``uv`` [H, V, C], ``ukv`` from :func:`latent_expand`; ``sinks`` and ``gate`` as for
    :func:`latent_attention`.  Decoding and short portions absorb the queries (q W_uk), attend the cache as it is stored and
    take the result through W_uv (``q_abs``: the first of these, done already); batches of longer portions write the visible rows' keys and values out first."""
    T = q.shape[0]
    dt = q.dtype
    if sinks is not None and (sinks.dtype != F32 or sinks.numel() != H):
        raise ValueError("latent_mix: sinks are fp32 [H]")
    if gate is not None and (gate.shape != (T, H) or gate.dtype != dt or gate.stride(1) != 1):
        raise ValueError("latent_mix: the gate is [T, H] of the queries' type with contiguous rows")
    if q.shape != (T, H * (Dn + R)) or cache.dim() != 2 or cache.shape[1] != C + R or uv.shape != (H, V, C):
        raise ValueError("latent_mix: queries [T, H (Dn + R)], a cache of C + R columns, uv [H, V, C]")
    nseq, max_qlen = b["cu_q"].shape[0] - 1, b.get("max_qlen", 0)
    ctx = b["block_tables"].shape[1] * block_size
    cap = min(T + nseq * (window - 1), nseq * ctx) if window else nseq * ctx
    aligned = (q.data_ptr() | cache.data_ptr()) % 16 == 0          # the two newer forms move whole vectors only
    if (LATENT_MFMA and ukv is not None and _gpu(q, cache) and aligned and max_qlen > 0 and 0 < LATENT_EXPAND_MIN * nseq <= T
            and not b.get("latent_absorbed") and cap < 1 << 24 and cap * H * (Dn + V) * q.element_size() <= LATENT_EXPAND_BYTES
            and _native().latent_prompt_ok(C, R, Dn, V)):
        rows, kbase, tiles, seg = _latent_keys(b, int(window), block_size, cap)
        nat = _native()
        if ukv.shape != (H * (Dn + V), C):
            raise ValueError("latent_mix: ukv is [H (Dn + V), C]")
        _p(cache, dt, "cache"), _p(ukv, dt, "ukv")
        try:
            kv = gemm(cache[:, :C], ukv.unsqueeze(0), a_rows=rows, tiles=tiles, rows=cap, seg=seg)
        except torch.OutOfMemoryError:      # no room for the keys and values: this batch's layers run absorbed
            b["latent_absorbed"] = True
        else:
            out = torch.empty(T, H * V, dtype=dt, device=q.device)
            nat.latent_prompt(out.data_ptr(), kv.data_ptr(), rows.data_ptr(), kbase.data_ptr(), _p(q), cache.data_ptr(), C, R, Dn,
                              V, _p(b["cu_q"], I32), _p(b["positions"], I32), nseq, int(max_qlen), H, int(window), float(scale),
                              _p(sinks), gate.data_ptr() if gate is not None else 0,
                              gate.stride(0) if gate is not None else 0, _f32(dt), -1)
            return out
    if q_abs is None:
        q_abs = torch.empty(T, H, C, dtype=dt, device=q.device)
        gemm(q.view(T, H, Dn + R)[:, :, :Dn].permute(1, 0, 2), uk_t, out=q_abs.permute(1, 0, 2))
    if LATENT_MFMA and max_qlen == 0 and dt == BF16 and _gpu(q, cache, sinks, gate) and aligned and \
            uv.data_ptr() % 16 == 0 and _native().latent_token_ok(C, R, Dn, V):
        # decoding: key splits of at least one 64-key step for about one workgroup per CU, joined by the kernel that takes
        # the sums through W_uv
        HP = (H + 15) // 16 * 16
        seen = min(b.get("max_keys", 0) or ctx, window or ctx, ctx)
        ns = max(1, min(256 // (T * (HP // 16)), (seen + 63) // 64, 32))
        pacc = torch.empty(T * HP * ns * C, dtype=F32, device=q.device)
        pml = torch.empty(T * HP * ns * 2, dtype=F32, device=q.device)
        out = torch.empty(T, H * V, dtype=dt, device=q.device)
        _native().latent_token(out.data_ptr(), pacc.data_ptr(), pml.data_ptr(), q_abs.data_ptr(), _p(q),
                               _p(cache, dt, "cache"), _p(uv, dt, "uv"), _p(b["block_tables"], I32),
                               b["block_tables"].shape[1], _p(b["tok_seq"], I32), _p(b["positions"], I32), T, C, R, H, Dn, V,
                               int(window), float(scale), block_size, ns, _p(sinks),
                               gate.data_ptr() if gate is not None else 0, gate.stride(0) if gate is not None else 0, -1)
        return out
    lat = latent_attention(q_abs, q, cache, b["block_tables"], b["tok_seq"], b["positions"], C, R, H, Dn, window, scale,
                           block_size, b.get("max_keys", 0), b["cu_q"], max_qlen, sinks=sinks, gate=gate)     # [T, H, C]
    a = torch.empty(T, H, V, dtype=dt, device=q.device)
    gemm(lat.permute(1, 0, 2), uv, out=a.permute(1, 0, 2))
    return a.view(T, H * V)


# ----------------------------------------------------------------------------- mixture of experts
def moe_route(logits: torch.Tensor, E: int, top: int, scale: float, score: str = "softmax"):
    """fp32 router logits [T, >= E] -> (expert ids int32 [T, top], weights fp32 [T, top]).  ``score``: "softmax"
    (weights renormalised over the chosen experts) or "sigmoid" (the chosen experts' scores as they are)."""
    if logits.dtype != F32:
        raise TypeError("router logits are fp32")
    if score not in ("softmax", "sigmoid"):
        raise ValueError(f"moe_route: unknown score {score!r}")
    if not _gpu(logits):
        return ref.moe_route(logits, E, top, scale, score)
    T = logits.shape[0]
    idx = torch.empty(T, top, dtype=I32, device=logits.device)
    w = torch.empty(T, top, dtype=F32, device=logits.device)
    _native().moe_route(idx.data_ptr(), w.data_ptr(), _p(logits), logits.stride(0), T, E, top, float(scale),
                        int(score == "sigmoid"), -1)
    return idx, w


def moe_align(topk_idx: torch.Tensor, E: int):
    """(sorted_tok [P], pos_of_pair [P], seg [E + 1], tiles [n, 3]) for the grouped GEMMs; no host sync."""
    if not _gpu(topk_idx):
        return ref.moe_align(topk_idx, E, GROUP_BM)
    T, top = topk_idx.shape
    P = T * top
    ntiles = (P + GROUP_BM - 1) // GROUP_BM + E
    dev = topk_idx.device
    sorted_tok = torch.empty(P, dtype=I32, device=dev)
    pos = torch.empty(P, dtype=I32, device=dev)
    seg = torch.empty(E + 1, dtype=I32, device=dev)
    tiles = torch.empty(ntiles, 3, dtype=I32, device=dev)
    _native().moe_align(sorted_tok.data_ptr(), pos.data_ptr(), seg.data_ptr(), tiles.data_ptr(), ntiles,
                        _p(topk_idx, I32, "topk_idx"), P, top, E, GROUP_BM, -1)
    return sorted_tok, pos, seg, tiles


def moe_table_align(ids: torch.Tensor, tables: torch.Tensor, E: int):
    """Experts named by a table instead of a router: the choices of token t in layer l are ``tables[l, ids[t]]`` (int32
    [L, vocab, top]).  They are known with the token ids, so all layers are sorted in one launch; per layer the tuple that
    :func:`moe_align` returns."""
    L, V, top = tables.shape
    if not _gpu(ids, tables):
        rows = tables[:, ids.long().clamp(0, V - 1)]
        return [ref.moe_align(rows[l], E, GROUP_BM) for l in range(L)]
    T = ids.shape[0]
    P = T * top
    n = (P + GROUP_BM - 1) // GROUP_BM + E
    st, pos, seg, tiles = (torch.empty(L, *s, dtype=I32, device=ids.device) for s in ((P,), (P,), (E + 1,), (n, 3)))
    _native().moe_table_align(st.data_ptr(), pos.data_ptr(), seg.data_ptr(), tiles.data_ptr(), n, _p(tables, I32, "tables"),
                              _p(ids, I32, "ids"), L, T, V, top, E, GROUP_BM, -1)
    return [(st[l], pos[l], seg[l], tiles[l]) for l in range(L)]


def moe_combine(D: torch.Tensor, pos_of_pair: torch.Tensor, topk_w: Optional[torch.Tensor],
                shared: Optional[torch.Tensor], logits: Optional[torch.Tensor], sg_col: int, top: int = 0,
                scale: float = 1.0) -> torch.Tensor:
    """z[t] = sum_k w[t, k] D[pos[t, k]] + sigmoid(logits[t, sg_col]) * shared[t]  (sg_col < 0: ungated).
    ``topk_w`` None (with ``top`` given): every choice has the weight ``scale`` (1 for experts whose weight scaled their
    input)."""
    top = topk_w.shape[1] if topk_w is not None else int(top)
    if top <= 0 or pos_of_pair.numel() % top:
        raise ValueError("moe_combine: the choices per token are needed")
    if sg_col >= 0 and logits is None:
        raise ValueError("moe_combine: a gated shared expert needs the router logits")
    if not _gpu(D, topk_w, shared):
        return ref.moe_combine(D, pos_of_pair, topk_w, shared, logits, sg_col, D.dtype, top, scale)
    T = pos_of_pair.numel() // top
    W = D.shape[1]
    z = torch.empty(T, W, dtype=D.dtype, device=D.device)
    _native().moe_combine(z.data_ptr(), _p(D), _p(pos_of_pair, I32), _p(topk_w, F32), float(scale), _p(shared, D.dtype, "shared"),
                          _p(logits, F32), logits.stride(0) if logits is not None else 0, sg_col, T, W, top,
                          _f32(D.dtype), -1)
    return z


def joint_experts(E: int, W: int, F: int) -> bool:
    """Whether a shared expert of the E others' size runs as one more group of their products: sizes that the big tiles take with
    any number of rows.  Two launches less a layer, and its rows fill the other groups' rounds: us, apart / joined (8 experts, top
    2; products of a layer, weights from memory): W = F = 2048, 1 token 30.4 / 25.1, 12 58.6 / 57.0, 32 61.2 / 58.8, 97 66.5 / 58.2, 333 83.7 /
    68.0, 1531 154 / 134, 2048 188 / 177; W = 4096, F = 3584, 1 65.5 / 62.6, 4 108.5 / 110.5, 32 155 / 151, 97 168 / 151, 200 187 / 180, 333 216 /
    194, 700 251 / 256, 1024 332 / 296, 1531 406 / 409, 2048 522 / 499: at most 3 % behind, where the rows of both end in part of a round, so
    not a choice of the step's."""
    return E + 1 <= GROUP_BIG_MAX_GROUPS and W % 64 == 0 and F % 64 == 0 and W >= 128 and F >= 128


class MoeBranch(NamedTuple):
    """The experts' output ahead of its combine, for the norm that follows (:func:`branchnorm`): row t is
    sum over ``top`` choices of ``scale`` D[pos[t, k]] + sigmoid(gate[t]) * shared[t] (``gate`` fp32 [T, 1] or None: 1).  With top + 1
    columns of ``pos`` and no ``shared`` the last one names the shared expert's row of ``D``."""
    D: torch.Tensor
    pos: torch.Tensor                  # int32, T x top or T x (top + 1) values
    top: int
    scale: float
    shared: Optional[torch.Tensor] = None
    gate: Optional[torch.Tensor] = None
    tokens: int = 0

    def select(self, rows: torch.Tensor) -> "MoeBranch":
        """The branch of these tokens."""
        pick = lambda t: None if t is None else t.index_select(0, rows)
        return self._replace(pos=self.pos.view(self.tokens, -1).index_select(0, rows), shared=pick(self.shared), gate=pick(self.gate),
                             tokens=rows.numel())

    def combined(self) -> torch.Tensor:
        pos, shared = self.pos.view(self.tokens, -1), self.shared
        if pos.shape[1] > self.top:
            shared, pos = self.D.index_select(0, pos[:, self.top].long()), pos[:, :self.top].contiguous()
        return moe_combine(self.D, pos.reshape(-1), None, shared, self.gate, 0 if self.gate is not None else -1, top=self.top,
                           scale=self.scale)

    def joins(self, x: torch.Tensor, w: torch.Tensor, out_dtype, next_w, dot_w) -> bool:
        """Whether the combine can go with the norm: one type, the sizes that either would ask for (the kernel itself looks at the
        alignment)."""
        D, shared, gate, W, dt = self.D, self.shared, self.gate, x.shape[1], w.dtype
        if D.dtype != dt or D.shape[1] != W or x.shape[0] != self.tokens or out_dtype not in (None, dt) or not D.is_contiguous():
            return False
        for t in (w, next_w, dot_w):
            if t is not None and (t.numel() != W or t.dtype != dt):
                return False
        if (next_w is not None and out_dtype is None) or (dot_w is not None and next_w is None):
            return False
        if shared is not None and (shared.dtype != dt or shared.shape != x.shape or not shared.is_contiguous()):
            return False
        return gate is None or (gate.dtype == F32 and gate.numel() == self.tokens and gate.is_contiguous())


# ----------------------------------------------------------------------------- windowed attention with pooled blocks
def pool_entries_per_page(block_size: int, P: int) -> int:
    """Pooled blocks of P tokens that can start inside one cache page."""
    return -(-block_size // P) if P > 0 else 0


def window_kv_write(kcache: torch.Tensor, vcache: torch.Tensor, qkv: torch.Tensor, koff: int, voff: int,
                    qb: Optional[torch.Tensor], kb: Optional[torch.Tensor], vb: Optional[torch.Tensor],
                    cos_sin: Optional[torch.Tensor], positions: torch.Tensor, slot_mapping: torch.Tensor, H: int, G: int,
                    D: int, V: int, dims: int, eps: float, unit: bool = True, *,
                    vfirst_in: Optional[torch.Tensor] = None, vfirst_out: Optional[torch.Tensor] = None,
                    lam: float = 0.0, half_layout: bool = False, qnw: Optional[torch.Tensor] = None,
                    knw: Optional[torch.Tensor] = None, head_qnw: Optional[torch.Tensor] = None,
                    head_knw: Optional[torch.Tensor] = None) -> None:
    """Prepares a projected row [q (H D) | ... k (G D at ``koff``) ... v (G V at ``voff``) ...] of every token: biases,
    rotation of the dimension pairs (2i, 2i + 1), i < dims / 2, by ``cos_sin[pos]`` = [cos | sin] (fp32), unit RMS per
    head of q and k (``unit``), value mixing v <- (1 - lam) v + lam ``vfirst_in`` [T, G V] fp32; the first mixing layer
    leaves its v in ``vfirst_out``.  q is rewritten in place; k and v go to the paged caches [slots, G, D] / [slots, G, V].
    ``half_layout``: the rotation pairs dimension i with i + dims / 2 instead.  ``qnw`` [H D] / ``knw`` [G D]: before the
    rotation the whole projection (all heads at once) is divided by its root mean square and multiplied by the weight.
    ``head_qnw`` / ``head_knw`` [D]: before the rotation every head is divided by its own root mean square and
    multiplied by the weight, which all heads share.
    ``kcache`` None (a layer that attends another layer's cache): only the queries are prepared."""
    dt = qkv.dtype
    if kcache is None:
        vcache, G, koff, voff = None, 0, 0, 0
    if qkv.dim() != 2 or qkv.stride(1) != 1:
        raise ValueError("window_kv_write: the projected rows must be contiguous")
    if koff + G * D > qkv.shape[1] or voff + G * V > qkv.shape[1] or H * D > qkv.shape[1]:
        raise ValueError("window_kv_write: part offsets exceed the projected row")
    if not _gpu(kcache, vcache, qkv):
        return ref.window_kv_write(kcache, vcache, qkv, koff, voff, qb, kb, vb, cos_sin, positions, slot_mapping,
                                   vfirst_in, vfirst_out, lam, H, G, D, V, dims, eps, unit, half_layout, qnw, knw,
                                   head_qnw, head_knw)
    T = qkv.shape[0]
    if cos_sin is not None and (cos_sin.shape[1] != dims or cos_sin.dtype != F32):
        raise ValueError("window_kv_write: the angle table must be fp32 [positions, dims]")
    for t in (vfirst_in, vfirst_out):
        if t is not None and (t.shape != (T, G * V) or t.dtype != F32):
            raise ValueError("window_kv_write: mixed values are fp32 [T, G V]")
    for t in (head_qnw, head_knw):
        if t is not None and t.numel() != D:
            raise ValueError("window_kv_write: per-head norm weights are [D]")
    _native().window_kv_write(_p(kcache, dt, "kcache"), _p(vcache, dt, "vcache"), qkv.data_ptr(), qkv.stride(0), koff,
                              voff, _p(qb, dt, "qb"), _p(kb, dt, "kb"), _p(vb, dt, "vb"), _p(cos_sin),
                              _p(positions, I32), _p(slot_mapping, I32), _p(vfirst_in), _p(vfirst_out), float(lam), T, H,
                              G, D, V, dims, float(eps), int(bool(unit)), int(bool(half_layout)), _p(qnw, dt, "qnw"),
                              _p(knw, dt, "knw"), _p(head_qnw, dt, "head_qnw"), _p(head_knw, dt, "head_knw"),
                              _f32(dt), -1)


def window_pool(kpool: torch.Tensor, vpool: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                block_tables: torch.Tensor, tok_seq: torch.Tensor, positions: torch.Tensor, P: int,
                block_size: int) -> None:
    """For every token of the batch that ends a block of P tokens ((pos + 1) % P == 0): the fp32 mean of the block's
    cached keys / values -> kpool / vpool [pages * ceil(block_size / P), G, D or V] (the block's entry lives with the
    page of its first token).  Call after :func:`window_kv_write` of the same batch."""
    if P <= 0:
        return
    if kpool.dtype != F32 or vpool.dtype != F32:
        raise TypeError("pooled keys / values are fp32")
    if not _gpu(kpool, vpool, kcache, vcache):
        return ref.window_pool(kpool, vpool, kcache, vcache, block_tables, tok_seq, positions, P, block_size)
    G, D, V = kcache.shape[1], kcache.shape[2], vcache.shape[2]
    _native().window_pool(_p(kpool), _p(vpool), _p(kcache), _p(vcache, kcache.dtype, "vcache"),
                          _p(block_tables, I32, "block_tables"), block_tables.shape[1], _p(tok_seq, I32),
                          _p(positions, I32), positions.shape[0], G, D, V, P, block_size, _f32(kcache.dtype), -1)


WINDOW_MFMA = os.environ.get("K8S_WINDOW_MFMA", "1") != "0"   # 0: always the plain-FMA attention kernel


def window_splits(T: int, G: int, window: int, P: int, max_pos: int, tile_rows: int) -> int:
    """Key splits of the plain windowed attention: one when the (token, key head) grid fills the chip several times over
    by itself, else enough splits of at least one tile each for about 1024 workgroups (a workgroup walks its tiles one
    after the other, so decoding wants them spread).  ``max_pos``: positions a token can have."""
    groups = T * G
    if groups >= 1024 or tile_rows <= 0:
        return 1
    keys = max_pos if window <= 0 else min(max_pos, window + (max_pos // P if P > 0 else 0))
    return max(1, min(-(-1024 // groups), -(-max(1, keys) // tile_rows), 16))


# Workgroups of the one-token kernel that run at once (its registers and 256 CUs): of 8 waves and of 4, by head size
_TOKEN_SLOTS = {64: (512, 1024), 96: (256, 768), 128: (256, 512)}


@functools.lru_cache(maxsize=4096)
def token_splits(T: int, G: int, keys: int, D: int, known: bool = True) -> int:
    """Key splits of the one-token kernel, whose workgroups have 8 waves while all of them (T x G) run at once, else 4.  Few tokens: one
    split for each 256 keys, a 32-key tile a wave, up to 256 workgroups; none for up to 1024 keys of at least 128 tokens x key heads,
    where two tiles a wave cost less than the merge's launch, and none for more than 512.  Between, by the rounds that the workgroups take,
    each as long as its waves' tiles, and the merge (two tiles); us, 1 / 2 / 3 / 4 splits: 40 tokens of 4 key heads of 128
    behind 4000 88 / 84 / 72 / 76, 56 of them 94 / 97 / 98 / 99, 80 142 / 150 / 124 / 130; of 64 dimensions, 40 57 / 47 / 39 / 46; of 96, 80 132 /
    100 / 114 / 102, behind 1000 36 / 32 / 36 / 35.  Not where ``keys`` is only what the block tables could hold (``known`` false: the
    tokens of a prompt whose query groups make no tile, 97 fresh ones 10.3 / 14.7 with three splits)."""
    n = max(1, T * G)
    if n <= 64 or n > 512 or not known or (n <= 256 and keys <= 1024):
        return 1 if n >= 128 and keys <= 1024 else max(1, min(256 // n, -(-max(1, keys) // 256), 16))
    wide, narrow = _TOKEN_SLOTS[D]
    waves, slots = (8, wide) if n <= wide else (4, narrow)
    tiles = -(-max(1, keys) // 32)

    def cost(s: int) -> int:
        return -(-n * s // slots) * -(-tiles // (s * waves)) + (2 if s > 1 else 0)

    return min(range(1, max(1, min(4, -(-tiles // waves))) + 1), key=cost)


def prompt_splits(groups: int, keys: int) -> int:
    """Key splits of the prompt kernel's ``groups`` workgroups: up to 256 of them (128, 512 fresh tokens: 1 20.0, 2 22.6, 4 22.6), of
    two 64-key steps at least, at most 6 (28 workgroups, 97 tokens behind 1000: 1 split 32.7 us, 2 24.5, 4 18.7, 6 17.3, 8 16.6; 52, 200
    tokens: 4 22.2, 6 25.4).  65 - 170 workgroups that may see more than 2048 keys: up to 512, as many as run at once (76, 300 tokens
    behind 4000: 1 split 107, 3 51.3, 6 42.9; behind 1000 40.1, 27.5, 26.9; 152: 1 108, 3 69.6, behind 1000 42.4, 36.7; 128, 500 behind
    1000: 1 44.1, 2 35.6, 4 33.6).  How many keys there are is only known on the device: 97 tokens behind none pay 3 us for the
    splits and their merge (9.7 in one piece)."""
    most = 512 if keys > 2048 and 64 < groups <= 170 else 256
    return max(1, min(most // max(1, groups), -(-max(1, keys) // 128), 6))


# fp32 portions: us of the plain-FMA kernel (a workgroup a token, key head and key split), head size and heads a key head -> (the splits'
# merge, per key of a split, whole tiles of them, and round of 512 workgroups, 1024 at 64 dimensions); of window_f32.hip, which has no
# splits, head size -> (fixed, per token of a workgroup, whose last keys it weighs token by token, per key).  Fitted to 901 batches of 2 - 97
# tokens behind 30 - 30000 (1 - 8 sequences, 1 - 16 heads a key head): rms error 12 - 26 % and 6 - 8 %.
_WINDOW_PLAIN_COST = {(64, 1): (3.1, 0.22), (64, 2): (3.3, 0.189), (64, 4): (4.1, 0.171), (64, 8): (2.8, 0.201), (64, 16): (6.2, 0.267),
                      (128, 1): (1.1, 0.386), (128, 2): (3.9, 0.302), (128, 4): (4.4, 0.272), (128, 8): (5.9, 0.259), (128, 16): (5.5, 0.471)}
_WINDOW_F32_COST = {64: (5.4, 0.536, 0.0202), 128: (6.9, 0.868, 0.0354)}


@functools.lru_cache(maxsize=4096)
def window_f32_plain(T: int, longest: int, H: int, G: int, D: int, keys: int, splits: int, tile_rows: int) -> bool:
    """Whether fp32 portions of ``T`` tokens, ``longest`` of one sequence, that see up to ``keys`` keys stay on the plain-FMA kernel and
    its ``splits``: few tokens behind many keys, since a workgroup of the other walks all of them.  Plain / window_f32.hip, us, 16 heads
    over 4 of 128: 2 tokens behind 250 19.8 / 17.3, 1000 33 / 41, 3000 59 / 104, 30000 471 / 1093; 8 behind 3000 70 / 106; 16 128.8 / 121.5; 24
    180 / 122; of 64, 8 behind 1000 15.6 / 26.5, 24 27.0 / 26.7; 8 heads over 8 of 64, 16 fresh tokens 12.2 / 14.7.  Within 5 % of each other
    the plain one: of the 901 two are more than 3 % slower than on it, 48 than on the other, 1.2 % from the faster one on average.  ``keys`` is
    what the launch knows; where there are fewer than it says, this is the time there was (2 behind 30 13.2 / 9.1)."""
    merge, key = _WINDOW_PLAIN_COST[D, H // G]
    fixed, token, each = _WINDOW_F32_COST[D]
    chain = -(-(-(-keys // splits)) // tile_rows) * tile_rows
    plain = (merge if splits > 1 else 0.0) + key * chain * max(1.0, T * G * splits / (1024 if D == 64 else 512))
    return plain < 1.05 * (fixed + token * min(longest, 16 * G // H) + each * keys)


def window_attention(q: torch.Tensor, gate: Optional[torch.Tensor], kcache: torch.Tensor, vcache: torch.Tensor,
                     kpool: Optional[torch.Tensor], vpool: Optional[torch.Tensor], block_tables: torch.Tensor,
                     tok_seq: torch.Tensor, positions: torch.Tensor, H: int, window: int, P: int, scale: float,
                     sink: bool, block_size: int, cu_q: Optional[torch.Tensor] = None, max_qlen: int = 0,
                     max_keys: int = 0, *, chunk: int = 0, softcap: float = 0.0, sinks: Optional[torch.Tensor] = None,
                     gate_per_head: bool = False, slopes: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Grouped-query attention over the paged caches [slots, G, D] / [slots, G, V]: the token at position p sees the
    tokens max(0, p - window + 1) .. p (``window`` <= 0: all) and, with ``P`` > 0, the pooled blocks that lie wholly
    before the window (b P + P - 1 <= p - window), all in one softmax; ``sink``: one more unit in the denominator.
    ``q`` [T, >= H D] (row stride free, the prepared queries first), ``gate`` [T, H V] (row stride free): the result is
    multiplied by sigmoid(gate); ``gate_per_head``: ``gate`` is [T, H], one number per head.  Returns [T, H V].
    ``chunk`` > 0 (instead of a window): positions are cut into chunks of that many, counted from 0, and a token sees
    the tokens of its own chunk up to itself.  ``softcap`` > 0: scores become softcap tanh(score / softcap).  ``sinks``
    [H] fp32 (with ``sink``): the extra term of head h is e^sinks[h] instead of 1.  ``slopes`` [H] fp32: slopes[h] (p - j)
    is taken off the score of the token at position j (not off the sink's; not with pooled blocks).
    ``cu_q`` / ``max_qlen`` (the sequences' query offsets and longest portion): bf16 portions of prompts whose sizes
    fit run on the matrix cores, tiles of consecutive tokens sharing the staged keys; so do bf16 tokens one by one
    (decoding, or query groups that make no tile) without pooled blocks, and fp32 portions of the usual sizes without them but few
    tokens behind many keys (:func:`window_f32_plain`); anything else on the plain-FMA kernel.  The keys of few tokens are split over
    several workgroups, but for those fp32 portions
    (``max_keys``: an upper bound of the positions any token sees, 0: the block tables' capacity)."""
    G, D, V = kcache.shape[1], kcache.shape[2], vcache.shape[2]
    if H % G:
        raise ValueError(f"window_attention: {H} query heads over {G} key heads")
    if chunk > 0 and window > 0:
        raise ValueError("window_attention: a window or chunks, not both")
    if window <= 0:
        P = 0
    if sinks is not None and (not sink or sinks.dtype != F32 or sinks.numel() != H):
        raise ValueError("window_attention: sinks are fp32 [H] and go with sink=True")
    if slopes is not None and (slopes.dtype != F32 or slopes.numel() != H or P > 0):
        raise ValueError("window_attention: slopes are fp32 [H] and do not go with pooled blocks")
    if not _gpu(q, kcache, vcache):
        return ref.window_attention(q, gate, kcache, vcache, kpool, vpool, block_tables, tok_seq, positions, H, G, D, V,
                                    window, P, scale, sink, block_size, q.dtype, chunk, softcap, sinks, gate_per_head,
                                    slopes)
    T = q.shape[0]
    dt = q.dtype
    if q.stride(1) != 1 or (gate is not None and (gate.stride(1) != 1 or gate.dtype != dt)):
        raise ValueError("window_attention: q and gate rows must be contiguous and of one dtype")
    out = torch.empty(T, H * V, dtype=dt, device=q.device)
    nat = _native()
    if (WINDOW_MFMA and dt == BF16 and cu_q is not None and max_qlen > 1 and nat.window_mfma_ok(H, G, D, V)
            and q.stride(0) % 8 == 0 and q.data_ptr() % 16 == 0):
        tile = nat.window_prompt_tile(H, G, D, V, int(P), block_size)
        ns, pacc, pml = 1, None, None
        if tile > 0:
            max_pos = max_keys or block_tables.shape[1] * block_size
            nseq = cu_q.shape[0] - 1     # (a batch of unequal portions has fewer tiles than its launch has workgroups)
            ns = prompt_splits(G * min(-(-int(max_qlen) // tile) * nseq, T // tile + nseq),
                               min(max_pos, (chunk or window + tile) if chunk > 0 or window > 0 else max_pos))
        if ns > 1:
            pacc = torch.empty(T * H * ns * V, dtype=F32, device=q.device)
            pml = torch.empty(T * H * ns * 2, dtype=F32, device=q.device)
        nat.window_attention_mfma(out.data_ptr(), _p(pacc), _p(pml), q.data_ptr(), q.stride(0), gate.data_ptr() if gate is not None else 0,
                                  gate.stride(0) if gate is not None else 0, _p(kcache, dt, "kcache"),
                                  _p(vcache, dt, "vcache"), _p(kpool, F32, "kpool"), _p(vpool, F32, "vpool"),
                                  _p(block_tables, I32, "block_tables"), block_tables.shape[1], _p(cu_q, I32, "cu_q"),
                                  _p(positions, I32), cu_q.shape[0] - 1, int(max_qlen), T, H, G, D, V, int(window), int(P),
                                  float(scale), int(bool(sink)), block_size, ns, int(chunk), float(softcap), _p(sinks),
                                  int(bool(gate_per_head)), _p(slopes), -1)
        return out
    max_pos = max_keys or block_tables.shape[1] * block_size
    span = chunk if chunk > 0 else window
    if (WINDOW_MFMA and dt == F32 and P <= 0 and cu_q is not None and max_qlen > 1 and nat.window_f32_ok(H, G, D, V)
            and q.stride(0) % 4 == 0 and (q.data_ptr() | kcache.data_ptr() | vcache.data_ptr()) % 16 == 0 and 1 < cu_q.shape[0] <= 65536):
        rows = nat.window_tile_rows(H, G, D, V)
        plain = rows > 0 and window_f32_plain(T, int(max_qlen), H, G, D, min(max_pos, span) if span > 0 else max_pos,
                                              window_splits(T, G, span, 0, max_pos, rows), rows)
        if not plain:
            nat.window_f32(out.data_ptr(), q.data_ptr(), q.stride(0), gate.data_ptr() if gate is not None else 0,
                           gate.stride(0) if gate is not None else 0, _p(kcache, dt, "kcache"), _p(vcache, dt, "vcache"),
                           _p(block_tables, I32, "block_tables"), block_tables.shape[1], _p(cu_q, I32, "cu_q"), _p(tok_seq, I32),
                           _p(positions, I32), T, cu_q.shape[0] - 1, int(max_qlen), H, G, D, V, int(window), float(scale),
                           int(bool(sink)), block_size, int(chunk), float(softcap), _p(sinks), int(bool(gate_per_head)), _p(slopes), -1)
            return out
    if (WINDOW_MFMA and dt == BF16 and P <= 0 and nat.window_token_ok(H, G, D, V, block_size) and q.stride(0) % 8 == 0
            and q.data_ptr() % 16 == 0):
        ns = token_splits(T, G, min(max_pos, chunk or window or max_pos), D, max_keys > 0)
        pacc = pml = None
        if ns > 1:
            pacc = torch.empty(T * H * ns * V, dtype=F32, device=q.device)
            pml = torch.empty(T * H * ns * 2, dtype=F32, device=q.device)
        nat.window_token(out.data_ptr(), _p(pacc), _p(pml), q.data_ptr(), q.stride(0),
                         gate.data_ptr() if gate is not None else 0, gate.stride(0) if gate is not None else 0,
                         _p(kcache, dt, "kcache"), _p(vcache, dt, "vcache"), _p(block_tables, I32, "block_tables"),
                         block_tables.shape[1], _p(tok_seq, I32), _p(positions, I32), T, H, G, D, int(window), float(scale),
                         int(bool(sink)), block_size, ns, int(chunk), float(softcap), _p(sinks), int(bool(gate_per_head)),
                         _p(slopes), -1)
        return out
    ns = window_splits(T, G, span, P, max_pos, nat.window_tile_rows(H, G, D, V))
    pacc = pml = None
    if ns > 1:
        pacc = torch.empty(T * H * ns * V, dtype=F32, device=q.device)
        pml = torch.empty(T * H * ns * 2, dtype=F32, device=q.device)
    nat.window_attention(out.data_ptr(), _p(pacc), _p(pml), q.data_ptr(), q.stride(0),
                         gate.data_ptr() if gate is not None else 0, gate.stride(0) if gate is not None else 0,
                         _p(kcache, dt, "kcache"), _p(vcache, dt, "vcache"), _p(kpool, F32, "kpool"),
                         _p(vpool, F32, "vpool"), _p(block_tables, I32, "block_tables"), block_tables.shape[1],
                         _p(tok_seq, I32), _p(positions, I32), T, H, G, D, V, int(window), int(P), float(scale),
                         int(bool(sink)), block_size, ns, int(chunk), float(softcap), _p(sinks), int(bool(gate_per_head)),
                         _p(slopes), _f32(dt), -1)
    return out


# ----------------------------------------------------------------------------- gated matrix-state recurrences
def gated_scan_max_dim() -> int:
    return 256


def gated_scan_record(kind: int, D: int, V: int) -> int:
    """fp32 values of one (slot, head) state record: S [D, V] (SCAN_MLSTM: then n [D] and the running maximum)."""
    return ref.gated_scan_record(kind, D, V)


# Batches of at least SCAN_CHUNK_MIN tokens run the recurrences as three passes over chunks of SCAN_CHUNK tokens (parallel
# over chunks); shorter ones (decoding, short portions) as one workgroup per sequence.
SCAN_CHUNK = int(os.environ.get("K8S_SCAN_CHUNK", "64"))
SCAN_CHUNK_MIN = int(os.environ.get("K8S_SCAN_CHUNK_MIN", "256"))
# SCAN_DECAY in bf16 with a portion of at least this many tokens runs on the matrix cores (0: never)
DECAY_MFMA_MIN = int(os.environ.get("K8S_DECAY_MFMA_MIN", "32"))


def gated_scan(proj: torch.Tensor, kind: int, cols: dict, normw: torch.Tensor, state: torch.Tensor, cu_q: torch.Tensor,
               seq_slots: torch.Tensor, positions: torch.Tensor, H: int, D: int, V: int, eps: float, out_dtype, *,
               fbias: Optional[torch.Tensor] = None, ibias: Optional[torch.Tensor] = None,
               lower: Optional[torch.Tensor] = None, cap: float = 0.0, chunk: Optional[int] = None,
               aux: Optional[torch.Tensor] = None, head_params: Optional[torch.Tensor] = None,
               groups: int = 0, max_qlen: int = 0) -> torch.Tensor:
    """A gated linear recurrence with a matrix state per head over a varlen batch; ``proj`` fp32 [T, ld] is the fused
    input projection with its parts at the column offsets ``cols``; ``state`` [slots, H, record] fp32 is updated in
    place (a portion at position 0 starts from zero).  Returns the normed (and, SCAN_MLSTM, gated) outputs [T, H V].
    SCAN_HGRN2: cols q, f, v; ``lower`` [H D], ``fbias`` [H D], ``normw`` [V].
    SCAN_MLSTM: cols q, k, v, i, f, g; ``ibias`` / ``fbias`` [H], ``cap`` > 0, ``normw`` [H V].
    SCAN_SSD (a scalar decay per head and token, set by a step size): ``proj`` holds v (the heads' inputs x, H V),
    k (B) and q (C) (``groups`` D each; head h uses group h // (H / groups)); ``aux`` fp32 [T, lda] holds f (the step
    size logits, H) and g (the output gate, H V) at ``cols``; ``head_params`` fp32 [3, H] = -exp(A_log), dt_bias, skip.
    dt = softplus(f + dt_bias); S <- exp(-exp(A_log) dt) S + dt B x^T; y = (S^T C + skip x) silu(g), returned in fp32
    without a norm (``normw`` None, ``out_dtype`` fp32).
    SCAN_DECAY (linear attention under a constant decay per head): ``proj`` in fp32 or bf16 holds q, k (``groups`` D each;
    head h uses group h // (H / groups)) and v (H V) before their activation; ``head_params`` fp32 [H] are the decays.
    S <- decay S + silu(k) silu(v)^T; y = S^T silu(q), returned in fp32 without a norm.  ``max_qlen``: the longest
    portion; bf16 portions of at least DECAY_MFMA_MIN tokens whose sizes fit run on the matrix cores (decay_scan.hip),
    anything else, or with ``chunk`` given, as the other kinds do."""
    if (proj.dtype != F32 and not (kind == SCAN_DECAY and proj.dtype == BF16)) or state.dtype != F32:
        raise TypeError("the recurrence's inputs and state are fp32")
    if proj.dim() != 2 or proj.stride(1) != 1:
        raise ValueError("gated_scan: projected rows must be contiguous")
    need = {SCAN_HGRN2: ("q", "f", "v"), SCAN_MLSTM: ("q", "k", "v", "i", "f", "g"),
            SCAN_SSD: ("q", "k", "v", "f", "g"), SCAN_DECAY: ("q", "k", "v")}[kind]
    G = int(groups) if kind in (SCAN_SSD, SCAN_DECAY) else H
    width = {"q": G * D, "k": G * D, "v": H * V, "g": H * V, "i": H, "f": H * D if kind == SCAN_HGRN2 else H}
    if kind == SCAN_SSD:
        if aux is None or head_params is None or G <= 0 or H % G:
            raise ValueError("gated_scan: SCAN_SSD needs aux, head_params and groups that divide the heads")
        if aux.dtype != F32 or aux.stride(1) != 1 or aux.shape[0] != proj.shape[0]:
            raise TypeError("gated_scan: aux is fp32 [T, lda] with contiguous rows")
        if head_params.dtype != F32 or head_params.shape != (3, H) or not head_params.is_contiguous():
            raise TypeError("gated_scan: head_params is contiguous fp32 [3, H]")
        if out_dtype != F32:
            raise TypeError("gated_scan: SCAN_SSD returns fp32")
    if kind == SCAN_DECAY:
        if head_params is None or G <= 0 or H % G:
            raise ValueError("gated_scan: SCAN_DECAY needs head_params and groups that divide the heads")
        if head_params.dtype != F32 or head_params.shape != (H,) or not head_params.is_contiguous():
            raise TypeError("gated_scan: the decays are contiguous fp32 [H]")
        if out_dtype != F32:
            raise TypeError("gated_scan: SCAN_DECAY returns fp32")
    for key in need:
        src = aux if kind == SCAN_SSD and key in ("f", "g") else proj
        if cols[key] < 0 or cols[key] + width[key] > src.shape[1]:
            raise ValueError(f"gated_scan: part {key!r} exceeds the projected row")
    if state.shape[1:] != (H, gated_scan_record(kind, D, V)):
        raise ValueError("gated_scan: state must be [slots, H, record]")
    if not _gpu(proj, state):
        return ref.gated_scan(proj, kind, cols, fbias, ibias, lower, normw, state, cu_q, seq_slots, positions, H, D, V,
                              eps, cap, out_dtype, aux, head_params, G)
    if max(D, V) > gated_scan_max_dim():
        raise ValueError(f"gated_scan: head sizes {D} x {V} exceed the kernel's {gated_scan_max_dim()}")
    T = proj.shape[0]
    out = torch.empty(T, H * V, dtype=out_dtype, device=proj.device)
    c = lambda key: int(cols.get(key, 0))
    nseq = cu_q.shape[0] - 1
    if (kind == SCAN_DECAY and chunk is None and proj.dtype == BF16 and 0 < DECAY_MFMA_MIN <= max_qlen
            and _native().decay_scan_ok(D, V) and proj.data_ptr() % 16 == 0
            and not any(n % 8 for n in (proj.stride(0), c("q"), c("k"), c("v")))):
        ws = torch.empty(_native().decay_scan_workspace(T, nseq, H, D, V), dtype=torch.uint8, device=proj.device) \
            if not _native().decay_scan_once(nseq, H, V, int(max_qlen)) else None
        _native().decay_scan(out.data_ptr(), proj.data_ptr(), proj.stride(0), c("q"), c("k"), c("v"), _p(head_params),
                             _p(state), _p(cu_q, I32), _p(seq_slots, I32), _p(positions, I32), nseq, H, D, V, H // G, T,
                             int(max_qlen), _p(ws), -1)
        return out
    Lc = (SCAN_CHUNK if T >= SCAN_CHUNK_MIN else 0) if chunk is None else int(chunk)
    ws = torch.empty(_native().gated_scan_workspace(T, nseq, H, D, V, Lc), dtype=F32, device=proj.device) if Lc > 0 \
        else None
    _native().gated_scan(out.data_ptr(), proj.data_ptr(), proj.stride(0), kind, c("q"), c("k"), c("v"), c("i"), c("f"), c("g"),
                         _p(fbias, out_dtype, "fbias"), _p(ibias, out_dtype, "ibias"), _p(lower, out_dtype, "lower"),
                         _p(normw, out_dtype, "normw"), _p(state), _p(cu_q, I32), _p(seq_slots, I32),
                         _p(positions, I32), nseq, H, D, V, float(eps), float(cap),
                         _f32(proj.dtype if kind == SCAN_DECAY else out_dtype), T, Lc, _p(ws),
                         aux.data_ptr() if aux is not None else 0, aux.stride(0) if aux is not None else 0,
                         _p(head_params), H // G, -1)
    return out


# ----------------------------------------------------------------------------- short convolutions, delta rule, RG-LRU
CONV_MAX_TAPS = 16


def short_conv(x: torch.Tensor, w: torch.Tensor, state: torch.Tensor, cu_q: torch.Tensor, tok_seq: torch.Tensor,
               seq_slots: torch.Tensor, positions: torch.Tensor, *, in_bias: Optional[torch.Tensor] = None,
               out_bias: Optional[torch.Tensor] = None, act: int = CONV_NONE, unit_cols: int = 0, unit_dim: int = 0,
               scale_cols: int = 0, scale: float = 1.0, unit_eps: float = 1e-6, residual: bool = False,
               out_dtype=F32) -> torch.Tensor:
    """Causal convolution over time per channel over a varlen batch, in fp32.  ``x`` fp32 [T, C] (row stride free),
    ``w`` fp32 [C, taps] (the last tap is the current token's); inputs are x + in_bias, zeros before position 0; the
    taps - 1 inputs before a portion come from ``state`` [slots, taps - 1, C] fp32, which then receives the portion's
    last inputs (a portion at position 0 starts from zeros).  Then out_bias, the activation (CONV_SILU), and, for the
    first ``unit_cols`` channels in groups of ``unit_dim``, v / sqrt(sum(v^2) + unit_eps); the first ``scale_cols``
    channels times ``scale``.  ``residual``: the token's own input is added to the result (x + conv(x)).  Returns
    [T, C] in ``out_dtype`` (fp32, or bf16 for a result that feeds a bf16 projection)."""
    T, C = x.shape
    taps = w.shape[1]
    if x.dtype != F32 or w.dtype != F32 or state.dtype != F32 or x.stride(1) != 1:
        raise TypeError("short_conv: inputs, taps and state are fp32 with contiguous rows")
    if w.shape[0] != C or taps < 1 or taps > CONV_MAX_TAPS or state.shape[1:] != (max(taps - 1, 0), C):
        raise ValueError("short_conv: taps [C, n] and state [slots, n - 1, C] must fit the input")
    if unit_cols and (unit_dim <= 0 or unit_cols % unit_dim or unit_cols > C or unit_dim > 256):
        raise ValueError("short_conv: unit groups must tile the leading channels")
    if scale_cols > C:
        raise ValueError("short_conv: scale_cols exceeds the channels")
    if not _gpu(x, w, state):
        return ref.short_conv(x, w, state, cu_q, seq_slots, positions, in_bias, out_bias, act, unit_cols, unit_dim,
                              scale_cols, scale, unit_eps, residual).to(out_dtype)
    out = torch.empty(T, C, dtype=out_dtype, device=x.device)
    _native().short_conv(out.data_ptr(), x.data_ptr(), x.stride(0), _p(w), _p(state), _p(cu_q, I32, "cu_q"),
                         _p(tok_seq, I32, "tok_seq"), _p(seq_slots, I32, "seq_slots"), _p(positions, I32, "positions"),
                         _p(in_bias, F32, "in_bias"), _p(out_bias, F32, "out_bias"), int(act), T, C, taps,
                         cu_q.shape[0] - 1, int(unit_cols), int(unit_dim), int(scale_cols), float(scale),
                         float(unit_eps), int(bool(residual)), _f32(out_dtype), -1)
    return out


def conv_kv(x: torch.Tensor, w: torch.Tensor, state: torch.Tensor, kcache: Optional[torch.Tensor],
            vcache: Optional[torch.Tensor], slot_mapping: torch.Tensor, cu_q: torch.Tensor, tok_seq: torch.Tensor,
            seq_slots: torch.Tensor, positions: torch.Tensor, q_cols: int, *, bias: Optional[torch.Tensor] = None,
            max_qlen: int = 0) -> torch.Tensor:
    """The causal convolution of :func:`short_conv` on an attention layer's projected rows ``x`` [T, >= C] = [q (``q_cols``)
    | k | v | ...] of the activation type (row stride free): ``bias`` [C] fp32 belongs to the projection (it is part of the
    convolution's inputs), ``w`` fp32 [taps, C] (the last tap is the current token's), ``state`` [slots, taps - 1, C] fp32.
    Keys and values go to the paged caches [slots, G, D] / [slots, G, V] (None: queries only, C = q_cols); returns the
    queries [T, q_cols].  ``max_qlen``: the longest portion (1: decoding, one launch)."""
    taps, C = w.shape
    ck = kcache[0].numel() if kcache is not None else 0
    cv = vcache[0].numel() if vcache is not None else 0
    if q_cols + ck + cv != C or x.dim() != 2 or x.shape[1] < C or x.stride(1) != 1:
        raise ValueError("conv_kv: the channels must be the leading columns q | k | v of contiguous rows")
    if taps < 1 or taps > CONV_MAX_TAPS or state.shape[1:] != (taps - 1, C) or (bias is not None and bias.numel() != C):
        raise ValueError("conv_kv: taps [n, C], state [slots, n - 1, C] and bias [C] must fit the input")
    if w.dtype != F32 or state.dtype != F32 or (bias is not None and bias.dtype != F32):
        raise TypeError("conv_kv: taps, bias and state are fp32")
    if not _gpu(x, w, state, kcache, vcache, bias):
        return ref.conv_kv(x, w, state, kcache, vcache, slot_mapping, cu_q, seq_slots, positions, q_cols, bias)
    T = x.shape[0]
    dt = x.dtype
    out = torch.empty(T, q_cols, dtype=dt, device=x.device)
    _native().conv_kv(out.data_ptr(), _p(kcache, dt, "kcache"), _p(vcache, dt, "vcache"), x.data_ptr(), x.stride(0), _p(w),
                      _p(bias), _p(state), _p(cu_q, I32, "cu_q"), _p(tok_seq, I32, "tok_seq"),
                      _p(seq_slots, I32, "seq_slots"), _p(positions, I32, "positions"), _p(slot_mapping, I32, "slot_mapping"),
                      T, cu_q.shape[0] - 1, q_cols, ck, cv, taps, int(max_qlen) or T, _f32(dt), -1)
    return out


def delta_scan_max_dim() -> int:
    return 256


def delta_scan(qkv: torch.Tensor, proj: torch.Tensor, cols: dict, neg_a: torch.Tensor, dt_bias: torch.Tensor,
               normw: torch.Tensor, state: torch.Tensor, cu_q: torch.Tensor, seq_slots: torch.Tensor,
               positions: torch.Tensor, H: int, G: int, D: int, V: int, eps: float, out_dtype,
               chunk: Optional[int] = None) -> torch.Tensor:
    """The gated delta rule with a matrix state per head over a varlen batch.  ``qkv`` fp32 [T, G D | G D | H V]: the
    prepared queries (unit vectors times D^-1/2), keys (unit vectors) and values; ``proj`` fp32 [T, ld] holds the
    columns ``cols`` b (H: beta = sigmoid), a (H: decay = exp(neg_a softplus(a + dt_bias))) and g (H V: output gate,
    silu); ``neg_a`` / ``dt_bias`` / ``normw`` fp32 [H] / [H] / [V].  Per head, with the queries / keys of head
    h // (H / G): S <- decay S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q; y = o / rms(o) * normw * silu(g).
    ``state`` [slots, H, D V] fp32 is updated in place (a portion at position 0 starts from zero).  [T, H V].
    Batches of at least SCAN_CHUNK_MIN tokens run as three passes over chunks of SCAN_CHUNK tokens, parallel over chunks
    (``chunk``: another chunk length, 0: one workgroup per sequence)."""
    T = qkv.shape[0]
    for t, n in ((qkv, "qkv"), (proj, "proj"), (state, "state"), (neg_a, "neg_a"), (dt_bias, "dt_bias"),
                 (normw, "normw")):
        if t.dtype != F32:
            raise TypeError(f"delta_scan: {n} is fp32")
    if H % G or qkv.shape[1] != 2 * G * D + H * V or not qkv.is_contiguous() or proj.stride(1) != 1:
        raise ValueError("delta_scan: qkv must be contiguous [T, G D | G D | H V]")
    for key, wd in (("b", H), ("a", H), ("g", H * V)):
        if cols[key] < 0 or cols[key] + wd > proj.shape[1]:
            raise ValueError(f"delta_scan: part {key!r} exceeds the projected row")
    if state.shape[1:] != (H, D * V):
        raise ValueError("delta_scan: state must be [slots, H, D V]")
    if not _gpu(qkv, proj, state):
        return ref.delta_scan(qkv, proj, cols, neg_a, dt_bias, normw, state, cu_q, seq_slots, positions, H, G, D, V, eps,
                              out_dtype)
    if max(D, V) > delta_scan_max_dim():
        raise ValueError(f"delta_scan: head sizes {D} x {V} exceed the kernel's {delta_scan_max_dim()}")
    out = torch.empty(T, H * V, dtype=out_dtype, device=qkv.device)
    nat = _native()
    nseq = cu_q.shape[0] - 1
    Lc = (SCAN_CHUNK if T >= SCAN_CHUNK_MIN else 0) if chunk is None else int(chunk)
    if Lc > 0 and not nat.delta_scan_chunks_ok(D, V):
        Lc = 0
    ws = torch.empty(nat.delta_scan_workspace(T, nseq, H, D, V, Lc), dtype=F32, device=qkv.device) if Lc > 0 else None
    nat.delta_scan(out.data_ptr(), _p(qkv), _p(proj), proj.stride(0), int(cols["b"]), int(cols["a"]), int(cols["g"]),
                   _p(neg_a), _p(dt_bias), _p(normw), _p(state), _p(cu_q, I32), _p(seq_slots, I32), _p(positions, I32),
                   nseq, H, G, D, V, float(eps), _f32(out_dtype), T, Lc, _p(ws), -1)
    return out


def rglru_scan(u: torch.Tensor, gates: torch.Tensor, gate_bias: torch.Tensor, decay_rate: torch.Tensor,
               proj: torch.Tensor, ycol: int, ybias: torch.Tensor, state: torch.Tensor, cu_q: torch.Tensor,
               seq_slots: torch.Tensor, positions: torch.Tensor, blocks: int, out_dtype, max_qlen: int = 0
               ) -> torch.Tensor:
    """The real-gated linear recurrent unit per channel over a varlen batch.  ``u`` fp32 [T, C] (the convolved
    branch); ``gates`` fp32 [T, blocks, 2 C / blocks]: per block the logits of the recurrence gate r, then of the
    input gate i (``gate_bias`` [blocks, 2 C / blocks] added, sigmoid); a = exp(decay_rate r) with ``decay_rate``
    [C] <= 0; S <- a S + sqrt(1 - a^2) i u; out = S gelu_tanh(proj[:, ycol + c] + ybias[c]).  ``state`` [slots, C]
    fp32 is updated in place (a portion at position 0 starts from zero).  ``max_qlen``: the longest portion (long
    portions are cut into time slices that run side by side and are joined exactly)."""
    T, C = u.shape
    for t, n in ((u, "u"), (gates, "gates"), (gate_bias, "gate_bias"), (decay_rate, "decay_rate"), (proj, "proj"),
                 (ybias, "ybias"), (state, "state")):
        if t.dtype != F32:
            raise TypeError(f"rglru_scan: {n} is fp32")
    if C % blocks or gates.numel() != T * 2 * C or not gates.is_contiguous() or not u.is_contiguous():
        raise ValueError("rglru_scan: gates must be contiguous [T, blocks, 2 C / blocks]")
    if ycol < 0 or ycol + C > proj.shape[1] or proj.stride(1) != 1 or state.shape[1:] != (C,):
        raise ValueError("rglru_scan: the gate branch exceeds the projected row, or state is not [slots, C]")
    if not _gpu(u, gates, state):
        return ref.rglru_scan(u, gates, gate_bias, decay_rate, proj, ycol, ybias, state, cu_q, seq_slots, positions, C,
                              blocks, out_dtype)
    out = torch.empty(T, C, dtype=out_dtype, device=u.device)
    _native().rglru_scan(out.data_ptr(), _p(u), _p(gates), _p(gate_bias), _p(decay_rate), _p(proj), proj.stride(0),
                         int(ycol), _p(ybias), _p(state), _p(cu_q, I32), _p(seq_slots, I32), _p(positions, I32),
                         cu_q.shape[0] - 1, C, blocks, int(max_qlen or T), _f32(out_dtype), -1)
    return out
