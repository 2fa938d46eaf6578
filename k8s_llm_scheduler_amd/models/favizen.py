"""Favizen: a decoder with an fp32 residual stream whose sublayers are normed on both sides,
``x <- x + norm1b(mixer(norm1(x))); x <- x + norm2b(ff(norm2(x)))`` (RMS norms with a weight per channel), two grouped-query
attentions in any order the config lists, both with a learned sink per head (one more term ``e^sink`` in the softmax's
denominator, no key, no value) and a sigmoid output gate of one number per head:

* ``attention``: no value projection -- a head's values are its keys as projected, before the rotation; rotary positions in
  the half layout (dimension i turns with i + dims / 2) on the first ``rot.dims`` dimensions with Llama-3.1 frequency
  scaling (``rot.scaling``: factor, low, high, original); a sliding window of ``mask.size`` tokens;
* ``attention_2``: biased projections, then a short causal convolution over time on every channel of q, k and v (``conv``
  taps); no rotation, a distance bias ``2^(-8 (h + 1) / heads) (i - j)`` taken off head h's scores; a chunked mask
  (positions are cut into chunks of ``mask.size`` counted from 0, a token sees its own chunk up to itself).  With
  ``kv_from: j`` the layer has no key / value projections and attends layer j's cache with its own queries.

The feed-forward of a layer is dense, ``W_down (g sigmoid(1.702 g) (u + 1))`` with ``g = min(W_gate h, limit)``,
``u = clamp(W_up h, -limit, limit)`` and biases on all three projections, or a mixture of such experts (without biases)
that has no router: a table names every token id's experts, which share the weight equally, and a shared expert is added
times ``sigmoid(w_sg . h)``.  The embedding is scaled by ``embedding.scale``, the logits by ``logit_scale``.

Optional parts are keyed by the config or by the presence of their tensor: no mask means every earlier token, no ``rot`` no
rotation, no ``conv`` no convolution, no ``.g`` / ``.sink`` / ``.b`` tensor none of that.

The model presents the engine's interface through :class:`~.stream.StreamModel`; caches: per attention layer with
projections of its own a paged K / V cache (layers with ``kv_from`` read another layer's), per convolution and request slot
its last inputs in fp32.  Every op is a kernel of :mod:`..ops.seqmix`; ``dtype=float32`` runs everything in true fp32.
Single rank (TP = 1).
"""

from __future__ import annotations

import math
from dataclasses import dataclass, field
from pathlib import Path
from typing import Dict, List, Optional

import torch

from ..ops import reference as ref
from ..ops import seqmix as sm
from ..parallel import TPGroup
from . import stream
from .stream import StreamModel, pick_rows

ARCHITECTURE = "Favizen"
MIXERS = ("attention", "attention_2")
F32 = torch.float32
SWISH_ALPHA = 1.702


# ----------------------------------------------------------------------------- configuration
@dataclass
class AttentionConfig:
    heads: int
    kv_heads: int
    dim: int
    vdim: int
    scale: float
    window: int = 0              # tokens a position sees, itself included; 0: every earlier one
    chunk: int = 0               # chunked mask instead of a window
    rot_dims: int = 0
    rot_base: float = 10000.0
    rot_scaling: Optional[dict] = None   # {"factor", "low", "high", "original"}
    distance: bool = False       # the distance bias on the scores
    tied_values: bool = False    # the values are the unrotated keys
    bias: bool = False           # biases on the q / k / v projections
    conv: int = 0                # taps of the convolution behind the projections; 0: none
    kv_from: Optional[int] = None


@dataclass
class MlpConfig:
    kind: str                    # dense | moe
    ff: int                      # of the dense layer, or of an expert
    limit: float = 0.0           # 0 (none in the configuration): no clamp
    experts: int = 0
    top: int = 0
    shared_ff: int = 0           # 0: no shared expert
    shared_limit: float = 0.0


@dataclass
class LayerConfig:
    type: str
    mixer: AttentionConfig
    mlp: Optional[MlpConfig] = None


@dataclass
class FavizenConfig:
    name: str
    vocab: int
    hidden: int
    layers: List[LayerConfig]
    rms_eps: float = 1e-5
    embed_scale: float = 1.0
    logit_scale: float = 1.0
    max_position: int = 1 << 20
    bos_id: int = 0
    eos_ids: tuple = ()
    extra: dict = field(default_factory=dict)
    token_ids_only = True    # checkpoints of this design ship no tokenizer: requests are token ids

    @property
    def num_layers(self) -> int:
        return len(self.layers)

    def validate_tp(self, tp: int) -> None:
        if tp != 1:
            raise ValueError(f"{self.name}: this design runs on one rank (tp={tp})")


def _attention_from(kind: str, d: dict) -> AttentionConfig:
    if kind not in MIXERS:
        raise ValueError(f"unknown mixer type {kind!r} (known: {', '.join(MIXERS)})")
    rot, size = d.get("rot") or {}, int((d.get("mask") or {}).get("size") or 0)
    dim, second, kv_from = int(d["dim"]), kind == "attention_2", d.get("kv_from")
    sc = rot.get("scaling")
    return AttentionConfig(heads=int(d["heads"]), kv_heads=int(d.get("kv_heads") or d["heads"]), dim=dim,
                           vdim=int(d.get("vdim") or dim), scale=float(d.get("scale", 1.0 / math.sqrt(dim))),
                           window=0 if second else size, chunk=size if second else 0,
                           rot_dims=int(rot.get("dims") or 0), rot_base=float(rot.get("base", 10000.0)),
                           rot_scaling={k: float(sc[k]) for k in ("factor", "low", "high", "original")} if sc else None,
                           distance=second, tied_values=not second, bias=second, conv=int(d.get("conv") or 0),
                           kv_from=None if kv_from is None else int(kv_from))


def _mlp_from(d: Optional[dict]) -> Optional[MlpConfig]:
    if d is None:
        return None
    kind = d.get("kind", "dense")
    if kind == "dense":
        return MlpConfig(kind, int(d["ff"]), float(d.get("limit") or 0.0))
    if kind != "moe":
        raise ValueError(f"unknown mlp kind {kind!r}")
    e, r, s = d["expert"], d["router"], d.get("shared")
    return MlpConfig(kind, int(e["ff"]), float(e.get("limit") or 0.0), int(r["experts"]), int(r["top"]),
                     int(s["ff"]) if s else 0, float(s.get("limit") or 0.0) if s else 0.0)


def config_from_json(c: dict, name: str = "favizen") -> FavizenConfig:
    return FavizenConfig(name=name, vocab=int(c["vocab"]), hidden=int(c["width"]),
                         layers=[LayerConfig(l["type"], _attention_from(l["type"], l["mixer"]), _mlp_from(l.get("mlp")))
                                 for l in c["layers"]],
                         rms_eps=float((c.get("norm") or {}).get("eps", 1e-5)),
                         embed_scale=float((c.get("embedding") or {}).get("scale", 1.0)),
                         logit_scale=float(c.get("logit_scale", 1.0)))


def config_to_json(cfg: FavizenConfig) -> dict:
    layers = []
    ff = lambda n, limit: {"ff": n, **({"limit": limit} if limit else {})}
    for L in cfg.layers:
        a, f = L.mixer, L.mlp
        m: dict = {"heads": a.heads, "kv_heads": a.kv_heads, "dim": a.dim, "vdim": a.vdim, "scale": a.scale}
        if a.window or a.chunk:
            m["mask"] = {"size": a.window or a.chunk}
        if a.rot_dims:
            m["rot"] = {"dims": a.rot_dims, "base": a.rot_base, **({"scaling": a.rot_scaling} if a.rot_scaling else {})}
        if a.conv:
            m["conv"] = a.conv
        if a.kv_from is not None:
            m["kv_from"] = a.kv_from
        mlp = None
        if f is not None and f.kind == "dense":
            mlp = {"kind": "dense", **ff(f.ff, f.limit)}
        elif f is not None:
            mlp = {"kind": "moe", "expert": ff(f.ff, f.limit), "router": {"experts": f.experts, "top": f.top},
                   "shared": ff(f.shared_ff, f.shared_limit) if f.shared_ff else None}
        layers.append({"type": L.type, "mixer": m, "mlp": mlp})
    return {"architecture": ARCHITECTURE, "vocab": cfg.vocab, "width": cfg.hidden, "layers": layers,
            "norm": {"eps": cfg.rms_eps}, "embedding": {"scale": cfg.embed_scale}, "logit_scale": cfg.logit_scale}


def _projections(a: AttentionConfig) -> List[tuple]:
    """(name, channels) of the layer's q / k / v projections."""
    parts = [("q", a.heads * a.dim)]
    if a.kv_from is None:
        parts.append(("k", a.kv_heads * a.dim))
        if not a.tied_values:
            parts.append(("v", a.kv_heads * a.vdim))
    return parts


def tensor_shapes(cfg: FavizenConfig) -> Dict[str, tuple]:
    """Checkpoint tensor names and shapes of a configuration."""
    W = cfg.hidden
    t: Dict[str, tuple] = {"embed": (cfg.vocab, W), "final.norm": (W,), "head": (cfg.vocab, W)}
    for i, L in enumerate(cfg.layers):
        p, a, f = f"l{i}.", L.mixer, L.mlp
        t.update({p + "norm1": (W,), p + "norm1b": (W,)})
        for name, n in _projections(a):
            t[f"{p}mix.{name}"] = (n, W)
            if a.bias:
                t[f"{p}mix.{name}.b"] = (n,)
            if a.conv:
                t[f"{p}mix.{name}.conv"] = (n, a.conv)
        t.update({p + "mix.sink": (a.heads,), p + "mix.g": (a.heads, W), p + "mix.o": (W, a.heads * a.vdim)})
        if f is None:
            continue
        t.update({p + "norm2": (W,), p + "norm2b": (W,)})
        q = p + "mlp."
        if f.kind == "dense":
            t.update({q + "gate": (f.ff, W), q + "gate.b": (f.ff,), q + "up": (f.ff, W), q + "up.b": (f.ff,),
                      q + "down": (W, f.ff), q + "down.b": (W,)})
            continue
        for e in range(f.experts):
            t.update({f"{q}e{e}.gate": (f.ff, W), f"{q}e{e}.up": (f.ff, W), f"{q}e{e}.down": (W, f.ff)})
        t[q + "table"] = (cfg.vocab, f.top)
        if f.shared_ff:
            t.update({q + "shared.gate": (f.shared_ff, W), q + "shared.up": (f.shared_ff, W),
                      q + "shared.down": (W, f.shared_ff), q + "shared.sg": (1, W)})
    return t


def random_tensors(cfg: FavizenConfig, seed: int = 0, device="cpu") -> Dict[str, torch.Tensor]:
    """Random bf16 weights of a configuration (benchmarks and tests): projections ~ N(0, 1 / fan_in), norm weights around
    one, biases and sinks of order one half, convolution taps of order 1 / sqrt(taps), embedding rows that start the stream
    at unit size; the experts' tables (int32) name different experts in every row."""
    g = torch.Generator(device=device).manual_seed(seed)
    out: Dict[str, torch.Tensor] = {}
    for name, shape in tensor_shapes(cfg).items():
        leaf = name.rsplit(".", 1)[-1]
        if leaf == "table":
            E = cfg.layers[int(name[1:name.index(".")])].mlp.experts
            out[name] = torch.rand(shape[0], E, generator=g, device=device).argsort(1)[:, :shape[1]].to(torch.int32)
            continue
        t = torch.randn(shape, generator=g, device=device)
        if leaf.startswith("norm"):
            t = 1.0 + t * 0.1
        elif leaf == "embed":
            t = t / max(abs(cfg.embed_scale), 1e-6)
        elif leaf in ("b", "sink"):
            t = t * 0.5
        else:
            t = t / math.sqrt(shape[-1])
        out[name] = t.to(torch.bfloat16)
    return out


def save_checkpoint(cfg: FavizenConfig, tensors: Dict[str, torch.Tensor], path: Path) -> None:
    stream.save_checkpoint(config_to_json(cfg), tensors, path)


def preset(name: str, width: int, vocab: int, order, *, heads: int, kv_heads: int, dim: int, window: int, rot_dims: int,
           side_heads: int, side_kv_heads: int, side_dim: int, chunk: int, conv: int = 4, ff: int = 0, experts: int = 0,
           top: int = 2, expert_ff: int = 0, shared_ff: int = 0, original: int = 4096, mlps=("dense",)) -> FavizenConfig:
    """Layers in ``order``: ``attention``, ``attention_2``, or ``shared`` (an ``attention_2`` on the keys and values of the
    last one before it that has its own); feed-forwards of the kinds ``mlps`` in turn."""
    layers: List[LayerConfig] = []
    owner = None
    for i, kind in enumerate(order):
        if kind == "attention":
            a = AttentionConfig(heads, kv_heads, dim, dim, 1.0 / math.sqrt(dim), window=window, rot_dims=rot_dims,
                                rot_base=500000.0, rot_scaling={"factor": 8.0, "low": 1.0, "high": 4.0,
                                                                "original": float(original)}, tied_values=True)
        else:
            a = AttentionConfig(side_heads, side_kv_heads, side_dim, side_dim, 1.0 / math.sqrt(side_dim), chunk=chunk,
                                distance=True, bias=True, conv=conv, kv_from=owner if kind == "shared" else None)
            owner = i if kind == "attention_2" else owner
        if mlps[i % len(mlps)] == "dense":
            f = MlpConfig("dense", ff, 7.0)
        else:
            f = MlpConfig("moe", expert_ff, 7.0, experts, top, shared_ff, 5.0)
        layers.append(LayerConfig("attention" if kind == "attention" else "attention_2", a, f))
    return FavizenConfig(name, vocab, width, layers, embed_scale=math.sqrt(width), logit_scale=0.5)


PRESETS = {
    # runs on the CPU in tests: every mixer and feed-forward, a shared cache, windows and chunks shorter than the prompts
    "favizen-tiny": preset("favizen-tiny", 80, 352, ("attention", "attention_2", "shared", "attention"), heads=6, kv_heads=2,
                           dim=16, window=24, rot_dims=12, side_heads=4, side_kv_heads=2, side_dim=24, chunk=28, conv=3, ff=72,
                           experts=5, top=2, expert_ff=40, shared_ff=56, original=64, mlps=("dense", "moe")),
    # layer shapes of a ~1B-class model (benchmarks, random weights)
    "favizen-1b": preset("favizen-1b", 2048, 32768, ("attention", "attention_2", "attention", "shared") * 2, heads=16,
                         kv_heads=4, dim=128, window=1024, rot_dims=64, side_heads=16, side_kv_heads=4, side_dim=128,
                         chunk=1024, ff=8192, experts=8, expert_ff=2048, shared_ff=2048, mlps=("dense", "moe")),
}


# ----------------------------------------------------------------------------- weights
@dataclass
class _Attention:
    cfg: AttentionConfig
    w_in: torch.Tensor                     # [q (| k (| v)) (| gate), W], rows padded to a multiple of 16
    cols: Dict[str, int]                   # column of every part in the product
    o: torch.Tensor                        # [W, H V]
    cos_sin: Optional[torch.Tensor]        # [positions, rot_dims] fp32
    biases: Dict[str, torch.Tensor]        # without a convolution: q, k, v biases
    bias: Optional[torch.Tensor]           # with one: fp32 [q | k | v]
    taps: Optional[torch.Tensor]           # fp32 [taps, q | k | v]
    sinks: Optional[torch.Tensor]          # fp32 [H]
    slopes: Optional[torch.Tensor]         # fp32 [H]
    gated: bool
    cache: int = -1                        # index into kv_cache: its own, or the one of the layer it reads
    state: int = -1                        # index into states


@dataclass
class _Glu:
    limit: float
    w_gu: torch.Tensor                     # [2 F, W] (experts: [E, 2 F, W]): gate | up
    w_down: torch.Tensor                   # [W, F] (experts: [E, W, F])
    b_gu: Optional[torch.Tensor] = None
    b_down: Optional[torch.Tensor] = None


@dataclass
class _Moe:
    cfg: MlpConfig
    experts: _Glu
    shared: Optional[_Glu]
    sg: Optional[torch.Tensor]             # [W]
    route: tuple                           # (key into the stacked tables, layer in them)
    joint: Optional[_Glu] = None           # experts and the shared one in one stack (the two above are views of it)


@dataclass
class _Layer:
    n1: torch.Tensor
    n1b: torch.Tensor
    mixer: _Attention
    n2: Optional[torch.Tensor]
    n2b: Optional[torch.Tensor]
    mlp: object                            # _Glu | _Moe | None


class FavizenModel(StreamModel):
    embeds_step = True

    def __init__(self, cfg: FavizenConfig, tp: Optional[TPGroup] = None, device="cpu", dtype=torch.bfloat16,
                 seed: int = 0, weights: Optional[str] = None, tensors: Optional[Dict[str, torch.Tensor]] = None,
                 max_model_len: int = 8192, weight_dtype: str = "bf16"):
        super().__init__(cfg, tp, device, dtype, seed, max_model_len, weight_dtype)
        self._rope: Dict[tuple, torch.Tensor] = {}
        if tensors is None:
            tensors = self._open(Path(weights)) if weights else random_tensors(cfg, seed, self.device)
        get = tensors if callable(tensors) else tensors.__getitem__
        self._build(get)

    # ------------------------------------------------------------------ weights
    def _f(self, t: torch.Tensor) -> torch.Tensor:
        """Small constants that enter fp32 arithmetic are kept in fp32."""
        return t.to(F32).to(self.device).contiguous()

    @staticmethod
    def _maybe(get, name: str) -> Optional[torch.Tensor]:
        try:
            return get(name)
        except KeyError:
            return None

    def _rope_table(self, a: AttentionConfig) -> Optional[torch.Tensor]:
        if not a.rot_dims:
            return None
        sc = a.rot_scaling
        key = (a.rot_dims, a.rot_base, tuple(sorted(sc.items())) if sc else None)
        if key not in self._rope:
            scaling = {"rope_type": "llama3", "factor": sc["factor"], "low_freq_factor": sc["low"],
                       "high_freq_factor": sc["high"], "original_max_position_embeddings": sc["original"]} if sc else None
            self._rope[key] = ref.rope_table(a.rot_dims, self.max_model_len, a.rot_base,
                                             scaling).to(self.device).contiguous()
        return self._rope[key]

    def _build_attention(self, get, p: str, a: AttentionConfig, where: str) -> _Attention:
        t, maybe = self._t, lambda name: self._maybe(get, p + name)
        H, G, D, V = a.heads, a.kv_heads, a.dim, a.vdim
        if H % G:
            raise ValueError(f"{where}: {H} query heads over {G} key / value heads")
        if a.rot_dims > D or a.rot_dims % 2:
            raise ValueError(f"{where}: rot.dims {a.rot_dims} must be even and at most dim {D}")
        if a.tied_values and V != D:
            raise ValueError(f"{where}: values that are the keys have the keys' size ({V} and {D})")
        names = [n for n, _ in _projections(a)]
        rows = [get(p + n) for n in names]
        C = sum(r.shape[0] for r in rows)
        if C != sum(n for _, n in _projections(a)):
            raise ValueError(f"{where}: the projections' rows do not fit the configured heads")
        # a checkpoint settles the optional parts by the tensors it holds
        taps = [maybe(n + ".conv") for n in names]
        conv = taps[0] is not None
        if conv:
            n_taps = taps[0].shape[1]
            if any(x is None or x.shape[1] != n_taps for x in taps) or n_taps > sm.CONV_MAX_TAPS:
                raise ValueError(f"{where}: every projection needs a convolution of the same taps, at most {sm.CONV_MAX_TAPS}")
            if a.rot_dims or a.tied_values:
                raise ValueError(f"{where}: a convolution goes with unrotated keys and projected values")
        a.conv = taps[0].shape[1] if conv else 0
        b = {n: maybe(n + ".b") for n in names}
        a.bias = b["q"] is not None
        bias, biases = None, {}
        if conv and a.bias:
            bias = self._f(torch.cat([b[n] for n in names]))
        elif a.bias:
            biases = {n: t(b[n]) for n in names}
        cols, at = {}, 0
        gate = maybe("g")
        if gate is not None:
            names, rows = names + ["g"], rows + [gate]
        for n, r in zip(names, rows):
            cols[n] = at
            at += r.shape[0]
        if a.tied_values:
            cols["v"] = cols.get("k", 0)
        if at % 16:                      # 16-byte aligned output rows for the matrix-core kernels
            rows.append(torch.zeros(16 - at % 16, rows[0].shape[1], dtype=rows[0].dtype, device=rows[0].device))
        slopes = None
        if a.distance:
            slopes = self._f(torch.exp2(-8.0 * torch.arange(1, H + 1, dtype=torch.float64) / H))
        sinks = maybe("sink")
        return _Attention(a, t(torch.cat(rows)), cols, t(get(p + "o")), self._rope_table(a), biases, bias,
                          self._f(torch.cat([x.T for x in taps], 1)) if conv else None,
                          self._f(sinks) if sinks is not None else None, slopes, gate is not None)

    def _build_mlp(self, get, p: str, f: MlpConfig, where: str):
        t = self._t
        if f.kind == "dense":
            parts = [self._maybe(get, f"{p}{n}.b") for n in ("gate", "up", "down")]
            glu = _Glu(f.limit, t(torch.cat([get(p + "gate"), get(p + "up")])), t(get(p + "down")))
            if parts[0] is not None:
                glu.b_gu, glu.b_down = t(torch.cat(parts[:2])), t(parts[2])
            return glu
        E = f.experts
        if not 0 < f.top <= E:
            raise ValueError(f"{where}: {f.top} of {E} experts per token")
        stack = lambda names: torch.stack([torch.cat([get(f"{p}e{e}.{n}") for n in names]) for e in range(E)])
        gate_up, down = stack(("gate", "up")), stack(("down",))
        shared = sg = joint = None
        if f.shared_ff:
            q = p + "shared."
            s_gate_up, s_down = torch.cat([get(q + "gate"), get(q + "up")]), get(q + "down")
            sg = self._maybe(get, q + "sg")
            sg = t(sg.reshape(-1)) if sg is not None else None
        table = get(p + "table").to(torch.int32).cpu()
        if table.shape != (self.cfg.vocab, f.top) or int(table.min()) < 0 or int(table.max()) >= E:
            raise ValueError(f"{where}: the experts' table must name {f.top} of {E} experts for every token id")
        if f.shared_ff == f.ff and self.dtype == torch.bfloat16 and sm.joint_experts(E, self.cfg.hidden, f.ff):
            # a shared expert of the others' size is one more of them, which every token has
            joint = _Glu(f.limit, t(torch.cat([gate_up, s_gate_up.unsqueeze(0)])), t(torch.cat([down, s_down.unsqueeze(0)])))
            experts = _Glu(f.limit, joint.w_gu[:E], joint.w_down[:E])
            shared = _Glu(f.shared_limit, joint.w_gu[E], joint.w_down[E])
            table = torch.cat([table, torch.full((self.cfg.vocab, 1), E, dtype=torch.int32)], 1)
        else:
            experts = _Glu(f.limit, t(gate_up), t(down))
            if f.shared_ff:
                shared = _Glu(f.shared_limit, t(s_gate_up), t(s_down))
        key = (E + (joint is not None), table.shape[1])
        group = self._tables.setdefault(key, [])
        group.append(table)
        return _Moe(f, experts, shared, sg, (key, len(group) - 1), joint)

    def _build(self, get) -> None:
        c, t = self.cfg, self._t
        self.embed = t(get("embed"))
        self.final_norm = t(get("final.norm"))
        self.lm_head = t(get("head"))
        self._tables: Dict[tuple, object] = {}        # (experts, top): the layers' tables
        self._kv_owners: List[_Attention] = []
        self._convs: List[_Attention] = []
        self.layers: List[_Layer] = []
        for i, L in enumerate(c.layers):
            p, a, where = f"l{i}.", L.mixer, f"layer {i}"
            w = self._build_attention(get, p + "mix.", a, where)
            if a.kv_from is None:
                w.cache = len(self._kv_owners)
                self._kv_owners.append(w)
            else:
                j = a.kv_from
                s = self.layers[j].mixer.cfg if 0 <= j < i else None
                if s is None or s.kv_from is not None:
                    raise ValueError(f"{where}: kv_from {j} must name an earlier layer with projections of its own")
                if (s.kv_heads, s.dim, s.vdim) != (a.kv_heads, a.dim, a.vdim):
                    raise ValueError(f"{where}: head sizes differ from layer {j}'s, whose cache it reads")
                w.cache = self.layers[j].mixer.cache
            if w.taps is not None:
                w.state = len(self._convs)
                self._convs.append(w)
            n2 = n2b = mlp = None
            if L.mlp is not None:
                n2, n2b = t(get(p + "norm2")), t(get(p + "norm2b"))
                mlp = self._build_mlp(get, p + "mlp.", L.mlp, where)
            self.layers.append(_Layer(t(get(p + "norm1")), t(get(p + "norm1b")), w, n2, n2b, mlp))
        self._tables = {k: torch.stack(v).to(self.device).contiguous() for k, v in self._tables.items()}

    def _weight_roots(self) -> tuple:
        return (self.embed, self.final_norm, self.lm_head, *self.layers, *(
            o for L in self.layers for o in (L.mixer, L.mlp, getattr(L.mlp, "experts", None), getattr(L.mlp, "shared", None))
            if o is not None))

    # ------------------------------------------------------------------ cache and state
    def _needs_state(self) -> bool:
        return bool(self._convs)

    def allocate_kv(self, num_blocks: int, block_size: int):
        """Per attention layer with projections of its own: paged keys [slots, G, D] and values [slots, G, V]."""
        self.block_size = block_size
        n = num_blocks * block_size
        self.kv_cache = [(torch.zeros(n, a.cfg.kv_heads, a.cfg.dim, dtype=self.dtype, device=self.device),
                          torch.zeros(n, a.cfg.kv_heads, a.cfg.vdim, dtype=self.dtype, device=self.device))
                         for a in self._kv_owners]
        return self.kv_cache

    def kv_bytes_per_block(self, block_size: int) -> int:
        eb = torch.finfo(self.dtype).bits // 8
        return max(1, sum(block_size * a.cfg.kv_heads * (a.cfg.dim + a.cfg.vdim) * eb for a in self._kv_owners))

    def allocate_state(self, slots: int) -> None:
        """Per convolution and request slot, fp32: the last taps - 1 projected rows."""
        self.state_slots = slots
        self.states = [torch.zeros(slots, w.taps.shape[0] - 1, w.taps.shape[1], dtype=F32, device=self.device)
                       for w in self._convs]

    def state_bytes_per_slot(self) -> int:
        return sum(4 * (w.taps.shape[0] - 1) * w.taps.shape[1] for w in self._convs)

    # ------------------------------------------------------------------ layers
    def _attention(self, w: _Attention, h, b) -> torch.Tensor:
        a = w.cfg
        H, G, D, V = a.heads, a.kv_heads, a.dim, a.vdim
        kc, vc = self.kv_cache[w.cache]
        own = (kc, vc) if a.kv_from is None else (None, None)
        proj = sm.linear(h, w.w_in)                                        # [T, q (| k (| v)) (| gate)]
        if w.taps is not None:
            q = sm.conv_kv(proj, w.taps, self.states[w.state], *own, b["slot_mapping"], b["cu_q"], b["tok_seq"],
                           b["seq_slots"], b["positions"], H * D, bias=w.bias, max_qlen=b.get("max_qlen", 1))
        else:
            sm.window_kv_write(*own, proj, w.cols.get("k", 0), w.cols.get("v", 0), w.biases.get("q"), w.biases.get("k"),
                               w.biases.get("v", w.biases.get("k") if a.tied_values else None), w.cos_sin, b["positions"],
                               b["slot_mapping"], H, G, D, V, a.rot_dims, self.cfg.rms_eps, False, half_layout=True)
            q = proj
        gate = proj[:, w.cols["g"]:w.cols["g"] + H] if w.gated else None
        y = sm.window_attention(q, gate, kc, vc, None, None, b["block_tables"], b["tok_seq"], b["positions"], H, a.window, 0,
                                a.scale, w.sinks is not None, self.block_size, b["cu_q"], b.get("max_qlen", 0),
                                b.get("max_keys", 0), chunk=a.chunk, sinks=w.sinks, gate_per_head=True, slopes=w.slopes)
        return sm.linear(y, w.o)

    @staticmethod
    def _glu(w: _Glu, h) -> torch.Tensor:
        return sm.linear(sm.linear_act(h, w.w_gu, sm.ACT_SWISH_CLAMP, w.limit, SWISH_ALPHA, bias=w.b_gu), w.w_down)

    def _moe(self, w: _Moe, h, sg, b) -> sm.MoeBranch:
        f, T = w.cfg, h.shape[0]
        key, l = w.route
        sorted_tok, pos, seg, tiles = b["routes"][key][l]
        if w.joint is not None:
            kw = dict(tiles=tiles, rows=T * (f.top + 1), seg=seg, common=T)
            g = sm.gemm_act(h, w.joint.w_gu, sm.ACT_SWISH_CLAMP, f.limit, SWISH_ALPHA, a_rows=sorted_tok,
                            common_limit=f.shared_limit, **kw)
            return sm.MoeBranch(sm.gemm(g, w.joint.w_down, **kw), pos, f.top, 1.0 / f.top, None, sg, T)
        P = T * f.top
        g = sm.gemm_act(h, w.experts.w_gu, sm.ACT_SWISH_CLAMP, f.limit, SWISH_ALPHA, a_rows=sorted_tok, tiles=tiles, rows=P,
                        seg=seg)
        d = sm.gemm(g, w.experts.w_down, tiles=tiles, rows=P, seg=seg)
        shared = self._glu(w.shared, h) if w.shared is not None else None
        return sm.MoeBranch(d, pos, f.top, 1.0 / f.top, shared, sg if shared is not None else None, T)

    def _blocks(self, ids, b, after=None):
        """The residual stream before the last layer's branch is added, and that branch: (x, branch, norm weight, bias)."""
        c, dt = self.cfg, self.dtype
        x = self._embed(ids, b, c.embed_scale)
        b["routes"] = {k: sm.moe_table_align(ids, t, k[0]) for k, t in self._tables.items()}
        pend = (None, None, None)        # branch, weight of the norm on it, its bias: not yet added

        def read(next_w, dot_w=None):
            branch, w, bias = pend
            return sm.branchnorm(x, branch, w, c.rms_eps, out_dtype=dt, bias=bias, next_w=next_w, dot_w=dot_w)

        for L in self.layers:
            pend = (self._attention(L.mixer, read(L.n1), b), L.n1b, None)
            if isinstance(L.mlp, _Moe):
                h, sg = (read(L.n2), None) if L.mlp.sg is None else read(L.n2, L.mlp.sg)
                pend = (self._moe(L.mlp, h, sg, b), L.n2b, None)
            elif L.mlp is not None:
                pend = (self._glu(L.mlp, read(L.n2)), L.n2b, L.mlp.b_down)
            if after is not None:
                sm.branchnorm(x, pend[0], pend[1], c.rms_eps, bias=pend[2])
                pend = (None, None, None)
                after.append(x.clone())
        return (x, *pend)

    def _forward(self, ids, b, rows) -> torch.Tensor:
        c = self.cfg
        x, branch, w, bias = self._blocks(ids, b)
        # the logits' factor rides on the final norm
        hf = sm.branchnorm(pick_rows(x, rows), pick_rows(branch, rows), w, c.rms_eps, out_dtype=self.dtype,
                           bias=bias, next_w=self.final_norm, gain=c.logit_scale)
        return sm.linear(hf, self.lm_head, out_dtype=F32).unsqueeze(0)     # [1, S, vocab]

    def residual_after_runs(self, ids, b) -> List[torch.Tensor]:
        """(debugging / tests) the fp32 residual stream after every layer."""
        after: List[torch.Tensor] = []
        self._blocks(ids, b, after)
        return after
