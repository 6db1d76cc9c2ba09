"""Layered decoder designs: models described layer by layer in a config.json (mixer type and sizes, feed-forward, shared caches),
next to the uniform Llama stack of model.py.

A design (DESIGNS) fixes what its checkpoints do not spell out — norm placement, activation, biases, whether the attention has a
sink and an output gate —; every size and every other constant comes from the configuration, per layer.  Mixers and feed-forwards
are looked up by name (MIXERS, MLPS), so a further design adds an entry and, where it needs one, a mixer.

Designs: Bolizen (latent attention) and Tefopel (time mixing with a recurrent state, attention over tied keys and values, layers that
use another layer's weights).

Two passes share one set of weights and one cache (paged.PagedCache: pages of rows, recurrent states per slot):
  prompt pass   ragged batch of portions (each any number of tokens, from any position), packed without padding; matrix products over a
                few rows by teal_rows.hip, larger ones by the vendor library, hand-written kernels for everything between them (csrc/teal_layered.hip, teal_latent.hip,
                teal_grouped.hip, teal_wkv.hip)
  step          one token per sequence; attention over the cached rows as they are, recurrences by one token
The residual stream is fp32 throughout.  dtype fp16 / bf16 (matrix products and activations) or float32 (everything).
"""
from __future__ import annotations

import collections
import json
from dataclasses import dataclass, field
from pathlib import Path
from typing import Any, Callable, Dict, List, Optional, Sequence

import numpy as np
import torch
import torch.nn as nn

from .. import runtime
from ..kernels import layered as K
from ..monkeypatch import to_column_major
from .paged import PAGE_SHIFT, PagedCache


def pad_to(n: int, k: int) -> int:
    return -(-n // k) * k


# ------------------------------------------------------------------------------------------------
# configuration
# ------------------------------------------------------------------------------------------------
@dataclass(frozen=True)
class Design:
    """what all checkpoints of a design have in common"""
    post_norms: bool = True          # a second norm on every sublayer's output, before the residual add
    norm_offset: float = 0.0         # added to the weights of the block's and the final norms (1: they are stored around zero)
    mlp_act: str = "gelu_tanh"
    mlp_gated: bool = True           # act(gate) * up, or act(up)
    mlp_bias: bool = True
    attn_sink: bool = True
    attn_gate: bool = True
    mixers: Sequence[str] = ("latent_attention",)


DESIGNS: Dict[str, Design] = {
    "Bolizen": Design(),
    "Tefopel": Design(post_norms=False, norm_offset=1.0, mlp_act="relu2", mlp_gated=False, mlp_bias=False, attn_gate=False, mixers=("wkv", "attention")),
}


@dataclass
class LatentAttentionArgs:
    heads: int
    dim: int                         # unrotated query / key dimensions per head
    rot_dim: int                     # rotated ones (one key part shared by the heads)
    vdim: int
    kv_rank: int
    scale: float
    rope_base: float
    window: Optional[int] = None     # a query attends to the most recent `window` positions, its own included; None: to all
    kv_from: Optional[int] = None    # reads the latents another layer caches
    sink: bool = True
    gate: bool = True

    @classmethod
    def parse(cls, d: Dict[str, Any], design: Design, shape=None) -> "LatentAttentionArgs":
        rot = d["rot"]
        if int(rot["dims"]) != int(d["rot_dim"]) or int(d["rot_dim"]) % 2:
            raise ValueError(f"latent_attention rotates all of its {d['rot_dim']} shared dimensions, in pairs (rot.dims = {rot['dims']})")
        window = (d.get("mask") or {}).get("size")
        kv_from = d.get("kv_from")
        return cls(heads=int(d["heads"]), dim=int(d["dim"]), rot_dim=int(d["rot_dim"]), vdim=int(d["vdim"]), kv_rank=int(d["kv_rank"]),
                   scale=float(d["scale"]), rope_base=float(rot["base"]), window=None if window is None else int(window),
                   kv_from=None if kv_from is None else int(kv_from), sink=design.attn_sink, gate=design.attn_gate)


@dataclass
class GroupedAttentionArgs:
    """grouped-query attention whose values are the unrotated keys"""
    heads: int
    kv_heads: int
    dim: int                         # per head, keys and values
    scale: float
    rot_dims: int                    # leading dimensions of a head that turn
    rope_base: float
    softcap: Optional[float] = None  # of the scores
    window: Optional[int] = None
    sink: bool = True
    kv_from: Optional[int] = None    # (every layer has keys of its own)

    @classmethod
    def parse(cls, d: Dict[str, Any], design: Design, shape=None) -> "GroupedAttentionArgs":
        rot, window, cap = d["rot"], (d.get("mask") or {}).get("size"), d.get("softcap")
        a = cls(heads=int(d["heads"]), kv_heads=int(d["kv_heads"]), dim=int(d["dim"]), scale=float(d["scale"]), rot_dims=int(rot["dims"]),
                rope_base=float(rot["base"]), softcap=None if cap is None else float(cap), window=None if window is None else int(window), sink=design.attn_sink)
        if int(d.get("vdim", a.dim)) != a.dim:
            raise ValueError(f"attention: the values are the keys, {a.dim} dimensions per head (vdim = {d['vdim']})")
        if a.heads % a.kv_heads:
            raise ValueError(f"attention: {a.heads} query heads over {a.kv_heads} key heads")
        if a.rot_dims % 2 or not 0 <= a.rot_dims <= a.dim:
            raise ValueError(f"attention: {a.rot_dims} rotated of {a.dim} dimensions")
        return a


@dataclass
class TimeMixArgs:
    heads: int
    dim: int                         # per head: key and value channels of the state
    decay_rank: int                  # of the low-rank map that makes the decays (the checkpoint's w1 has it)
    kv_from: Optional[int] = None

    @classmethod
    def parse(cls, d: Dict[str, Any], design: Design, shape=None) -> "TimeMixArgs":
        w1 = shape("mix.w1") if shape is not None else None
        rank = w1[0] if w1 is not None else d.get("decay_rank")
        if rank is None:
            raise ValueError("wkv: the rank of the decay path is in the checkpoint's mix.w1 (or decay_rank of a synthetic configuration)")
        return cls(heads=int(d["heads"]), dim=int(d["dim"]), decay_rank=int(rank))


@dataclass
class MLPArgs:
    ff: int
    act: str = "gelu_tanh"
    bias: bool = True

    @classmethod
    def parse(cls, d: Dict[str, Any], design: Design) -> "MLPArgs":
        return cls(ff=int(d["ff"]), act=design.mlp_act, bias=design.mlp_bias)


@dataclass
class LayerArgs:
    kind: str
    mixer: Any
    mlp_kind: Optional[str] = None
    mlp: Any = None
    weights_of: Optional[int] = None  # the layer whose weights this one uses (caches and states are its own)


@dataclass
class LayeredArgs:
    architecture: str
    vocab_size: int
    dim: int
    norm_eps: float
    layers: List[LayerArgs]
    logit_softcap: Optional[float] = None
    block_size: int = 1 << 20        # positions are rotated by angle, not by table: the cache is the only limit
    design: Design = field(default_factory=Design)

    @property
    def n_layer(self) -> int:
        return len(self.layers)

    @classmethod
    def from_dict(cls, d: Dict[str, Any], shapes: Optional[Dict[str, tuple]] = None) -> "LayeredArgs":
        """d: a parsed config.json; shapes: the checkpoint's tensors (sizes that only a tensor has)"""
        arch = d.get("architecture")
        if arch not in DESIGNS:
            raise KeyError(f"no layered design named {arch!r} (known: {sorted(DESIGNS)})")
        design, layers = DESIGNS[arch], []
        sources = [cls._source(d["layers"], i) for i in range(len(d["layers"]))]
        for i, (j, ld) in enumerate(zip(sources, d["layers"])):
            if j is not None and any(ld.get(k) != d["layers"][j].get(k) for k in ("type", "mixer", "mlp")):
                raise ValueError(f"layer {i} uses the weights of layer {j}, which is described differently")
            kind, mlp = ld["type"], ld.get("mlp")
            if kind not in MIXERS or kind not in design.mixers:
                raise ValueError(f"layer {i}: unknown mixer {kind!r} for {arch}")
            if mlp is not None and mlp["kind"] not in MLPS:
                raise ValueError(f"layer {i}: unknown feed-forward {mlp['kind']!r}")
            at = f"l{i if j is None else j}."
            shape = None if shapes is None else (lambda n, at=at: shapes.get(at + n))
            layers.append(LayerArgs(kind, MIXERS[kind].args.parse(ld["mixer"], design, shape), mlp["kind"] if mlp else None,
                                    MLPArgs.parse(mlp, design) if mlp else None, j))
        for i, ly in enumerate(layers):
            j = ly.mixer.kv_from
            if j is None:
                continue
            if not 0 <= j < i or layers[j].kind != ly.kind or layers[j].mixer.kv_from is not None:
                raise ValueError(f"layer {i}: kv_from {j} must name an earlier layer with latents of its own")
            a, b = ly.mixer, layers[j].mixer
            if (a.kv_rank, a.rot_dim, a.rope_base) != (b.kv_rank, b.rot_dim, b.rope_base):
                raise ValueError(f"layer {i}: latent size and rotation differ from layer {j}'s")
        cap = d.get("logit_softcap")
        return cls(arch, int(d["vocab"]), int(d["width"]), float(d["norm"]["eps"]), layers, None if cap is None else float(cap), design=design)

    @staticmethod
    def _source(layers, i: int) -> Optional[int]:
        """the layer that holds layer i's weights, or None"""
        seen, j = {i}, layers[i].get("weights_of")
        if j is None:
            return None
        while 0 <= int(j) < len(layers) and int(j) not in seen:
            seen.add(int(j))
            if layers[int(j)].get("weights_of") is None:
                return int(j)
            j = layers[int(j)]["weights_of"]
        raise ValueError(f"layer {i}: weights_of leads to no layer with weights of its own")

    @classmethod
    def from_name(cls, name: str, n_layer: Optional[int] = None) -> "LayeredArgs":
        return cls.from_dict(named_config(name, n_layer))


# name -> sizes of a synthetic model: like the named Llama shapes of model.transformer_configs, for runs without a checkpoint.
# share: layers that read the latents of the one before them follow each owner in runs of this many (0: every layer owns its own)
layered_configs: Dict[str, Dict[str, Any]] = {
    "Bolizen-tiny-test": dict(architecture="Bolizen", n_layer=4, width=128, vocab=256, ff=384, heads=2, dim=24, rot_dim=8, vdim=40, kv_rank=64, window=48, share=1),
    "Bolizen-1B": dict(architecture="Bolizen", n_layer=16, width=2048, vocab=32000, ff=5632, heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, window=4096, share=1),
    "Bolizen-7B": dict(architecture="Bolizen", n_layer=32, width=4096, vocab=32000, ff=11008, heads=32, dim=128, rot_dim=64, vdim=128, kv_rank=512, window=4096, share=1),
    # period: a time-mixing layer (without a feed-forward) comes first in every run of this many layers; repeat: the other runs' use its weights
    "Tefopel-tiny-test": dict(architecture="Tefopel", n_layer=5, width=128, vocab=256, ff=320, heads=4, kv_heads=2, dim=32, rot=16, window=48, wkv_heads=4, wkv_dim=32, decay_rank=8,
                              period=3, repeat=True),
    "Tefopel-1B": dict(architecture="Tefopel", n_layer=24, width=2048, vocab=32000, ff=8192, heads=16, kv_heads=8, dim=128, rot=64, window=4096, wkv_heads=32, wkv_dim=64, decay_rank=64,
                       period=4, repeat=False),
    "Tefopel-7B": dict(architecture="Tefopel", n_layer=40, width=4096, vocab=32000, ff=16384, heads=32, kv_heads=16, dim=128, rot=64, window=4096, wkv_heads=64, wkv_dim=64,
                       decay_rank=64, period=4, repeat=False),
}


def is_layered_name(name: str) -> bool:
    return name in layered_configs


def named_config(name: str, n_layer: Optional[int] = None) -> Dict[str, Any]:
    """the config.json of a named synthetic model"""
    c = layered_configs[name]
    layers = []
    if c["architecture"] == "Tefopel":
        for i in range(n_layer or c["n_layer"]):
            if i % c["period"] == 0:
                ly = {"type": "wkv", "mixer": dict(heads=c["wkv_heads"], dim=c["wkv_dim"], decay_rank=c["decay_rank"]), "mlp": None}
                if c["repeat"] and i:
                    ly["weights_of"] = 0
            else:
                ly = {"type": "attention", "mlp": {"kind": "dense", "ff": c["ff"]},
                      "mixer": dict(heads=c["heads"], kv_heads=c["kv_heads"], dim=c["dim"], vdim=c["dim"], mask={"size": c["window"]}, rot={"base": 10000.0, "dims": c["rot"]},
                                    scale=c["dim"] ** -0.5, softcap=50.0)}
            layers.append(ly)
        return {"architecture": "Tefopel", "layers": layers, "norm": {"eps": 1e-6}, "vocab": c["vocab"], "width": c["width"]}
    for i in range(n_layer or c["n_layer"]):
        mixer = dict(heads=c["heads"], dim=c["dim"], rot_dim=c["rot_dim"], vdim=c["vdim"], kv_rank=c["kv_rank"], mask={"size": c["window"]},
                     rot={"base": 10000.0, "dims": c["rot_dim"]}, scale=(c["dim"] + c["rot_dim"]) ** -0.5)
        owner = i - i % (c["share"] + 1)
        if owner != i:
            mixer["kv_from"] = owner
        layers.append({"type": "latent_attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": c["ff"]}})
    return {"architecture": c["architecture"], "layers": layers, "logit_softcap": 30.0, "norm": {"eps": 1e-6}, "vocab": c["vocab"], "width": c["width"]}


# ------------------------------------------------------------------------------------------------
# the two passes' shared metadata
# ------------------------------------------------------------------------------------------------
class PromptBatch:
    """A ragged batch of prompt portions: per entry a slot, its first position and its tokens, packed back to back.

    Everything a pass reads from it on the device lies in one buffer (`dev`, contents `flat`); two batches with the same `shape` differ
    in the buffer's contents only, so a captured pass serves all of them."""

    def __init__(self, cache: PagedCache, entries, device):
        """entries: [(slot, start, tokens)]; the cache already has room for them and `sync` has run"""
        self.cache = cache
        toks, pos, row, krow, slots, run, self.spans = [], [], [], [], [], [], []
        q0 = k0 = 0
        for slot, start, tokens in entries:
            n = len(tokens)
            p = np.arange(start, start + n, dtype=np.int64)
            klo = 0 if cache.window is None else max(0, start - cache.window + 1)
            keys = np.arange(klo, start + n, dtype=np.int64)
            span = np.full(pad_to(len(keys), K.TILE), -1, dtype=np.int64)
            span[: len(keys)] = cache.rows(slot, keys)
            toks.append(np.asarray(tokens, dtype=np.int64)), pos.append(p), row.append(cache.rows(slot, p)), krow.append(span)
            slots.append(np.full(n, slot)), run.append(np.where(np.arange(n) == 0, n, 0))
            self.spans.append((q0, n, start, k0, klo))
            q0 += n
            k0 += len(span)
        self.n_tokens, self.n_keys = q0, k0
        self.flat = np.concatenate([np.concatenate(x) for x in (toks, pos, row, slots, run)] + krow + [np.asarray(self.spans).ravel()]).astype(np.int32)
        dev = torch.from_numpy(self.flat).to(device)
        self.dev, self.tokens, self.pos, self.row = dev, dev[:q0], dev[q0:2 * q0], dev[2 * q0:3 * q0]
        self.slot, self.run = dev[3 * q0:4 * q0], dev[4 * q0:5 * q0]  # per token; run: tokens of the portion on its first one, else 0
        self.key_row = dev[5 * q0:5 * q0 + k0]
        self.seqs = dev[5 * q0 + k0:].view(-1, 5)
        self.device = device
        self.tickets: Optional[torch.Tensor] = None  # counters of the running pass (LayeredTransformer._run)
        self._tiles: Dict[int, torch.Tensor] = {}
        self.packed: Dict[int, Any] = {}  # owner layer -> (latents, rotated key parts) of every key row of the batch

    @property
    def shape(self) -> tuple:
        """(tokens, first position) of every entry"""
        return tuple((n, start) for _, n, start, _, _ in self.spans)

    @property
    def longest(self) -> int:
        return max(n for _, n, _, _, _ in self.spans)

    def tiles(self, size: int) -> torch.Tensor:
        if size not in self._tiles:
            # (those with most keys before them first: they take longest)
            t = sorted(((i, q) for i, (_, n, _, _, _) in enumerate(self.spans) for q in range(0, n, size)), key=lambda t: -(self.spans[t[0]][2] + t[1]))
            self._tiles[size] = torch.tensor(t, dtype=torch.int32).to(self.device)
        return self._tiles[size]


@dataclass
class StepBatch:
    """one token per sequence; all tensors int32 on the device"""
    cache: PagedCache
    tokens: torch.Tensor
    pos: torch.Tensor
    slot: torch.Tensor
    max_pos: int                     # no position of the batch is larger (chooses how far the attention is split; not a limit)
    tickets: Optional[torch.Tensor] = None  # counters of the running pass (LayeredTransformer._run)


# ------------------------------------------------------------------------------------------------
# modules
# ------------------------------------------------------------------------------------------------
def _weight(*shape) -> nn.Parameter:
    return nn.Parameter(torch.zeros(*shape), requires_grad=False)


def padded_rows(rows: int, cols: int, lin: nn.Linear, ref: torch.Tensor) -> torch.Tensor:
    """uninitialised input rows of `lin` whose columns past `cols` are zero"""
    y = torch.empty(rows, lin.in_features, device=ref.device, dtype=ref.dtype)
    if lin.in_features > cols:
        y[:, cols:].zero_()
    return y


class LatentAttention(nn.Module):
    """Latent attention with an optional window, sink, output gate and a cache shared between layers (csrc/teal_latent.hip).

    `proj` holds the projections that read the mixer's input as one image, [q | gate | latent + shared key part], every segment
    padded with zero rows to whole 64-column tiles; `wo` reads the padded concatenation of the heads."""

    args = LatentAttentionArgs
    MAX_SPLITS = 64
    SITES = ("q", "g", "kv", "o")  # inputs of matrix products that can be masked
    from_residual = False          # takes the normed input h (True: the residual and the norm's weight)

    def __init__(self, cfg: LayeredArgs, index: int, a: LatentAttentionArgs):
        super().__init__()
        self.a, self.index, self.eps = a, index, cfg.norm_eps
        self.nq, self.nv = a.heads * (a.dim + a.rot_dim), a.heads * a.vdim
        self.g0 = pad_to(self.nq, 64)
        self.kv0 = self.g0 + (pad_to(self.nv, 64) if a.gate else 0)
        self.nkv = a.kv_rank + a.rot_dim
        n = self.kv0 + (pad_to(self.nkv, 64) if a.kv_from is None else 0)
        self.proj = nn.Linear(cfg.dim, n, bias=False)
        self.wo = nn.Linear(pad_to(self.nv, 64), cfg.dim, bias=False)
        self.uk, self.uv = _weight(a.heads * a.dim, a.kv_rank), _weight(self.nv, a.kv_rank)
        self.kv_norm = _weight(a.kv_rank) if a.kv_from is None else None
        self.sink = _weight(a.heads) if a.sink else None
        self.register_buffer("inv_freq", torch.zeros(max(1, a.rot_dim // 2)), persistent=False)

    def owner(self, index: Optional[int] = None) -> int:
        """the layer whose cache layer `index` (this mixer's own by default; another one that uses its weights) reads"""
        return self.a.kv_from if self.a.kv_from is not None else self.index if index is None else index

    @property
    def window(self) -> int:
        return K.NO_WINDOW if self.a.window is None else self.a.window

    def init_buffers(self):
        i = torch.arange(0, self.a.rot_dim, 2, dtype=torch.float64)
        self.inv_freq = (float(self.a.rope_base) ** (-i / max(1, self.a.rot_dim))).to(device=self.uk.device, dtype=torch.float32)

    def cache_width(self) -> Optional[int]:
        return pad_to(self.nkv, 32) if self.a.kv_from is None else None

    def state_shapes(self) -> Dict[str, tuple]:
        return {}

    def tensors(self, get: Callable[[str], torch.Tensor]) -> None:
        """fill from a checkpoint's tensors, by name inside the mixer"""
        a, w = self.a, self.proj.weight
        w[: self.nq] = get("q")
        if a.gate:
            w[self.g0:self.g0 + self.nv] = get("g")
        if a.kv_from is None:
            w[self.kv0:self.kv0 + self.nkv] = get("dkv")
            self.kv_norm.copy_(get("dkv.norm"))
        self.uk.copy_(get("uk"))
        self.uv.copy_(get("uv"))
        if a.sink:
            self.sink.copy_(get("sink"))
        self.wo.weight[:, : self.nv] = get("o")

    def shapes(self) -> Dict[str, tuple]:
        a, d = self.a, self.proj.in_features
        out = {"q": (self.nq, d), "uk": (a.heads * a.dim, a.kv_rank), "uv": (self.nv, a.kv_rank), "o": (d, self.nv)}
        if a.kv_from is None:
            out.update({"dkv": (self.nkv, d), "dkv.norm": (a.kv_rank,)})
        if a.sink:
            out["sink"] = (a.heads,)
        if a.gate:
            out["g"] = (self.nv, d)
        return out

    def _gate(self, proj):
        return proj[:, self.g0:self.g0 + self.nv] if self.a.gate else None

    def prompt_tile(self, b: PromptBatch) -> int:
        return K.prompt_tile(self.a.dim, self.a.rot_dim, self.a.vdim, b.longest, self.uk.dtype)

    def prompt(self, h: torch.Tensor, b: PromptBatch, index: Optional[int] = None) -> torch.Tensor:
        a, owner = self.a, self.owner(index)
        pool = b.cache.pools[owner]
        own = a.kv_from is None
        proj = K.linear(self.proj, h, b.tickets)
        K.latent_prompt_rows(proj, self.kv0 if own else -1, b.pos, b.row if own else None, self.inv_freq, self.kv_norm, self.eps, a.heads, a.dim, a.rot_dim,
                             a.kv_rank, pool if own else None)
        if own:
            b.packed[owner] = K.latent_gather(pool, b.key_row, a.kv_rank, a.rot_dim)
        c, kr = b.packed[owner]
        k, vt = torch.matmul(c, self.uk.T), torch.matmul(self.uv, c.T)
        tile = self.prompt_tile(b)
        y = K.prompt_attention(proj, k, kr, vt, self.sink, self._gate(proj), padded_rows(b.n_tokens, self.nv, self.wo, h), b.seqs, b.tiles(tile), tile, a.heads, a.dim,
                                      a.rot_dim, a.vdim, self.window, a.scale)
        return K.linear(self.wo, y, b.tickets, slabs=True)

    def splits(self, batch: int, max_pos: int, dtype: torch.dtype) -> int:
        """workgroups the cached rows of one sequence are split over: one per CU in all (of a scalar kernel two), one 32-key tile each at least.
        (Two per CU: attention and merge of 16 tokens at 1000 positions 21.4 us, one: 19.6; at 16 heads 20.1 and 16.2; 64 tokens at 250: 29.0, 28.6)"""
        groups, total = (self.a.heads, 512) if dtype == torch.float32 else (-(-self.a.heads // 16), 256)
        tiles = min(self.window, max_pos + 1) // 32 + 1
        return max(1, min(tiles, total // (batch * groups), self.MAX_SPLITS))

    def qcat_shape(self, cache: PagedCache, index: int) -> tuple:
        return self.a.heads, cache.pools[self.owner(index)].shape[-1]

    def attend(self, proj: torch.Tensor, b: StepBatch, y: Optional[torch.Tensor] = None, buffers=None, index: Optional[int] = None) -> torch.Tensor:
        """the step's attention on a computed projection: append the cache row, attend, merge -> the wo projection's input"""
        a, n, pool = self.a, proj.shape[0], b.cache.pools[self.owner(index)]
        own = a.kv_from is None
        splits = self.splits(n, b.max_pos, proj.dtype)
        if buffers is None:
            qcat = K.step_qcat(n, a.heads, pool.shape[-1], proj.dtype, proj.device)
            part = K.step_part(n, a.heads, splits, a.kv_rank, proj.device)
        else:
            qcat, part = buffers
        K.latent_step_query(proj, self.kv0 if own else -1, b.pos, b.slot, b.cache.table, PAGE_SHIFT, self.inv_freq, self.kv_norm, self.eps, self.uk, a.heads,
                            a.dim, a.rot_dim, a.kv_rank, pool, qcat)
        K.step_attention(qcat, pool, b.pos, b.slot, b.cache.table, PAGE_SHIFT, a.kv_rank, a.rot_dim, self.window, a.scale, splits, part)
        y = padded_rows(n, self.nv, self.wo, proj) if y is None else y
        return K.latent_step_merge(part, splits, self.uv, self.sink, self._gate(proj), y, n, a.heads, a.kv_rank, a.vdim)

    def step(self, h: torch.Tensor, b: StepBatch, index: Optional[int] = None) -> torch.Tensor:
        return K.linear(self.wo, self.attend(K.linear(self.proj, h, b.tickets), b, index=index), b.tickets, slabs=True)

    def linears(self):
        return [self.proj, self.wo]


class GroupedAttention(nn.Module):
    """Grouped-query attention over tied keys and values — a head's value is its key before rotation — with partial rotation, an optional
    score cap, window and sink (csrc/teal_grouped.hip; the attention kernels are those of csrc/teal_latent.hip).

    `proj` = [q | k], each padded with zero rows to whole 64-column tiles.  A cached row holds, per key head, the key and the rotated
    copy of its turning dimensions."""

    args = GroupedAttentionArgs
    MAX_SPLITS = 64
    SITES = ("q", "k", "o")
    from_residual = False

    def __init__(self, cfg: LayeredArgs, index: int, a: GroupedAttentionArgs):
        super().__init__()
        self.a, self.index = a, index
        self.nv, self.nk = a.heads * a.dim, a.kv_heads * a.dim
        self.k0 = pad_to(self.nv, 64)
        self.proj = nn.Linear(cfg.dim, self.k0 + pad_to(self.nk, 64), bias=False)
        self.wo = nn.Linear(pad_to(self.nv, 64), cfg.dim, bias=False)
        self.sink = _weight(a.heads) if a.sink else None
        self.register_buffer("inv_freq", torch.zeros(max(1, a.rot_dims // 2)), persistent=False)

    def owner(self, index: Optional[int] = None) -> int:
        return self.index if index is None else index

    @property
    def window(self) -> int:
        return K.NO_WINDOW if self.a.window is None else self.a.window

    @property
    def group(self) -> int:
        return self.a.heads // self.a.kv_heads

    @property
    def row(self) -> int:
        """elements of a key head's segment of the cached row"""
        return pad_to(self.a.dim + self.a.rot_dims, 32)

    def init_buffers(self):
        i = torch.arange(0, self.a.rot_dims, 2, dtype=torch.float64)
        self.inv_freq = (float(self.a.rope_base) ** (-i / max(1, self.a.rot_dims))).to(device=self.wo.weight.device, dtype=torch.float32)

    def cache_width(self) -> Optional[int]:
        return self.a.kv_heads * self.row

    def state_shapes(self) -> Dict[str, tuple]:
        return {}

    def tensors(self, get: Callable[[str], torch.Tensor]) -> None:
        self.proj.weight[: self.nv] = get("q")
        self.proj.weight[self.k0:self.k0 + self.nk] = get("k")
        if self.a.sink:
            self.sink.copy_(get("sink"))
        self.wo.weight[:, : self.nv] = get("o")

    def shapes(self) -> Dict[str, tuple]:
        d = self.proj.in_features
        out = {"q": (self.nv, d), "k": (self.nk, d), "o": (d, self.nv)}
        if self.a.sink:
            out["sink"] = (self.a.heads,)
        return out

    def prompt_tile(self, b: PromptBatch) -> int:
        return K.prompt_tile(self.a.dim, 0, self.a.dim, b.longest, self.wo.weight.dtype)

    def prompt(self, h: torch.Tensor, b: PromptBatch, index: Optional[int] = None) -> torch.Tensor:
        a, pool = self.a, b.cache.pools[self.owner(index)]
        proj = K.linear(self.proj, h, b.tickets)
        K.grouped_prompt_rows(proj, self.k0, b.pos, b.row, self.inv_freq, a.heads, a.kv_heads, a.dim, a.rot_dims, pool)
        k, vt = K.grouped_gather(pool, b.key_row, a.kv_heads, a.dim, a.rot_dims)
        tile = self.prompt_tile(b)
        y = K.prompt_attention(proj, k, None, vt, self.sink, None, padded_rows(b.n_tokens, self.nv, self.wo, h), b.seqs, b.tiles(tile), tile, a.heads, a.dim, 0, a.dim,
                               self.window, a.scale, self.group, a.softcap)
        return K.linear(self.wo, y, b.tickets, slabs=True)

    def splits(self, batch: int, max_pos: int, dtype: torch.dtype) -> int:
        groups = self.a.heads if dtype == torch.float32 else self.a.kv_heads * -(-self.group // 16)
        tiles = min(self.window, max_pos + 1) // 32 + 1
        return max(1, min(tiles, 512 // (batch * groups), self.MAX_SPLITS))

    def qcat_shape(self, cache: PagedCache, index: int) -> tuple:
        return self.a.heads, self.row

    def attend(self, proj: torch.Tensor, b: StepBatch, y: Optional[torch.Tensor] = None, buffers=None, index: Optional[int] = None) -> torch.Tensor:
        """the step's attention on a computed projection: append the cache row, attend, merge -> the wo projection's input"""
        a, n, pool = self.a, proj.shape[0], b.cache.pools[self.owner(index)]
        splits = self.splits(n, b.max_pos, proj.dtype)
        if buffers is None:
            qcat = K.step_qcat(n, a.heads, self.row, proj.dtype, proj.device)
            part = K.step_part(n, a.heads, splits, a.dim, proj.device)
        else:
            qcat, part = buffers
        K.grouped_step_attention(proj, self.k0, b.pos, b.slot, b.cache.table, PAGE_SHIFT, self.inv_freq, a.heads, a.kv_heads, a.dim, a.rot_dims, pool, self.window, a.scale,
                                 a.softcap, splits, qcat, part)
        y = padded_rows(n, self.nv, self.wo, proj) if y is None else y
        return K.grouped_step_merge(part, splits, self.sink, y, n, a.heads, a.dim)

    def step(self, h: torch.Tensor, b: StepBatch, index: Optional[int] = None) -> torch.Tensor:
        return K.linear(self.wo, self.attend(K.linear(self.proj, h, b.tickets), b, index=index), b.tickets, slabs=True)

    def linears(self):
        return [self.proj, self.wo]


class TimeMix(nn.Module):
    """Time mixing with a decaying matrix state per head (csrc/teal_wkv.hip).  Works on the fp32 residual: the token shift comes between
    the norm and the first rounding.

    `proj` = [r | k | v | g | w1], each padded with zero rows to whole 64-column tiles; every segment reads a mix of its own."""

    args = TimeMixArgs
    SITES = ("rkvg", "w", "o")
    MIXES = ("r", "k", "v", "g", "w")
    from_residual = True

    def __init__(self, cfg: LayeredArgs, index: int, a: TimeMixArgs):
        super().__init__()
        if a.dim > 256:
            raise ValueError(f"wkv: {a.dim} channels per head (at most 256)")
        self.a, self.index, self.eps, self.norm_offset = a, index, cfg.norm_eps, cfg.design.norm_offset
        self.nv = a.heads * a.dim
        self.seg = pad_to(self.nv, 64)
        self.proj = nn.Linear(cfg.dim, 4 * self.seg + pad_to(a.decay_rank, 64), bias=False)
        self.wo = nn.Linear(self.seg, cfg.dim, bias=False)
        self.mu = _weight(5, cfg.dim)
        self.w2, self.w0 = _weight(self.nv, a.decay_rank), _weight(self.nv)
        self.u, self.norm = _weight(a.heads, a.dim), _weight(self.nv)
        self.mixed = nn.Identity()  # (what the projections read passes through here: calibration hooks)

    def owner(self, index: Optional[int] = None) -> int:
        return self.index if index is None else index

    def init_buffers(self):
        pass

    def cache_width(self) -> Optional[int]:
        return None

    def state_shapes(self) -> Dict[str, tuple]:
        a = self.a
        return {"shift": (2, self.proj.in_features), "wkv": (2, a.heads, a.dim, a.dim)}

    def tensors(self, get: Callable[[str], torch.Tensor]) -> None:
        w = self.proj.weight
        for i, n in enumerate(self.MIXES):
            self.mu[i] = get("mu." + n)
            t = get(n if n != "w" else "w1")
            w[i * self.seg:i * self.seg + t.shape[0]] = t
        self.w2.copy_(get("w2"))
        self.w0.copy_(get("w0"))
        self.u.copy_(get("u"))
        self.norm.copy_(get("norm"))
        self.wo.weight[:, : self.nv] = get("o")

    def shapes(self) -> Dict[str, tuple]:
        a, d = self.a, self.proj.in_features
        out = {"mu." + n: (d,) for n in self.MIXES}
        out.update({n: (self.nv, d) for n in "rkvg"})
        out.update({"w1": (a.decay_rank, d), "w2": (self.nv, a.decay_rank), "w0": (self.nv,), "u": (a.heads, a.dim), "norm": (self.nv,), "o": (d, self.nv)})
        return out

    def prompt_tile(self, b: PromptBatch) -> Optional[int]:
        return None

    def _project(self, x, norm_w, b, run, index):
        """-> r, k, v, g [rows, heads * dim], z [rows, rank]"""
        mixes = self.mixed(K.wkv_mix(x, norm_w, self.norm_offset, self.eps, self.mu, b.pos, b.slot, run, b.cache.states[self.owner(index), "shift"]))
        w, n = self.proj.weight, (self.nv,) * 4 + (self.a.decay_rank,)
        return [K.linear(None, mixes[i], b.tickets, weight=w[i * self.seg:i * self.seg + n[i]]) for i in range(5)]

    def prompt(self, x: torch.Tensor, norm_w: torch.Tensor, b: PromptBatch, index: Optional[int] = None) -> torch.Tensor:
        a = self.a
        r, k, v, g, z = self._project(x, norm_w, b, b.run, index)
        o = K.wkv_scan(r, k, v, K.wkv_decay(z, self.w2, self.w0), self.u, b.seqs, b.slot, b.cache.states[self.owner(index), "wkv"], b.longest)
        return K.linear(self.wo, K.wkv_out(o, self.norm, g, self.eps, padded_rows(b.n_tokens, self.nv, self.wo, r), a.heads, a.dim), b.tickets, slabs=True)

    def advance(self, r, k, v, g, z, b: StepBatch, y: Optional[torch.Tensor] = None, index: Optional[int] = None) -> torch.Tensor:
        """the step behind the projections -> the wo projection's input"""
        y = padded_rows(r.shape[0], self.nv, self.wo, r) if y is None else y
        return K.wkv_step(r, k, v, g, z, self.w2, self.w0, self.u, self.norm, self.eps, b.pos, b.slot, b.cache.states[self.owner(index), "wkv"], y)

    def step(self, x: torch.Tensor, norm_w: torch.Tensor, b: StepBatch, index: Optional[int] = None) -> torch.Tensor:
        return K.linear(self.wo, self.advance(*self._project(x, norm_w, b, None, index), b, index=index), b.tickets, slabs=True)

    def linears(self):
        return [self.proj, self.wo]


class GatedMLP(nn.Module):
    """down(act(gate h + b) * (up h + b)) (+ b, added by the residual kernel); gate | up as one image, both padded to whole tiles"""

    SITES = ("gate", "up", "down")

    def __init__(self, cfg: LayeredArgs, a: MLPArgs):
        super().__init__()
        self.a, self.fp = a, pad_to(a.ff, 64)
        self.gate_up = nn.Linear(cfg.dim, 2 * self.fp, bias=False)
        self.down = nn.Linear(self.fp, cfg.dim, bias=False)
        self.gate_up_bias = _weight(2 * self.fp) if a.bias else None
        self.down_bias = _weight(cfg.dim) if a.bias else None

    def tensors(self, get: Callable[[str], torch.Tensor]) -> None:
        ff, fp = self.a.ff, self.fp
        self.gate_up.weight[:ff] = get("gate")
        self.gate_up.weight[fp:fp + ff] = get("up")
        self.down.weight[:, :ff] = get("down")
        if self.a.bias:
            self.gate_up_bias[:ff] = get("gate.b")
            self.gate_up_bias[fp:fp + ff] = get("up.b")
            self.down_bias.copy_(get("down.b"))

    def shapes(self) -> Dict[str, tuple]:
        ff, d = self.a.ff, self.down.out_features
        out = {"gate": (ff, d), "up": (ff, d), "down": (d, ff)}
        if self.a.bias:
            out.update({"gate.b": (ff,), "up.b": (ff,), "down.b": (d,)})
        return out

    def forward(self, h: torch.Tensor, tickets: Optional[torch.Tensor] = None) -> torch.Tensor:
        return K.linear(self.down, K.gated_linear(self.gate_up, h, self.a.act, self.gate_up_bias, tickets), tickets, slabs=True)

    def linears(self):
        return [self.gate_up, self.down]


class PlainMLP(nn.Module):
    """down(act(up h + b)) (+ b, added by the residual kernel), padded to whole tiles"""

    SITES = ("up", "down")

    def __init__(self, cfg: LayeredArgs, a: MLPArgs):
        super().__init__()
        self.a, self.fp = a, pad_to(a.ff, 64)
        self.up = nn.Linear(cfg.dim, self.fp, bias=False)
        self.down = nn.Linear(self.fp, cfg.dim, bias=False)
        self.up_bias = _weight(self.fp) if a.bias else None
        self.down_bias = _weight(cfg.dim) if a.bias else None

    def tensors(self, get: Callable[[str], torch.Tensor]) -> None:
        self.up.weight[: self.a.ff] = get("up")
        self.down.weight[:, : self.a.ff] = get("down")
        if self.a.bias:
            self.up_bias[: self.a.ff] = get("up.b")
            self.down_bias.copy_(get("down.b"))

    def shapes(self) -> Dict[str, tuple]:
        ff, d = self.a.ff, self.down.out_features
        out = {"up": (ff, d), "down": (d, ff)}
        if self.a.bias:
            out.update({"up.b": (ff,), "down.b": (d,)})
        return out

    def forward(self, h: torch.Tensor, tickets: Optional[torch.Tensor] = None) -> torch.Tensor:
        return K.linear(self.down, K.linear(self.up, h, tickets, act=self.a.act, bias=self.up_bias), tickets, slabs=True)

    def linears(self):
        return [self.up, self.down]


MIXERS = {"latent_attention": LatentAttention, "attention": GroupedAttention, "wkv": TimeMix}
MLPS = {"dense": lambda design: GatedMLP if design.mlp_gated else PlainMLP}


class LayeredBlock(nn.Module):
    """a layer's weights; layers that use another's are the same object in LayeredTransformer.layers, at an index of their own"""

    def __init__(self, cfg: LayeredArgs, index: int):
        super().__init__()
        ly = cfg.layers[index]
        self.mix = MIXERS[ly.kind](cfg, index, ly.mixer)
        self.mlp = MLPS[ly.mlp_kind](cfg.design)(cfg, ly.mlp) if ly.mlp_kind else None
        post = cfg.design.post_norms
        self.norm1, self.norm1b = _weight(cfg.dim), _weight(cfg.dim) if post else None
        self.norm2 = _weight(cfg.dim) if self.mlp is not None else None
        self.norm2b = _weight(cfg.dim) if self.mlp is not None and post else None


class GraphedPrompt:
    """prompt passes replayed from a hipGraph per shape of the batch: a pass of a short prompt is hundreds of launches of a few
    microseconds.  A shape's first use runs eagerly (the warm-up a capture needs), its second is captured."""

    MAX_TOKENS, MAX_GRAPHS = 256, 8  # longer prompts keep the GPU busy by themselves; least recently used graphs go first

    def __init__(self, model: "LayeredTransformer"):
        self.model = model
        self._seen: set = set()
        self._graphs: "collections.OrderedDict[tuple, tuple]" = collections.OrderedDict()

    def __call__(self, b: PromptBatch, want: Sequence[int]) -> Optional[torch.Tensor]:
        key = (b.shape, tuple(want), b.cache.version, id(b.cache))
        if b.n_tokens > self.MAX_TOKENS or not len(want) or (key not in self._graphs and key not in self._seen):
            if len(self._seen) >= 1024:
                self._seen.clear()
            self._seen.add(key)
            return self.model.prompt_pass(b, want)
        if key not in self._graphs:
            rows = torch.tensor(list(want), dtype=torch.int32).to(b.device)
            for ly in self.model.layers:
                tile = ly.mix.prompt_tile(b)
                if tile is not None:
                    b.tiles(tile)  # (host-built: before the capture)
            torch.cuda.synchronize()
            while len(self._graphs) >= self.MAX_GRAPHS:
                self._graphs.popitem(last=False)
            g = torch.cuda.CUDAGraph()
            with runtime.graph_capture(g):
                logits = self.model.prompt_pass(b, rows)
            self._graphs[key] = (g, b, rows, logits)
        self._graphs.move_to_end(key)
        g, static, _, logits = self._graphs[key]
        static.dev.copy_(torch.from_numpy(b.flat))
        g.replay()
        return logits.clone()


class LayeredTransformer(nn.Module):
    def __init__(self, config: LayeredArgs):
        super().__init__()
        self.config = config
        self.tok_embeddings = nn.Embedding(config.vocab_size, config.dim)
        own = {i: LayeredBlock(config, i) for i, ly in enumerate(config.layers) if ly.weights_of is None}
        self.layers = nn.ModuleList(own[i if ly.weights_of is None else ly.weights_of] for i, ly in enumerate(config.layers))
        self.norm = _weight(config.dim)
        self.output: Optional[nn.Linear] = None  # the embedding table as the head's image (finalize)
        self.max_batch_size = self.max_seq_length = -1
        self.cache: Optional[PagedCache] = None

    def own_layers(self):
        """(index, block) of the layers that have weights of their own"""
        return [(i, b) for i, b in enumerate(self.layers) if self.config.layers[i].weights_of is None]

    # ---- weights ---------------------------------------------------------------------------------------------------
    def tensor_shapes(self) -> Dict[str, tuple]:
        """every checkpoint tensor of this configuration, by name"""
        d = self.config.dim
        out = {"embed": (self.config.vocab_size, d), "final.norm": (d,)}
        for i, b in self.own_layers():
            out.update({f"l{i}.{n}": (d,) for n in ("norm1", "norm1b", "norm2", "norm2b") if getattr(b, n) is not None})
            out.update({f"l{i}.mix.{n}": s for n, s in b.mix.shapes().items()})
            if b.mlp is not None:
                out.update({f"l{i}.mlp.{n}": s for n, s in b.mlp.shapes().items()})
        return out

    @torch.no_grad()
    def load_tensors(self, get: Callable[[str], torch.Tensor]) -> "LayeredTransformer":
        shapes = self.tensor_shapes()

        def checked(name):
            t = get(name)
            if tuple(t.shape) != shapes[name]:
                raise ValueError(f"{name}: shape {tuple(t.shape)}, the configuration needs {shapes[name]}")
            return t

        self.tok_embeddings.weight.copy_(checked("embed"))
        self.norm.copy_(checked("final.norm"))
        for i, b in self.own_layers():
            for n in ("norm1", "norm1b", "norm2", "norm2b"):
                if getattr(b, n) is not None:
                    getattr(b, n).copy_(checked(f"l{i}.{n}"))
            b.mix.tensors(lambda n, i=i: checked(f"l{i}.mix.{n}"))
            if b.mlp is not None:
                b.mlp.tensors(lambda n, i=i: checked(f"l{i}.mlp.{n}"))
        return self.finalize()

    @torch.no_grad()
    def finalize(self) -> "LayeredTransformer":
        """after the weights are in place: derived buffers, and the layout the decode kernels stream (16-bit: the transposed image of
        every projection, monkeypatch.to_column_major; the head's image is padded to whole 64-column tiles)"""
        w = self.tok_embeddings.weight
        for p in self.parameters():
            p.requires_grad_(False)
        head = nn.Linear(1, 1, bias=False)
        if w.dtype == torch.float32:
            head.weight = nn.Parameter(w.data, requires_grad=False)
        else:
            padded = torch.zeros(pad_to(w.shape[0], 64), w.shape[1], dtype=w.dtype, device=w.device)
            padded[: w.shape[0]] = w
            head.weight = nn.Parameter(padded, requires_grad=False)
            to_column_major(head)
        self.output = head
        for _, b in self.own_layers():
            b.mix.init_buffers()
            if w.dtype != torch.float32:
                for lin in b.mix.linears() + (b.mlp.linears() if b.mlp is not None else []):
                    to_column_major(lin)
        return self.eval()

    # ---- cache -----------------------------------------------------------------------------------------------------
    def new_cache(self, max_tokens: int, max_requests: int = 8) -> PagedCache:
        w = self.tok_embeddings.weight
        windows = [b.a.window for b in (ly.mix for ly in self.layers) if hasattr(b.a, "window")]
        widths = {i: b.mix.cache_width() for i, b in enumerate(self.layers) if b.mix.cache_width() is not None}
        states = {(i, n): s for i, b in enumerate(self.layers) for n, s in b.mix.state_shapes().items()}
        return PagedCache(widths, w.dtype, w.device, max_tokens, max_requests, None if None in windows else max(windows, default=1), states)

    def setup_caches(self, max_batch_size: int, max_seq_length: int):
        """model.Transformer's interface: room for max_batch_size sequences of max_seq_length positions, slots 0 .. max_batch_size - 1"""
        if self.max_seq_length >= max_seq_length and self.max_batch_size >= max_batch_size:
            return
        self.max_seq_length, self.max_batch_size = pad_to(max_seq_length, 8), max_batch_size
        self.cache = self.new_cache(max_batch_size * self.max_seq_length, max_batch_size)
        for _ in range(max_batch_size):
            self.cache.extend(self.cache.open(), self.max_seq_length)
        self.cache.sync()
        self._slots = torch.arange(max_batch_size, dtype=torch.int32, device=self.tok_embeddings.weight.device)

    def cache_key(self):
        """what launch descriptors and captured graphs hold pointers to"""
        return (self.max_seq_length, self.cache.version, id(self.cache))

    # ---- passes ----------------------------------------------------------------------------------------------------
    def _run(self, b, mixer, want: Optional[torch.Tensor], n_want: int, hook=None) -> Optional[torch.Tensor]:
        """embedding -> layers -> logits of the rows `want` (None: every row) of the batch b; mixer(layer's mixer, its inputs, index) = its
        pass over the normed input, or (mixers that say so) over the residual and the norm's weight"""
        cfg, w = self.config, self.tok_embeddings.weight
        norm = dict(eps=cfg.norm_eps, norm_offset=cfg.design.norm_offset, dtype=w.dtype)
        x = torch.empty(b.tokens.numel(), cfg.dim, device=w.device, dtype=torch.float32)

        def entry(i):
            """what the residual kernel leaves for layer i: its normed input, or nothing"""
            return dict(pre_w=None if self.layers[i].mix.from_residual else self.layers[i].norm1)

        # a few rows: the products are teal_rows_gemm's, which need a set of counters that no other pass uses at the same time
        rows = min(x.shape[0], n_want or x.shape[0])
        b.tickets = torch.empty(K.TICKETS, device=w.device, dtype=torch.int32) if w.dtype != torch.float32 and rows <= K.ROWS_MAX else None
        h = K.resid_norm(x, tokens=b.tokens, embed=w, **entry(0), **norm, zero=b.tickets)
        for i, layer in enumerate(self.layers):
            last = i + 1 == len(self.layers)
            after = dict(pre_w=self.norm if n_want else None) if last else entry(i + 1)
            if last and hook is None and n_want:
                after["rows"] = want  # nothing reads the other rows any more
            first = after if layer.mlp is None else dict(pre_w=layer.norm2)
            y = mixer(layer.mix, (x, layer.norm1) if layer.mix.from_residual else (h,), i)
            h = K.resid_norm(x, y=y, post_w=layer.norm1b, **first, **norm)
            if layer.mlp is not None:
                h = K.resid_norm(x, y=layer.mlp(h, b.tickets), y_bias=layer.mlp.down_bias, post_w=layer.norm2b, **after, **norm)
            if hook is not None:
                hook(i, x)
        if not n_want:
            return None
        if hook is not None and want is not None:
            h = h[want.long()]
        return K.head(self.output, h, cfg.vocab_size, cfg.logit_softcap, b.tickets)

    @torch.no_grad()
    def prompt_pass(self, b: PromptBatch, want, hook=None) -> Optional[torch.Tensor]:
        """logits (fp32) of the packed rows `want` (a sequence, or int32 on the device); the cache rows of every token are written"""
        w = want if torch.is_tensor(want) else torch.tensor(list(want), dtype=torch.int32).to(b.tokens.device) if len(want) else None
        return self._run(b, lambda m, ins, i: m.prompt(*ins, b, i), w, 0 if w is None else w.numel(), hook)

    @torch.no_grad()
    def step_pass(self, b: StepBatch, hook=None) -> torch.Tensor:
        """logits (fp32 [batch, vocab]) of one token per sequence"""
        return self._run(b, lambda m, ins, i: m.step(*ins, b, i), None, b.tokens.numel(), hook)

    @torch.no_grad()
    def forward(self, idx: torch.Tensor, input_pos: Optional[torch.Tensor] = None) -> torch.Tensor:
        """model.Transformer's interface: idx [B, S] at positions input_pos [S] of slots 0 .. B - 1 -> logits [B, S, vocab].  S = 1 keeps
        everything on the device (capturable into a hipGraph)."""
        assert self.cache is not None, "Caches must be initialized first"
        B, S = idx.shape
        if S == 1:
            pos = input_pos.to(torch.int32).expand(B).contiguous()
            b = StepBatch(self.cache, idx.view(-1).to(torch.int32), pos, self._slots[:B], self.max_seq_length - 1)
            return self.step_pass(b).view(B, 1, -1)
        start = int(input_pos[0])
        assert start + S <= self.max_seq_length
        toks = idx.cpu().numpy()
        b = PromptBatch(self.cache, [(i, start, toks[i]) for i in range(B)], idx.device)
        return self.prompt_pass(b, range(B * S)).view(B, S, -1)

    def prefill(self, graph: bool = True):
        """generate()'s `prefill` callable: the prompt of slot 0 -> logits [1, 1, vocab] of its last token"""
        run = GraphedPrompt(self) if graph else self.prompt_pass

        @torch.no_grad()
        def call(prompt: torch.Tensor) -> torch.Tensor:
            b = PromptBatch(self.cache, [(0, 0, prompt.view(-1).cpu().numpy())], prompt.device)
            return run(b, [b.n_tokens - 1]).view(1, 1, -1)

        return call


# ------------------------------------------------------------------------------------------------
# construction
# ------------------------------------------------------------------------------------------------
def _empty(cfg: LayeredArgs, device, dtype) -> LayeredTransformer:
    with torch.device("meta"):
        model = LayeredTransformer(cfg).to(dtype)
    model = model.to_empty(device=device)
    with torch.no_grad():
        for p in model.parameters():
            p.zero_()  # (padding rows stay zero)
    return model


def load_layered_checkpoint(path, device, dtype: torch.dtype) -> LayeredTransformer:
    """a folder with config.json and model.safetensors"""
    from safetensors import safe_open
    path = Path(path)
    with open(path / "config.json") as f:
        raw = json.load(f)
    with safe_open(str(path / "model.safetensors"), framework="pt", device="cpu") as st:
        model = _empty(LayeredArgs.from_dict(raw, {n: tuple(st.get_slice(n).get_shape()) for n in st.keys()}), device, dtype)
        return model.load_tensors(lambda n: st.get_tensor(n).to(device=device, dtype=dtype))


@torch.no_grad()
def build_layered_model(cfg: LayeredArgs, device, dtype: torch.dtype, seed: int = 1234, std: float = 0.02) -> LayeredTransformer:
    """random weights at the exact shapes: N(0, std^2) matrices, unit norms, zero biases and sinks, slow decays, even token shifts"""
    g = torch.Generator(device=device).manual_seed(seed)
    model = _empty(cfg, device, dtype)
    shapes = model.tensor_shapes()

    def get(name):
        shape = shapes[name]
        if len(shape) == 1:
            block_norm = name == "final.norm" or name.split(".")[1].startswith("norm")
            fill = 1.0 - cfg.design.norm_offset if block_norm else 1.0 if "norm" in name else -4.0 if name.endswith(".w0") else 0.5 if ".mu." in name else 0.0
            return torch.full(shape, fill, device=device, dtype=dtype)
        return (torch.randn(shape, device=device, dtype=torch.float32, generator=g) * std).to(dtype)

    return model.load_tensors(get)


def is_layered_checkpoint(path) -> bool:
    """does this folder (or a file in it) belong to a layered design?"""
    path = Path(path)
    cfg = (path if path.is_dir() else path.parent) / "config.json"
    if not cfg.is_file():
        return False
    with open(cfg) as f:
        return json.load(f).get("architecture") in DESIGNS
