"""Python side of the layered designs' kernels (include/teal_hip.h: teal_layer_*, teal_gated_act, teal_logit_softcap,
teal_latent_*, teal_grouped_*, teal_wkv_*): shape checks, dtype codes and the launch on the current stream.  PyTorch owns every buffer.

Activations and weights fp16, bf16 or true fp32; there is no CPU path."""
from __future__ import annotations

import ctypes
from typing import Optional

import torch

from .. import _lib, runtime

F32 = 2
ACTS = {"silu": 0, "gelu_tanh": 1, "relu2": 2, "silu_rounded": 3}  # (silu_rounded: gate | up products of teal_rows_gemm only)
NO_WINDOW = 1 << 30  # a window wider than any sequence: plain causal attention
TILE = 64            # packed key spans of a prompt pass are padded to this many rows


def dtype_code(dt: torch.dtype) -> int:
    return F32 if dt == torch.float32 else runtime.dtype_code(dt)


def _p(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _run(name: str, *args) -> None:
    rc = getattr(_lib.load(), name)(*args, runtime.stream_ptr())
    if rc != 0:
        _lib.check(rc, name)


def _rows(t: torch.Tensor) -> int:
    """row stride of a 2-D tensor whose columns are contiguous"""
    assert t.dim() == 2 and (t.stride(1) == 1 or t.shape[1] == 1), (t.shape, t.stride())
    return t.stride(0)


class RowsGemm(ctypes.Structure):  # teal_rows_gemm_t
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "w", "w_up", "bias", "bias_up", "y", "part")] + [("part_bytes", ctypes.c_size_t), ("tickets", ctypes.c_void_p)] + \
        [(n, ctypes.c_int) for n in ("M", "K", "N", "ldx", "ld", "ldy", "mode", "act", "n_valid")] + [("softcap", ctypes.c_float)]


ROWS_MAX, ROWS_PAIR_MAX = 64, 32  # rows of teal_rows_gemm; of its gate | up form: past them the vendor's product and gated_act are faster (64 rows, 4096 ->
# 2 x 11008: 55 us against 44 + 6; 32 rows: 38 us against 38 + 6)
ROWS_ROUNDED, ROWS_SLABS, ROWS_F32 = 0, 1, 2
TICKETS = 256


def rows_weight(lin) -> Optional[torch.Tensor]:
    """the weight of a plain linear whose product may bypass the module, else None (hooks, another class, a bias)"""
    if type(lin) is not torch.nn.Linear or lin.bias is not None or lin._forward_hooks or lin._forward_pre_hooks:
        return None
    return lin.weight


def _image(x, w) -> bool:
    """x [M, K] and the column-major w [N, K] as the products' kernels take them: one 16-bit type, aligned, in reach of a 32-bit offset"""
    return (w.dtype in (torch.float16, torch.bfloat16) and x.dtype == w.dtype and w.is_cuda and w.stride(0) == 1 and w.stride(1) >= w.shape[0] and not w.stride(1) & 7
            and x.stride(1) == 1 and not x.stride(0) & 7 and not (w.data_ptr() | x.data_ptr()) & 15 and w.shape[1] * w.stride(1) * 2 <= 0xFFF00000)


def rows_split(x, w, paired: bool = False) -> int:
    """slices teal_rows_gemm takes for x [M, K] and the column-major w [N, K]; 0: not a case for it"""
    M, (N, Kd) = x.shape[0], w.shape
    if paired:
        N //= 2
    if M > (ROWS_PAIR_MAX if paired else ROWS_MAX) or (N & 7) or not _image(x, w):
        return 0
    return int(_lib.load().teal_rows_split(M, Kd, N, int(paired)))


def tile_split(x, w, images: int = 1, slabs: bool = False) -> int:
    """slices teal_tile_gemm takes for more rows than teal_rows_gemm does (w: one of `images` of its shape); 0: not a case for it"""
    M, (N, Kd) = x.shape[0], w.shape
    if M <= ROWS_MAX or not _image(x, w) or x.stride(0) < Kd or M * x.stride(0) * 2 > 0xFFF00000:
        return 0
    return int(_lib.load().teal_tile_split(M, Kd, N, images, int(slabs)))


def _tile_gemm(x, w, N, y, y_up=None, w_up=None, slabs=False):
    _run("teal_tile_gemm", x.data_ptr(), x.stride(0), w.data_ptr(), w_up, w.stride(1), None if slabs else y.data_ptr(), _p(y_up), y.stride(-2), y.data_ptr() if slabs else None,
         x.shape[0], w.shape[1], N, runtime.dtype_code(x.dtype))
    return y


def _rows_gemm(x, w, N, split, mode, tickets, y, w_up=None, bias=None, bias_up=None, act=-1, n_valid=0, softcap=0.0):
    tile = 64 if w_up is not None else 128
    part = None
    if split > 1 and mode != ROWS_SLABS:
        part = torch.empty(split * x.shape[0] * (-(-N // tile) * 128), device=x.device, dtype=torch.float32)
    a = RowsGemm(x=x.data_ptr(), w=w.data_ptr(), w_up=w_up, bias=_p(bias), bias_up=_p(bias_up), y=y.data_ptr(), part=_p(part), part_bytes=0 if part is None else part.numel() * 4,
                 tickets=_p(tickets), M=x.shape[0], K=w.shape[1], N=N, ldx=x.stride(0), ld=w.stride(1), ldy=y.stride(-2), mode=mode, act=act, n_valid=n_valid, softcap=softcap)
    _run("teal_rows_gemm", ctypes.byref(a), runtime.dtype_code(x.dtype))
    return y


def linear(lin, x, tickets=None, slabs: bool = False, weight=None, act: Optional[str] = None, bias=None):
    """act(x W^T + bias) of a linear (or of rows of its weight).  With `tickets` (zero counters, left zero: one set per pass) a few rows go through
    teal_rows_gemm; `slabs`: the result may be the product's fp32 partial sums [slices, rows, columns] instead (of a few rows, or teal_tile_gemm's of
    more), for resid_norm to add"""
    if slabs and act is None and weight is None and x.shape[0] > ROWS_MAX and (w := rows_weight(lin)) is not None and (split := tile_split(x, w, slabs=True)):
        return _tile_gemm(x, w, w.shape[0], torch.empty(split, x.shape[0], w.shape[0], device=x.device, dtype=torch.float32), slabs=True)
    w = (rows_weight(lin) if tickets is not None else None) if weight is None else weight
    split = rows_split(x, w) if w is not None and tickets is not None else 0
    if split == 0:
        y = lin(x) if weight is None else torch.nn.functional.linear(x, weight)
        return y if act is None else gated_act(y, y.shape[1], 0, act, bias)
    M, N = x.shape[0], w.shape[0]
    if slabs and act is None:
        return _rows_gemm(x, w, N, split, ROWS_SLABS, None, torch.empty(split, M, N, device=x.device, dtype=torch.float32))
    return _rows_gemm(x, w, N, split, ROWS_ROUNDED, tickets, torch.empty(M, N, device=x.device, dtype=x.dtype), bias=bias, act=-1 if act is None else ACTS[act])


def gated_linear(lin, x, act: str, bias=None, tickets=None):
    """act(gate + bias) * (up + bias) of a linear whose output is [gate | up]"""
    w = rows_weight(lin) if tickets is not None else None
    N = lin.out_features // 2
    split = rows_split(x, w, True) if w is not None and not N & 63 else 0
    if split == 0:
        return gated_act(lin(x), N, N, act, bias)
    y = torch.empty(x.shape[0], N, device=x.device, dtype=x.dtype)
    return _rows_gemm(x, w, N, split, ROWS_ROUNDED, tickets, y, w_up=w.data_ptr() + 2 * N, bias=None if bias is None else bias[:N], bias_up=None if bias is None else bias[N:],
                      act=ACTS[act])


def gated_pair(gate, up, x, act: str, tickets=None):
    """round(act(gate)) * up of two linears of one shape and layout, or None: not a case for teal_rows_gemm"""
    w, u = (rows_weight(lin) if tickets is not None else None for lin in (gate, up))
    if w is None or u is None or w.shape != u.shape or w.stride() != u.stride() or u.data_ptr() & 15 or x.shape[0] > ROWS_PAIR_MAX or w.shape[0] & 63:
        return None
    if rows_split(x, w) == 0:
        return None
    split = int(_lib.load().teal_rows_split(x.shape[0], w.shape[1], w.shape[0], 1))
    return _rows_gemm(x, w, w.shape[0], split, ROWS_ROUNDED, tickets, torch.empty(x.shape[0], w.shape[0], device=x.device, dtype=x.dtype), w_up=u.data_ptr(), act=ACTS[act])


def both(gate, up, x):
    """(gate(x), up(x)) of two linears"""
    w, u = rows_weight(gate), rows_weight(up)
    if w is None or u is None or w.shape != u.shape or w.stride() != u.stride() or u.dtype != w.dtype or u.data_ptr() & 15 or not tile_split(x, w, 2):
        return gate(x), up(x)
    y = torch.empty(2, x.shape[0], w.shape[0], device=x.device, dtype=x.dtype)
    _tile_gemm(x, w, w.shape[0], y[0], y[1], u.data_ptr())
    return y[0], y[1]


def head(lin, h, vocab: int, cap: Optional[float], tickets=None):
    """fp32 logits [rows, vocab], soft-capped"""
    w = rows_weight(lin) if tickets is not None else None
    split = rows_split(h, w) if w is not None else 0
    if split == 0:
        return softcap(lin(h), vocab, cap)
    out = torch.empty(h.shape[0], vocab, device=h.device, dtype=torch.float32)
    return _rows_gemm(h, w, w.shape[0], split, ROWS_F32, tickets, out, n_valid=vocab, softcap=float(cap or 0.0))


def resid_norm(x, *, tokens=None, embed=None, y=None, y_bias=None, post_w=None, pre_w=None, eps=1e-6, rows=None, dtype=None, norm_offset=0.0, zero=None):
    """x (fp32 [T, D], in place) = embedding rows | x, + [post norm](y + bias); returns h = RMSNorm(x) * (norm_offset + pre_w) (rows of
    `rows`, packed).  y: 16-bit, or slabs of `linear`; zero: counters to clear on the way"""
    assert x.dtype == torch.float32 and x.is_contiguous()
    n = x.shape[0] if rows is None else rows.numel()
    slabs = y is not None and y.dim() == 3
    dtype = dtype or (pre_w if pre_w is not None else embed if embed is not None else y).dtype
    h = torch.empty(n, x.shape[1], device=x.device, dtype=dtype) if pre_w is not None else None
    head = (_p(x), n, x.shape[1], _p(tokens), _p(embed), 0 if embed is None else embed.shape[0], _p(y))
    tail = (_p(y_bias), _p(post_w), _p(pre_w), float(norm_offset), float(eps), _p(h), _p(rows))
    if slabs:
        assert y.dtype == torch.float32 and y.is_contiguous()
        _run("teal_layer_resid_norm_slabs", *head, y.shape[0], y.shape[1], y.shape[2], *tail, _p(zero), 0 if zero is None else zero.numel(), dtype_code(dtype))
    elif zero is not None:
        assert y is None
        _run("teal_layer_resid_norm_slabs", *head, 0, 0, 0, *tail, _p(zero), zero.numel(), dtype_code(dtype))
    else:
        _run("teal_layer_resid_norm", *head, 0 if y is None else _rows(y), *tail, dtype_code(dtype))
    return h


def gated_act(gu, n_cols: int, up0: int, act: str, bias=None, out=None):
    """act(gate + bias) * (up + bias): gate = gu[:, :n_cols], up = gu[:, up0:up0 + n_cols]; bias laid out like a row of gu.  up0 = 0:
    act(gate + bias) alone"""
    if out is None:
        out = torch.empty(gu.shape[0], n_cols, device=gu.device, dtype=gu.dtype)
    _run("teal_gated_act", _p(gu), _rows(gu), up0, _p(bias), None if bias is None or not up0 else bias.data_ptr() + up0 * bias.element_size(), _p(out), _rows(out),
         gu.shape[0], n_cols, ACTS[act], dtype_code(gu.dtype))
    return out


def softcap(logits, vocab: int, cap: Optional[float], out=None):
    """fp32 [rows, vocab] = cap * tanh(logits / cap)"""
    if out is None:
        out = torch.empty(logits.shape[0], vocab, device=logits.device, dtype=torch.float32)
    _run("teal_logit_softcap", _p(logits), _rows(logits), _p(out), logits.shape[0], vocab, float(cap or 0.0), dtype_code(logits.dtype))
    return out


def sample_rows(logits, rng, temperature: float, top_k: Optional[int], out=None, pos=None, history=None):
    """one token per row of fp32 logits; rng int64 [rows, 2] {seed, draw counter}; temperature <= 0: the largest logit"""
    assert logits.dtype == torch.float32 and rng.dtype == torch.int64 and rng.is_contiguous() and rng.numel() >= 2 * logits.shape[0]
    if out is None:
        out = torch.empty(logits.shape[0], dtype=torch.int32, device=logits.device)
    _run("teal_sample_rows", _p(logits), _rows(logits), logits.shape[0], logits.shape[1], int(top_k or 0), float(temperature), _p(rng), _p(out), _p(pos), _p(history),
         0 if history is None else history.shape[-1])
    return out


def latent_prompt_rows(proj, kv0, pos, row, inv_freq, norm_w, eps, heads, dim, rot, rank, pool):
    """rotate proj's queries in place; kv0 >= 0: write each token's cache row"""
    assert pos.dtype == torch.int32 and pos.numel() == proj.shape[0]
    _run("teal_latent_prompt_rows", _p(proj), _rows(proj), kv0, proj.shape[0], _p(pos), _p(row), _p(inv_freq), _p(norm_w), float(eps), heads, dim, rot, rank,
         _p(pool), 0 if pool is None else pool.shape[-1], dtype_code(proj.dtype))


def latent_gather(pool, row, rank, rot):
    """(c [n, rank], kr [n, rot]) of the cache rows `row` (negative: zeros)"""
    n = row.numel()
    c = torch.empty(n, rank, device=pool.device, dtype=pool.dtype)
    kr = torch.empty(n, rot, device=pool.device, dtype=pool.dtype)
    _run("teal_latent_gather", _p(pool), pool.shape[-1], _p(row), n, rank, rot, _p(c), _p(kr), dtype_code(pool.dtype))
    return c, kr


def prompt_tile(dim, rot, vdim, n_queries, dtype) -> int:
    return int(_lib.load().teal_layer_prompt_tile(dim, rot, vdim, n_queries, dtype_code(dtype)))


def prompt_attention(q, k, kr, vt, sink, gate, out, seqs, tiles, tile, heads, dim, rot, vdim, window, scale, group=1, softcap=None):
    """flash attention over packed keys; `group` query heads per key / value head"""
    assert k.is_contiguous() and (kr is None or kr.is_contiguous()) and vt.is_contiguous() and k.shape[0] == vt.shape[1]
    assert seqs.dtype == tiles.dtype == torch.int32 and seqs.shape[1] == 5 and tiles.shape[1] == 2
    _run("teal_layer_prompt_attention", _p(q), _rows(q), _p(k), _p(kr), _p(vt), k.shape[0], _p(sink), _p(gate), 0 if gate is None else _rows(gate), _p(out),
         _rows(out), _p(seqs), _p(tiles), tiles.shape[0], tile, heads, group, dim, rot, vdim, int(window), float(scale), float(softcap or 0.0), dtype_code(q.dtype))
    return out


def step_qcat(batch, heads, ldq, dtype, device):
    """the step's query rows: fp32, or a high and a low 16-bit row"""
    return torch.empty(batch, heads, *(() if dtype == torch.float32 else (2,)), ldq, device=device, dtype=dtype)


def step_part(batch, heads, splits, rank, device):
    """the splits' partial results: weighted values (padded to 4), max, sum"""
    return torch.empty(batch * heads * splits * (-(-rank // 4) * 4 + 4), device=device, dtype=torch.float32)


def latent_step_query(proj, kv0, pos, slot, table, page_shift, inv_freq, norm_w, eps, uk, heads, dim, rot, rank, pool, qcat):
    assert uk.is_contiguous() and table.is_contiguous() and pos.dtype == slot.dtype == table.dtype == torch.int32
    _run("teal_latent_step_query", _p(proj), _rows(proj), kv0, proj.shape[0], _p(pos), _p(slot), _p(table), table.shape[1], page_shift, _p(inv_freq), _p(norm_w),
         float(eps), _p(uk), heads, dim, rot, rank, _p(pool), pool.shape[-1], _p(qcat), qcat.shape[-1], dtype_code(proj.dtype))


def step_attention(qcat, pool, pos, slot, table, page_shift, rank, rot, window, scale, splits, part, group=None, softcap=None):
    """`group` heads share a segment of the cached row (None: all of them, one segment)"""
    assert part.dtype == torch.float32
    heads = qcat.shape[1]
    _run("teal_layer_step_attention", _p(qcat), qcat.shape[-1], _p(pool), pool.shape[-1], _p(pos), _p(slot), _p(table), table.shape[1], page_shift, qcat.shape[0],
         heads, group or heads, rank, rot, int(window), float(scale), float(softcap or 0.0), splits, _p(part), part.numel() * 4, dtype_code(qcat.dtype))


def latent_step_merge(part, splits, uv, sink, gate, y, batch, heads, rank, vdim):
    assert uv.is_contiguous()
    _run("teal_latent_step_merge", _p(part), splits, _p(uv), _p(sink), _p(gate), 0 if gate is None else _rows(gate), _p(y), _rows(y), batch, heads, rank, vdim,
         dtype_code(y.dtype))
    return y


def grouped_prompt_rows(proj, k0, pos, row, inv_freq, heads, kv_heads, dim, rot, pool):
    """rotate proj's queries in place; write each token's cache row"""
    assert pos.dtype == row.dtype == torch.int32 and pos.numel() == proj.shape[0]
    _run("teal_grouped_prompt_rows", _p(proj), _rows(proj), k0, proj.shape[0], _p(pos), _p(row), _p(inv_freq), heads, kv_heads, dim, rot, _p(pool),
         pool.shape[-1] // kv_heads, dtype_code(proj.dtype))


def grouped_gather(pool, row, kv_heads, dim, rot):
    """(rotated keys [n, kv_heads * dim], values transposed [kv_heads * dim, n]) of the cache rows `row` (negative: zeros)"""
    n = row.numel()
    k = torch.empty(n, kv_heads * dim, device=pool.device, dtype=pool.dtype)
    vt = torch.empty(kv_heads * dim, n, device=pool.device, dtype=pool.dtype)
    _run("teal_grouped_gather", _p(pool), pool.shape[-1] // kv_heads, _p(row), n, kv_heads, dim, rot, _p(k), _p(vt), dtype_code(pool.dtype))
    return k, vt


def grouped_step_attention(proj, k0, pos, slot, table, page_shift, inv_freq, heads, kv_heads, dim, rot, pool, window, scale, softcap, splits, qcat, part):
    """the token's cache row and the split attention of one token per sequence"""
    assert table.is_contiguous() and pos.dtype == slot.dtype == table.dtype == torch.int32 and part.dtype == torch.float32
    assert qcat.shape[-1] == pool.shape[-1] // kv_heads and qcat.numel() >= proj.shape[0] * heads * qcat.shape[-1] * (1 if proj.dtype == torch.float32 else 2)
    _run("teal_grouped_step_attention", _p(proj), _rows(proj), k0, proj.shape[0], _p(pos), _p(slot), _p(table), table.shape[1], page_shift, _p(inv_freq), heads, kv_heads,
         dim, rot, _p(pool), pool.shape[-1] // kv_heads, int(window), float(scale), float(softcap or 0.0), splits, _p(qcat), _p(part), part.numel() * 4,
         dtype_code(proj.dtype))


def grouped_step_merge(part, splits, sink, y, batch, heads, dim):
    _run("teal_grouped_step_merge", _p(part), splits, _p(sink), _p(y), _rows(y), batch, heads, dim, dtype_code(y.dtype))
    return y


def wkv_mix(x, norm_w, norm_offset, eps, mu, pos, slot, run, shift):
    """the token-shifted inputs [n_mix, rows, width] of time mixing, from the fp32 residual rows; `shift` [slots, 2, width] is updated"""
    assert x.dtype == shift.dtype == torch.float32 and x.is_contiguous() and mu.is_contiguous() and pos.numel() == slot.numel() == x.shape[0]
    assert pos.dtype == slot.dtype == torch.int32
    out = torch.empty(mu.shape[0], *x.shape, device=x.device, dtype=mu.dtype)
    _run("teal_wkv_mix", _p(x), x.shape[0], x.shape[1], _p(norm_w), float(norm_offset), float(eps), _p(mu), mu.shape[0], _p(pos), _p(slot), _p(run), _p(shift), _p(out),
         dtype_code(mu.dtype))
    return out


def wkv_decay(z, w2, w0):
    out = torch.empty(z.shape[0], w2.shape[0], device=z.device, dtype=torch.float32)
    _run("teal_wkv_decay", _p(z), _rows(z), _p(w2), _p(w0), w2.shape[1], z.shape[0], w2.shape[0], _p(out), dtype_code(z.dtype))
    return out


def wkv_scan(r, k, v, w, u, seqs, slot, state, longest):
    """the recurrence over a prompt's portions (the longest has `longest` rows) -> fp32 [rows, heads * dim]; `state` [slots, 2, heads, dim, dim]
    is updated"""
    heads, dim = u.shape
    assert _rows(r) == _rows(k) == _rows(v) and w.dtype == state.dtype == torch.float32 and w.is_contiguous() and seqs.dtype == torch.int32 and seqs.shape[1] == 5
    o = torch.empty(r.shape[0], heads * dim, device=r.device, dtype=torch.float32)
    chunks = torch.empty(_lib.load().teal_wkv_chunk_bytes(r.shape[0], seqs.shape[0], heads, dim) // 4, device=r.device, dtype=torch.float32)
    _run("teal_wkv_scan", _p(r), _p(k), _p(v), _rows(r), _p(w), _p(u), _p(seqs), seqs.shape[0], r.shape[0], longest, _p(slot), _p(state), _p(chunks), chunks.numel() * 4,
         _p(o), heads, dim, dtype_code(r.dtype))
    return o


def wkv_out(o, norm, g, eps, y, heads, dim):
    _run("teal_wkv_out", _p(o), _p(norm), _p(g), _rows(g), float(eps), _p(y), _rows(y), o.shape[0], heads, dim, dtype_code(y.dtype))
    return y


def wkv_step(r, k, v, g, z, w2, w0, u, norm, eps, pos, slot, state, y):
    """one token per sequence, from the projections to W_o's input"""
    heads, dim = u.shape
    assert _rows(r) == _rows(k) == _rows(v) == _rows(g) and state.dtype == torch.float32
    _run("teal_wkv_step", _p(r), _p(k), _p(v), _p(g), _rows(r), _p(z), _rows(z), _p(w2), _p(w0), w2.shape[1], _p(u), _p(norm), float(eps), _p(pos), _p(slot), _p(state),
         _p(y), _rows(y), r.shape[0], heads, dim, dtype_code(y.dtype))
    return y
