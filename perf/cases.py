"""The work that users of this framework have it do, as cases that can be timed and checked.

A case is a dict of plain values; `listed()` names the standing ones and `draw(rng)` makes more of the same ranges.  `prepare` builds
what a program holds before the call (weights, caches, engine), `run` is one pass through the public entry points, `exact` the same
result in 64 bits from torch alone.  Weights are random at the named shapes (fewer layers than the full models: every layer does the
same work), scaled so that a residual stream stays near the embedding it started from: the next token is then certain, as it mostly is
in a trained model, and a sampled continuation is the same for every correct implementation.

Paths:
  gemv            one call of the sparse GEMV operator on one token
  llama_decode    a few tokens decoded at batch 1 from a filled cache (the device-resident loop: hipGraph, fused sampler)
  llama_prompt    the prompt pass that generate() runs under --compile
  layered_step    a decode step of a batch, replayed from a hipGraph
  layered_prompt  a ragged batch of prompts through the batched serving engine
  layered_generate  generate() at batch 1: prompt, then fused decoding
"""
from __future__ import annotations

import math
import zlib

import torch

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS_LLAMA = 1e-5


def listed():
    return [
        # a projection swapped by hand into somebody's own model: the operator at the reference benchmark's square shape.  Launch latency.
        {"name": "gemv_4096", "path": "gemv", "Z": 4096, "N": 4096, "dtype": "fp16", "sparsity": 0.5},
        # the headline: chat decoding of a 7B model at half of its activations
        {"name": "7b_decode_s50", "path": "llama_decode", "model": "7B", "n_layer": 8, "dtype": "fp16", "weights": 16, "sparsity": 0.5, "context": 500, "tokens": 16},
        # a long document in the cache of a grouped-query model
        {"name": "8b_decode_s40_long", "path": "llama_decode", "model": "llama-3-8b", "n_layer": 4, "dtype": "bf16", "weights": 16, "sparsity": 0.4, "context": 7000,
         "tokens": 16},
        # the widest model that fits one card
        {"name": "70b_decode_s50", "path": "llama_decode", "model": "70B", "n_layer": 2, "dtype": "fp16", "weights": 16, "sparsity": 0.5, "context": 1000, "tokens": 16},
        # group-quantised weights under the same sparsity
        {"name": "7b_decode_int4_s50", "path": "llama_decode", "model": "7B", "n_layer": 8, "dtype": "fp16", "weights": 4, "sparsity": 0.5, "context": 500, "tokens": 16},
        # the reference harness's own prompt ("Hello, my name is" and the like): counted by its tokens per second
        {"name": "7b_prompt_7", "path": "llama_prompt", "model": "7B", "n_layer": 8, "dtype": "fp16", "tokens": 7},
        # a chat turn
        {"name": "7b_prompt_301", "path": "llama_prompt", "model": "7B", "n_layer": 8, "dtype": "fp16", "tokens": 301},
        # a document to summarise
        {"name": "8b_prompt_3000", "path": "llama_prompt", "model": "llama-3-8b", "n_layer": 8, "dtype": "bf16", "tokens": 3000},
        # serving: sixteen requests in flight
        {"name": "bolizen_step_b16", "path": "layered_step", "model": "Bolizen-7B", "n_layer": 4, "dtype": "bf16", "batch": 16, "context": 1000},
        # serving: requests of different lengths admitted together
        {"name": "bolizen_prompt_3k", "path": "layered_prompt", "model": "Bolizen-7B", "n_layer": 4, "dtype": "bf16", "batch": 5, "tokens": 3000},
        # one user of a recurrent design: prompt and answer
        {"name": "tefopel_generate", "path": "layered_generate", "model": "Tefopel-7B", "n_layer": 4, "dtype": "bf16", "tokens": 100, "new": 33},
        # time mixing over long prompts
        {"name": "tefopel_prompt_3k", "path": "layered_prompt", "model": "Tefopel-7B", "n_layer": 4, "dtype": "bf16", "batch": 3, "tokens": 3000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["gemv", "llama_decode", "llama_decode", "llama_prompt", "llama_prompt", "layered_step", "layered_prompt", "layered_generate"])
    if path == "gemv":  # any rows, 16-byte columns
        return {"path": path, "Z": _log(rng, 500, 16000), "N": 8 * _log(rng, 64, 2000), "dtype": rng.choice(["fp16", "bf16"]), "sparsity": round(rng.uniform(0.25, 0.75), 2)}
    if path == "llama_decode":
        model, n_layer, dtype, context = rng.choice([("7B", 8, "fp16", (8, 1900)), ("13B", 6, "fp16", (8, 1900)), ("llama-3-8b", 4, "bf16", (8, 7500)), ("70B", 2, "fp16", (8, 1900))])
        return {"path": path, "model": model, "n_layer": n_layer, "dtype": dtype, "weights": rng.choice([16, 16, 8, 4]), "sparsity": round(rng.uniform(0.25, 0.65), 2),
                "context": _log(rng, *context), "tokens": rng.randint(5, 16)}
    if path == "llama_prompt":
        model, n_layer, dtype, most = rng.choice([("7B", 8, "fp16", 2000), ("llama-3-8b", 8, "bf16", 3000)])
        return {"path": path, "model": model, "n_layer": rng.randint(4, n_layer), "dtype": dtype, "tokens": _log(rng, 2, most)}
    design = rng.choice(["Bolizen-1B", "Bolizen-7B", "Tefopel-1B", "Tefopel-7B"])
    c = {"path": path, "model": design, "n_layer": 4, "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if path == "layered_step":
        c["batch"] = _log(rng, 2, 64)
        c["context"] = _log(rng, 60, min(4000, 16000 // c["batch"]))
    elif path == "layered_prompt":
        c["batch"] = rng.randint(1, 6)
        c["tokens"] = _log(rng, 40 * c["batch"], 3000)
    else:
        c["tokens"], c["new"] = _log(rng, 4, 300), rng.randint(9, 33)
    return c


# ------------------------------------------------------------------------------------------------
# tensors from a seed
# ------------------------------------------------------------------------------------------------
def _gen(seed, name):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))


def _randn(seed, name, shape, std, dtype, mean=0.0):
    return (torch.randn(shape, device=DEV, dtype=torch.float32, generator=_gen(seed, name)) * std + mean).to(dtype)


def _tokens(seed, name, n, vocab):
    return torch.randint(0, vocab, (n,), device=DEV, generator=_gen(seed, name), dtype=torch.int64)


# ------------------------------------------------------------------------------------------------
# the Llama stack
# ------------------------------------------------------------------------------------------------
class _LlamaWeights:
    """Weights of a Llama stack by name; `matrix(name, work)` is what the matrix products compute with, in the type `work`."""

    def __init__(self, c, seed):
        from teal_amd.gpt_fast.model import ModelArgs
        a = ModelArgs.from_name(c["model"])
        a.n_layer = c["n_layer"]
        self.args, self.seed, self.dtype, self.bits = a, seed, DTYPES[c["dtype"]], c.get("weights", 16)
        self.kv = a.n_local_heads * a.head_dim
        # unit projections; a feed-forward adds `part` of the residual's size, attention less.  Under thresholds a small error of the input
        # moves values across them and comes out as its square root: a stack whose layers add much is chaotic, whatever computes it
        one, part = a.dim ** -0.5, 0.05 if c["path"] == "llama_decode" else 0.5
        self.shapes = {"wqkv": (a.dim + 2 * self.kv, a.dim, one), "wo": (a.dim, a.dim, 2 * part * one), "w1": (a.intermediate_size, a.dim, one),
                       "w3": (a.intermediate_size, a.dim, one), "w2": (a.dim, a.intermediate_size, part / 0.6 * a.intermediate_size ** -0.5)}

    def embed(self):
        return _randn(self.seed, "embed", (self.args.vocab_size, self.args.dim), 1.0, self.dtype)

    def norm(self, name):
        return _randn(self.seed, name, (self.args.dim,), 0.05, self.dtype, 1.0)

    def plain(self, layer, name):
        """16-bit [N, Z]"""
        n, z, std = self.shapes[name]
        return _randn(self.seed, f"{layer}.{name}", (n, z), std, self.dtype)

    def output(self):
        """row j is the embedding of token j - 1: token t is followed by t + 1"""
        return (torch.roll(self.embed(), 1, 0) * 0.1).to(self.dtype)

    def int8(self, w):
        """(int8 [N, Z], scale [N])"""
        s = (w.float().abs().amax(1) / 127).to(self.dtype)
        return (w.float() / s.float()[:, None]).round().clamp(-127, 127).to(torch.int8), s

    def int4(self, layer, name, group=32):
        """(0..15 as int32 [N, Z], bf16 [Z / group, N, 2] of scales and zeros)"""
        n, z, std = self.shapes[name]
        g = _gen(self.seed, f"{layer}.{name}")
        q = torch.randint(0, 16, (n, z), device=DEV, dtype=torch.int32, generator=g)
        s = (torch.rand(z // group, n, device=DEV, generator=g) * 0.5 + 0.75) * (std / 4.61)
        return q, torch.stack([s, 0.5 * s], dim=-1).to(torch.bfloat16)

    def matrix(self, layer, name, work):
        if name == "output":
            w = self.output()
            if self.bits != 8:
                return w.to(work)
            q, s = self.int8(w)
            return q.to(work) * s.to(work)[:, None]
        if self.bits == 4:
            q, sz = self.int4(layer, name)
            s, z = (sz[..., i].to(work).T.repeat_interleave(32, dim=1) for i in (0, 1))
            return (q.to(work) - 8) * s + z
        if self.bits == 8:
            q, s = self.int8(self.plain(layer, name))
            return q.to(work) * s.to(work)[:, None]
        return self.plain(layer, name).to(work)

    def caches(self, layer, context):
        a = self.args
        return tuple(_randn(self.seed, f"{layer}.{n}", (a.n_local_heads, context, a.head_dim), s, self.dtype) for n, s in (("k", 2.5), ("v", 1.0)))


def _llama_model(W, seq):
    """the framework's model over these weights, caches set up"""
    from teal_amd import quantize
    from teal_amd.gpt_fast.model import Transformer
    with torch.device("meta"):
        model = Transformer(W.args).to(W.dtype)
        if W.bits == 8:
            quantize.convert_for_runtime_int8(model, W.dtype)
        elif W.bits == 4:
            quantize.convert_for_runtime_int4(model, 32)
    model = model.to_empty(device=DEV).eval()
    for p in model.parameters():
        p.requires_grad_(False)

    def fill(lin, layer, name):
        if name != "output" and W.bits == 4:
            q, sz = W.int4(layer, name)
            lin.weight.copy_(quantize.pack_int4_colmajor(q))
            lin.scales_and_zeros.copy_(sz)
        elif W.bits == 8:
            q, s = W.int8(W.output() if name == "output" else W.plain(layer, name))
            lin.weight.copy_(q)
            lin.scales.copy_(s)
        else:
            lin.weight.copy_(W.output() if name == "output" else W.plain(layer, name))

    model.tok_embeddings.weight.copy_(W.embed())
    model.norm.weight.copy_(W.norm("norm"))
    fill(model.output, -1, "output")
    for i, b in enumerate(model.layers):
        b.attention_norm.weight.copy_(W.norm(f"{i}.attention_norm"))
        b.ffn_norm.weight.copy_(W.norm(f"{i}.ffn_norm"))
        for n, lin in (("wqkv", b.attention.wqkv), ("wo", b.attention.wo), ("w1", b.feed_forward.w1), ("w2", b.feed_forward.w2), ("w3", b.feed_forward.w3)):
            fill(lin, i, n)
    model.setup_caches(max_batch_size=1, max_seq_length=seq)
    return model


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _turn(x, cos, sin):
    """adjacent pairs of x [T, heads, d] by the angles of cos, sin [T, d / 2]"""
    u, v = x[..., 0::2], x[..., 1::2]
    c, s = cos[:, None], sin[:, None]
    return torch.stack((u * c - v * s, v * c + u * s), dim=-1).flatten(-2)


def _softmax_attend(q, k, v, start, scale, window=None, cap=None, sink=None):
    """causal attention of q [T, heads, d] at positions start.. over k [S, kv heads, d], v [S, kv heads, e]: [T, heads, e]"""
    T, S, rep = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    p, j = torch.arange(start, start + T, device=DEV)[:, None], torch.arange(S, device=DEV)[None]
    hidden = (j > p) if window is None else (j > p) | (j <= p - window)
    out = torch.empty(T, q.shape[1], v.shape[2], device=DEV, dtype=q.dtype)
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // rep].T) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(hidden, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink[h].expand(T, 1)], dim=1)
        s = torch.softmax(s, dim=1)[:, :S]
        out[:, h] = s @ v[:, h // rep]
    return out


def _llama(W, tokens, start, work, thresholds=None, sparsity=None):
    """The stack over `tokens` at positions start .. behind caches of that many rows, in the type `work`: (logits, [(k rows, v rows)], thresholds).
    thresholds: what falls to zero at each projection's input; sparsity: they are taken from these tokens, per site."""
    a, T = W.args, tokens.numel()
    inv = 1.0 / (a.rope_base ** (torch.arange(0, a.head_dim, 2, device=DEV)[: a.head_dim // 2].float() / a.head_dim))
    ang = torch.outer(torch.arange(start, start + T, device=DEV).float(), inv)
    cos, sin = (f(ang).to(W.dtype).to(work) for f in (torch.cos, torch.sin))  # (the model holds its rotation table in 16 bits)
    found, rows = [], []

    def site(x, layer, name):
        """x with its small values zeroed: what the projection `name` reads"""
        if thresholds is None and sparsity is None:
            return x
        mag = x.to(W.dtype).float().abs()
        if thresholds is None:
            flat = mag.flatten()
            found[layer][name] = float("%.4g" % torch.quantile(flat[:: max(1, flat.numel() // 200000)], sparsity))
        return x * (mag > (found if thresholds is None else thresholds)[layer][name])

    x = W.embed()[tokens].to(work)
    for i in range(a.n_layer):
        found.append({})
        h = site(_rms(x, W.norm(f"{i}.attention_norm").to(work), EPS_LLAMA), i, "q")
        q, k, v = (h @ W.matrix(i, "wqkv", work).T).split([a.dim, W.kv, W.kv], dim=-1)
        k, v = _turn(k.view(T, -1, a.head_dim), cos, sin), v.view(T, -1, a.head_dim)
        rows.append((k, v))
        kk, vv = k, v
        if start:
            ck, cv = W.caches(i, start)
            kk, vv = torch.cat([ck.transpose(0, 1).to(work), k]), torch.cat([cv.transpose(0, 1).to(work), v])
        y = _softmax_attend(_turn(q.view(T, -1, a.head_dim), cos, sin), kk, vv, start, a.head_dim ** -0.5).reshape(T, a.dim)
        x = x + site(y, i, "o") @ W.matrix(i, "wo", work).T
        h = site(_rms(x, W.norm(f"{i}.ffn_norm").to(work), EPS_LLAMA), i, "gate")
        m = torch.nn.functional.silu(h @ W.matrix(i, "w1", work).T) * (h @ W.matrix(i, "w3", work).T)
        x = x + site(m, i, "down") @ W.matrix(i, "w2", work).T
    for th in found:
        if th:
            th.update(k=th["q"], v=th["q"], up=th["gate"])
    return _rms(x, W.norm("norm").to(work), EPS_LLAMA) @ W.matrix(-1, "output", work).T, rows, found


def _thresholds(W, c, first):
    """what keeps 1 - sparsity of the inputs of every projection on the tokens about to be decoded"""
    tokens = (first + torch.arange(4, device=DEV)) % W.args.vocab_size
    return _llama(W, tokens, c["context"], torch.float32, sparsity=c["sparsity"])[2]


# ------------------------------------------------------------------------------------------------
# layered designs
# ------------------------------------------------------------------------------------------------
def _layered_config(c):
    from teal_amd.gpt_fast.layered import named_config
    return named_config(c["model"], c["n_layer"])


def _layered_tensor(cfg, seed, dtype, name, shape):
    """a checkpoint tensor: sublayers add little to the residual, decays are slow, token shifts uneven, norms near their neutral value"""
    tefopel = cfg["architecture"] == "Tefopel"
    leaf = name.split(".")[-1]
    std, mean = 0.02, 0.0
    if name == "embed":
        std = 0.05
    elif leaf in ("norm1b", "norm2b"):
        std, mean = 0.002, 0.02
    elif leaf in ("norm1", "norm2") or name == "final.norm":
        std, mean = 0.05, 0.0 if tefopel else 1.0
    elif leaf == "norm":
        std, mean = 0.05, 1.0
    elif leaf == "w0":
        std, mean = 1.0, -4.0
    elif ".mu." in name:
        std, mean = 0.1, 0.5
    elif leaf in ("sink", "b", "u"):
        std = 0.3 if leaf != "b" else 0.02
    elif tefopel and leaf in ("o", "down"):
        std = 0.0005
    return _randn(seed, name, shape, std, dtype, mean)


def _layered_model(c, seed):
    from teal_amd.gpt_fast.layered import LayeredArgs, LayeredTransformer
    cfg, dtype = _layered_config(c), DTYPES[c["dtype"]]
    with torch.device("meta"):
        model = LayeredTransformer(LayeredArgs.from_dict(cfg)).to(dtype)
    model = model.to_empty(device=DEV)
    with torch.no_grad():
        for p in model.parameters():
            p.zero_()
    shapes = model.tensor_shapes()
    return model.load_tensors(lambda n: _layered_tensor(cfg, seed, dtype, n, shapes[n]))


class _Layered:
    """the designs in 64 bits, one sequence at a time"""

    def __init__(self, c, seed):
        self.cfg, self.seed, self.dtype = _layered_config(c), seed, DTYPES[c["dtype"]]
        self.kept = {}

    def w(self, name, *shape):
        if name not in self.kept:
            self.kept[name] = _layered_tensor(self.cfg, self.seed, self.dtype, name, shape)
        return self.kept[name].double()

    def rot(self, x, base, dims):
        i = torch.arange(0, dims, 2, device=DEV, dtype=torch.float64)
        ang = torch.outer(torch.arange(x.shape[0], device=DEV, dtype=torch.float64), float(base) ** (-i / max(1, dims)))
        return torch.cat([_turn(x[..., :dims], ang.cos(), ang.sin()), x[..., dims:]], dim=-1)

    def latent(self, h, n, a, store, i):
        T, H, D, R, V, K, width = h.shape[0], a["heads"], a["dim"], a["rot_dim"], a["vdim"], a["kv_rank"], h.shape[1]
        base = a["rot"]["base"]
        q = (h @ self.w(n + ".q", H * (D + R), width).T).view(T, H, D + R)
        q = torch.cat([q[..., :D], self.rot(q[..., D:], base, R)], dim=-1)
        if a.get("kv_from") is None:
            kv = h @ self.w(n + ".dkv", K + R, width).T
            store[i] = _rms(kv[:, :K], self.w(n + ".dkv.norm", K), self.cfg["norm"]["eps"]), self.rot(kv[:, None, K:], base, R)
        c, kr = store[i if a.get("kv_from") is None else a["kv_from"]]
        k = torch.cat([(c @ self.w(n + ".uk", H * D, K).T).view(T, H, D), kr.expand(T, H, R)], dim=-1)
        v = (c @ self.w(n + ".uv", H * V, K).T).view(T, H, V)
        y = _softmax_attend(q, k, v, 0, a["scale"], a["mask"]["size"], sink=self.w(n + ".sink", H)).reshape(T, H * V)
        return (y * torch.sigmoid(h @ self.w(n + ".g", H * V, width).T)) @ self.w(n + ".o", width, H * V).T

    def tied(self, h, n, a):
        T, H, G, D, width = h.shape[0], a["heads"], a["kv_heads"], a["dim"], h.shape[1]
        q = self.rot((h @ self.w(n + ".q", H * D, width).T).view(T, H, D), a["rot"]["base"], a["rot"]["dims"])
        v = (h @ self.w(n + ".k", G * D, width).T).view(T, G, D)
        k = self.rot(v, a["rot"]["base"], a["rot"]["dims"])
        y = _softmax_attend(q, k, v, 0, a["scale"], a["mask"]["size"], a["softcap"], self.w(n + ".sink", H))
        return y.reshape(T, H * D) @ self.w(n + ".o", width, H * D).T

    def wkv(self, h, n, a):
        T, H, D, rank, width = h.shape[0], a["heads"], a["dim"], a["decay_rank"], h.shape[1]
        prev = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
        mixed = {s: h + (prev - h) * self.w(n + ".mu." + s, width) for s in "rkvgw"}
        r, k, v = ((mixed[s] @ self.w(n + "." + s, H * D, width).T).view(T, H, D) for s in "rkv")
        z = torch.tanh(mixed["w"] @ self.w(n + ".w1", rank, width).T) @ self.w(n + ".w2", H * D, rank).T + self.w(n + ".w0", H * D)
        decay, u = torch.exp(-torch.exp(z)).view(T, H, D, 1), self.w(n + ".u", H, D)[:, :, None]
        S, out = torch.zeros(H, D, D, device=DEV, dtype=torch.float64), torch.empty(T, H, D, device=DEV, dtype=torch.float64)
        for t in range(T):
            kv = k[t, :, :, None] * v[t, :, None, :]
            out[t] = ((S + u * kv) * r[t, :, :, None]).sum(1)
            S = decay[t] * S + kv
        out = _rms(out, 1.0, self.cfg["norm"]["eps"]).reshape(T, H * D)
        g = mixed["g"] @ self.w(n + ".g", H * D, width).T
        return (out * self.w(n + ".norm", H * D) * torch.nn.functional.silu(g)) @ self.w(n + ".o", width, H * D).T

    def logits(self, tokens, last):
        """of the last `last` of `tokens`"""
        cfg, width, eps = self.cfg, self.cfg["width"], self.cfg["norm"]["eps"]
        tefopel = cfg["architecture"] == "Tefopel"
        one = 1.0 if tefopel else 0.0
        x, store = self.w("embed", cfg["vocab"], width)[tokens], {}
        for i, ly in enumerate(cfg["layers"]):
            n, a = f"l{i}", ly["mixer"]
            h = _rms(x, one + self.w(n + ".norm1", width), eps)
            y = self.wkv(h, n + ".mix", a) if ly["type"] == "wkv" else self.tied(h, n + ".mix", a) if tefopel else self.latent(h, n + ".mix", a, store, i)
            x = x + (y if tefopel else _rms(y, self.w(n + ".norm1b", width), eps))
            if ly["mlp"] is None:
                continue
            h, ff, m = _rms(x, one + self.w(n + ".norm2", width), eps), ly["mlp"]["ff"], n + ".mlp"
            if tefopel:
                x = x + torch.relu(h @ self.w(m + ".up", ff, width).T).square() @ self.w(m + ".down", width, ff).T
            else:
                g = torch.nn.functional.gelu(h @ self.w(m + ".gate", ff, width).T + self.w(m + ".gate.b", ff), approximate="tanh")
                y = (g * (h @ self.w(m + ".up", ff, width).T + self.w(m + ".up.b", ff))) @ self.w(m + ".down", width, ff).T + self.w(m + ".down.b", width)
                x = x + _rms(y, self.w(n + ".norm2b", width), eps)
        out = _rms(x[-last:], one + self.w("final.norm", width), eps) @ self.w("embed", cfg["vocab"], width).T
        cap = cfg.get("logit_softcap")
        return out if cap is None else cap * torch.tanh(out / cap)


def _ragged(c):
    """how many tokens each request of a ragged batch brings: uneven shares, odd ones among them"""
    shares = [1.0 + 1.7 * (i * 0.618 % 1.0) for i in range(c["batch"])]
    lens = [max(1, int(c["tokens"] * s / sum(shares))) for s in shares]
    lens[0] += c["tokens"] - sum(lens)
    return lens


# ------------------------------------------------------------------------------------------------
@torch.no_grad()
def prepare(case, seed):
    c, path = case, case["path"]
    if path == "gemv":
        from teal_amd.monkeypatch import to_column_major
        dtype = DTYPES[c["dtype"]]
        lin = torch.nn.Linear(1, 1, bias=False)
        lin.weight = torch.nn.Parameter(_randn(seed, "w", (c["N"], c["Z"]), 0.02, dtype), requires_grad=False)
        to_column_major(lin)
        x = _randn(seed, "x", (1, 1, c["Z"]), 1.0, dtype)
        return {"path": path, "x": x, "w": lin.weight, "tau": _gemv_tau(c)}
    if path == "llama_decode":
        from teal_amd.gpt_fast.engine import DecodeEngine
        from teal_amd.monkeypatch import monkeypatch_layer
        W = _LlamaWeights(c, seed)
        first = _tokens(seed, "first", 1, W.args.vocab_size)
        model = _llama_model(W, c["context"] + 16)
        ths = _thresholds(W, c, first)
        for i, layer in enumerate(model.layers):
            monkeypatch_layer(i, layer, c["sparsity"], None, DEV, thresholds=ths[i])
            kc, vc = layer.attention.kv_cache.k_cache, layer.attention.kv_cache.v_cache
            kc[0, :, : c["context"]], vc[0, :, : c["context"]] = W.caches(i, c["context"])
        eng = DecodeEngine(model, ths)
        eng.manual_seed(seed)
        return {"path": path, "model": model, "engine": eng, "first": first.to(torch.int32), "context": c["context"], "tokens": c["tokens"]}
    if path == "llama_prompt":
        from teal_amd.gpt_fast.generate import GraphedPrefill, relayout_for_engine
        from teal_amd.gpt_fast.prefill import FusedPrefill
        from teal_amd.monkeypatch import monkeypatch_layer
        W = _LlamaWeights(c, seed)
        model = _llama_model(W, c["tokens"] + 64)
        for i, layer in enumerate(model.layers):  # (a prompt is dense: the thresholds are for the tokens after it)
            monkeypatch_layer(i, layer, 0.5, None, DEV, thresholds=dict.fromkeys(("q", "k", "v", "o", "gate", "up", "down"), 0.5))
        relayout_for_engine(model)
        return {"path": path, "model": model, "prefill": FusedPrefill(model, graph=True, fallback=GraphedPrefill(model)),
                "prompt": _tokens(seed, "prompt", c["tokens"], W.args.vocab_size).to(torch.int32)}
    model = _layered_model(c, seed)
    vocab = model.config.vocab_size
    if path == "layered_step":
        from teal_amd import runtime
        runtime.init()
        model.setup_caches(c["batch"], c["context"] + 8)
        toks = _tokens(seed, "prompt", c["batch"] * (c["context"] + 1), vocab).view(c["batch"], -1)
        every = toks[:, : c["context"]]
        portion = max(1, 8192 // c["batch"])  # (the prompts enter in portions)
        for lo in range(0, c["context"], portion):
            hi = min(c["context"], lo + portion)
            if hi - lo == 1:
                model(every[:, lo:hi].to(torch.int32), torch.tensor([lo], device=DEV, dtype=torch.int32))
            else:
                model(every[:, lo:hi], torch.arange(lo, hi, device=DEV))
        idx, pos = torch.zeros(c["batch"], 1, device=DEV, dtype=torch.int32), torch.zeros(1, device=DEV, dtype=torch.int32)
        new, at = toks[:, -1:].to(torch.int32), torch.tensor([c["context"]], device=DEV, dtype=torch.int32)
        idx.copy_(new)
        pos.copy_(at)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model(idx, pos)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with runtime.graph_capture(graph):
            logits = model(idx, pos)
        return {"path": path, "model": model, "graph": graph, "idx": idx, "pos": pos, "new": new, "at": at, "logits": logits}
    if path == "layered_prompt":
        from teal_amd.gpt_fast.serving import BatchEngine
        lens = _ragged(c)
        toks = _tokens(seed, "prompt", c["tokens"], vocab).tolist()
        prompts = [toks[sum(lens[:i]):sum(lens[: i + 1])] for i in range(len(lens))]
        return {"path": path, "engine": BatchEngine(model, max_tokens=c["tokens"] + 64 * c["batch"], max_requests=c["batch"], graphs=True), "prompts": prompts}
    from teal_amd.gpt_fast.generate import EngineDecoder
    model.setup_caches(1, c["tokens"] + c["new"])
    return {"path": path, "model": model, "decoder": EngineDecoder(model, None, True, 0.8, 200), "prefill": model.prefill(graph=True), "new": c["new"],
            "prompt": _tokens(seed, "prompt", c["tokens"], vocab).to(torch.int32)}


def _gemv_tau(c):
    """|N(0, 1)| is below this in a `sparsity` share of cases"""
    return float("%.4g" % (math.sqrt(2) * torch.erfinv(torch.tensor(c["sparsity"], dtype=torch.float64)).item()))


def _kept(cache):
    """what a batch leaves for its next tokens: cached rows and recurrent states"""
    return {"rows": [cache.pools[i] for i in sorted(cache.pools)], "states": [cache.states[i] for i in sorted(cache.states)]}


@torch.no_grad()
def run(state):
    s, path = state, state["path"]
    if path == "gemv":
        from teal_amd.kernels.sparse_gemv import splitk_sparse_gemv
        return splitk_sparse_gemv(s["x"], s["w"], s["tau"], 0)
    if path == "llama_decode":
        eng = s["engine"]
        tokens = eng.decode_n(s["first"], s["context"], s["tokens"], temperature=0.8, top_k=200)
        caches = [layer.attention.kv_cache for layer in s["model"].layers]
        return {"tokens": tokens, "logits": eng.logits, "k": [x.k_cache for x in caches], "v": [x.v_cache for x in caches]}
    if path == "llama_prompt":
        logits = s["prefill"](s["prompt"])
        caches = [layer.attention.kv_cache for layer in s["model"].layers]
        return {"logits": logits, "k": [x.k_cache for x in caches], "v": [x.v_cache for x in caches]}
    if path == "layered_step":
        s["idx"].copy_(s["new"])
        s["pos"].copy_(s["at"])
        s["graph"].replay()
        return {"logits": s["logits"], **_kept(s["model"].cache)}
    if path == "layered_prompt":
        logits = s["engine"].step([(i, p, [len(p) - 1]) for i, p in enumerate(s["prompts"])])
        for i in range(len(s["prompts"])):
            s["engine"].release(i)
        return {"logits": logits, **_kept(s["engine"].cache)}
    from teal_amd.gpt_fast.generate import generate
    tokens = generate(s["model"], s["prompt"], s["new"], s["decoder"], temperature=0.8, top_k=200, prefill=s["prefill"])
    return {"tokens": tokens, "logits": s["decoder"].model.logits}


@torch.no_grad()
def exact(case, seed):
    c, path = case, case["path"]
    if path == "gemv":
        dtype = DTYPES[c["dtype"]]
        w, x = _randn(seed, "w", (c["N"], c["Z"]), 0.02, dtype), _randn(seed, "x", (1, 1, c["Z"]), 1.0, dtype)
        return (x.double() * (x.float().abs() > torch.tensor(_gemv_tau(c), dtype=torch.float32, device=DEV))) @ w.double().T
    if path in ("llama_decode", "llama_prompt"):
        W = _LlamaWeights(c, seed)
        a, decode = W.args, path == "llama_decode"
        start = c["context"] if decode else 0
        if decode:
            first = _tokens(seed, "first", 1, a.vocab_size)
            tokens = (first + torch.arange(c["tokens"] + 1, device=DEV)) % a.vocab_size
            logits, rows, _ = _llama(W, tokens[:-1], start, torch.float64, thresholds=_thresholds(W, c, first))
        else:
            logits, rows, _ = _llama(W, _tokens(seed, "prompt", c["tokens"], a.vocab_size), 0, torch.float64)
        seq = -(-(start + 16 if decode else c["tokens"] + 64) // 8) * 8
        out = {"k": [], "v": []}
        for i, pair in enumerate(rows):
            before = W.caches(i, start) if start else (None, None)
            for name, old, new in zip(("k", "v"), before, pair):
                t = torch.zeros(1, a.n_local_heads, seq, a.head_dim, device=DEV, dtype=torch.float64)
                if old is not None:
                    t[0, :, :start] = old.double()
                t[0, :, start:start + new.shape[0]] = new.transpose(0, 1)
                out[name].append(t)
        if decode:
            return {"tokens": tokens[1:].to(torch.int32), "logits": logits[-1:].view(1, 1, -1), **out}
        return {"logits": (logits[-1:] if c["tokens"] <= 16 else logits).unsqueeze(0), **out}  # (a short prompt's pass returns its last token's)
    M = _Layered(c, seed)
    vocab = M.cfg["vocab"]
    if path == "layered_step":
        toks = _tokens(seed, "prompt", c["batch"] * (c["context"] + 1), vocab).view(c["batch"], -1)
        return {"logits": torch.cat([M.logits(t, 1) for t in toks])}
    if path == "layered_prompt":
        return {"logits": torch.cat([M.logits(t, 1) for t in _tokens(seed, "prompt", c["tokens"], vocab).split(_ragged(c))])}
    prompt = _tokens(seed, "prompt", c["tokens"], vocab)
    tokens = torch.cat([prompt, prompt[-1:].expand(c["new"])])  # (tied embeddings: a token follows itself)
    return {"tokens": tokens.to(torch.int32), "logits": M.logits(tokens[:-1], 1).view(1, 1, -1)}


# ------------------------------------------------------------------------------------------------
def _layered_sizes(c):
    """(weights of all layers without the head, head, per layer and token of context: cached elements, score and value flops)"""
    cfg = _layered_config(c)
    d, total, cached, attend, window = cfg["width"], 0, 0, 0, 1
    for ly in cfg["layers"]:
        a = ly["mixer"]
        if ly["type"] == "wkv":
            total += 5 * d * a["heads"] * a["dim"] + a["decay_rank"] * (d + a["heads"] * a["dim"])
        elif ly["type"] == "attention":
            total += d * a["dim"] * (2 * a["heads"] + a["kv_heads"])
            cached += a["kv_heads"] * (a["dim"] + a["rot"]["dims"])
            attend += 4 * a["heads"] * a["dim"]
            window = a["mask"]["size"]
        else:
            total += d * a["heads"] * (a["dim"] + a["rot_dim"] + 2 * a["vdim"]) + a["heads"] * a["kv_rank"] * (a["dim"] + a["vdim"])
            total += 0 if a.get("kv_from") is not None else d * (a["kv_rank"] + a["rot_dim"])
            cached += a["kv_rank"] + a["rot_dim"]
            attend += 2 * a["heads"] * (a["dim"] + a["rot_dim"] + a["vdim"])
            window = a["mask"]["size"]
        if ly["mlp"] is not None:
            total += (2 if cfg["architecture"] == "Tefopel" else 3) * d * ly["mlp"]["ff"]
    return total, d * cfg["vocab"], cached, attend, window


def work(case):
    c, path = case, case["path"]
    if path == "gemv":
        kept = (1 - c["sparsity"]) * c["Z"] * c["N"]
        return {"bytes": 2 * (kept + c["Z"] + c["N"]), "flops": 2 * kept}
    if path in ("llama_decode", "llama_prompt"):
        from teal_amd.gpt_fast.model import ModelArgs
        a = ModelArgs.from_name(c["model"])
        kv = a.n_local_heads * a.head_dim
        layer = a.dim * (2 * a.dim + 2 * kv) + 3 * a.dim * a.intermediate_size
        total, head, T = c["n_layer"] * layer, a.dim * a.vocab_size, c["tokens"]
        if path == "llama_decode":
            size = {16: 2.0, 8: 1.0, 4: 0.625}[c["weights"]]
            kept = (1 - c["sparsity"]) * total
            past = c["n_layer"] * 2 * kv * c["context"]
            return {"bytes": T * (kept * size + head * (1 if c["weights"] == 8 else 2) + 2 * past), "flops": T * 2 * (kept + head + past * a.n_head // a.n_local_heads)}
        shown = 1 if T <= 16 else T
        return {"bytes": 2 * (total + head + T * (2 * kv * c["n_layer"] + a.dim) + shown * a.vocab_size),
                "flops": 2 * T * total + 2 * shown * head + 2 * T * T * a.dim * c["n_layer"]}
    total, head, cached, attend, window = _layered_sizes(c)
    if path == "layered_step":
        past = c["batch"] * min(c["context"], window)
        return {"bytes": 2 * (total + head + past * cached) + 4 * c["batch"] * _layered_config(c)["vocab"], "flops": c["batch"] * 2 * (total + head) + past * attend}
    if path == "layered_prompt":
        return {"bytes": 2 * (total + head + c["tokens"] * cached), "flops": 2 * c["tokens"] * total + 2 * c["batch"] * head + sum(n * n // 2 for n in _ragged(c)) * attend}
    T, new = c["tokens"], c["new"]
    return {"bytes": new * 2 * (total + head), "flops": 2 * (T + new) * total + 2 * new * head + (T + new) ** 2 // 2 * attend}


def tolerance(case):
    # about four times the distance from 64 bits (`exact`), measured: 16-bit activations between the layers, and where inputs are masked
    # a value next to its threshold that falls on either side of it
    half = case["dtype"] == "fp16"
    if case["path"] == "gemv":
        return {"rel": 0.001 if half else 0.007}
    if case["path"] == "llama_decode":
        return {"rel": 0.03, "differ": 0.0}
    return {"rel": 0.006 if half else 0.03, "differ": 0.0}
