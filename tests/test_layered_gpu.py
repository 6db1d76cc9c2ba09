"""GPU: the layered designs against the plain restatement (oracle/layered_oracle.py, float64): whole prompts, token by token, portions,
unequal batches, reused pages and states, the fused step and its graphs, sampling, the scheduler, the command line and the trace replay.

32-bit models are held to 2e-5 of the logits' rms per position, which tells every mechanism apart (tests/test_layered.py plants
mistakes in the oracle); 16-bit models to their rounding."""
import copy
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from layered_models import CONFIGS, TEFOPEL, error, random_config, random_tefopel, random_tensors, random_tokens, save_checkpoint
from oracle import layered_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
TOL = {F32: 2e-5, BF16: 0.06, F16: 0.01}


def close(e, dtype):
    """per-position errors within the format's tolerance; in 16 bits a query whose two best keys nearly tie may stand out by rounding
    alone, so there one position in ten may exceed it, six-fold at most (a wrong key is an error of order 1)"""
    if dtype == F32:
        return float(e.max()) < TOL[dtype]
    return float(e.max()) < 6 * TOL[dtype] and int((e > TOL[dtype]).sum()) <= max(1, len(e) // 10)


_cache = {}


def setup(name, dtype, tmp_path_factory):
    """(config, tensors, model on the GPU, {(T, seed): (tokens, oracle logits)}) — built once per session"""
    from teal_amd import runtime
    from teal_amd.gpt_fast import registry
    runtime.init()
    key = (name, dtype)
    if key not in _cache:
        cfg = CONFIGS[name]
        t = random_tensors(cfg, 1)
        path = save_checkpoint(tmp_path_factory.mktemp(name), cfg, t)
        _cache[key] = (cfg, t, registry.load_model(path, DEV, dtype))
    return _cache[key]


def expected(name, cfg, t, n, seed):
    key = ("want", name, n, seed)
    if key not in _cache:
        toks = random_tokens(cfg, n, seed)
        _cache[key] = (toks, O.forward(cfg, t, toks))
    return _cache[key]


def poison(eng):
    """NaN in every cache row no live sequence has written, in every free slot's state and in the half of a live one's that the next token
    does not read: nothing may read them"""
    used = np.zeros(eng.cache.n_pages * 64, dtype=bool)
    for s, pages in enumerate(eng.cache.slots):
        if pages is not None:
            pos = np.arange(eng.cache.lengths[s])
            pos = pos[np.asarray([pages[p >> 6] >= 0 for p in pos], dtype=bool)] if len(pos) else pos
            used[eng.cache.rows(s, pos)] = True
    rows = torch.from_numpy(np.nonzero(~used)[0]).to(DEV)
    for layer, pool in eng.cache.pools.items():
        pool[rows] = float("nan")
    for state in eng.cache.states.values():
        for s, pages in enumerate(eng.cache.slots):
            if pages is None or eng.cache.lengths[s] == 0:
                state[s] = float("nan")
            else:
                state[s, eng.cache.lengths[s] & 1] = float("nan")


def engine(model, **kw):
    from teal_amd.gpt_fast.serving import BatchEngine
    return BatchEngine(model, **{"max_tokens": 256, "max_requests": 2, **kw})


ALL = [(n, d) for n in CONFIGS for d in (F32, BF16)] + [("even", F16), ("heads", F16), ("t-even", F16)]


def widest(cfg):
    """the widest window of a configuration"""
    return max((ly["mixer"]["mask"]["size"] for ly in cfg["layers"] if "mask" in ly["mixer"]), default=1)


# ---- row kernels -------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
@pytest.mark.parametrize("D", [64, 70, 2048, 5120])
def test_residual_norm_rows(dtype, D):
    from teal_amd.kernels import layered as K
    T, V, eps = 9, 40, 1e-3
    r = lambda *s: torch.randn(*s, device=DEV)  # noqa: E731
    emb, y, bias = r(V, D).to(dtype), (3 * r(T, D)).to(dtype), r(D).to(dtype)
    post, pre = (1 + 0.2 * r(D)).to(dtype), (1 + 0.2 * r(D)).to(dtype)
    tok = torch.randint(0, V, (T,), device=DEV, dtype=torch.int32)
    x = torch.full((T, D), float("nan"), device=DEV)
    h = K.resid_norm(x, tokens=tok, embed=emb, pre_w=pre, eps=eps)
    assert torch.equal(x, emb[tok.long()].float())
    ref = O.rms_norm(x.double(), pre.double(), eps)
    tol = 1e-5 if dtype == F32 else 2 ** -8 if dtype == BF16 else 2 ** -10
    assert h.dtype == dtype and ((h.double() - ref).abs() <= tol * (1 + ref.abs())).all()
    want = x.double() + O.rms_norm(y.double() + bias.double(), post.double(), eps)
    x2 = x.clone()
    h = K.resid_norm(x2, y=y, y_bias=bias, post_w=post, pre_w=pre, eps=eps)
    assert (x2.double() - want).abs().max() < 1e-5
    ref = O.rms_norm(want, pre.double(), eps)
    assert ((h.double() - ref).abs() <= tol * (1 + ref.abs())).all()
    x3, rows = x.clone(), torch.tensor([7, 0, 3], device=DEV, dtype=torch.int32)  # a subset, packed; the other rows stay
    h3 = K.resid_norm(x3, y=y, y_bias=bias, post_w=post, pre_w=pre, eps=eps, rows=rows)
    assert torch.equal(h3, h[rows.long()]) and torch.equal(x3[1], x[1]) and torch.equal(x3[7], x2[7])
    x4 = x.clone()
    assert K.resid_norm(x4, y=y, dtype=dtype) is None and torch.allclose(x4, x + y.float(), atol=1e-6)  # no norms: a plain add


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("n,up0", [(128, 128), (77, 90), (4104, 4104)])
def test_gated_activation_and_soft_cap(dtype, n, up0):
    from teal_amd.kernels import layered as K
    gu, b = (2 * torch.randn(5, up0 + n, device=DEV)).to(dtype), torch.randn(up0 + n, device=DEV).to(dtype)
    g, u = gu[:, :n].double(), gu[:, up0:up0 + n].double()
    tol = 1e-5 if dtype == F32 else 2 ** -7
    for act, f in (("gelu_tanh", O.gelu_tanh), ("silu", torch.nn.functional.silu)):
        ref = f(g + b[:n].double()) * (u + b[up0:up0 + n].double())
        assert ((K.gated_act(gu, n, up0, act, b).double() - ref).abs() <= tol * (1 + ref.abs())).all()
        ref = f(g) * u
        assert ((K.gated_act(gu, n, up0, act).double() - ref).abs() <= tol * (1 + ref.abs())).all()
    z = (9 * torch.randn(3, n + 8, device=DEV)).to(dtype)
    assert torch.allclose(K.softcap(z, n, 5.0).double(), 5 * torch.tanh(z[:, :n].double() / 5), atol=1e-5)
    assert torch.equal(K.softcap(z, n, None), z[:, :n].float())


@pytest.mark.parametrize("V", [33, 1000, 32000, 128256])
def test_sampler_rows(V):
    from teal_amd.kernels import layered as K
    B = 4
    x = 3 * torch.randn(B, V + 3, device=DEV)[:, :V]
    x[1] = x[1].round()               # ties everywhere
    x[2] *= 1e-3                      # a flat row
    x[3, : V // 2] = -50.0
    rng = torch.tensor([[11 + i, 0] for i in range(B)], device=DEV)
    pos, hist = torch.zeros(B, dtype=torch.int32, device=DEV), torch.full((B, 6), -1, dtype=torch.int32, device=DEV)
    assert torch.equal(K.sample_rows(x, rng.clone(), 0.0, None).long(), x.argmax(-1))
    for k in (1, 2, 7, min(200, V - 1), V):
        kth = x.topk(k, -1).values[:, -1:]
        allowed = x >= kth
        for rep in range(6):
            t = K.sample_rows(x, rng, 1.5, k, pos=pos, history=hist).long()
            assert allowed.gather(1, t[:, None]).all(), (V, k)
    assert (pos == 30).all() and (rng[:, 1] == 30).all() and (hist >= 0).all()
    # the frequencies of a small distribution
    p = torch.tensor([[0.5, 0.25, 0.15, 0.1]], device=DEV)
    rng = torch.tensor([[5, 0]], device=DEV)
    n = torch.zeros(4)
    for _ in range(1500):
        n[int(K.sample_rows(p.log() * 0.7, rng, 0.7, None))] += 1
    assert (n / 1500 - p[0].cpu()).abs().max() < 0.05


@pytest.mark.parametrize("V", [4, 4096, 8192, 8196, 32768, 32772])
def test_sampler_rows_in_registers(V):
    """rows that the sampler keeps in registers (aligned, whole 16 bytes) draw the same tokens as those it reads from memory on each pass, at the
    ends of each register count; with ties, infinities, NaN and rows of one value"""
    from teal_amd.kernels import layered as K
    x = 3 * torch.randn(6, V, device=DEV)
    x[1] = x[1].round()
    x[2] = 0.25
    x[3, ::3], x[3, 1::7] = float("nan"), -float("inf")
    x[4, V // 2] = float("inf")
    x[5] = float("nan")
    loose = torch.empty(6, V + 1, device=DEV)[:, :V].copy_(x)
    rng = torch.tensor([[11 + i, 0] for i in range(6)], device=DEV)
    for temperature, k in ((0.0, None), (1.5, None), (0.8, 1), (0.8, min(200, V - 1)), (1e3, V - 1)):
        for rep in range(3):
            r2 = rng.clone()
            assert torch.equal(K.sample_rows(x, rng, temperature, k), K.sample_rows(loose, r2, temperature, k)), (temperature, k)
            assert torch.equal(rng, r2)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("B,heads,dim,rot,vdim,rank", [(5, 26, 32, 8, 33, 32), (16, 8, 96, 0, 64, 272), (17, 8, 128, 64, 100, 512), (33, 4, 160, 16, 17, 544), (8, 16, 64, 24, 128, 2048)])
def test_step_products_on_matrix_cores(B, heads, dim, rot, vdim, rank, dtype):
    """the absorbed query and the merge of several tokens at the ends of their tiles (16 and 4 tokens, 64 columns, 4 and 16 steps), with sink and gate and splits
    that got nothing.  The query's two halves: fp32 sums of exact products, then half a step of the low part; the merge: one rounding at the end, of fp32 sums
    (every partial sum is below the sum of the sizes: 2^-19 of it)"""
    from teal_amd.kernels import layered as K
    from teal_amd import runtime
    runtime.init()
    torch.manual_seed(B)
    r = lambda *s: torch.randn(*s, device=DEV)  # noqa: E731
    ldq, nq, pages = -(-(rank + rot) // 32) * 32, heads * (dim + rot), 3
    ldp = -(-(nq + rank + rot) // 8) * 8
    proj, uk, uv = r(B, ldp).to(dtype), (0.1 * r(heads * dim, rank)).to(dtype), (0.1 * r(heads * vdim, rank)).to(dtype)
    pos = torch.randint(0, 64 * pages, (B,), device=DEV, dtype=torch.int32)
    slot, table = torch.randperm(B, device=DEV).int(), torch.randperm(B * pages, device=DEV).int().view(B, pages).contiguous()
    inv, norm_w = torch.rand(max(1, rot // 2), device=DEV), r(rank).to(dtype)
    qcat = torch.full((B, heads, 2, ldq), 7.0, device=DEV, dtype=dtype)
    caches = [torch.full((B * pages * 64, ldq), 3.0, device=DEV, dtype=dtype) for _ in range(2)]
    K.latent_step_query(proj, nq, pos, slot, table, 6, inv, norm_w, 1e-5, uk, heads, dim, rot, rank, caches[0], qcat)
    one = torch.full((B, heads, 2, ldq), 9.0, device=DEV, dtype=dtype)
    for b in range(B):  # token by token: the kernel of few tokens
        K.latent_step_query(proj[b:b + 1], nq, pos[b:b + 1], slot[b:b + 1], table, 6, inv, norm_w, 1e-5, uk, heads, dim, rot, rank, caches[1], one[b:b + 1])
    assert torch.equal(caches[0], caches[1])
    assert torch.equal(qcat[..., rank:], one[..., rank:])
    q = proj[:, :nq].view(B, heads, dim + rot)[..., :dim].double()
    w = uk.double().view(heads, dim, rank)
    want = torch.stack([q[:, h] @ w[h] for h in range(heads)], 1)
    size = torch.stack([q[:, h].abs() @ w[h].abs() for h in range(heads)], 1)
    got = qcat[..., :rank].double().sum(2)
    step = 2.0 ** (-22 if dtype is F16 else -16)
    assert ((got - want).abs() <= step * want.abs() + 2.0 ** -19 * size + 2.0 ** -24).all()
    for splits in (1, 7, 20):
        part = torch.full((B, heads, splits, (rank + 3) // 4 * 4 + 4), float("nan"), device=DEV)
        part[..., :rank], part[..., -4], part[..., -3] = r(B, heads, splits, rank), 3 * r(B, heads, splits), 1 + torch.rand(B, heads, splits, device=DEV)
        if splits > 1:
            part[1, :, splits - 1, :rank], part[1, :, splits - 1, -4], part[1, :, splits - 1, -3] = 0.0, -float("inf"), 0.0
        for sink, gate in ((None, None), (r(heads).to(dtype), r(B, heads * vdim + 5).to(dtype)[:, :heads * vdim])):
            y = torch.full((B + 1, heads * vdim + 3), 7.0, device=DEV, dtype=dtype)
            K.latent_step_merge(part, splits, uv, sink, gate, y[:B], B, heads, rank, vdim)
            f = torch.exp2(part[..., -4].double())
            den = (f * part[..., -3].double()).sum(-1) + (0 if sink is None else sink.double().exp())
            o = (part[..., :rank].double() * f[..., None]).sum(2) / den[..., None]
            big = (part[..., :rank].double().abs() * f[..., None]).sum(2) / den[..., None]
            v = uv.double().view(heads, vdim, rank)
            want = torch.stack([o[:, h] @ v[h].T for h in range(heads)], 1).reshape(B, -1)
            size = torch.stack([big[:, h] @ v[h].abs().T for h in range(heads)], 1).reshape(B, -1)
            if gate is not None:
                want = want * gate.double().sigmoid()
            err = (y[:B, :heads * vdim].double() - want).abs()
            assert (err <= 2.0 ** (-11 if dtype is F16 else -8) * want.abs() + 2.0 ** -19 * size + 2.0 ** -24).all(), (splits, float(err.max()))
            assert (y[B] == 7).all() and (y[:, heads * vdim:] == 7).all()


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("dim,rot,vdim,cap", [(128, 64, 128, None), (40, 8, 72, None), (64, 0, 64, 30.0), (136, 48, 200, None), (192, 64, 256, 80.0), (96, 16, 104, 20.0)])
def test_prompt_attention_by_pieces_and_by_elements(dim, rot, vdim, cap, dtype):
    """rows in whole 16 bytes are loaded in pieces, others element by element: the same products in the same order, so the same results.  Portions
    that end inside a tile, a window, 64 and 128 queries to a workgroup; keys past a portion's last are never seen (they are NaN)"""
    from teal_amd.kernels import layered as K
    from teal_amd import runtime
    runtime.init()
    torch.manual_seed(dim)
    heads, group = 4, 2
    spans = [(0, 130, 70, 0, 0), (130, 1, 0, 256, 0), (131, 77, 0, 320, 0)]  # q0, nq, start, k0, klo (keys padded to 64 rows)
    T, S = 208, 320 + 128
    r = lambda *s: torch.randn(*s, device=DEV).to(dtype)  # noqa: E731
    q, k, vt = r(T, heads * (dim + rot)), r(S, heads // group * dim), r(heads // group * vdim, S)
    kr, gate, sink = (r(S, rot) if rot else None), r(T, heads * vdim), r(heads)
    for q0, nq, start, k0, klo in spans:
        end = k0 + start + nq - klo
        k[end:k0 + -(-(end - k0) // 64) * 64] = float("nan")
    loose = torch.empty(T, heads * (dim + rot) + 3, device=DEV, dtype=dtype)[:, :heads * (dim + rot)].copy_(q)
    seqs = torch.tensor(spans, dtype=torch.int32, device=DEV)
    for tile in (64, 128) if vdim <= 128 else (64,):
        tiles = torch.tensor([(i, a) for i, s in enumerate(spans) for a in range(0, s[1], tile)], dtype=torch.int32, device=DEV)
        for window in (1 << 30, 50):
            out = [torch.zeros(T, heads * vdim, device=DEV, dtype=dtype) for _ in range(2)]
            for y, x in zip(out, (q, loose)):
                K.prompt_attention(x, k, kr, vt, sink, gate, y, seqs, tiles, tile, heads, dim, rot, vdim, window, (dim + rot) ** -0.5, group=group, softcap=cap)
            assert out[0].isfinite().all() and out[0].abs().sum() > 0
            assert torch.equal(out[0], out[1])


# ---- the mixer alone: one key stands out ----------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("window", [1, 2, 63, 64, 65, 96, 300])
def test_a_key_at_the_windows_edge(dtype, window):
    """Query p asks for the key of position j with a score far above all others, j just inside and just outside the window, at page
    borders and at the start: the answer is j's value inside, anything else's outside.  In the prompt pass and in the step."""
    from teal_amd import runtime
    from teal_amd.gpt_fast.layered import LayeredArgs, LayeredTransformer, PromptBatch, StepBatch, _empty
    from layered_models import config, mixer
    runtime.init()
    H, D, R, V, rank, T, W = 2, 16, 8, 16, 64, 200, 64
    cfg = config(W, 16, [(mixer(H, D, R, V, rank, window, scale=1.0), None)])
    t = random_tensors(cfg, 9)
    t["l0.mix.sink"] = torch.tensor([-1.0, 2.0]).to(torch.bfloat16)
    model = _empty(LayeredArgs.from_dict(cfg), DEV, dtype)
    model.load_tensors(lambda n: t[n].to(DEV, dtype))
    mix = model.layers[0].mix
    Wd = {k: v.double() for k, v in t.items()}
    h = torch.randn(T, W, dtype=torch.float64).to(torch.bfloat16).double()
    a = cfg["layers"][0]["mixer"]
    # the input of query p is built so that W_uk^T W_q h has a large component along j's latent (a least-squares preimage)
    pairs = [(p, p - d) for p in (40, 63, 64, 65, 127, 128, 130, 199) for d in (0, window - 1, window, window // 2) if p - d >= 0]
    pairs += [(window - 1, 0), (window, 0)] if window < T else [(150, 0)]
    h = h.clone()
    seen = set()
    plan = []
    for p, j in pairs:
        if p in seen or p == j:
            continue
        seen.add(p)
        plan.append((p, j))
    targets = {j for _, j in plan}
    plan = [(p, j) for p, j in plan if p not in targets]  # (a target's own input stays as it is)
    c, kr = O.latents(h, Wd, "l0.mix", a, cfg["norm"]["eps"])
    M = torch.cat([Wd["l0.mix.uk"][n * D:(n + 1) * D].T @ Wd["l0.mix.q"].view(H, D + R, W)[n, :D] for n in range(H)])  # [H rank, W]
    for p, j in plan:
        h[p] = (torch.linalg.lstsq(M, torch.cat([c[j]] * H)[:, None]).solution[:, 0] * 3).to(torch.bfloat16).double()
    c, kr = O.latents(h, Wd, "l0.mix", a, cfg["norm"]["eps"])
    want = O.latent_attention(h, c, kr, Wd, "l0.mix", a)
    wide = O.latent_attention(h, c, kr, Wd, "l0.mix", dict(a, mask={"size": window + 1}))
    moved = (wide - want).norm(dim=-1) / want.norm(dim=-1)
    if window < T - 1:
        assert float(moved.max()) > 0.5  # a window one token wider answers otherwise somewhere
    tol = 5e-5 if dtype == F32 else 0.1
    cache = model.new_cache(T, 1)
    s = cache.open()
    cache.extend(s, T)
    cache.sync()
    hd = h.to(DEV, dtype)
    got = mix.prompt(hd, PromptBatch(cache, [(s, 0, [0] * T)], DEV))
    rel = lambda g, w: ((g.double().cpu() - w).norm(dim=-1) / want.norm(dim=-1).mean()).max()  # noqa: E731
    assert float(rel(got, want)) < tol
    for pool in cache.pools.values():
        pool.zero_()
    out = []
    for p in range(T):
        b = StepBatch(cache, torch.zeros(1, dtype=torch.int32, device=DEV), torch.tensor([p], dtype=torch.int32, device=DEV),
                      torch.tensor([s], dtype=torch.int32, device=DEV), p)
        out.append(mix.step(hd[p:p + 1], b))
    assert float(rel(torch.cat(out), want)) < tol


def test_no_window_and_no_sink(tmp_path_factory):
    """the mixer's options: attention over everything before a position, and a softmax without a sink"""
    from teal_amd.gpt_fast.layered import LayeredArgs, _empty
    from layered_models import config, mixer
    cfg = config(64, 50, [(mixer(2, 16, 8, 16, 32, 0), 64)])
    del cfg["layers"][0]["mixer"]["mask"]
    t = random_tensors(cfg, 4)
    toks = random_tokens(cfg, 150, 1)
    for sink in (True, False):
        args = LayeredArgs.from_dict(cfg)
        args.layers[0].mixer.sink = sink
        model = _empty(args, DEV, F32).load_tensors(lambda n: t[n].to(DEV, F32))
        tt = t if sink else dict(t, **{"l0.mix.sink": torch.full_like(t["l0.mix.sink"], -1e4)})
        want = O.forward(cfg, tt, toks)
        eng = engine(model)
        assert float(error(eng.step([(0, toks[:90], range(90))]), want[:90]).max()) < TOL[F32]
        for p in range(90, 150):
            assert float(error(eng.step([(0, toks[p:p + 1], [0])]), want[p:p + 1]).max()) < TOL[F32] * 3


# ---- time mixing: every kernel alone -------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
@pytest.mark.parametrize("W", [64, 70, 2048, 4096])
def test_token_shift(dtype, W):
    """whole sequences, portions of even and odd length (down to one token), two sequences side by side; over poisoned state"""
    from teal_amd.kernels import layered as K
    eps, n = 1e-3, 11
    nw, mu = (0.3 * torch.randn(W, device=DEV)).to(dtype), torch.rand(5, W, device=DEV).to(dtype)
    x = torch.randn(2, n, W, device=DEV) * 2
    h = O.rms_norm(x.double().cpu(), 1 + nw.double().cpu(), eps)
    want = torch.stack([torch.stack([O.token_shift(h[b], m) for m in mu.double().cpu()]) for b in range(2)])
    tol = 1e-5 if dtype == F32 else 2 ** -8 if dtype == BF16 else 2 ** -10
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    for cuts in ([11], [4, 7], [1, 2, 1, 3, 4], [1] * 11):
        shift = torch.full((5, 2, W), float("nan"), device=DEV)
        at = 0
        for c in cuts:
            rows = x[:, at:at + c].reshape(2 * c, W).contiguous()
            run = None if c == 1 else i32([c] + [0] * (c - 1)).repeat(2)
            got = K.wkv_mix(rows, nw, 1.0, eps, mu, i32(range(at, at + c)).repeat(2), i32([3] * c + [1] * c), run, shift)
            ref = want[:, :, at:at + c].transpose(0, 1).reshape(5, 2 * c, W)
            assert got.dtype == dtype and ((got.double().cpu() - ref).abs() <= tol * (1 + ref.abs())).all(), (cuts, at)
            at += c
            last = shift[[3, 1], (at - 1) & 1].double().cpu()
            assert (last - h[:, at - 1]).abs().max() < 1e-5 * h.abs().max()
        assert shift[[0, 2, 4]].isnan().all()


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("rank,C", [(5, 33), (16, 300), (64, 1024), (100, 40), (300, 70)])
def test_decays(dtype, rank, C):
    from teal_amd.kernels import layered as K
    z, w2, w0 = (1.5 * torch.randn(37, rank + 3, device=DEV)).to(dtype)[:, :rank], torch.randn(C, rank, device=DEV).to(dtype), (2 * torch.randn(C, device=DEV)).to(dtype)
    W = {"m.w1": torch.eye(rank, dtype=torch.float64), "m.w2": w2.double().cpu(), "m.w0": w0.double().cpu()}
    want = O.wkv_decay(z.double().cpu(), W, "m")
    got = K.wkv_decay(z, w2, w0)
    assert got.dtype == F32 and (got.double().cpu() - want).abs().max() < 2e-5


@pytest.mark.parametrize("dtype", [F32, BF16, F16])
@pytest.mark.parametrize("H,D", [(3, 5), (2, 16), (1, 24), (3, 32), (2, 64), (1, 100), (2, 128), (1, 250), (1, 256)])
def test_recurrence(dtype, H, D):
    """whole sequences, portions and single tokens give the recurrence's outputs and end in its state, in slots of any order; decays
    near 1 (a value from the start shows at the end) and near 0"""
    from teal_amd.kernels import layered as K
    n = 75
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    C = H * D
    r, k, v, g = ((torch.randn(2, n, C) * s).to(dtype) for s in (1, 1, 1, 1))
    k[:, 0], v[:, 0] = 4.0, 4.0  # (the first token's pair stands out)
    u, norm = torch.randn(H, D).to(dtype), (1 + 0.2 * torch.randn(C)).to(dtype)
    rank = 4
    z = torch.randn(2, n, rank).to(dtype)
    w2, w0 = torch.randn(C, rank).to(dtype), torch.where(torch.arange(C) % 3 == 0, 1.0, torch.where(torch.arange(C) % 3 == 1, -2.0, -7.0)).to(dtype)
    d = lambda x: x.double()  # noqa: E731
    W = {"m.w1": torch.eye(rank, dtype=torch.float64), "m.w2": d(w2), "m.w0": d(w0)}
    o, y = [], []
    for b in range(2):
        w = O.wkv_decay(d(z[b]), W, "m").view(n, H, D)
        ob = torch.stack([O.wkv_recurrence(*(d(t[b]).view(n, H, D)[:, h] for t in (r, k, v)), w[:, h], d(u)[h]) for h in range(H)], 1)
        o.append(ob.reshape(n, C))
        gb = d(g[b])
        y.append((ob / torch.sqrt((ob * ob).mean(-1, keepdim=True) + 1e-4)).reshape(n, C) * d(norm) * gb * torch.sigmoid(gb))
    dev = [t.to(DEV) for t in (r, k, v, g, z)]
    w2, w0, u, norm = (t.to(DEV) for t in (w2, w0, u, norm))
    rel = lambda a, b: float((a.double().cpu() - b).abs().max() / b.abs().max())  # noqa: E731
    ytol = 3e-5 if dtype == F32 else 2 ** -7 if dtype == BF16 else 2 ** -9
    slots = [2, 0]
    for cuts in ([75], [32, 43], [1, 2, 15, 17, 40], [16, 59]):
        state, at = torch.full((4, 2, H, D, D), float("nan"), device=DEV), 0
        for c in cuts:
            part = [t[:, at:at + c].reshape(2 * c, -1).contiguous() for t in dev]
            w = K.wkv_decay(part[4], w2, w0)
            got = K.wkv_scan(*part[:3], w, u, i32([[0, c, at, 0, 0], [c, c, at, 0, 0]]), i32([slots[0]] * c + [slots[1]] * c), state, c)
            ref = torch.cat([t[at:at + c] for t in o])
            assert rel(got, ref) < 2e-5, (cuts, at)
            gy = K.wkv_out(got, norm, part[3], 1e-4, torch.empty(2 * c, C, device=DEV, dtype=dtype), H, D)
            assert rel(gy, torch.cat([t[at:at + c] for t in y])) < ytol
            at += c
        whole = state[slots, (n - 1) & 1].clone()
        assert not whole.isnan().any() and state[[1, 3]].isnan().all()
    # after a prompt of 40: token by token
    state = torch.full((4, 2, H, D, D), float("nan"), device=DEV)
    part = [t[:, :40].reshape(80, -1).contiguous() for t in dev]
    K.wkv_scan(*part[:3], K.wkv_decay(part[4], w2, w0), u, i32([[0, 40, 0, 0, 0], [40, 40, 0, 0, 0]]), i32([slots[0]] * 40 + [slots[1]] * 40), state, 40)
    for start in (40, 0):
        for p in range(start, n if start else 3):
            r1, k1, v1, g1, z1 = (t[:, p].contiguous() for t in dev)
            for _ in range(2):  # (a repeated step repeats)
                gy = K.wkv_step(r1, k1, v1, g1, z1, w2, w0, u, norm, 1e-4, i32([p, p]), i32(slots), state, torch.empty(2, C, device=DEV, dtype=dtype))
            assert rel(gy, torch.stack([t[p] for t in y])) < ytol, p
        if start:
            assert rel(state[slots, (n - 1) & 1], whole.double().cpu()) < 1e-5
            state.fill_(float("nan"))


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("window", [1, 2, 63, 64, 65, 96, 300])
@pytest.mark.parametrize("heads,kv,dim,rot", [(2, 1, 32, 16), (2, 2, 32, 32), (3, 1, 20, 6)])
def test_a_tied_key_at_the_windows_edge(dtype, window, heads, kv, dim, rot):
    """Query p asks for the (rotated) key of position j far above all others, j just inside and just outside the window, at page borders and
    at the start; capped scores and a sink next to it.  In the prompt pass and in the step."""
    from teal_amd import runtime
    from teal_amd.gpt_fast.layered import LayeredArgs, PromptBatch, StepBatch, _empty
    from layered_models import tefopel, tied
    runtime.init()
    T, W = 200, 128
    cfg = tefopel(W, 16, [(tied(heads, kv, dim, rot, window, base=700.0, scale=0.7, cap=25.0), None)])
    t = random_tensors(cfg, 9, peak=1.0)
    t["l0.mix.sink"] = torch.linspace(-1, 3, heads).to(torch.bfloat16)
    model = _empty(LayeredArgs.from_dict(cfg), DEV, dtype).load_tensors(lambda n: t[n].to(DEV, dtype))
    mix, a = model.layers[0].mix, cfg["layers"][0]["mixer"]
    Wd = {k: v.double() for k, v in t.items()}
    h = torch.randn(T, W, dtype=torch.float64).to(torch.bfloat16).double()
    plan = {}  # query -> the position it asks for: the window's last, the first outside, one in the middle
    for i, p in enumerate((40, 63, 64, 65, 66, 100, 127, 128, 129, 130, 198, 199)):
        plan[p] = p - (window, window - 1, window, window // 2)[i % 4]
    plan.update({window - 1: 0, window: 0} if window < T else {150: 0})
    plan = {p: j for p, j in plan.items() if 0 <= j < p}
    plan = {p: j for p, j in plan.items() if p not in plan.values()}
    keys = (h @ Wd["l0.mix.k"].T).view(T, kv, dim)
    pinv = torch.linalg.pinv(Wd["l0.mix.q"])
    for p, j in plan.items():  # the query that, turned to p, points along the key turned to j
        turned = O.rotate_pairs(keys[j:j + 1], torch.tensor([j - p]), rot, 700.0)[0]
        h[p] = (pinv @ torch.cat([turned[n // (heads // kv)] for n in range(heads)])).to(torch.bfloat16).double()
    want = O.tied_attention(h, Wd, "l0.mix", a)
    moved = (O.tied_attention(h, Wd, "l0.mix", dict(a, mask={"size": window + 1})) - want).norm(dim=-1) / want.norm(dim=-1)
    if window < T - 1:
        assert float(moved.max()) > 0.5  # a window one token wider answers otherwise somewhere
    tol = 5e-5 if dtype == F32 else 0.1
    cache = model.new_cache(T, 1)
    s = cache.open()
    cache.extend(s, T)
    cache.sync()
    hd = h.to(DEV, dtype)
    got = mix.prompt(hd, PromptBatch(cache, [(s, 0, [0] * T)], DEV))
    rel = lambda g, w: ((g.double().cpu() - w).norm(dim=-1) / want.norm(dim=-1).mean()).max()  # noqa: E731
    assert float(rel(got, want)) < tol
    for pool in cache.pools.values():
        pool.zero_()
    out = []
    for p in range(T):
        b = StepBatch(cache, torch.zeros(1, dtype=torch.int32, device=DEV), torch.tensor([p], dtype=torch.int32, device=DEV),
                      torch.tensor([s], dtype=torch.int32, device=DEV), p)
        out.append(mix.step(hd[p:p + 1], b))
    assert float(rel(torch.cat(out), want)) < tol


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_squared_relu_and_norms_around_zero(dtype):
    from teal_amd.kernels import layered as K
    tol = 1e-5 if dtype == F32 else 2 ** -7
    for n in (128, 77, 4104):
        z = (2 * torch.randn(5, n, device=DEV)).to(dtype)
        ref = torch.relu(z.double()) ** 2
        got = K.gated_act(z, n, 0, "relu2")
        assert ((got.double() - ref).abs() <= tol * (1 + ref.abs())).all() and torch.equal(got == 0, ref.to(dtype) == 0)
        b = torch.randn(n, device=DEV).to(dtype)
        ref = torch.relu(z.double() + b.double()) ** 2
        assert ((K.gated_act(z, n, 0, "relu2", b).double() - ref).abs() <= tol * (1 + ref.abs())).all()
        x, w = torch.randn(5, n, device=DEV), (1e-2 * torch.randn(n, device=DEV)).to(dtype)  # (1 + w is no 16-bit number)
        got = K.resid_norm(x.clone(), pre_w=w, eps=1e-4, norm_offset=1.0)
        ref = O.rms_norm(x.double(), 1 + w.double(), 1e-4)
        assert ((got.double() - ref).abs() <= (1e-5 if dtype == F32 else 2 ** -8) * (1 + ref.abs())).all()


# ---- whole models ---------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("name,dtype", ALL)
def test_whole_prompts(name, dtype, tmp_path_factory):
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    eng = engine(model)
    for n, seed in ((1, 1), (2, 1), (33, 2), (160, 3)):
        toks, want = expected(name, cfg, t, n, seed)
        poison(eng)
        e = error(eng.step([(n, toks, range(n))]), want)
        assert close(e, dtype), (n, int(e.argmax()), float(e.max()))
        eng.release(n)


@pytest.mark.parametrize("name", list(CONFIGS))
def test_residual_after_every_layer(name, tmp_path_factory):
    """32-bit: the residual stream layer by layer, of a prompt and of a decoded token"""
    cfg, t, model = setup(name, F32, tmp_path_factory)
    toks, want = random_tokens(cfg, 50, 6), []
    O.forward(cfg, t, toks, layers_out=want)
    eng, got, step = engine(model), [], []
    eng.step([("a", toks[:49], [48])], hook=lambda i, x: got.append(x.double().cpu()))
    eng.step([("a", toks[49:], [0])], hook=lambda i, x: step.append(x.double().cpu()))
    assert len(got) == len(step) == len(want) == len(cfg["layers"])
    for i, w in enumerate(want):
        assert (got[i] - w[:49]).abs().max() < 1e-4 * w.abs().max(), i
        assert (step[i] - w[49:]).abs().max() < 1e-4 * w.abs().max(), i


@pytest.mark.parametrize("name,dtype", ALL)
def test_token_by_token_equals_the_prompt(name, dtype, tmp_path_factory):
    """decoding from the second token on, through several pages and windows, over poisoned memory"""
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    toks, want = expected(name, cfg, t, 160, 3)
    eng = engine(model)
    got = [eng.step([("a", toks[:1], [0])])]
    for p in range(1, 160):
        poison(eng)
        got.append(eng.step([("a", toks[p:p + 1], [0])]))
    e = error(torch.cat(got), want)
    assert close(e, dtype), (int(e.argmax()), float(e.max()))
    assert eng.cache.pages_in_use <= 1 + -(-widest(cfg) // 64)


@pytest.mark.parametrize("name,dtype", [("ragged", F32), ("even", F32), ("even", BF16), ("heads", BF16), ("t-ragged", F32), ("t-even", F32), ("t-even", BF16), ("t-heads", BF16),
                                        ("t-large", F32)])
@pytest.mark.parametrize("sizes", [[2], [3, 1], [7, 64], [65, 31], [100, 1, 1, 2]])
def test_portions_of_a_prompt(name, dtype, sizes, tmp_path_factory):
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    toks, want = expected(name, cfg, t, 160, 3)
    eng, got, at, k = engine(model), [], 0, 0
    while at < 160:
        n = min(sizes[k % len(sizes)], 160 - at)
        poison(eng)
        got.append(eng.step([("a", toks[at:at + n], range(n))]))
        at, k = at + n, k + 1
    assert close(error(torch.cat(got), want), dtype)


@pytest.mark.parametrize("name,dtype", [("ragged", F32), ("even", F32), ("even", BF16), ("heads", BF16), ("large", BF16), ("t-ragged", F32), ("t-even", F32), ("t-even", BF16),
                                        ("t-heads", F32), ("t-large", BF16), ("t-recurrent", F32)])
def test_unequal_batch_and_reused_pages(name, dtype, tmp_path_factory):
    """requests of different lengths start together, decode together and end one after the other; later requests get their slots and
    pages; a portion and a running request share a step.  Everything equals each request alone."""
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    toks, want = expected(name, cfg, t, 160, 3)
    other, want2 = expected(name, cfg, t, 33, 2)
    eng = engine(model, max_tokens=64, max_requests=1)  # (the cache has to grow on the way)
    check = lambda got, w: close(error(got, w), dtype)  # noqa: E731
    start = {"a": 1, "b": 33, "c": 64, "d": 100}
    for rnd in range(2):
        poison(eng)
        got = eng.step([(r, toks[:n], [0, n - 1] if n > 1 else [0]) for r, n in start.items()])
        rows = [i for n in start.values() for i in ([0, n - 1] if n > 1 else [0])]
        assert check(got, want[rows])
        live = dict(start)
        for k in range(40):
            poison(eng)
            got = eng.step([(r, toks[p:p + 1], [0]) for r, p in live.items()])
            assert check(got, want[list(live.values())]), (rnd, k)
            live = {r: p + 1 for r, p in live.items()}
            if k % 12 == 11:
                eng.release(next(iter(live)))
                live.pop(next(iter(live)))
        eng.step([("e", other[:20], []), *[(r, toks[p:p + 1], []) for r, p in live.items()]])  # a prompt next to running requests
        live = {r: p + 1 for r, p in live.items()}
        poison(eng)
        got = eng.step([("e", other[20:], [12]), *[(r, toks[p:p + 1], [0]) for r, p in live.items()]])
        assert check(got, torch.cat([want2[32:33], want[list(live.values())]]))
        for r in ["e", *live]:
            eng.release(r)
        assert eng.cache.pages_in_use == 0


@pytest.mark.parametrize("name,dtype", ALL)
def test_wide_batches(name, dtype, tmp_path_factory):
    """batches past eight (a workgroup then serves four tokens per weight read), not a multiple of four, and one past the tiles' rows"""
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    toks, want = expected(name, cfg, t, 160, 3)
    eng = engine(model, max_tokens=4096, max_requests=32)
    for B in (10, 23):
        at = {r: 1 + 5 * r for r in range(B)}
        eng.step([(r, toks[:p], []) for r, p in at.items()])
        for _ in range(3):
            poison(eng)
            got = eng.step([(r, toks[p:p + 1], [0]) for r, p in at.items()])
            assert close(error(got, want[list(at.values())]), dtype), B
            at = {r: p + 1 for r, p in at.items()}
        for r in at:
            eng.release(r)


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_long_decoding_far_keys(dtype, tmp_path):
    """hundreds of decoded tokens over many pages, most of them given back on the way; windows of several pages"""
    from layered_models import config, mixer
    from teal_amd.gpt_fast import registry
    cfg = config(64, 120, [(mixer(2, 24, 8, 24, 40, 300), 80), (mixer(3, 16, 8, 16, 40, 190, kv_from=0), None), (mixer(1, 32, 8, 32, 64, 10), 40)])
    t = random_tensors(cfg, 2)
    model = registry.load_model(save_checkpoint(tmp_path / "m", cfg, t), DEV, dtype)
    toks = random_tokens(cfg, 620, 5)
    want = O.forward(cfg, t, toks)
    eng = engine(model, max_tokens=64, max_requests=1)
    got = [eng.step([("a", toks[:40], [39])])]
    for p in range(40, 620):
        if p % 50 == 0:
            poison(eng)
        got.append(eng.step([("a", toks[p:p + 1], [0])]))
    assert close(error(torch.cat(got), want[39:]), dtype) and eng.cache.pages_in_use <= 6


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_long_decoding_with_states(dtype, tmp_path):
    """hundreds of decoded tokens through windows of several pages and through states that hardly decay"""
    from layered_models import tefopel, tied, time_mix
    from teal_amd.gpt_fast import registry
    cfg = tefopel(64, 120, [(time_mix(2, 32), None), (tied(2, 1, 32, 8, 300), 80), 0, (tied(3, 3, 16, 16, 190), None), (time_mix(1, 64), 40)])
    t = random_tensors(cfg, 2)
    for i in (0, 4):
        t[f"l{i}.mix.w0"] -= 3.0
    model = registry.load_model(save_checkpoint(tmp_path / "m", cfg, t), DEV, dtype)
    toks = random_tokens(cfg, 620, 5)
    want = O.forward(cfg, t, toks)
    other = O.forward(cfg, t, [(toks[0] + 1) % 120] + toks[1:])
    assert float(error(other, want)[-1]) > 50 * TOL[F32]  # the first token still shows at the end
    eng = engine(model, max_tokens=64, max_requests=1)
    got = [eng.step([("a", toks[:40], [39])])]
    for p in range(40, 620):
        if p % 50 == 0:
            poison(eng)
        got.append(eng.step([("a", toks[p:p + 1], [0])]))
    assert close(error(torch.cat(got), want[39:]), dtype) and eng.cache.pages_in_use <= 6


def test_bad_steps_are_refused(tmp_path_factory):
    cfg, t, model = setup("even", F32, tmp_path_factory)
    eng = engine(model)
    for entries in ([("a", [], [])], [("a", [256], [])], [("a", [-1], [])], [("a", [1], [1])], [("a", [1], []), ("a", [2], [])]):
        with pytest.raises(ValueError):
            eng.step(entries)
    assert not eng.slot and eng.cache.pages_in_use == 0
    assert eng.step([("a", [1, 2], [])]) is None and eng.length("a") == 2


# ---- the fused step --------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("name,dtype", [("even", BF16), ("even", F16), ("heads", BF16), ("large", BF16), ("t-even", BF16), ("t-even", F16), ("t-heads", BF16), ("t-large", BF16),
                                        ("t-recurrent", BF16)])
def test_fused_step_equals_the_unfused_one(name, dtype, tmp_path_factory):
    from teal_amd.gpt_fast.layered import StepBatch
    from teal_amd.gpt_fast.layered_engine import LayeredEngine
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    assert LayeredEngine.supports(model, need_caches=False) is None
    toks, want = expected(name, cfg, t, 160, 3)
    eng = engine(model)
    assert eng.fused is not None
    eng.step([("a", toks[:70], [])])
    pairs = []
    for p in range(70, 160):
        s = eng.slot["a"]
        eng.cache.extend(s, p + 1)
        eng.cache.sync()
        dev = torch.tensor([[toks[p]], [p], [s]], dtype=torch.int32, device=DEV)
        plain = model.step_pass(StepBatch(eng.cache, dev[0], dev[1], dev[2], p)).clone()
        fused = eng._decode(dev, p)  # (the same position twice: states repeat)
        pairs.append((error(fused, want[p:p + 1]), error(fused, plain.double().cpu())))
    assert all(close(torch.cat(e), dtype) for e in zip(*pairs))


def test_fused_step_needs_whole_chunks(tmp_path_factory):
    from teal_amd.gpt_fast.engine import pick_engine
    cfg, t, model = setup("ragged", BF16, tmp_path_factory)  # 72 wide: no fused form, the engine keeps the unfused step
    cls, why = pick_engine(model, need_caches=False)
    assert cls is None and "width" in why and engine(model).fused is None


@pytest.mark.parametrize("name,dtype,batch", [("even", BF16, 1), ("heads", BF16, 1), ("even", BF16, 3), ("ragged", F32, 2), ("t-even", BF16, 1), ("t-even", BF16, 3), ("t-ragged", F32, 2)])
def test_graph_replays_equal_eager_steps(name, dtype, batch, tmp_path_factory):
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    toks, _ = expected(name, cfg, t, 160, 3)
    a, b = engine(model, max_requests=4, max_tokens=1024), engine(model, max_requests=4, max_tokens=1024, graphs=True)
    for e in (a, b):
        e.step([(r, toks[: 50 + r], []) for r in range(batch)])
    for k in range(60):
        step = [(r, [toks[50 + r + k]], [0]) for r in range(batch)]
        x, y = a.step(step), b.step(step)
        torch.cuda.synchronize()
        assert float(error(y, x.double().cpu()).max()) < (1e-5 if dtype == F32 else TOL[dtype] / 4), k
    assert b._graphs


@pytest.mark.parametrize("name,dtype", [("even", BF16), ("ragged", F32), ("heads", BF16), ("t-even", BF16), ("t-ragged", F32)])
def test_graphed_prompts_equal_eager_ones(name, dtype, tmp_path_factory):
    """the same shapes again and again with other tokens and on other pages: every replay against the oracle"""
    cfg, t, model = setup(name, dtype, tmp_path_factory)
    eng = engine(model, max_tokens=1024, max_requests=4, graphs=True)
    toks, want = expected(name, cfg, t, 160, 3)
    other, want2 = expected(name, cfg, t, 33, 2)
    eng.step([("keep", toks[:90], [])])  # (occupies the first pages)
    for rep in range(5):
        got = eng.step([("x", toks[:20], [19]), ("y", other[:33], [0, 32])])
        assert close(error(got, torch.cat([want[19:20], want2[[0, 32]]])), dtype), rep
        got = eng.step([("x", toks[20:40], [19])])  # a portion
        assert close(error(got, want[39:40]), dtype), rep
        eng.release("x"), eng.release("y")
        got = eng.step([("x", other[:20], [19]), ("y", toks[:33], [0, 32])])
        assert close(error(got, torch.cat([want2[19:20], want[[0, 32]]])), dtype), rep
        eng.release("y"), eng.release("x")
        poison(eng)
        if rep == 2:
            eng.release("keep")
    assert len(eng.prompt._graphs) == 2
    assert close(error(eng.step([("long", toks, [0, 159])]), want[[0, 159]]), dtype)


@pytest.mark.parametrize("name", ["even", "t-even"])
def test_sparsity_masks_the_projections(name, tmp_path_factory):
    """thresholds of the fused step = the unfused step on masked activations"""
    from teal_amd.gpt_fast.layered import StepBatch
    from teal_amd.gpt_fast.layered_engine import LayeredEngine, calibrate_thresholds
    from teal_amd.gpt_fast.layered import GatedMLP, TimeMix
    cfg, t, model = setup(name, BF16, tmp_path_factory)
    ths = calibrate_thresholds(model, 0.4)
    toks = random_tokens(cfg, 60, 8)
    eng = engine(model)
    eng.step([("a", toks[:40], [])])
    s = eng.slot["a"]
    eng.cache.extend(s, 41)
    eng.cache.sync()
    dev = torch.tensor([[toks[40]], [40], [s]], dtype=torch.int32, device=DEV)
    fused = LayeredEngine(model, ths, cache=eng.cache, max_seq=64)
    fused.slot = dev[2]
    got = fused(dev[0], dev[1]).view(1, -1).clone()
    hooks, kept = [], []

    def mask(lin, tau, n=None):
        def pre(_m, args):
            keep = args[0].float().abs() > tau
            if n is not None:
                keep[n:] = True  # (time mixing: the decay path's input is not masked)
            kept.append(float(keep.float().mean()))
            return (args[0] * keep,)
        hooks.append(lin.register_forward_pre_hook(pre))

    for i, b in model.own_layers():
        th = ths[i]
        if isinstance(b.mix, TimeMix):
            mask(b.mix.mixed, th["rkvg"], 4)
        else:
            mask(b.mix.proj, th["q"])
        mask(b.mix.wo, th["o"])
        if b.mlp is not None:
            first, down = b.mlp.linears()
            mask(first, th["gate" if isinstance(b.mlp, GatedMLP) else "up"]), mask(down, th["down"])
    plain = model.step_pass(StepBatch(eng.cache, dev[0], dev[1], dev[2], 40)).clone()
    for h in hooks:
        h.remove()
    dense = model.step_pass(StepBatch(eng.cache, dev[0], dev[1], dev[2], 40))
    assert (0.4 if name == "even" else 0.3) < sum(kept) / len(kept) < 0.8
    assert float(error(got, plain.double().cpu())) < 0.12 < float(error(dense, plain.double().cpu()))


@pytest.mark.parametrize("make", [random_config, random_tefopel])
@pytest.mark.parametrize("seed", range(12))
def test_random_configurations(seed, make, tmp_path):
    """the whole path on configurations of all kinds: a batch of prompts, then decoding together and alone, 32-bit and bf16"""
    from teal_amd.gpt_fast import registry
    cfg = make(seed)
    t = random_tensors(cfg, seed, peak=2.0)
    path = save_checkpoint(tmp_path / "m", cfg, t)
    n = 105
    toks = random_tokens(cfg, n, seed)
    want = O.forward(cfg, t, toks)
    for dtype in (F32, BF16):
        model = registry.load_model(path, DEV, dtype)
        eng = engine(model)
        assert (eng.fused is not None) == (dtype == BF16 and cfg["width"] % 64 == 0)
        first = {"a": 70, "b": 1, "c": 34}
        errs = [error(eng.step([(r, toks[:k], range(k)) for r, k in first.items()]), torch.cat([want[:k] for k in first.values()]))]
        poison(eng)
        live = dict(first)
        for k in range(35):
            if k == 12:
                for r in ("b", "c"):
                    eng.release(r)
                    live.pop(r)
                poison(eng)
            got = eng.step([(r, [toks[p]], [0]) for r, p in live.items()])
            errs.append(error(got, want[list(live.values())]))
            live = {r: p + 1 for r, p in live.items()}
        e = torch.cat(errs)
        assert close(e, dtype), (cfg, dtype, int(e.argmax()), float(e.max()))


# ---- generation ------------------------------------------------------------------------------------------------------------
def greedy(cfg, t, prompt, n):
    seq = list(prompt)
    for _ in range(n):
        seq.append(int(O.forward(cfg, t, seq)[-1].argmax()))
    return seq[len(prompt):]


@pytest.mark.parametrize("name", ["even", "t-even"])
def test_greedy_generation_equals_the_oracle(name, tmp_path_factory):
    """32-bit: more requests than run at once, of unequal lengths, whole prompts and portions, eager and from graphs"""
    from teal_amd.gpt_fast.serving import Request, generate_batch
    cfg, t, model = setup(name, F32, tmp_path_factory)
    reqs = [(random_tokens(cfg, n, 20 + n), m) for n, m in ((1, 9), (30, 6), (66, 8), (5, 1), (12, 10))]
    want = [greedy(cfg, t, p, m) for p, m in reqs]
    for kw in ({}, {"max_batch": 2}, {"portion": 7}, {"max_batch": 3, "graphs": False}):
        assert generate_batch(model, [Request(p, m) for p, m in reqs], **kw) == want, kw
    # sampling: a request's stream depends on its own seed alone
    r = [Request(p, m) for p, m in reqs]
    alone = [generate_batch(model, r[i:i + 1], temperature=1.0, top_k=20, seed=50 + i)[0] for i in range(5)]
    assert generate_batch(model, r, temperature=1.0, top_k=20, seed=50) == alone


@pytest.mark.parametrize("name,named", [("even", "Bolizen-tiny-test"), ("t-even", "Tefopel-tiny-test")])
def test_generate_entry_point_and_command_line(name, named, tmp_path_factory):
    """generate() with the fused engine (bf16: every chosen token is within rounding of the oracle's best) and the CLI's main"""
    from teal_amd.gpt_fast import generate as G
    cfg, t, model = setup(name, BF16, tmp_path_factory)
    path = save_checkpoint(tmp_path_factory.mktemp("cli"), cfg, t)
    prompt = random_tokens(cfg, 20, 3)
    base = ["--checkpoint_path", str(path), "--num_samples", "1", "--max_new_tokens", "70", "--temperature", "0", "--compile"]
    run = lambda *a: G.main(G.build_parser().parse_args([*base, *a]))  # noqa: E731
    res = run("--precision", "bf16", "--prompt_ids", ",".join(map(str, prompt)))
    seq = res["sequences"][0]
    assert res["decoder"] == "EngineDecoder" and seq[:20] == prompt and len(seq) == 90
    lg = O.forward(cfg, t, seq)
    gap = (lg.max(-1).values - lg.gather(1, torch.tensor(seq[1:] + [0])[:, None])[:, 0])[19:-1]
    assert float(gap.max()) < 3 * TOL[BF16] * float(lg.pow(2).mean().sqrt())
    res = run("--precision", "fp32", "--prompt_ids", "1,2,3;" + " ".join(map(str, prompt)), "--max_new_tokens", "5")
    assert [s[-5:] for s in res["sequences"]] == [greedy(cfg, t, [1, 2, 3], 5), greedy(cfg, t, prompt, 5)]
    res = G.main(G.build_parser().parse_args(["--synthetic", named, "--precision", "bf16", "--num_samples", "2", "--max_new_tokens", "12", "--compile",
                                              "--sparsity", "0.3"]))
    assert len(res["sequences"]) == 2 and res["thresholds"] is not None
    with pytest.raises(SystemExit):
        G.main(G.build_parser().parse_args(["--synthetic", "7B", "--precision", "fp32"]))


@pytest.mark.parametrize("name", ["even", "t-even"])
def test_module_interface(name, tmp_path_factory):
    """forward(idx, input_pos) as model.Transformer's: prompt of a batch, then a captured single-token step"""
    from teal_amd.gpt_fast.generate import GraphedDecoder
    cfg, t, model = setup(name, F32, tmp_path_factory)
    toks, want = expected(name, cfg, t, 160, 3)
    model.setup_caches(2, 170)
    idx = torch.tensor([toks[:50], toks[:50]], device=DEV)
    lg = model(idx, torch.arange(50, device=DEV))
    assert lg.shape == (2, 50, 256) and float(error(lg[1], want[:50]).max()) < TOL[F32]
    dec = GraphedDecoder(model, True, 0.0, None)
    cur, pos = torch.tensor([[toks[50]]], device=DEV, dtype=torch.int), torch.tensor([50], device=DEV, dtype=torch.int)
    dec.capture(cur, pos)
    for p in range(50, 90):
        got = dec(torch.tensor([[toks[p]]], device=DEV, dtype=torch.int), torch.tensor([p], device=DEV, dtype=torch.int))
        assert float(want[p].max() - want[p][int(got)]) < 1e-4, p  # (capped logits tie)
    model.max_seq_length = model.max_batch_size = -1


@pytest.mark.parametrize("name", ["even", "t-even"])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_trace_replay(dtype, name, tmp_path, tmp_path_factory):
    cfg, t, model = setup(name, F32, tmp_path_factory)
    toks, want = expected(name, cfg, t, 160, 3)
    path = save_checkpoint(tmp_path / "m", cfg, t)
    steps = [{"step": 0, "entries": [{"id": "x", "tokens": toks[:40], "want": [0, 39]}, {"id": "y", "tokens": toks[:1], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "x", "tokens": toks[40:41], "want": [0]}, {"id": "y", "tokens": toks[1:2], "want": [0]}], "end": ["y"]},
             {"step": 2, "entries": [{"id": "x", "tokens": toks[41:42], "want": []}], "end": []},
             {"step": 3, "entries": [{"id": "x", "tokens": toks[42:43], "want": [0]}], "end": ["x"]}]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([os.path.join(root, "bin", "trace_run"), "--model", str(path), "--dtype", dtype, "--out", str(tmp_path), "--max-tokens", "64"],
                       input="".join(json.dumps(s) + "\n" for s in steps), text=True, capture_output=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [ln for ln in r.stdout.splitlines() if ln.startswith("done")] == [f"done {i}" for i in range(4)]
    read = lambda i: torch.from_numpy(np.fromfile(tmp_path / f"{i}.f32", dtype="<f4").reshape(-1, 256))  # noqa: E731
    tol = TOL[getattr(torch, dtype)]
    assert float(error(read(0), want[[0, 39]]).max()) < tol and float(error(read(1), want[[40, 1]]).max()) < tol
    assert float(error(read(3), want[[42]]).max()) < tol and not (tmp_path / "2.f32").exists()
