"""GPU: the fused prompt pass of any length (teal_amd/csrc/teal_prompt.hip, prefill.PromptPass) — its kernels against float64, the pass against
the op-by-op modules, and what keeps a model on the modules."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = {0: torch.float16, 1: torch.bfloat16}
STEP = {0: 2.0 ** -10, 1: 2.0 ** -7}  # two roundings to 16 bits


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("T,heads,kv,hd,max_seq,order", [(1, 2, 2, 64, 8, "asc"), (2, 4, 1, 128, 64, "asc"), (31, 2, 1, 64, 65, "perm"), (64, 2, 2, 128, 64, "asc"),
                                                         (129, 4, 2, 128, 200, "late"), (257, 8, 2, 64, 333, "perm"), (640, 2, 1, 128, 640, "asc")])
def test_prompt_attention(T, heads, kv, hd, max_seq, order, dtype):
    """part tiles of queries and keys, positions in any order and behind rows that were there before, large scores late in a row (the running
    maximum is replaced) and in its first tile (it is kept)"""
    from teal_amd import _lib, runtime
    L, dt = _lib.load(), DT[dtype]
    runtime.init()
    g = torch.Generator(device=DEV).manual_seed(T + hd)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g).to(dt)  # noqa: E731
    qkv, kc, vc = r(T, (heads + 2 * kv) * hd + 8), r(kv, max_seq, hd), r(kv, max_seq, hd)
    qkv[:, : heads * hd] *= 3
    kc[:, max_seq // 2] *= 4
    pos = torch.arange(T, device=DEV) if order == "asc" else torch.arange(max_seq - T, max_seq, device=DEV) if order == "late" else torch.randperm(max_seq, device=DEV, generator=g)[:T]
    pos = pos.to(torch.int32 if hd == 64 else torch.int64)
    out = torch.full((T, heads * hd + 4), float("nan"), device=DEV, dtype=dt)
    rc = L.teal_prompt_attention(qkv.data_ptr(), qkv.stride(0), kc.data_ptr(), vc.data_ptr(), pos.data_ptr(), int(pos.dtype == torch.int64), out.data_ptr(), out.stride(0), T,
                                 heads, kv, hd, max_seq, hd ** -0.5, dtype, runtime.stream_ptr())
    assert rc == 0
    q = qkv[:, : heads * hd].double().view(T, heads, hd)
    seen = torch.arange(max_seq, device=DEV)[None] <= pos[:, None].long()
    for h in range(heads):
        s = (q[:, h] @ kc[h // (heads // kv)].double().T) * hd ** -0.5
        p = torch.softmax(s.masked_fill(~seen, float("-inf")), dim=1)
        v = vc[h // (heads // kv)].double()
        # weights and the result are each rounded once to 16 bits
        tol = STEP[dtype] * (p @ v.abs() + (p @ v).abs()) + 1e-5
        assert bool(((out[:, h * hd:(h + 1) * hd].double() - p @ v).abs() <= tol).all())
    assert bool(torch.isnan(out[:, heads * hd:]).all())


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("T,D", [(1, 8), (3, 2048), (5, 4104), (2, 8200), (2, 16384)])
def test_prompt_norm(T, D, dtype):
    from teal_amd import _lib, runtime
    L, dt = _lib.load(), DT[dtype]
    g = torch.Generator(device=DEV).manual_seed(D)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    emb, w, y, slabs = r(11, D).to(dt), r(D).to(dt), r(T, D).to(dt), r(3, T, D)
    norm = lambda h: (h.float() * torch.rsqrt(h.float().square().mean(-1, keepdim=True) + 1e-5)).to(dt) * w  # noqa: E731
    h, x, zero = torch.empty(T, D, device=DEV, dtype=dt), torch.empty(T, D, device=DEV, dtype=dt), torch.full((256,), 3, device=DEV, dtype=torch.int32)
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731

    def call(emb_=None, tok=None, y_=None, s_=None, z=None):
        rc = L.teal_prompt_norm(p(emb_), 11, p(tok), int(tok is not None and tok.dtype == torch.int64), h.data_ptr(), p(y_), p(s_), 3, w.data_ptr(), x.data_ptr(), T, D, 1e-5, p(z),
                                256, dtype, runtime.stream_ptr())
        assert rc == 0

    close = lambda a, b: bool(((a.float() - b.float()).abs() <= 2 * STEP[dtype] * (b.float().abs() + 1e-3)).all())  # noqa: E731  (a step to the side per rounding)
    for it in (torch.int32, torch.int64):
        tok = torch.randint(0, 11, (T,), device=DEV, generator=g).to(it)
        call(emb, tok, z=zero)
        assert torch.equal(h, emb[tok.long()]) and close(x, norm(h)) and not zero.any()
        want = h + y
        call(y_=y)
        assert torch.equal(h, want) and close(x, norm(h))
        want = (h.float() + ((slabs[0] + slabs[1]) + slabs[2]).to(dt).float()).to(dt)
        call(s_=slabs)
        assert torch.equal(h, want) and close(x, norm(h))
    assert L.teal_prompt_norm(None, 0, None, 0, h.data_ptr(), None, None, 0, w.data_ptr(), x.data_ptr(), T, D + 4, 1e-5, None, 0, dtype, runtime.stream_ptr()) == -3


def _model(arch, dt, seq, **kw):
    from teal_amd.gpt_fast import generate as G
    model = G.build_synthetic_model(arch, DEV, dt, seed=21, n_layer=2)
    G.apply_sparsity(model, sparsity=0.5, hist_path=None, greedy_lookup=None, synthetic=True, decode_calibration=False)
    model.max_seq_length = -1
    model.setup_caches(1, seq)
    return model


@pytest.mark.parametrize("arch,dt,relayout", [("7B", torch.float16, True), ("llama-3-8b", torch.bfloat16, False), ("tiny-gqa-test", torch.float16, True)])
def test_prompt_pass_equals_modules(arch, dt, relayout):
    """whole prompts on both sides of the row products' limits, and a portion behind earlier rows; logits of every token, cache rows, rows outside
    the prompt untouched"""
    from teal_amd.gpt_fast import generate as G
    from teal_amd.gpt_fast.prefill import PromptPass
    seq = 128 if arch.startswith("tiny") else 416
    model = _model(arch, dt, seq)
    if relayout:
        G.relayout_for_engine(model)
    assert PromptPass.supports(model) is None
    g = torch.Generator(device=DEV).manual_seed(3)
    tol = 0.004 if dt == torch.float16 else 0.03  # (relative, two layers; about four times what is seen)
    with torch.no_grad():
        for T, start in ((2, 0), (17, 0), (33, 5), (64, 0), (65, 0), (seq - 100, 90)):
            idx = torch.randint(0, model.config.vocab_size, (1, T), device=DEV, generator=g)
            pos, got = torch.arange(start, start + T, device=DEV), {}
            for fused in (False, True):
                for b in model.layers:
                    for c in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache):
                        c[:, :, start:].zero_()
                model.fused_decode = fused
                logits = model(idx.to(torch.int32 if T & 1 else torch.int64), pos)
                got[fused] = [logits.float()] + [c.float().clone() for b in model.layers for c in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache)]
                assert logits.shape == (1, T, model.config.vocab_size)
            for a, b in zip(got[False], got[True]):
                assert float((a - b).norm()) <= tol * float(a.norm()), (T, start)
            for c in got[True][1:]:
                assert not c[:, :, start + T:].any()


def test_prompt_pass_leaves_other_models_alone():
    from teal_amd.gpt_fast import generate as G
    from teal_amd.gpt_fast.prefill import PromptPass
    model = _model("tiny-gqa-test", torch.float16, 64)
    assert PromptPass.supports(model) is None
    at, ff = model.layers[1].attention, model.layers[0].feed_forward
    seen = []
    for m in (at, ff, model.layers[0], model.norm):  # hooks are called
        h = m.register_forward_pre_hook(lambda mod, a: seen.append(type(mod).__name__))
        assert PromptPass.supports(model) is not None
        with torch.no_grad():
            model(torch.zeros(1, 5, dtype=torch.int32, device=DEV), torch.arange(5, device=DEV))
        h.remove()
    assert len(seen) == 4
    op, at.gemv2 = at.gemv2, lambda *a: seen.append("op") or op(*a)  # an operator of the caller's own
    assert PromptPass.supports(model) == "replaced operators"
    with torch.no_grad():
        model(torch.zeros(1, 5, dtype=torch.int32, device=DEV), torch.arange(5, device=DEV))
    assert seen[-1] == "op"
    at.gemv2 = op
    fwd, ff.forward = ff.forward, lambda x: x  # a forward of the caller's own
    assert PromptPass.supports(model) is not None
    ff.forward = fwd
    assert PromptPass.supports(model) is None
    plain = G.build_synthetic_model("tiny-gqa-test", DEV, torch.float16, seed=1)  # never patched: the dense baseline
    plain.setup_caches(1, 64)
    assert PromptPass.supports(plain) is not None
    model.max_seq_length = model.max_batch_size = -1
    model.setup_caches(2, 64)  # batched caches
    assert PromptPass.supports(model) is not None
