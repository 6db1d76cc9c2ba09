"""GPU: the matrix products over a few rows on the matrix cores (teal_amd/csrc/teal_rows_core.h) at the sizes where tiles, slices and
producers end.

fp32 sums of exact products: |error| <= K * 2^-24 * sum |x w|, loosely bounded by 2^-18 * sum |x w| at these K (the sums run over waves
and slices).  Where a producer makes x (rsqrt, exp), an element next to a rounding boundary may come out one 16-bit step to the side:
a few steps of the largest element are allowed on top."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = {0: torch.float16, 1: torch.bfloat16}


def _image(Z, N, dtype, seed, pad=64):
    g = torch.Generator(device=DEV).manual_seed(seed)
    buf = torch.full((Z, N + pad), float("nan"), device=DEV, dtype=DT[dtype])  # (nothing may read the padding)
    buf[:, :N] = (torch.randn(Z, N, device=DEV, generator=g) * 0.05).to(DT[dtype])
    return buf


def _close(got, x, w, dtype, steps=0):
    want, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    step = 2.0 ** (-10 if dtype == 0 else -7)
    tol = 2.0 ** -18 * size + steps * step * float(x.abs().max()) * float(w.abs().max())
    err = (got.double() - want).abs()
    assert bool((err <= tol).all()), (float((err / tol).max()), float(err.max()))


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("Z,n0,n1,T", [(256, 256, 0, 1), (768, 512, 256, 8), (1280, 256, 0, 9), (4352, 256, 256, 16), (11008, 4096, 0, 7), (16384, 256, 0, 13)])
def test_prompt_gemm_producers(Z, n0, n1, T, dtype):
    """every producer of teal_prefill_gemm; one slice and several, slices of unequal length, one and two images, 8 and 16 token slots"""
    from teal_amd import _lib, runtime
    from teal_amd.gpt_fast.prefill import IN_NORM, IN_SILU_MUL, IN_XT, PrefillIn
    L, dt, R = _lib.load(), DT[dtype], 8 if T <= 8 else 16
    runtime.init()
    g = torch.Generator(device=DEV).manual_seed(Z + T)
    W0, W1 = _image(Z, n0, dtype, 1), _image(Z, n1, dtype, 2) if n1 else None
    w = torch.cat([W0[:, :n0]] + ([W1[:, :n1]] if n1 else []), dim=1)
    N, eps = n0 + n1, 1e-5
    h = torch.zeros(Z, R, device=DEV, dtype=dt)
    h[:, :T] = torch.randn(Z, T, device=DEV, generator=g).to(dt)
    norm_w = (1 + 0.1 * torch.randn(Z, device=DEV, generator=g)).to(dt)
    nwg = -(-Z // 256)
    sumsq = torch.zeros(64, R, device=DEV)
    sumsq[0] = h.float().square().sum(0)  # (any split over the producing workgroups is as good)
    gu = torch.randn(3, 2 * Z, R, device=DEV, generator=g)
    rstd = torch.rsqrt(sumsq.sum(0) / Z + eps)
    gate, up = (gu[0] + gu[1] + gu[2]).to(dt).float().split(Z)
    xs = {IN_XT: (h, 0), IN_NORM: (((h.float() * rstd).to(dt).float() * norm_w.float()[:, None]).to(dt), 4),
          IN_SILU_MUL: (((gate / (1 + torch.exp(-gate))).to(dt).float() * up).to(dt), 4)}
    split = ctypes.c_int(0)
    for mode, (x, steps) in xs.items():
        if mode == IN_NORM and nwg > 64:
            continue
        slabs = torch.full((16 * N * R,), float("nan"), device=DEV)
        gin = PrefillIn(mode=mode, xt=h.data_ptr(), sumsq=sumsq.data_ptr(), nwg=nwg, norm_w=norm_w.data_ptr(), eps=eps, gu_slabs=gu.data_ptr(), gu_split=3)
        rc = L.teal_prefill_gemm(ctypes.byref(gin), W0.data_ptr(), W0.stride(0), n0, None if W1 is None else W1.data_ptr(), 0 if W1 is None else W1.stride(0), n1,
                                 slabs.data_ptr(), slabs.numel() * 4, Z, T, dtype, ctypes.byref(split), runtime.stream_ptr())
        assert rc == 0 and 1 <= split.value <= 16
        got = slabs[: split.value * N * R].view(split.value, N, R).sum(0)[:, :T].T
        _close(got, x[:, :T].T.float(), w.float(), dtype, steps)


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("M,K,N", [(1, 32, 8), (2, 96, 72), (16, 4096, 4096), (17, 288, 136), (32, 1056, 264), (33, 4096, 200), (64, 11008, 384), (5, 16384, 64)])
def test_rows_gemm(M, K, N, dtype):
    """every output of teal_rows_gemm: part tiles of rows and columns, one slice and several (fewer steps than waves, unequal slices), rows of x
    and y further apart than their columns; slabs and complete sums agree bit for bit; the counters come back zero"""
    from teal_amd import _lib, runtime
    from teal_amd.kernels import layered as Kn
    runtime.init()
    dt = DT[dtype]
    g = torch.Generator(device=DEV).manual_seed(K + M)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    img = _image(K, 2 * N, dtype, 3)
    w, wu = img[:, :N].T, img[:, N:2 * N].T
    x = torch.full((M, K + 24), float("nan"), device=DEV, dtype=dt)[:, :K]
    x.copy_(r(M, K).to(dt))
    bias, bias_up = r(N).to(dt), r(N).to(dt)
    tickets = torch.zeros(Kn.TICKETS, device=DEV, dtype=torch.int32)
    split = Kn.rows_split(x, w)
    assert split == _lib.load().teal_rows_split(M, K, N, 0) >= 1
    slabs = Kn._rows_gemm(x, w, N, split, Kn.ROWS_SLABS, None, torch.full((split, M, N), float("nan"), device=DEV))
    _close(slabs.sum(0), x.float(), w.T.float(), dtype)
    total = slabs[0].clone()
    for k in range(1, split):
        total += slabs[k]
    logits = torch.full((M, N + 3), float("nan"), device=DEV)
    Kn._rows_gemm(x, w, N, split, Kn.ROWS_F32, tickets, logits, n_valid=N - 3)
    assert torch.equal(logits[:, : N - 3], total[:, : N - 3]) and bool(torch.isnan(logits[:, N - 3:]).all())
    out = torch.full((M, N + 4), float("nan"), device=DEV, dtype=dt)
    for _ in range(3):
        Kn._rows_gemm(x, w, N, split, Kn.ROWS_ROUNDED, tickets, out)
        assert torch.equal(out[:, :N], total.to(dt)) and bool(torch.isnan(out[:, N:]).all())
    step = 2.0 ** (-10 if dtype == 0 else -7)
    act = Kn.linear(None, x, tickets, weight=w, act="relu2", bias=bias)
    want = torch.relu(total + bias.float()).square()
    assert bool(((act.float() - want).abs() <= step * want + 1e-6).all())
    if N % 64 == 0 and M <= Kn.ROWS_PAIR_MAX:
        lin = torch.nn.Linear(1, 1, bias=False, device=DEV)
        lin.weight, lin.out_features = torch.nn.Parameter(img[:, : 2 * N].T, requires_grad=False), 2 * N
        both = torch.cat([bias, bias_up])
        got = Kn.gated_linear(lin, x, "gelu_tanh", both, tickets)
        z, u = (x.double() @ w.T.double() + bias.double()), x.double() @ wu.T.double() + bias_up.double()
        want = torch.nn.functional.gelu(z, approximate="tanh") * u
        size = x.double().abs() @ w.T.double().abs()
        # (the sums' own bound goes through a slope of at most 1.13 and the other factor)
        assert bool(((got.double() - want).abs() <= step * want.abs() + 2.0 ** -17 * size * (1 + z.abs() + u.abs()) + 1e-6).all())
        calls = []
        lin.register_forward_pre_hook(lambda m, a: calls.append(1))  # a hooked module is called, not passed by
        again = Kn.gated_linear(lin, x, "gelu_tanh", both, tickets)
        assert calls and bool(((again.double() - want).abs() <= 4 * step * (want.abs() + z.abs() + u.abs() + z.abs() * u.abs())).all())
    torch.cuda.synchronize()
    assert not tickets.any()


def test_rows_gemm_refuses():
    from teal_amd.kernels import layered as Kn
    w = torch.zeros(256, 128 + 8, device=DEV, dtype=torch.float16)[:, :128].T
    x = torch.zeros(4, 256, device=DEV, dtype=torch.float16)
    assert Kn.rows_split(x, w) >= 1
    assert Kn.rows_split(x.float(), w) == 0 and Kn.rows_split(x.bfloat16(), w) == 0 and Kn.rows_split(x, w.contiguous()) == 0
    assert Kn.rows_split(torch.zeros(65, 256, device=DEV, dtype=torch.float16), w) == 0
    assert Kn.rows_split(torch.zeros(4, 260, device=DEV, dtype=torch.float16)[:, 2:258], w) == 0    # rows not on 16 bytes
    assert Kn.rows_split(torch.zeros(4, 264, device=DEV, dtype=torch.float16)[:, :248], w[:, :248]) == 0  # K not a multiple of 32
    # what is refused there still has its product
    a, b = torch.randn(3, 248, device=DEV).half(), torch.randn(248, 16, device=DEV).half().T
    assert torch.equal(Kn.linear(None, a, torch.zeros(256, device=DEV, dtype=torch.int32), weight=b), torch.nn.functional.linear(a, b))


@pytest.mark.parametrize("D", [64, 1003, 4096])
def test_resid_norm_adds_slabs(D):
    """slabs in slab order, rows picked out of them, counters cleared"""
    from teal_amd.kernels import layered as Kn
    T, S = 7, 3
    x, y = torch.randn(T, D, device=DEV), torch.randn(S, T, D, device=DEV)
    post, pre = (torch.randn(D, device=DEV).to(torch.bfloat16) for _ in range(2))
    rows = torch.tensor([5, 1], device=DEV, dtype=torch.int32)
    s = (y[0] + y[1]) + y[2]
    norm = lambda t: t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-5)  # noqa: E731
    want = x + norm(s) * post.float()
    got, zero = x.clone(), torch.full((256,), 7, device=DEV, dtype=torch.int32)
    h = Kn.resid_norm(got, y=y, post_w=post, pre_w=pre, eps=1e-5, rows=rows, zero=zero)
    assert torch.allclose(got[rows.long()], want[rows.long()], atol=1e-5, rtol=1e-5) and torch.equal(got[0], x[0]) and not zero.any()
    assert torch.allclose(h.float(), (norm(want) * pre.float())[rows.long()], atol=1e-2, rtol=2 ** -7)


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("M,K,N", [(1, 64, 16), (47, 256, 272), (65, 320, 2064), (161, 4096, 496), (320, 11008, 256), (640, 2048, 1024)])
def test_tile_gemm(M, K, N, dtype):
    """every output of teal_tile_gemm: part tiles of rows and columns, one slice and several (unequal ones), one image and two, rows of x, of the
    images and of y further apart than their columns; nothing outside the result is written"""
    from teal_amd import _lib, runtime
    L, dt = _lib.load(), DT[dtype]
    runtime.init()
    g = torch.Generator(device=DEV).manual_seed(K + M)
    x = torch.full((M, K + 8), float("nan"), device=DEV, dtype=dt)
    x[:, :K] = torch.randn(M, K, device=DEV, generator=g).to(dt)
    img = _image(K, 2 * N, dtype, 3)
    y = torch.full((M + 1, 2 * N + 8), 7.0, device=DEV, dtype=dt)

    def run(images, slabs):
        up = images == 2
        rc = L.teal_tile_gemm(x.data_ptr(), K + 8, img.data_ptr(), img.data_ptr() + 2 * N if up else None, img.stride(0), None if slabs is not None else y.data_ptr(),
                              y.data_ptr() + 2 * N if up else None, y.stride(0), None if slabs is None else slabs.data_ptr(), M, K, N, dtype, runtime.stream_ptr())
        assert rc == 0

    def rounded(cols):
        want = (x[:, :K].double() @ img[:, :cols].double())
        err, size = (y[:M, :cols].double() - want).abs(), x[:, :K].double().abs() @ img[:, :cols].double().abs()
        assert bool((err <= 2.0 ** -18 * size + 2.0 ** (-11 if dtype == 0 else -8) * want.abs() + 2.0 ** -25).all())
        assert bool((y[:M, cols:] == 7).all()) and bool((y[M] == 7).all())

    run(1, None)
    rounded(N)
    run(2, None)
    rounded(2 * N)
    if (split := L.teal_tile_split(M, K, N, 1, 1)) > 0:
        slabs = torch.full((split + 1, M, N), float("nan"), device=DEV)
        run(1, slabs)
        assert bool(slabs[split].isnan().all())
        _close(slabs[:split].sum(0), x[:, :K].float(), img[:, :N].float(), dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_tile_products_of_linears(dtype):
    """the linears of a prompt by either route: partial sums, gate and up; others (a hook) keep the module's"""
    from teal_amd import runtime
    from teal_amd.kernels import layered as Kn
    from teal_amd.monkeypatch import to_column_major
    runtime.init()
    torch.manual_seed(0)

    def lin(n, k):
        m = torch.nn.Linear(k, n, bias=False, device=DEV, dtype=dtype)
        m.weight.data = (torch.randn(n, k, device=DEV) * k ** -0.5).to(dtype)
        to_column_major(m)
        return m

    step = 2.0 ** (-10 if dtype is torch.float16 else -7)
    x, down, gate, up = torch.randn(100, 1024, device=DEV).to(dtype), lin(512, 1024), lin(8192, 1024), lin(8192, 1024)
    y = Kn.linear(down, x, slabs=True)
    assert y.dim() == 3 and y.dtype == torch.float32
    assert (y.sum(0) - x.float() @ down.weight.float().T).abs().max() < 1e-4  # (sums of 1024 products near 1)
    assert Kn.tile_split(x, gate.weight, 2) == 1
    for a, lin_ in zip(Kn.both(gate, up, x), (gate, up)):
        assert (a.float() - x.float() @ lin_.weight.float().T).abs().max() < 4 * step
    down.register_forward_hook(lambda *a: None)
    assert Kn.linear(down, x, slabs=True).dim() == 2
