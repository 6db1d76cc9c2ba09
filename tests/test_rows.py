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
