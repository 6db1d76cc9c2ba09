"""GPU: the int4 GEMV at the sizes where its units, slices and the LDS end: one unit, slices of unequal length, fewer units than waves, the longest
vector in one slice (128 KB of activations), every group size; nothing, half and everything kept."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("Z,N,G,prepared", [(32, 128, 32, True), (64, 256, 64, True), (544, 384, 32, True), (1280, 128, 256, True), (4352, 640, 128, True), (65536, 128, 256, False),
                                            (65536, 128, 32, True)])
def test_int4_units(Z, N, G, prepared, dtype):
    from teal_amd import _lib, quantize, runtime
    L = _lib.load()
    runtime.init()
    dt = (torch.float16, torch.bfloat16)[dtype]
    g = torch.Generator(device=DEV).manual_seed(Z + N)
    q = torch.randint(0, 16, (N, Z), device=DEV, dtype=torch.int32, generator=g)
    packed = quantize.pack_int4_colmajor(q)
    packed[:, N:] = 0xAB
    sz = (torch.randn(Z // G, N, 2, device=DEV, generator=g) * 0.01).to(torch.bfloat16)
    x = torch.randn(Z, device=DEV, generator=g).to(dt)
    scale, zero = (sz[..., i].double().T.repeat_interleave(G, dim=1) for i in (0, 1))
    y = torch.empty(N, device=DEV, dtype=dt)
    nbytes = int(L.teal_workspace_bytes(Z, N))
    ws = runtime.new_workspace(Z, N) if prepared else torch.empty(nbytes // 4 + 1, device=DEV)  # (not prepared: one slice)
    for tau in (1e9, 0.6745, -1.0):
        rc = L.teal_sparse_qkv_gemv_i4(x.data_ptr(), packed.data_ptr(), sz.data_ptr(), y.data_ptr(), tau, tau, tau, Z, N, N, 0, packed.stride(0), G, dtype, ws.data_ptr(),
                                       ws.numel() * 4, runtime.stream_ptr())
        assert rc == 0
        xm = torch.where(x.float().abs() > tau, x, torch.zeros_like(x)).double()
        want = ((q.double() - 8) * scale + zero) @ xm
        # per unit of 32 rows the biased sum (bias at most 1032) is exact to 2^-22 or so of its terms' sizes; one rounding at the end
        units = xm.abs().view(-1, 32).sum(1)
        tol = 2.0 ** -21 * 1040 * (scale.abs()[:, ::32] @ units) + 2.0 ** (-11 if dtype == 0 else -8) * want.abs() + 2.0 ** -18 * (zero.abs()[:, ::32] @ units) + 1e-7
        err = (y.double() - want).abs()
        assert bool((err <= tol).all()), (tau, float((err / tol).max()))
