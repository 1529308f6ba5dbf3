"""The output projection of a few tokens that takes its norm with it (hdla_rows_gemm_norm) by eight waves and, from more than 1024 channels on, sixteen: channels that leave waves a
short share or none."""
import ctypes

import pytest
import torch

from hdla_hip import _lib

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(1, 20), (16, 100)])
@pytest.mark.parametrize("K", [512, 1024, 1056, 1152, 2016, 2048, 2080, 4096])
def test_shares_of_the_channels(K, M, N):
    gen = torch.Generator().manual_seed(K + M)
    gated, w = torch.randn(M, K, generator=gen), torch.randn(N, K, generator=gen).bfloat16()
    weight, parts = 1.0 + 0.1 * torch.randn(K, generator=gen), 4
    sums = gated.double().square().view(M, parts, K // parts).sum(-1).float()
    buf = torch.cat([gated.flatten(), sums.flatten()]).to(DEV)
    out = torch.full((M + 1, N + 4), 7.0, dtype=torch.bfloat16, device=DEV)
    bf, f32 = _lib.dtype_code(torch.bfloat16), _lib.dtype_code(torch.float32)
    nd, wd, gd = _lib.HdlaNormDims(M, 1, K, bf, f32, 1, K ** 0.5, 1e-5), w.to(DEV), weight.to(DEV)
    assert _lib.load().hdla_rows_gemm_norm(M, N, K, buf.data_ptr(), parts, ctypes.byref(nd), gd.data_ptr(), wd.data_ptr(), K, out.data_ptr(), N + 4,
                                           _lib.current_stream(DEV)) == 0
    x = gated.double() / (gated.double().square().mean(-1, keepdim=True) + 1e-5).sqrt() * weight.double()
    x = x.bfloat16().double()
    got, want = out[:M, :N].double().cpu(), x @ w.double().T
    # the result's rounding (2^-8 of it), and x's where its last bit is another one: half a unit (2^-8) of single elements of x, here of all of them
    bound = want.abs() * 2.0 ** -8 + ((x * w.double()[:, None]).square().sum(-1).sqrt() * 2.0 ** -8 * 4).T + 1e-6 * K ** 0.5
    assert ((got - want).abs() <= bound).all()
    assert bool((out[M:] == 7.0).all() and (out[:, N:] == 7.0).all())
