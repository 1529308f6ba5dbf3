"""The layer's products of some hundred rows (hdla_tile_gemm): edges of tiles, of the waves' shares of K and of its last block, both orders of W, against float64."""
import ctypes

import pytest
import torch

from hdla_hip import _lib

DEV = "cuda"


def _fn():
    f, i, q, p = _lib.load().hdla_tile_gemm, ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p
    f.argtypes, f.restype = [i, i, i, p, q, p, q, i, p, q, p], ctypes.c_int
    return f


def test_what_is_refused():
    f, ok = _fn(), 4096
    call = lambda M=8, N=64, K=64, x=ok, ldx=64, w=ok, ldw=64, turned=0, y=ok, ldy=64: f(M, N, K, x, ldx, w, ldw, turned, y, ldy, None)
    assert call(M=0) == 0
    for kw in (dict(M=-1), dict(N=0), dict(N=60), dict(K=0), dict(K=60), dict(N=72, ldy=72, ldw=72, turned=1), dict(ldx=56), dict(ldw=56), dict(ldy=56), dict(x=None), dict(w=None),
               dict(y=None), dict(x=ok + 8), dict(w=ok + 8), dict(y=ok + 8), dict(ldx=68), dict(ldw=68), dict(ldy=68)):
        assert call(**kw) != 0, kw


# 32 x 32, 64 x 32 and 64 x 64 tiles (TG_UNITS); one row, a row more and less than a tile's; K of one eight, of less than a block for each wave, of a last block of one to seven eights
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (31, 64, 64), (33, 72, 40), (64, 128, 256), (65, 192, 264), (100, 1024, 1024), (100, 3216, 1024), (129, 3216, 520), (63, 8256, 72),
                                   (484, 904, 256), (257, 2048, 904), (1000, 1024, 136), (1025, 960, 320)])
def test_against_float64(M, N, K):
    f, gen = _fn(), torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=gen).bfloat16(), torch.randn(N, K, generator=gen).bfloat16()
    want = (x.double() @ w.double().T).to(DEV)
    nan = float("nan")
    # rows farther apart than they are long, and nothing but NaN between them
    xs = torch.full((M, K + 8), nan, dtype=torch.bfloat16)
    xs[:, :K] = x
    xs = xs.to(DEV)
    for turned in (0, 1) if N % 64 == 0 else (0,):
        ws = torch.full((K, N + 16) if turned else (N, K + 16), nan, dtype=torch.bfloat16)
        ws[:, :N if turned else K] = w.T if turned else w
        ws = ws.to(DEV)
        y = torch.full((M + 1, N + 8), nan, dtype=torch.bfloat16, device=DEV)
        assert f(M, N, K, xs.data_ptr(), xs.stride(0), ws.data_ptr(), ws.stride(0), turned, y.data_ptr(), y.stride(0), torch.cuda.current_stream().cuda_stream) == 0
        got = y[:M, :N].double()
        # rounding to bf16: half a unit, at most 2^-8 of each value; sums of K products in 32 bits: K 2^-24 of the sum of their absolute values
        bound = want.abs() * 2.0 ** -8 + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T).to(DEV)
        assert ((got - want).abs() <= bound).all()
        assert torch.isnan(y[M]).all() and torch.isnan(y[:, N:]).all()
