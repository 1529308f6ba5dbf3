"""hdla_weight_grad (csrc/wgrad.hip) through the C ABI against the float64 product of the same bf16 operands: one rounding of the result, so 2e-3.
Rows that fill no stage or pair of stages, one and several shares, one and many tiles, operands within wider ones, values that are none."""
import pytest
import torch

from hdla_hip import _lib
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
P = _lib.ptr


def _call(dy, x, N, K):
    lib, M = _lib.load(), dy.shape[0]
    nws = lib.hdla_weight_grad_workspace_bytes(M, N, K)
    ws = torch.full((max(nws, 16),), 0xff, dtype=torch.uint8, device=DEV)
    dw = torch.full((N, K), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert lib.hdla_weight_grad(M, N, K, P(dy), dy.stride(0), P(x), x.stride(0), P(dw), P(ws), nws, _lib.current_stream(DEV)) == 0
    return dw, nws


@pytest.mark.parametrize("M", [1, 63, 64, 65, 127, 128, 129, 500, 1023, 1025, 2200, 5000])
@pytest.mark.parametrize("N,K", [(128, 128), (256, 384), (1024, 1024)])
def test_against_float64(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    dy = torch.randn(M, N + 64, generator=g).bfloat16().to(DEV)[:, 32:32 + N]
    x = torch.randn(M, K + 8, generator=g).bfloat16().to(DEV)[:, 8:]
    dw, nws = _call(dy, x, N, K)
    assert (nws > 0) == (M >= 1024)
    assert O.rel_l2(dw, dy.double().t() @ x.double()) <= 2e-3


def test_many_tiles_and_refusals():
    g = torch.Generator().manual_seed(1)
    dy, x = torch.randn(300, 3328, generator=g).bfloat16().to(DEV), torch.randn(300, 1024, generator=g).bfloat16().to(DEV)
    dw, nws = _call(dy, x, 3328, 1024)
    assert nws == 0 and O.rel_l2(dw, dy.double().t() @ x.double()) <= 2e-3
    lib, st = _lib.load(), _lib.current_stream(DEV)
    call = lambda M=300, N=128, K=128, ldy=3328, ldx=1024, y=P(dy), ws=None, n=0: lib.hdla_weight_grad(M, N, K, y, ldy, P(x), ldx, P(dw), ws, n, st)
    assert [call(N=120), call(K=64), call(M=0), call(ldy=100), call(ldx=1020)] == [-2] * 5
    assert call(y=None) == -1 and call(y=dy.data_ptr() + 2) == -6 and lib.hdla_weight_grad_workspace_bytes(2048, 128, 128) > 0
    assert lib.hdla_weight_grad(2048, 128, 128, P(dy), 128, P(x), 128, P(dw), None, 0, st) == -5


@pytest.mark.parametrize("M", [65, 1025, 1030, 2200, 5000])
@pytest.mark.parametrize("N,K", [(128, 128), (256, 384)])
def test_every_row_counts_once(M, N, K):
    """Small whole numbers, most of them zero, whose sums bf16 holds: the bits, at rows that fill neither the last stage nor the last share."""
    g = torch.Generator().manual_seed(M)
    dy = (torch.randint(-1, 2, (M, N), generator=g) * (torch.rand(M, N, generator=g) < 0.1)).bfloat16().to(DEV)
    x = (torch.randint(-1, 2, (M, K), generator=g) * (torch.rand(M, K, generator=g) < 0.1)).bfloat16().to(DEV)
    dy[-1], x[-1] = 1, 1                                           # (the row that those past the end are read from)
    want = dy.double().t() @ x.double()
    assert want.abs().max() <= 256
    assert torch.equal(_call(dy, x, N, K)[0].double(), want)


@pytest.mark.parametrize("M", [100, 1025, 2200])                  # one share; the last one's last stage of one row; several stages
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -3.3895313892515355e38])
def test_a_value_that_is_none_stays_in_its_row(value, M):
    g = torch.Generator().manual_seed(2)
    dy, x = torch.randn(M, 256, generator=g).bfloat16().to(DEV), torch.rand(M, 128, generator=g).bfloat16().to(DEV) + 0.5
    clean = _call(dy, x, 256, 128)[0]
    dy[M - 1, 77] = value                                          # (in the last row, which the rows past the end are read from)
    dw = _call(dy, x, 256, 128)[0]
    rest = torch.arange(256, device=DEV) != 77
    assert torch.equal(dw[rest], clean[rest])
    want = (dy[:, 77].double() @ x.double()).float().bfloat16()
    assert torch.equal(dw[77].isnan(), want.isnan()) and torch.equal(dw[77].isinf(), want.isinf())
