"""The layer's own matrix products (csrc/lowrank.hip, csrc/skinny.hip) through the C ABI against float64 products of the same
bf16 operands: one rounding of the result, so 2e-3 (logsigmoid is taken of the rounded f, as the kernels do)."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from hdla_hip import _lib
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
P = _lib.ptr


def _rn(seed, *s):
    return torch.randn(*s, generator=torch.Generator().manual_seed(seed)).bfloat16().to(DEV)


@pytest.mark.parametrize("rows,d,D", [(1, 128, 64), (17, 256, 128), (64, 1024, 64), (100, 384, 128), (4100, 256, 64), (4096, 128, 128)])
def test_low_rank_pair(rows, d, D):
    lib, st = _lib.load(), _lib.current_stream(DEV)
    ld, cf, cg = 2 * D + 40, 8, D + 16                             # gaps before, between and behind the two ranges
    u = _lib.HdlaUpDims(rows, d, D, ld, cf, cg)
    y, wf, wg = _rn(1, rows, ld), _rn(2, d, D) * 0.2, _rn(3, d, D) * 0.2
    f, lf, gate = (torch.full((rows, d), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(3))
    assert lib.hdla_layer_up_fwd(ctypes.byref(u), P(y), P(wf), P(wg), P(f), P(lf), P(gate), st) == 0
    f0, g0 = y[:, cf:cf + D].double(), y[:, cg:cg + D].double()
    assert O.rel_l2(f, f0 @ wf.double().t()) <= 2e-3 and O.rel_l2(gate, g0 @ wg.double().t()) <= 2e-3
    assert O.rel_l2(lf, F.logsigmoid(f.double())) <= 2e-3
    lf2 = torch.empty_like(lf)
    assert lib.hdla_layer_up_fwd(ctypes.byref(u), P(y), P(wf), P(wg), None, P(lf2), P(gate), st) == 0
    assert torch.equal(lf, lf2)
    dlf, dg = _rn(4, rows, d), _rn(5, rows, d)
    dy = torch.full((rows, ld), 7.0, dtype=torch.bfloat16, device=DEV)
    assert lib.hdla_layer_down(ctypes.byref(u), P(wf), P(wg), P(f), P(dlf), P(dg), P(dy), st) == 0
    df = (dlf.double() * torch.sigmoid(-f.double())).bfloat16().double()
    assert O.rel_l2(dy[:, cf:cf + D], df @ wf.double()) <= 2e-3 and O.rel_l2(dy[:, cg:cg + D], dg.double() @ wg.double()) <= 2e-3
    rest = torch.ones(ld, dtype=torch.bool, device=DEV)
    rest[cf:cf + D] = rest[cg:cg + D] = False
    assert bool((dy[:, rest] == 7.0).all())
    dwf, dwg = torch.empty_like(wf), torch.empty_like(wg)
    nws = lib.hdla_layer_up_wgrad_workspace_bytes(ctypes.byref(u))
    ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
    assert lib.hdla_layer_up_wgrad(ctypes.byref(u), P(y), P(f), P(dlf), P(dg), P(dwf), P(dwg), P(ws), nws, st) == 0
    assert O.rel_l2(dwf, df.t() @ f0) <= 2e-3 and O.rel_l2(dwg, dg.double().t() @ g0) <= 2e-3
    assert lib.hdla_layer_up_wgrad(ctypes.byref(u), P(y), P(f), P(dlf), P(dg), P(dwf), P(dwg), P(ws), nws - 1, st) == -5
    assert lib.hdla_layer_up_fwd(ctypes.byref(_lib.HdlaUpDims(rows, d, 96, ld, cf, cg)), P(y), P(wf), P(wg), None, P(lf), P(gate), st) == -2


@pytest.mark.parametrize("rows,d,D", [(2047, 128, 64), (2048, 384, 64), (2079, 256, 64), (5000, 640, 64), (31, 128, 128), (33, 384, 64), (4129, 384, 128)])
def test_low_rank_pair_at_the_lines(rows, d, D):
    """Where a dispatch goes another way (rows), and with tiles of 32 rows and of 64 columns that are not all there."""
    test_low_rank_pair(rows, d, D)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(20, 32), (16, 160), (200, 1056), (1040, 2048)])
def test_rows_gemm(M, N, K):
    lib, st = _lib.load(), _lib.current_stream(DEV)
    x, w = _rn(6, M, K + 8), _rn(7, N, K)
    y = torch.full((M + 1, N + 4), 7.0, dtype=torch.bfloat16, device=DEV)
    assert lib.hdla_rows_gemm(M, N, K, P(x), K + 8, P(w), K, P(y), N + 4, st) == 0
    assert O.rel_l2(y[:M, :N], x[:, :K].double() @ w.double().t()) <= 2e-3
    assert bool((y[M:] == 7.0).all() and (y[:, N:] == 7.0).all())
    assert lib.hdla_rows_gemm(65, N, K, P(x), K + 8, P(w), K, P(y), N + 4, st) == -2
    assert lib.hdla_rows_gemm(M, N, K - 8, P(x), K + 8, P(w), K, P(y), N + 4, st) == -2


@pytest.mark.parametrize("M", [16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(4095, 64), (4096, 512), (4116, 544), (4127, 2080)])
def test_rows_gemm_many_columns(M, N, K):
    """Both sides of the line from which a workgroup takes 32 rows of W, with a last one of few; blocks of K that the waves share unevenly."""
    lib, st = _lib.load(), _lib.current_stream(DEV)
    ld = (N + 3) // 4 * 4
    x, w = _rn(8, M, K), _rn(9, N, K)
    y = torch.full((M + 1, ld), 7.0, dtype=torch.bfloat16, device=DEV)
    assert lib.hdla_rows_gemm(M, N, K, P(x), K, P(w), K, P(y), ld, st) == 0
    # bf16 result of an exact sum of K products, up to K fp32 roundings: half a bf16 step each way, 2^-9 at most, on average 2^-9 / sqrt(3)
    assert O.rel_l2(y[:M, :N], x.double() @ w.double().t()) <= 2e-3
    assert bool((y[M:] == 7.0).all() and (y[:, N:] == 7.0).all())


@pytest.mark.parametrize("rows,width,pad", [((1,), 8, 0), ((3, 0, 5), 24, 1), ((64, 64, 64, 16, 16, 4), 256, 12), ((129, 1, 1, 1, 1, 1, 1, 1), 1016, 0),
                                            ((1024, 1024, 1024, 64, 64, 16), 1024, 112)])
def test_stacked_rows(rows, width, pad):
    """Whole pieces copied, so bit for bit; what lies behind the output stays."""
    lib, st = _lib.load(), _lib.current_stream(DEV)
    parts = [_rn(7 + i, r, width) for i, r in enumerate(rows)]
    total = sum(rows) + pad
    buf = torch.full(((total + 3) * width,), 7.0, dtype=torch.bfloat16, device=DEV)
    pp = (ctypes.c_void_p * len(rows))(*[t.data_ptr() for t in parts])
    rr = (ctypes.c_int64 * len(rows))(*rows)
    assert lib.hdla_stack_rows(pp, rr, len(rows), width, P(buf), total, st) == 0
    want = torch.cat(parts + [torch.zeros(pad, width, dtype=torch.bfloat16, device=DEV)])
    assert torch.equal(buf[:total * width].view(total, width), want) and (buf[total * width:] == 7.0).all()
    assert lib.hdla_stack_rows(pp, rr, len(rows), width, P(buf), sum(rows) - 1, st) != 0
    assert lib.hdla_stack_rows(pp, rr, len(rows), width - 1, P(buf), total, st) != 0
