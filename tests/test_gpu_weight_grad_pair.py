"""hdla_weight_grad_pair (csrc/wgrad.hip): two weight gradients over the same rows in one launch.  Small whole numbers, most of them zero, whose sums bf16
holds, so that every tile and row counts once to the bit.  Few tiles in shares; as many as there are workgroups; one, some and 256 more; rows that
fill neither a stage nor a share."""
import ctypes

import pytest
import torch

from hdla_hip import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _arr(kind, values):
    return (kind * 2)(*values)


def _call(M, N, K, dy, x, room=None):
    lib = _lib.load()
    n, k = _arr(ctypes.c_int32, N), _arr(ctypes.c_int32, K)
    nws = lib.hdla_weight_grad_pair_workspace_bytes(M, n, k)
    ws = torch.full((max(nws, 16),), 0xff, dtype=torch.uint8, device=DEV)
    dw = [torch.full((N[i], K[i]), float("nan"), dtype=torch.bfloat16, device=DEV) for i in range(2)]
    p = lambda t: _arr(ctypes.c_void_p, [_lib.ptr(a) for a in t])
    s = lambda t: _arr(ctypes.c_int64, [a.stride(0) for a in t])
    rc = lib.hdla_weight_grad_pair(M, n, k, p(dy), s(dy), p(x), s(x), p(dw), _lib.ptr(ws), nws if room is None else room, None, _lib.current_stream(DEV))
    return rc, dw, nws


@pytest.mark.parametrize("M", [1, 65, 128, 511, 1025, 2200, 8192])
@pytest.mark.parametrize("N,K", [((128, 128), (128, 256)), ((1792, 512), (512, 512)), ((2048, 512), (1920, 512)), ((2048, 128), (2048, 128)),
                                 ((3328, 1024), (1024, 1024)), ((2048, 2048), (2048, 2048))])
def test_every_row_counts_once(M, N, K):
    g = torch.Generator().manual_seed(M + N[0])
    rare = lambda r, c: torch.randint(-1, 2, (r, c), generator=g) * (torch.rand(r, c, generator=g) < 0.08)
    dy = [rare(M, n + 64).bfloat16().to(DEV)[:, 32:32 + n] for n in N]
    x = [rare(M, k + 8).bfloat16().to(DEV)[:, 8:] for k in K]
    for t in dy + x:
        t[-1] = 1
    rc, dw, _ = _call(M, N, K, dy, x)
    assert rc == 0
    for i in range(2):
        want = dy[i].float().t() @ x[i].float()
        assert want.abs().max() <= 256
        assert torch.equal(dw[i].float(), want), i


def test_refusals():
    z = torch.zeros(2048, 4096, dtype=torch.bfloat16, device=DEV)
    assert _call(2048, (128, 128), (128, 128), [z, z], [z, z], room=0)[0] == -5
    assert _call(2048, (128, 100), (128, 128), [z, z], [z, z])[0] == -2
    assert _call(2048, (4096, 128), (1152, 128), [z, z], [z, z])[0] == -2      # 288 tiles
    assert _call(2048, (128, 128), (128, 128), [z, z[:, 1:]], [z, z])[0] == -6
