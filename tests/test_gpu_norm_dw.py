"""hdla_normalize_bwd_as: the weight's gradient in the weight's own type is the fp32 one rounded once, for every layout of the partial sums."""
import ctypes

import pytest
import torch

from hdla_hip import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
P = _lib.ptr


@pytest.mark.parametrize("rows,G,E", [(0, 1, 64), (1, 1, 16), (7, 2, 48), (300, 1, 1024), (4100, 16, 64), (33, 1, 4096), (5, 1, 16384)])
@pytest.mark.parametrize("gate_pos", [0, 1, 2])
def test_rounded_once(rows, G, E, gate_pos):
    lib, g = _lib.load(), torch.Generator().manual_seed(rows + E)
    x, gate, do = (torch.randn(rows, G * E, generator=g).bfloat16().to(DEV) for _ in range(3))
    w = (1 + 0.1 * torch.randn(G * E, generator=g)).bfloat16().to(DEV)
    d = _lib.HdlaNormDims(rows, G, E, 0, 0, gate_pos, E ** 0.5, 1e-5)
    nws = lib.hdla_normalize_workspace_bytes(ctypes.byref(d))
    out = []
    for f, dt in ((lib.hdla_normalize_bwd, torch.float32), (lib.hdla_normalize_bwd_as, torch.bfloat16)):
        dx, dgate, dw = torch.empty_like(x), torch.empty_like(x), torch.full((G * E,), float("nan"), dtype=dt, device=DEV)
        ws = torch.empty(max(nws, 16), dtype=torch.uint8, device=DEV)
        assert f(ctypes.byref(d), P(x), P(w), P(gate) if gate_pos else None, P(do), P(dx), P(dgate) if gate_pos else None, P(dw), P(ws), nws,
                 _lib.current_stream(DEV)) == 0
        out.append((dx, dw))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1].bfloat16(), out[1][1])
