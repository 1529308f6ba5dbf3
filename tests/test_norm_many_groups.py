"""The norm over more groups a row than a launch has workgroups to give each (65536): groups of up to 512 16-byte pieces are a wavefront's there, four a
workgroup, and only wider ones are refused."""
import ctypes

import pytest
import torch

from hdla_hip import _lib
from hdla_hip.normalize import normalize_fn


def _room(G, E, rows=4, dtype=_lib.HDLA_BF16):
    d = _lib.HdlaNormDims(rows, G, E, dtype, _lib.HDLA_FP32, 1, 1.0, 1e-5)
    return _lib.load().hdla_normalize_workspace_bytes(ctypes.byref(d))


@pytest.mark.parametrize("dtype,n", [(_lib.HDLA_BF16, 8), (_lib.HDLA_FP32, 4)])
@pytest.mark.parametrize("pieces", [129, 256, 512])
def test_what_is_taken(dtype, n, pieces):
    E = n * pieces
    # partial rows of the weight's gradient, 4 E bytes each: one for each group at the least
    for G in (65535, 65536, 65540, 200000, 262144):
        room = _room(G, E, dtype=dtype)
        assert room >= 4 * G * E and room % (4 * G * E) == 0, G
    # no multiple of four: the launch would meet its groups again after more than 65536 workgroups
    for G in (65537, 131074, 262148):
        assert _room(G, E, dtype=dtype) == 0, G
    assert _room(65536, n * 513, dtype=dtype) > 0 and _room(65540, n * 513, dtype=dtype) == 0


@pytest.mark.gpu
def test_against_float64():
    G, E = 65540, 1032
    g = torch.Generator(device="cuda").manual_seed(3)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, do, w = rn(1, G * E).bfloat16().requires_grad_(), rn(1, G * E).bfloat16(), (1.0 + 0.1 * rn(G * E)).requires_grad_()
    o = normalize_fn(x, w, c=E ** 0.5, eps=1e-5, num_groups=G)
    dx, dw = torch.autograd.grad(o, (x, w), do)
    X, D, W = x.detach().view(G, E).double(), do.view(G, E).double(), w.detach().view(G, E).double()
    r = torch.rsqrt((X * X).mean(-1, keepdim=True) + 1e-5)
    want = [X * r * W, r * (D * W - X * r * r * (D * W * X).mean(-1, keepdim=True)), D * X * r]
    errs = [((a.view(G, E).double() - b).norm() / b.norm()).item() for a, b in zip((o.detach(), dx, dw), want)]
    # rounded once to bf16 (2^-9, rms 1.66e-3); one product of 32-bit values
    assert max(errs[:2]) <= 3e-3 and errs[2] <= 4e-7, errs
