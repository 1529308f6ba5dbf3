"""The gated norm where its launch changes: groups of more than two 16-byte pieces a lane of a wavefront (a workgroup has them), the rows from which a lane's sums
for the weight's gradient are folded (every four), and the grid of the backward kernel with two pieces a lane."""
import pytest
import torch

from hdla_hip.normalize import normalize_fn

pytestmark = pytest.mark.gpu


def _reference(x, w, gate, pos, eps):
    s = torch.sigmoid(gate)
    z = x * s if pos == "pre" else x
    o = z / torch.sqrt((z * z).mean(-1, keepdim=True) + eps) * w
    return o * s if pos == "post" else o


# bf16 outputs are rounded once (2^-9, rms 1.66e-3); 32-bit sums stay below 2.1e-7, the longest here
@pytest.mark.parametrize("rows,E,dtype,pos", [
    (1, 1032, torch.bfloat16, "pre"), (3, 1024, torch.bfloat16, "pre"), (4099, 1032, torch.bfloat16, "post"), (4100, 2056, torch.bfloat16, "pre"),
    (16400, 1024, torch.bfloat16, "pre"), (13000, 776, torch.bfloat16, "post"), (4097, 516, torch.float32, "pre"), (8300, 516, torch.float32, "post"),
    (2050, 1028, torch.float32, "pre"), (4100, 2052, torch.float32, "pre")])
def test_against_float64(rows, E, dtype, pos):
    g = torch.Generator(device="cuda").manual_seed(rows + E)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, gate, do = (rn(rows, E).to(dtype) for _ in range(3))
    w = 1.0 + 0.1 * rn(E)
    leaves = [t.requires_grad_() for t in (x, gate, w)]
    o = normalize_fn(x, w, gate=gate, gate_pos=pos, c=E ** 0.5, eps=1e-5)
    got = [o.detach(), *torch.autograd.grad(o, leaves, do)]
    X, G, W = (t.detach().double().requires_grad_() for t in leaves)
    r = _reference(X, W, G, pos, 1e-5)
    want = [r.detach(), *torch.autograd.grad(r, [X, G, W], do.double())]
    errs = [((a.double() - b).norm() / b.norm()).item() for a, b in zip(got, want)]
    assert max(errs[:3]) <= (3e-3 if dtype == torch.bfloat16 else 4e-7) and errs[3] <= 4e-7, errs
