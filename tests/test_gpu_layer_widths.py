"""Training steps of the layer on both sides of the lines that its concatenated weight's rows are padded by (whole 128-row tiles, where the weight's gradient is then the library's
own), and that its products' kernels are chosen by, next to the layer's Python code."""
import pytest
import torch

from hdla_hip.layer import HDLA_Custom

DEV = "cuda"


# rows of the weight 3 d + 2 D + H: short of a tile, over one; 1024 rows; more tiles than there are compute units (d = 2048); 64 rows and 65
@pytest.mark.gpu
@pytest.mark.parametrize("B,T,d,H", [(1, 1, 128, 2), (2, 33, 256, 4), (1, 64, 128, 2), (1, 65, 512, 8), (1, 1023, 128, 2), (1, 1024, 128, 2), (3, 100, 512, 4), (1, 70, 2048, 16)])
def test_against_the_python_code(B, T, d, H):
    torch.manual_seed(3)
    with torch.device(DEV):
        m = HDLA_Custom(d, H, token_mixer_init_type=2, rescale_type=0).bfloat16().train()
        x, do = torch.randn(B, T, d).bfloat16().requires_grad_(), torch.randn(B, T, d).bfloat16()
    names = ["x", *(n for n, _ in m.named_parameters())]

    def step():
        y = m(x)[0]
        return [y.detach(), *torch.autograd.grad(y, [x, *m.parameters()], do)]

    got = step()
    m._forward_native = lambda *_: None
    want = step()
    # every stage of both rounds its result to bf16 (2^-9 of it at the most), a dozen of them one behind the other, in other orders of sums
    for n, a, b in zip(["y", *names], got, want):
        assert a.shape == b.shape and torch.isfinite(a.float()).all(), n
        rel = (a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)
        assert rel <= 12 * 2.0 ** -8, (n, float(rel))
