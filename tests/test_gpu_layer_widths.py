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
    # every stage of both rounds its result to bf16 (2^-8 of it at the most), a dozen of them one behind the other, in other orders of sums
    for n, a, b in zip(["y", *names], got, want):
        assert a.shape == b.shape and torch.isfinite(a.float()).all(), n
        rel = (a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)
        assert rel <= 12 * 2.0 ** -8, (n, float(rel))


# rows that the layer's own products take, on both sides of the number of their tiles with and without the padding (257 .. 320 of 1024 channels), and that are the BLAS library's
@pytest.mark.gpu
@pytest.mark.parametrize("B,T,d,H", [(1, 33, 1024, 16), (1, 65, 512, 8), (1, 257, 1024, 16), (4, 80, 1024, 16), (1, 321, 1024, 16), (2, 500, 1024, 16), (1, 700, 512, 4), (1, 1023, 768, 6), (1, 1024, 768, 6)])
def test_outputs_with_and_without_gradients(B, T, d, H):
    """The same bits, as a recomputation in place of a pass without gradients expects them; so are the gradients behind one."""
    from torch.utils.checkpoint import checkpoint
    torch.manual_seed(4)
    with torch.device(DEV):
        m = HDLA_Custom(d, H, token_mixer_init_type=2, rescale_type=0).bfloat16().train()
        x, do = torch.randn(B, T, d).bfloat16().requires_grad_(), torch.randn(B, T, d).bfloat16()
    y = m(x)[0]
    want = torch.autograd.grad(y, [x, *m.parameters()], do)
    with torch.no_grad():
        assert torch.equal(m(x)[0], y)
        m.eval()
        assert torch.equal(m(x)[0], y)
        m.train()
    y2 = checkpoint(lambda t: m(t)[0], x, use_reentrant=True)
    assert torch.equal(y2, y)
    for p in [x, *m.parameters()]:
        p.grad = None
    y2.backward(do)
    for p, w in zip([x, *m.parameters()], want):
        assert torch.equal(p.grad, w)
