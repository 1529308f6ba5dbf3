"""The gradients of few (chunk, head) pairs, by one launch in which each workgroup does its own pair, flagged or not, next to the same sequences in a batch of more pairs, whose flagged
ones are a launch of their own: both kernels have one text."""
import pytest
import torch

from hdla_hip import chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

DEV = "cuda"


# pairs of a sequence; repeated they pass 256 (K = V = 64 with decays of the inputs' type: 512).  strong: channels that lose more than e^-70 within eight tokens in some pairs, in none, in all
@pytest.mark.gpu
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("strong", ["some", "none", "all"])
@pytest.mark.parametrize("K,V,gk,T,H,times", [(64, 64, torch.bfloat16, 512, 16, 2), (64, 64, torch.bfloat16, 33, 2, 100), (64, 64, torch.float32, 250, 16, 2), (128, 128, torch.bfloat16, 250, 16, 2),
                                              (64, 128, torch.bfloat16, 17, 1, 140), (128, 64, torch.float32, 100, 3, 16)])
def test_few_and_many(K, V, gk, T, H, times, strong, form):
    inp = make_inputs(41, 1, T, H, K, V, gk_div=16.0)
    k = torch.nn.functional.normalize(inp.k, dim=-1)
    beta = 2.0 * torch.rand(1, T, H, 1, generator=torch.Generator().manual_seed(5))
    g = inp.gk.clone()
    if strong != "none":
        g[:, ::3, :, :5] = -18.0
        if strong == "some":
            g[:, : T // 2, ::2] = inp.gk[:, : T // 2, ::2]
    x = [t.bfloat16() for t in [inp.q, k, inp.v] + ([inp.a, inp.b] if form == "ab" else [beta])] + [g.to(gk)]
    op = (lambda *a, **kw: chunk_hrdplr_delta_rule(*a, 2, **kw)) if form == "ab" else chunk_hdla_delta_rule

    def grads(n):
        leaves = [t.repeat(n, *[1] * (t.dim() - 1)).to(DEV).requires_grad_() for t in x]
        o, ht = op(*leaves, scale=0.7, output_final_state=True, keep_forward=False)
        do = inp.do.bfloat16().repeat(n, 1, 1, 1).to(DEV)
        return torch.autograd.grad([o, ht], leaves, [do, torch.zeros_like(ht)])

    with pytest.MonkeyPatch.context() as mp:
        mp.setenv("HDLA_HIP_ROUTE", "plain")                     # the classic kernels in one segment, whatever the number of lanes
        few, many = grads(1), grads(times)
    for i, (a, b) in enumerate(zip(few, many)):
        assert torch.isfinite(a.float()).all(), i
        for n in (0, times - 1):
            assert torch.equal(a[0], b[n]), (i, n)
