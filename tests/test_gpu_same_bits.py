"""Outputs and gradients of some calls of every kind of chunk_grad kernel (few pairs and many, common ones and flagged, decays of the inputs' type and fp32) and of packed sequences on the
fused route, bit for bit what they have been: which multiply is fused with which add and where a sequence is cut are part of the kernels, and no matter of what else a file has, how it is
compiled or what a sequence is packed with."""
import hashlib

import pytest
import torch

from hdla_hip import chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

DEV, BF, F32 = "cuda", torch.bfloat16, torch.float32

# form, route, element type, type of the decays, K, V, heads, lengths (packed where there are several), strong decays: digest
CASES = [
    (("ab", "plain", BF, BF, 64, 64, 16, (1100,), False), "3fc9d92c2656c186"),
    (("ab", "plain", BF, BF, 128, 128, 16, (500,), True), "890ea1eb968d4005"),
    (("ab", "plain", BF, F32, 64, 128, 5, (17, 333), True), "e87b434f5acc3822"),
    (("ab", "plain", BF, F32, 128, 64, 16, (500,), False), "a6ae86a25ad1037f"),
    (("beta", "plain", BF, BF, 64, 64, 16, (1100,), True), "715af2b346258485"),
    (("beta", "plain", BF, BF, 128, 128, 16, (300, 211), False), "473c9e8a24438656"),
    (("beta", "plain", BF, F32, 128, 128, 3, (200,), True), "3ac7b31692f489eb"),
    (("beta", "plain", BF, BF, 64, 128, 16, (500,), False), "2fd06501c701c114"),
    (("beta", "plain", BF, BF, 128, 64, 2, (99,), False), "98b269fcf0029ca7"),
    (("beta", "auto", BF, BF, 64, 64, 2, (256,), False), "410e8294307728a6"),
    (("beta", "fused", BF, BF, 64, 64, 16, (2048,), False), "8a4c0b87794f070b"),
    (("ab", "fused", BF, F32, 64, 64, 3, (700,), True), "ce98f932aee3720b"),
    (("beta", "fused", BF, BF, 64, 64, 16, (2000, 17, 983), False), "e469513fe0726ae3"),
    (("ab", "fused", BF, BF, 64, 64, 2, (48, 1200, 300, 5), True), "16e908c0b85e6754"),
    (("beta", "plain", F32, F32, 64, 64, 8, (501,), False), "254d916e912087e3"),
    (("ab", "plain", F32, F32, 128, 64, 2, (64, 30), True), "f51379d2e86e56e8"),
]


def digest(form, route, dtype, gk_dtype, K, V, H, lens, strong):
    inp = make_inputs(7, 1, sum(lens), H, K, V, n_states=len(lens))
    beta = 2.0 * torch.rand(1, sum(lens), H, 1, generator=torch.Generator().manual_seed(3))
    g = inp.gk.clone()
    if strong:
        g[:, ::3, :, :5] = -18.0
    x = [inp.q, inp.k, inp.v] + ([inp.a, inp.b] if form == "ab" else [beta]) + [g]
    leaves = [t.to(dtype).to(DEV).requires_grad_() for t in x[:-1]] + [g.to(gk_dtype).to(DEV).requires_grad_(), inp.h0.to(DEV).requires_grad_()]
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], device=DEV) if len(lens) > 1 else None
    kw = dict(scale=0.7, initial_state=leaves[-1], output_final_state=True, cu_seqlens=cu)
    with pytest.MonkeyPatch.context() as mp:
        mp.setenv("HDLA_HIP_ROUTE", route)
        o, ht = chunk_hrdplr_delta_rule(*leaves[:-1], 2, **kw) if form == "ab" else chunk_hdla_delta_rule(*leaves[:-1], **kw)
        out = [o, ht, *torch.autograd.grad([o, ht], leaves, [inp.do.to(o), inp.dht.to(DEV)])]
    h = hashlib.sha1()
    for t in out:
        h.update(t.detach().contiguous().view(torch.uint8).cpu().numpy().tobytes())
    return h.hexdigest()[:16]


@pytest.mark.gpu
@pytest.mark.parametrize("case,want", CASES, ids=[" ".join(str(x).replace("torch.", "") for x in c) for c, _ in CASES])
def test_same_bits(case, want):
    assert digest(*case) == want
