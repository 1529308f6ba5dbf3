"""u and w where the backward pass forms them again from (I - A_ab)^-1, A_ak, the sums over channels and the inputs: lengths at
the edges of a chunk, packed sequences, strong decays, decays in the inputs' type (rebuilt) and fp32 (read from the workspace).
Against the float64 recurrence at the operators' stated tolerances (5e-3 forward, 1e-2 backward for bf16), and bit for bit where the same kernels
run on a kept workspace, on a recomputed one and on one whose buffers the classic route leaves to be looked at."""
import pytest
import torch

from hdla_hip import chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def _step(form, K, V, lens, gk_dtype, keep, strong=False):
    g = torch.Generator().manual_seed(sum(lens) + K + 3 * V)
    T, H, N = sum(lens), 2, len(lens)
    rn = lambda *s: torch.randn(*s, generator=g)
    unit = lambda: torch.nn.functional.normalize(rn(1, T, H, K), dim=-1)
    q, k, v = unit(), unit(), rn(1, T, H, V)
    beta, log_f = 2.0 * torch.rand(1, T, H, 1, generator=g), torch.nn.functional.logsigmoid(rn(1, T, H, K))
    if strong:
        log_f[..., 5] = -14.0
    h0, do, dht = rn(N, H, K, V), rn(1, T, H, V), rn(N, H, K, V)
    a, b = O.parameterize_a_b(beta, k, log_f)
    x = [q, k, v] + ([beta] if form == "beta" else [a, b]) + [log_f]
    types = [BF] * (len(x) - 1) + [gk_dtype]
    cu = torch.tensor([sum(lens[:i]) for i in range(N + 1)]) if N > 1 else None

    leaves = [t.to(d).double().requires_grad_() for t, d in zip(x, types)]
    ab = O.parameterize_a_b(leaves[3], leaves[1], leaves[4]) if form == "beta" else leaves[3:5]
    h = h0.double().requires_grad_()
    o, ht = O.recurrence(*leaves[:3], *ab, leaves[-1], 1.0, h, cu_seqlens=cu)
    ref = [o, ht] + list(torch.autograd.grad([o, ht], leaves + [h], [do.to(BF).double(), dht.double()]))

    leaves = [t.to(d).to(DEV).requires_grad_() for t, d in zip(x, types)]
    h = h0.to(DEV).requires_grad_()
    kw = dict(scale=1.0, initial_state=h, output_final_state=True, cu_seqlens=None if cu is None else cu.to(DEV), keep_forward=keep)
    o, ht = chunk_hdla_delta_rule(*leaves, **kw) if form == "beta" else chunk_hrdplr_delta_rule(*leaves, 2, chunk_size=16, **kw)
    got = [o, ht] + list(torch.autograd.grad([o, ht], leaves + [h], [do.to(BF).to(DEV), dht.to(DEV)]))
    return [t.detach() for t in got], [t.detach() for t in ref]


@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("lens", [(1,), (16,), (47,), (15, 1, 33)])
@pytest.mark.parametrize("K,V", [(64, 64), (128, 128), (64, 128), (128, 64)])
@pytest.mark.parametrize("form,gk_dtype", [("beta", BF), ("beta", torch.float32), ("ab", BF)])
def test_rebuilt_operands(form, gk_dtype, K, V, lens, strong, monkeypatch):
    outs = {}
    for route, keep in (("auto", None), ("classic", False), ("classic", True)):
        monkeypatch.setenv("HDLA_HIP_ROUTE", route)
        got, ref = outs[route, keep] = _step(form, K, V, lens, gk_dtype, keep, strong)
        errs = [O.rel_l2(x, r) for x, r in zip(got, ref)]
        print(form, gk_dtype, K, V, lens, strong, route, keep, [f"{e:.1e}" for e in errs], flush=True)
        # (dbeta: one value a token, here 2 to 98 in all, in which the two ranks' parts, rounded to 2^-9 each, cancel to a quarter and less of
        # their size: 2 x 2^-9 x 4 of single values, up to twice that at the worst of them; 2.8e-2 with u and w as the forward pass had them)
        dbeta = errs.pop(5) if form == "beta" else 0.
        assert max(errs[:2]) <= 5e-3 and max(errs[2:]) <= 1e-2 and dbeta <= 3.2e-2, (errs, dbeta)
    for x, y in zip(outs["classic", False][0], outs["classic", True][0]):
        assert torch.equal(x, y)
    if (K, V) != (64, 64):                                # (there the library's own choice may be another route)
        for x, y in zip(outs["classic", False][0], outs["auto", None][0]):
            assert torch.equal(x, y)
