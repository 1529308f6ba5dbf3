"""The token-serial kernel over both forms of its grid (fewer than 256 workgroups; 256 and more, a head's column blocks as neighbours)
and over tokens requested ahead: a call over many sequences against one call each (the same arithmetic in the same order, so the
same bits), and against the float64 recurrence (bf16 outputs: 8 bits; the state in fp32 over T tokens)."""
import pytest
import torch

from hdla_hip import fused_recurrent_dplr_delta_rule, fused_recurrent_hdla_delta_rule
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("N,H,K,V,T", [(51, 5, 64, 64, 3), (64, 4, 64, 64, 1), (17, 15, 64, 64, 2), (25, 5, 64, 128, 4), (43, 3, 128, 128, 1),
                                       (16, 8, 128, 128, 5), (9, 7, 128, 256, 2), (64, 4, 128, 64, 3), (33, 2, 256, 256, 2), (70, 1, 64, 256, 6)])
def test_grid_forms(dtype, reverse, N, H, K, V, T):
    inp = make_inputs(900 + N, N, T, H, K, V, gk_div=2.0, n_states=N)
    q, k, v, a, b, gk = [t.to(dtype).to(DEV) for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)]
    h0 = inp.h0.to(DEV)
    beta = torch.rand(N, T, H, generator=torch.Generator().manual_seed(N)).to(dtype).to(DEV)
    kw = dict(scale=0.7, output_final_state=True, reverse=reverse)

    def dplr(s):
        return fused_recurrent_dplr_delta_rule(q[s], k[s], v[s], a[s], b[s], gk[s], 2, initial_state=h0[s], **kw)

    def hdla(s):
        return fused_recurrent_hdla_delta_rule(q[s], k[s], v[s], beta[s], gk[s], initial_state=h0[s], **kw)

    for f in (dplr, hdla):
        o, ht = f(slice(None))
        for n in (0, 1, N // 2, N - 1):
            o_1, ht_1 = f(slice(n, n + 1))
            assert torch.equal(o[n], o_1[0]) and torch.equal(ht[n], ht_1[0]), (f.__name__, n)
    o, ht = dplr(slice(None))
    o_r, ht_r = O.recurrence(*[t.cpu().double() for t in (q, k, v, a, b, gk)], 0.7, inp.h0.double(), reverse=reverse)
    tol = 5e-3 if dtype == torch.bfloat16 else 1e-5
    assert O.rel_l2(o, o_r) <= tol and O.rel_l2(ht, ht_r) <= 1e-5


@pytest.mark.parametrize("lengths", [[0, 1, 5, 0, 2] * 20, [3, 0, 7]])
def test_packed_with_empty_sequences(lengths):
    cu = torch.tensor([0] + lengths).cumsum(0)
    N, total = len(lengths), sum(lengths)
    inp = make_inputs(950, 1, total, 3, 64, 128, gk_div=2.0, n_states=N)
    t = [x.to(DEV) for x in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)]
    o, ht = fused_recurrent_dplr_delta_rule(*t, 2, scale=0.7, initial_state=inp.h0.to(DEV), output_final_state=True, cu_seqlens=cu.to(DEV))
    o_r, ht_r = O.recurrence(*[x.cpu().double() for x in t], 0.7, inp.h0.double(), cu_seqlens=cu)
    assert O.rel_l2(o, o_r) <= 1e-5 and O.rel_l2(ht, ht_r) <= 1e-5
    empty = [n for n in range(N) if lengths[n] == 0]
    assert torch.equal(ht[empty].cpu(), inp.h0[empty])
