"""Inputs that arrive as whole row pieces and change lanes in LDS (prep and chunk_grad kernels): every head shape, both forms
of the operator and both types of the decays, at lengths that leave the last chunk one row, all but one, exactly full and one over,
against the float64 recurrence with autograd through it (bf16: outputs 5e-3, gradients 1e-2; fp32: 1e-5)."""
import pytest
import torch

from hdla_hip import chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
TOL = {"bf16": (5e-3, 1e-2), "bf16_gk32": (5e-3, 1e-2), "fp32": (1e-5, 1e-5)}


@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("types", list(TOL))
@pytest.mark.parametrize("K,V", [(64, 64), (128, 128), (64, 128), (128, 64)])
@pytest.mark.parametrize("T,H,cu", [(1, 3, None), (15, 2, None), (16, 1, None), (17, 33, None), (47, 2, (0, 1, 18, 18, 47))])
def test_rows_into_fragments(T, H, cu, K, V, types, form, monkeypatch):
    if (K, V) == (64, 64):
        monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")       # the kernels of the other shapes, at this one
    dt = torch.float32 if types == "fp32" else torch.bfloat16
    gdt = torch.bfloat16 if types == "bf16" else torch.float32
    N = 1 if cu is None else len(cu) - 1
    inp = make_inputs(7, 1, T, H, K, V, gk_div=4.0, n_states=N)
    names = ["q", "k", "v"] + (["a", "b"] if form == "ab" else []) + ["gk"]
    x = {n: getattr(inp, n).to(gdt if n == "gk" else dt) for n in names}
    if form == "beta":
        x["k"] = torch.nn.functional.normalize(inp.k, dim=-1).to(dt)
        x["beta"] = (2.0 * torch.rand(1, T, H, 1, generator=torch.Generator().manual_seed(5))).to(dt)
    table = None if cu is None else torch.tensor(cu, dtype=torch.int64)

    def run(dev, wide):
        lv = {n: (t.double() if wide else t).to(dev).requires_grad_() for n, t in x.items()}
        h0 = (inp.h0.double() if wide else inp.h0).to(dev).requires_grad_()
        c = None if table is None else table.to(dev)
        if wide:
            a, b = (lv["a"], lv["b"]) if form == "ab" else O.parameterize_a_b(lv["beta"], lv["k"], lv["gk"])
            o, ht = O.recurrence(lv["q"], lv["k"], lv["v"], a, b, lv["gk"], 0.7, h0, cu_seqlens=c)
        elif form == "ab":
            o, ht = chunk_hrdplr_delta_rule(*[lv[n] for n in names], 2, scale=0.7, initial_state=h0, output_final_state=True,
                                            chunk_size=16, cu_seqlens=c)
        else:
            o, ht = chunk_hdla_delta_rule(lv["q"], lv["k"], lv["v"], lv["beta"], lv["gk"], scale=0.7, initial_state=h0,
                                          output_final_state=True, cu_seqlens=c)
        g = torch.autograd.grad([o, ht], list(lv.values()) + [h0], [inp.do.to(dt).to(o), inp.dht.to(ht)])
        return [o.detach(), ht.detach()], dict(zip(list(lv) + ["h0"], g))

    (o, ht), g = run("cuda", False)
    (ro, rht), rg = run("cpu", True)
    tol_o, tol_g = TOL[types]
    errs = {"o": O.rel_l2(o, ro), "ht": O.rel_l2(ht, rht), **{n: O.rel_l2(g[n], rg[n]) for n in g}}
    print(T, H, K, V, types, form, {n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
    assert errs["o"] <= tol_o and errs["ht"] <= tol_o, errs
    # dbeta is one number a token and head: with a handful of them nothing averages out the roundings of the four 8-bit factors
    # (k, the decayed copy, the state gradient, the result) of their sums, 2^-8 each at the worst
    tol_beta = max(tol_g, 4 * 2.0 ** -8) if dt == torch.bfloat16 and T * H < 16 else tol_g
    assert all(errs[n] <= (tol_beta if n == "beta" else tol_g) for n in g), errs
