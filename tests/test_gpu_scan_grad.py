"""The scans of the backward pass for 2-byte elements where their loops can go wrong, as test_gpu_scan_out.py has it for the forward
pass: few chunks, ragged ends, every number of column blocks in a workgroup, time segments in both directions, packed sequences
of unequal and no length, either scan by itself.  Against autograd through the float64 recurrence; tolerance: that of every bf16 gradient."""
import pytest
import torch

from hdla_hip import chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV, TOL = "cuda", 1e-2


def _check(inp, heads, cu=None, scale=0.9):
    leaves = [t.bfloat16() for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)] + [inp.h0]
    do, dht = inp.do.bfloat16(), inp.dht
    ref = [(t[:, heads] if i == 6 else t[:, :, heads]).double().requires_grad_() for i, t in enumerate(leaves)]
    o_r, ht_r = O.recurrence(*ref[:6], scale, ref[6], cu_seqlens=cu)
    want = torch.autograd.grad([o_r, ht_r], ref, [do[:, :, heads].double(), dht[:, heads].double()])
    got = [t.to(DEV).requires_grad_() for t in leaves]
    o, ht = chunk_hrdplr_delta_rule(*got[:6], 2, scale=scale, initial_state=got[6], output_final_state=True, cu_seqlens=cu)
    grads = torch.autograd.grad([o, ht], got, [do.to(DEV), dht.to(DEV)])
    errs = [O.rel_l2(x[:, heads] if i == 6 else x[:, :, heads], y) for i, (x, y) in enumerate(zip(grads, want))]
    print(["%.2e" % e for e in errs], flush=True)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("K,V", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 64, 79, 113, 160])
def test_few_chunks(K, V, T, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    _check(make_inputs(1500 + T, 2, T, 2, K, V, gk_div=2.0), [0, 1])


@pytest.mark.parametrize("K,V,H", [(64, 64, 32), (64, 64, 33), (64, 64, 65), (64, 128, 16), (64, 128, 17), (64, 128, 33), (128, 64, 32), (128, 64, 33),
                                   (128, 64, 65), (128, 128, 16), (128, 128, 17), (128, 128, 33)])
def test_column_blocks_of_a_workgroup(K, V, H, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    _check(make_inputs(1600 + H, 1, 100, H, K, V, gk_div=4.0), [0, H // 2, H - 1])


@pytest.mark.parametrize("K,V", [(64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("T,segments", [(40, 2), (100, 3), (230, 4), (330, 7)])
def test_time_segments(K, V, T, segments, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    _check(make_inputs(1700 + T, 1, T, 3, K, V, gk_div=8.0), [0, 2])


@pytest.mark.parametrize("K,V", [(64, 128), (128, 128)])
@pytest.mark.parametrize("segments", [1, 3])
def test_packed_sequences(K, V, segments, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    cu = torch.tensor([0, 5, 5, 101, 117, 300])
    _check(make_inputs(1800, 1, 300, 2, K, V, gk_div=4.0, n_states=5), [0, 1], cu=cu)


@pytest.mark.parametrize("K,V,segments", [(64, 64, 1), (64, 128, 1), (128, 64, 1), (128, 128, 1), (64, 128, 4), (128, 64, 4), (128, 128, 4)])
@pytest.mark.parametrize("where,value", [("do", float("nan")), ("do", float("inf")), ("dht", float("nan")), ("v", float("nan"))])
def test_a_value_that_is_none_stays_with_its_head(K, V, segments, where, value, monkeypatch):
    """In chunk 9 of one head, or in its final state's gradient: the other heads and sequences keep their gradients' bits, and what comes
    behind a gradient does as well."""
    if segments == 1:
        monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    T = 330
    inp = make_inputs(1850, 2, T, 3, K, V, gk_div=8.0)
    t = [x.bfloat16().to(DEV) for x in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)] + [inp.h0.to(DEV)]
    do, dht = inp.do.bfloat16().to(DEV), inp.dht.to(DEV)

    def run():
        x = [y.clone().requires_grad_() for y in t]
        return torch.autograd.grad(chunk_hrdplr_delta_rule(*x[:6], 2, scale=0.9, initial_state=x[6], output_final_state=True), x, [do, dht])

    clean = run()
    if where == "dht":
        dht[1, 2, 3, 5] = value
    else:
        (do if where == "do" else t[2])[1, 150, 2, 5] = value
    for i, (g, g_0) in enumerate(zip(run(), clean)):
        if i == 6:
            assert torch.equal(g[0], g_0[0]) and torch.equal(g[1, :2], g_0[1, :2])
            assert where == "v" or not torch.isfinite(g[1, 2]).all()
            continue
        r = g.shape[1] // T
        bad = torch.zeros(2, T * r, 3, dtype=torch.bool)
        bad[1, :(160 * r if where == "do" else None), 2] = True
        assert torch.equal(g[~bad], g_0[~bad]), i
        assert where == "v" or i == 0 or not torch.isfinite(g[1, :144 * r, 2].float()).all(), i
