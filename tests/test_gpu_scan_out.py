"""The forward pass's scan for 2-byte elements where its loops can go wrong: sequences of fewer chunks than it has slots in LDS or
registers in flight, ragged ends, every number of column blocks in a workgroup, time segments, packed sequences of unequal
and no length.  Against the float64 recurrence; tolerance: that of every bf16 output (operands rounded to 8 bits)."""
import pytest
import torch

from hdla_hip import chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV, TOL = "cuda", 5e-3


def _check(inp, heads, cu=None, scale=0.9):
    leaves = [t.bfloat16() for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)]
    o_r, ht_r = O.recurrence(*[t[:, :, heads].double() for t in leaves], scale, inp.h0[:, heads].double(), cu_seqlens=cu)
    with torch.no_grad():
        o, ht = chunk_hrdplr_delta_rule(*[t.to(DEV) for t in leaves], 2, scale=scale, initial_state=inp.h0.to(DEV), output_final_state=True,
                                        cu_seqlens=cu)
    errs = O.rel_l2(o[:, :, heads], o_r), O.rel_l2(ht[:, heads], ht_r)
    print(["%.2e" % e for e in errs], flush=True)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("K,V", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 48, 64, 79, 96, 113, 160, 250])
def test_few_chunks(K, V, T, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    _check(make_inputs(500 + T, 2, T, 2, K, V, gk_div=2.0), [0, 1])


@pytest.mark.parametrize("K,V", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("H", [3, 32, 33, 64, 65, 129])
def test_column_blocks_of_a_workgroup(K, V, H, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    _check(make_inputs(600 + H, 1, 100, H, K, V, gk_div=4.0), [0, H // 2, H - 1])


@pytest.mark.parametrize("K,V", [(64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("T,segments", [(40, 2), (100, 3), (230, 4), (330, 7)])
def test_time_segments(K, V, T, segments, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    _check(make_inputs(700 + T, 1, T, 3, K, V, gk_div=8.0), [0, 2])


@pytest.mark.parametrize("K,V", [(64, 128), (128, 128)])
@pytest.mark.parametrize("segments", [1, 3])
def test_packed_sequences(K, V, segments, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    cu = torch.tensor([0, 5, 5, 101, 117, 300])
    inp = make_inputs(800, 1, 300, 2, K, V, gk_div=4.0, n_states=5)
    _check(inp, [0, 1], cu=cu)


@pytest.mark.parametrize("K,V,segments", [(64, 64, 1), (64, 128, 1), (128, 64, 1), (128, 128, 1), (64, 128, 4), (128, 64, 4), (128, 128, 4)])
@pytest.mark.parametrize("where,value", [("q", float("nan")), ("k", float("nan")), ("v", float("nan")), ("v", float("inf")), ("gk", float("nan")), ("h0", float("nan")),
                                         ("h0", -float("inf"))])
def test_a_value_that_is_none_stays_with_its_head(K, V, segments, where, value, monkeypatch):
    """In chunk 9 of one head, or its initial state: the other heads and sequences and the chunks before it keep their bits."""
    if segments == 1:
        monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    inp = make_inputs(850, 2, 330, 3, K, V, gk_div=8.0)
    t = [x.bfloat16().to(DEV) for x in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)] + [inp.h0.to(DEV)]
    run = lambda: chunk_hrdplr_delta_rule(*t[:6], 2, scale=0.9, initial_state=t[6], output_final_state=True)
    with torch.no_grad():
        o_0, ht_0 = run()
        if where == "h0":
            t[6][1, 2, 3, 5] = value
        else:
            t[{"q": 0, "k": 1, "v": 2, "gk": 5}[where]][1, 150, 2, 5] = value
        o, ht = run()
    bad = torch.zeros(2, 330, 3, dtype=torch.bool)
    bad[1, 0 if where == "h0" else 144:, 2] = True
    assert torch.equal(o[~bad], o_0[~bad]) and torch.equal(ht[0], ht_0[0]) and torch.equal(ht[1, :2], ht_0[1, :2])
    hit = o[1, 160:, 2] if where != "q" else o[1, 150, 2]
    assert not torch.isfinite(hit.float()).all()
    assert torch.isfinite(ht[1, 2]).all() == (where == "q")
