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
