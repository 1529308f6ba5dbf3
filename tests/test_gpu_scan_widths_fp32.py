"""fp32, V = 128: the scans of many sequences have all column blocks of a head in a workgroup, those of few have half of them.  Column blocks do not meet in
a scan, so outputs and gradients have the bits of a call for each sequence by itself."""
import pytest
import torch

from hdla_hip import chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("B", [8, 9, 16, 20])              # of 16 heads: half, all, all, half (forward pass); half, half, all, half (backward pass)
def test_the_bits_of_each_sequence_by_itself(K, B, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", "1")
    inp = make_inputs(2300 + B, B, 37, 16, K, 128, gk_div=4.0)
    x = [t.to(DEV) for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk, inp.h0)]
    do, dht = inp.do.to(DEV), inp.dht.to(DEV)

    def run(x, do, dht):
        x = [t.clone().requires_grad_() for t in x]
        o, ht = chunk_hrdplr_delta_rule(*x[:6], 2, scale=0.9, initial_state=x[6], output_final_state=True)
        return [o.detach(), ht.detach()] + list(torch.autograd.grad([o, ht], x, [do, dht]))

    whole = run(x, do, dht)
    for n in (0, B // 2, B - 1):
        for i, (a, b) in enumerate(zip(whole, run([t[n:n + 1] for t in x], do[n:n + 1], dht[n:n + 1]))):
            assert torch.equal(a[n:n + 1], b), (n, i)
