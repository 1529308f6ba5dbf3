"""fp32: the scans of many sequences have all column blocks of a head in a workgroup, those of few have half of them, or two of them with two waves each that
share the channels.  Column blocks do not meet in a scan, and the sums over channels are those of two halves whoever forms them, so outputs and gradients have
the bits of a call for each sequence by itself."""
import pytest
import torch

from hdla_hip import chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


# of 16 heads: at K = V = 64 the first three are two waves' a block in the forward pass, the first two in the backward pass; at K = V = 128 all column blocks are
# a workgroup's at 9 and 16 in the forward pass, at 16 in the backward pass
@pytest.mark.parametrize("K,V", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("B", [2, 4, 8, 9, 16, 20])
def test_the_bits_of_each_sequence_by_itself(K, V, B, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", "1")
    inp = make_inputs(2300 + B, B, 61, 16, K, V, gk_div=4.0)
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
