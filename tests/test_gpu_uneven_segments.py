"""Packed sequences of unequal lengths on the fused route, whose time segments are equal in number: against the classic route, which cuts none of these, the passes among each other,
and the same sequence beside others."""
import ctypes

import pytest
import torch

from hdla_hip import _lib, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O
from test_gpu_fused import _dev, backward, forward
from test_gpu_graph import _capture

pytestmark = pytest.mark.gpu
DEV = "cuda"

# Equal and unequal lengths; sequences of one token, of none, at the front, the end and between; tokens of no sequence; one long sequence beside a short one;
# 64 sequences, most of them empty, and 65; lengths of whole chunks and of a token more or less.
CUTS = [
    (2, (0, 4100, 5600, 7600, 8192)), (3, (0, 300, 1000, 3500, 3700)), (4, (0, 0, 17, 1500, 1500, 1501, 2100, 2100)), (2, (5, 2300, 2310, 2900)), (1, (0, 10000, 10016)),
    (1, (0, 257, 514, 770)), (16, (0, 2000, 2047, 3000)), (12, (0, 1597, 3421)), (1, (0, 16, 33, 1040, 1600)), (1, tuple([0] * 40 + [9000, 9600] + [17000] * 23)), (1, tuple([0] * 41 + [9000, 9600] + [17000] * 23)),
]


@pytest.mark.parametrize("gk", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,cu", CUTS)
def test_against_classic_route(H, cu, gk):
    """The tolerances of the route's own segments against the classic one (test_gpu_fused.py): rounding to 2 bytes once more at each boundary."""
    T, N = cu[-1] + 3, len(cu) - 1
    x, cud = _dev(make_inputs(61, 1, T, H, 64, 64, gk_div=8.0, n_states=N), gk), torch.tensor(cu, device=DEV)
    dims = _lib.make_dims(1, T, H, 64, 64, 2, N, torch.bfloat16, gk, 0.7, cud, route=_lib.ROUTE_FUSED)
    slots = _lib.boundary(dims, DEV).numel() // (H * 64 * 64 * 4)
    assert slots > N or N > 64                                    # segments there are
    o_c, ht_c, _ = forward(x, _lib.ROUTE_CLASSIC, 0, cu=cud)
    o, ht, bnd = forward(x, _lib.ROUTE_FUSED, 0, cu=cud, boundary=True)
    assert O.rel_l2(o, o_c) <= 3e-3 and O.rel_l2(ht, ht_c) <= 3e-3
    for n in range(N):
        assert O.rel_l2(ht[n], ht_c[n]) <= 6e-3, n                # (no sequence has another's: a state that is not its own would be 1 off)
    g_c = backward(x, _lib.ROUTE_CLASSIC, 0, cu=cud)
    kept, own = backward(x, _lib.ROUTE_FUSED, 0, cu=cud, bnd=bnd), backward(x, _lib.ROUTE_FUSED, 0, cu=cud)
    errs = {n: max(O.rel_l2(g[n], g_c[n]) for g in (kept, own)) for n in g_c}
    assert all(e <= 6e-3 for e in errs.values()), errs
    if N <= 64:                                                   # the states entering the segments are where the host's count of them says
        counts = [slots // N] * N
        # a record is 16 x 16 tiles [value block][key block], lane 16 g + c's four elements of one: keys 4 g + i of value column c
        rec = bnd.view(torch.float32).view(slots * H, 4, 4, 4, 16, 4).permute(0, 2, 3, 5, 1, 4).reshape(slots * H, 64, 64)
        first = 0
        for n, count in enumerate(counts):
            chunks = -(-(cu[n + 1] - cu[n]) // 16)
            per = -(-chunks // count)
            for s in range(1, count):
                if s * per >= chunks:
                    continue
                begin, end = cu[n], cu[n] + s * per * 16
                y = {t: x[t][:, begin:end].contiguous() for t in ("q", "k", "v", "gk")} | {t: x[t][:, 2 * begin:2 * end].contiguous() for t in ("a", "b")}
                y["h0"] = x["h0"][n:n + 1].contiguous()
                state = forward(y, _lib.ROUTE_CLASSIC, 0)[1][0]
                mine = torch.stack([rec[first * H + h * count + s] for h in range(H)])
                assert O.rel_l2(mine, state) <= 6e-3, (n, s)
            first += count


def test_operator_records_and_inputs_only():
    """What a forward pass leaves for the backward one is that of its segments: training through the operator, with the record, without it (saved-tensor hooks) and replayed from a graph."""
    cu, H = (0, 40, 3000, 3700, 3700, 4600), 8
    inp = make_inputs(62, 1, cu[-1], H, 64, 64, gk_div=8.0, n_states=5)
    x = [getattr(inp, n).bfloat16().to(DEV).requires_grad_() for n in ("q", "k", "v", "a", "b", "gk")] + [inp.h0.to(DEV).requires_grad_()]
    do, dht, cud = inp.do.bfloat16().to(DEV), inp.dht.to(DEV), torch.tensor(cu, device=DEV)
    run = lambda: chunk_hrdplr_delta_rule(*x[:6], 2, scale=0.7, initial_state=x[6], output_final_state=True, cu_seqlens=cud)

    def train():
        o, ht = run()
        # detached: a graph kept from one stream keeps the leaves' accumulators, and with them that stream joins a capture on another
        return [o.detach(), ht.detach(), *torch.autograd.grad([o, ht], x, [do, dht])]

    eager = train()
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(run(), eager))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        hooked = train()
    assert all(O.rel_l2(a, b) <= 6e-3 for a, b in zip(hooked, eager))
    graph, out = _capture(train)
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, eager))
        train()
        torch.cuda.synchronize()


@pytest.mark.parametrize("H,lens,others", [(16, (700, 1150, 1150), (700, 2290, 10)), (16, (1150, 700, 1150), (10, 1840, 1150)), (16, (40, 1960), (1960, 40)), (2, (700, 33, 767, 500), (500, 700, 40, 760))])
def test_a_sequence_beside_others(H, lens, others):
    """What a sequence gives and gets is its own: the same bits whatever the lengths of those packed with it, as many and as long in all."""
    inp = make_inputs(63, 1, sum(lens), H, 64, 64, gk_div=4.0, n_states=len(lens))

    def run(order, at):                                           # the first sequence of `lens` at place `at`, others of the same numbers
        cu = [sum(order[:i]) for i in range(len(order) + 1)]
        def place(t, r=1):
            t = t.clone()
            mine, T = t[:, :r * lens[0]].clone(), t.shape[1]
            return torch.cat([t[:, T - r * cu[at]:], mine, t[:, r * lens[0]:T - r * cu[at]]], 1)
        x = [place(getattr(inp, n), 2 if n in "ab" else 1).bfloat16().to(DEV).requires_grad_() for n in ("q", "k", "v", "a", "b", "gk")]
        h0, dht = (torch.cat([t[len(lens) - at:], t[:1], t[1:len(lens) - at]]).to(DEV) for t in (inp.h0, inp.dht))
        h0.requires_grad_()
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("HDLA_HIP_ROUTE", "fused")
            o, ht = chunk_hrdplr_delta_rule(*x, 2, scale=0.7, initial_state=h0, output_final_state=True, cu_seqlens=torch.tensor(cu, device=DEV))
            g = torch.autograd.grad([o, ht], x + [h0], [place(inp.do).bfloat16().to(DEV), dht])
        tok = lambda t, r=1: t[0, r * cu[at]:r * cu[at + 1]]
        return [tok(o), ht[at], *[tok(t, 2 if i in (3, 4) else 1) for i, t in enumerate(g[:6])], g[6][at]]

    for a, b in zip(run(lens, 0), run(others, others.index(lens[0]))):
        assert torch.equal(a, b)
