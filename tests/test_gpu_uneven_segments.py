"""Packed sequences on the fused route in time segments by their lengths (share_segments, prep.hip), as many in all as in equal numbers: against the classic route, which cuts
none of these, and the passes among each other."""
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

# Equal and unequal lengths; sequences of one token, of none, at the front, the end and between; tokens of no sequence; more segments than the long one may have (64, eight chunks each);
# 64 sequences, most of them empty, and 65, which are cut in equal numbers; lengths of whole chunks and of a token more or less.
CUTS = [
    (2, (0, 4100, 5600, 7600, 8192)), (3, (0, 300, 1000, 3500, 3700)), (4, (0, 0, 17, 1500, 1500, 1501, 2100, 2100)), (2, (5, 2300, 2310, 2900)), (1, (0, 10000, 10016)),
    (1, (0, 257, 514, 770)), (16, (0, 2000, 2047, 3000)), (12, (0, 1597, 3421)), (1, (0, 16, 33, 1040, 1600)), (1, tuple([0] * 40 + [9000, 9600] + [17000] * 23)), (1, tuple([0] * 41 + [9000, 9600] + [17000] * 23)),
]


def _chunk_segments(cu, slots):
    """share_segments on the host: segments of each sequence"""
    chunks = [-(-(e - b) // 16) for b, e in zip(cu, cu[1:])]
    of = lambda length: [max(1, min(64, c // 8, -(-c // length))) for c in chunks]
    length = max(8, -(-sum(chunks) // slots))
    while sum(of(length)) > slots:
        length += 1
    even = slots // len(chunks)
    return of(length) if max(chunks) > length * even else [even] * len(chunks)


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
        counts = _chunk_segments(cu, slots)
        assert sum(counts) <= slots
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
