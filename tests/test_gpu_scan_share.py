"""Few packed sequences whose workgroups in the scans are as wide as their lengths make them (scan_out_share_kernel, scan_grad_share_kernel): every
width in one launch, empty sequences, more workgroups than the device holds, the first count of sequences that is too many.  Column
blocks do not meet in a scan, so outputs and gradients have the bits of a call for each sequence by itself."""
import ctypes

import pytest
import torch

import hdla_hip.chunk as CK
from hdla_hip import _lib, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"

LENS = {
    "one long": [37, 700, 21, 16, 0, 65],
    "falling": [16 * n for n in (40, 30, 20, 12, 6, 3, 1)],
    "two": [333, 64],
    "equal": [50] * 9,
    "32": [400] + [17] * 30 + [0],
    "33": [400] + [17] * 31 + [0],
    "all empty but one": [0, 0, 90, 0],
}


@pytest.mark.parametrize("K,V,H", [(64, 64, 40), (64, 128, 20), (128, 64, 24), (128, 128, 17), (128, 128, 129)])
@pytest.mark.parametrize("lens", sorted(LENS))
@pytest.mark.parametrize("keep", [False, True])
def test_the_bits_of_each_sequence_by_itself(K, V, H, lens, keep, monkeypatch):
    monkeypatch.setenv("HDLA_HIP_ROUTE", "classic")
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", "1")
    lens = LENS[lens]
    if H > 100 and len(lens) > 10:
        pytest.skip("as many workgroups with fewer sequences")
    N, T = len(lens), sum(lens)
    cu = torch.tensor([0] + lens).cumsum(0)
    inp = make_inputs(2100 + T, 1, T, H, K, V, gk_div=4.0, n_states=N)
    x = [t.bfloat16().to(DEV) for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)] + [inp.h0.to(DEV)]
    do, dht = inp.do.bfloat16().to(DEV), inp.dht.to(DEV)

    def run(x, do, dht, cu=None):
        x = [t.clone().requires_grad_() for t in x]
        o, ht = chunk_hrdplr_delta_rule(*x[:6], 2, scale=0.9, initial_state=x[6], output_final_state=True, cu_seqlens=cu, keep_forward=keep)
        return [o.detach(), ht.detach()] + list(torch.autograd.grad([o, ht], x, [do, dht]))

    whole = run(x, do, dht, cu.to(DEV))
    for n in sorted(range(N), key=lambda n: -lens[n])[:4] + [N - 1]:
        s, e = int(cu[n]), int(cu[n + 1])
        if s == e:
            assert torch.equal(whole[1][n], x[6][n]) and torch.equal(whole[8][n], dht[n])
            continue
        cut = lambda t, r: t[:, s * r:e * r]
        r = [1, 1, 1, 2, 2, 1]
        alone = run([cut(t, k) for t, k in zip(x, r)] + [x[6][n:n + 1]], cut(do, 1), dht[n:n + 1])
        parts = [cut(whole[0], 1), whole[1][n:n + 1]] + [cut(t, k) for t, k in zip(whole[2:8], r)] + [whole[8][n:n + 1]]
        for i, (a, b) in enumerate(zip(parts, alone)):
            assert torch.equal(a, b), (n, i)


# (H, segments) of three sequences at V = 128: the scan of the forward pass in workgroups of one column block fits the device up to 10 heads, the two
# of the backward pass up to 5
@pytest.mark.parametrize("H,segments,widths", [(5, 1, {"fwd": False, "bwd": False, "keep": False}), (6, 1, {"fwd": False, "bwd": True, "keep": True}),
                                               (11, 1, {"fwd": True, "bwd": True, "keep": True}), (11, 4, {"fwd": False, "bwd": False, "keep": True})])
def test_widths_are_chosen_where_a_scan_asks_for_them(H, segments, widths):
    lens, K, V = [400, 130, 60], 64, 128
    T, N, plan = sum(lens), len(lens), (_lib.ROUTE_AUTO, segments)
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0)
    inp = make_inputs(2101, 1, T, H, K, V, gk_div=4.0, n_states=N)
    x = [t.bfloat16().to(DEV) for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)] + [0.9, inp.h0.to(DEV)]
    dims = CK._dims(x[0], x[2], x[5], 0.9, cu, N, plan)
    ws = {"keep": CK.chunk_hrdplr_fwd(*x, True, cu, keep=True, plan=plan)[2],
          "bwd": CK.chunk_hrdplr_bwd(*x, inp.do.bfloat16().to(DEV), inp.dht.to(DEV), cu, keep_workspace=True, plan=plan)[7],
          "fwd": _lib.workspace(dims, _lib.PASS_FWD, x[0].device)}
    P, o = _lib.ptr, torch.empty_like(x[2])
    assert _lib.load().hdla_chunk_fwd_b(ctypes.byref(dims), *[P(t) for t in x[:5]], None, P(x[5]), P(x[7]), P(o), None, None, 0, P(ws["fwd"]),
                                        ws["fwd"].numel(), _lib.current_stream(x[0].device)) == 0
    for name, p in (("fwd", _lib.PASS_FWD), ("bwd", _lib.PASS_BWD), ("keep", _lib.PASS_FWD_KEEP)):
        at = _lib.workspace_layout(dims, p)["CHUNK_OFF"] + 4 * (N + 1)
        order = ws[name][at:at + 4 * N].view(torch.int32).tolist()
        assert [e & 0x0fffffff for e in order] == [0, 1, 2] and any(e >> 28 for e in order) == widths[name], (name, order)
