"""What the kernels of 2-byte elements hand each other in the place of u and v^T: the two ranks of A_ak, from which the scans (and, with the HDLA
parameterisation, chunk_grad) form u, and that parameterisation's sums over the channels.  Read from the workspace at hdla_ws_layout's offsets, against the
stage-by-stage restatement."""
import ctypes

import pytest
import torch

import gpu_util as G
from hdla_hip import _lib
from hdla_hip.synthetic import make_inputs
from oracle import chunk_stages as CS
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def _buffers(form, B, T, H, K, V, route, segments, kept):
    """The workspace of a backward pass (or of a forward pass that keeps it) and its layout, and the operands."""
    inp = make_inputs(61, B, T, H, K, V, gk_div=1.0)
    k, beta = torch.nn.functional.normalize(inp.k, dim=-1), 2.0 * torch.rand(B, T, H, generator=torch.Generator().manual_seed(8))
    x = {n: t.to(BF) for n, t in (("q", inp.q), ("k", k), ("v", inp.v), ("a", inp.a), ("b", inp.b), ("gk", inp.gk), ("beta", beta), ("do", inp.do))}
    d, P, lib = {n: t.to(DEV) for n, t in x.items()}, _lib.ptr, _lib.load()
    a, b, bt = (d["a"], d["b"], None) if form == "ab" else (None, None, d["beta"])
    h0 = inp.h0.to(DEV)
    dims = _lib.make_dims(B, T, H, K, V, 2, B, BF, BF, 0.7, None, route=route, segments=segments)
    pass_ = _lib.PASS_FWD_KEEP if kept else _lib.PASS_BWD
    ws = torch.full((lib.hdla_workspace_bytes(ctypes.byref(dims), pass_),), 255, dtype=torch.uint8, device=DEV)
    head = [P(t) for t in (d["q"], d["k"], d["v"], a, b, bt, d["gk"], h0)]
    stream = _lib.current_stream(DEV)
    if kept:
        o, ht = torch.empty_like(d["v"]), torch.empty_like(h0)
        assert lib.hdla_chunk_fwd_keep(ctypes.byref(dims), *head, P(o), P(ht), P(ws), ws.numel(), stream) == 0
    else:
        g = [torch.empty_like(d[n]) for n in ("q", "k", "v")] + ([torch.empty_like(a), torch.empty_like(b), None] if form == "ab" else
                                                                  [None, None, torch.empty_like(bt)]) + [torch.empty_like(d["gk"]), torch.empty_like(h0)]
        assert lib.hdla_chunk_bwd_b(ctypes.byref(dims), *head, P(d["do"]), None, *[P(t) for t in g], None, 0, P(ws), ws.numel(), stream) == 0
    torch.cuda.synchronize()
    return ws, _lib.workspace_layout(dims, pass_), {n: t.double() for n, t in x.items()}


@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("B,T,H,K,V,route,segments,kept", [
    (2, 40, 2, 64, 64, _lib.ROUTE_PLAIN, 0, False), (1, 35, 2, 128, 128, _lib.ROUTE_CLASSIC, 0, False), (1, 16, 3, 64, 128, _lib.ROUTE_AUTO, 0, False),
    (1, 65, 2, 128, 64, _lib.ROUTE_AUTO, 2, False), (2, 40, 2, 64, 64, _lib.ROUTE_PLAIN, 0, True), (1, 90, 2, 128, 128, _lib.ROUTE_AUTO, 3, True),
    (2, 40, 2, 64, 64, _lib.ROUTE_FUSED, 1, False), (1, 150, 3, 64, 64, _lib.ROUTE_FUSED, 2, False)])
def test_a_ak_and_the_sums(B, T, H, K, V, route, segments, kept, form):
    ws, L, x = _buffers(form, B, T, H, K, V, route, segments, kept)
    a, b = (x["a"], x["b"]) if form == "ab" else (t.to(BF).double() for t in O.parameterize_a_b(x["beta"], x["k"], x["gk"]))
    p = CS.prep(x["q"], x["k"], x["v"], a, b, x["gk"], 0.7)
    nch = L["nch"]
    slots = lambda t: t.permute(1, 0, 2, *range(3, t.dim())).reshape(H, nch, *t.shape[3:])
    assert L["AAK"] > 0 and L["AAK_STRIDE"] in (1024, 2048)
    assert O.rel_l2(G.pair_tiles(ws, L["AAK"], BF, H, nch, 2, stride=L["AAK_STRIDE"]), slots(p["Aak"])) <= 1e-2
    if form == "beta":
        f = x["k"] ** 2 * torch.exp(x["gk"])
        s = CS._chunks(CS._pad_T(f, -(-T // 16) * 16), 16).sum(-1)
        got, want = G.rows(ws, L["SUM"], torch.float32, H, nch, 16), slots(s)
        real = want > 0                                       # (rows past the end: never used)
        assert bool(real.any()) and O.rel_l2(got[real], want[real]) <= 1e-5       # 64 or 128 positive terms in 32 bits


@pytest.mark.parametrize("pass_", [_lib.PASS_FWD, _lib.PASS_BWD, _lib.PASS_FWD_KEEP])
@pytest.mark.parametrize("K,V,gk", [(64, 64, BF), (128, 128, BF), (64, 128, torch.float32), (128, 64, BF)])
def test_ks_gated_copy_under_the_classic_route(K, V, gk, pass_):
    """With the HDLA parameterisation no kernel reads it: for those who look, it is what the same k has beside plain a, b."""
    B, T, H, P, lib = 2, 40, 3, _lib.ptr, _lib.load()
    inp = make_inputs(62, B, T, H, K, V, gk_div=1.0)
    k, beta = torch.nn.functional.normalize(inp.k, dim=-1), 2.0 * torch.rand(B, T, H, generator=torch.Generator().manual_seed(8))
    d = {n: t.to(BF).to(DEV) for n, t in (("q", inp.q), ("k", k), ("v", inp.v), ("a", inp.a), ("b", inp.b), ("beta", beta), ("do", inp.do))}
    d["gk"], h0 = inp.gk.to(gk).to(DEV), inp.h0.to(DEV)
    dims = _lib.make_dims(B, T, H, K, V, 2, B, BF, gk, 0.7, None, route=_lib.ROUTE_CLASSIC, segments=0)
    L, got = _lib.workspace_layout(dims, pass_), []
    for form in ("ab", "beta"):
        ws = torch.full((lib.hdla_workspace_bytes(ctypes.byref(dims), pass_),), 255, dtype=torch.uint8, device=DEV)
        head = [P(d["q"]), P(d["k"]), P(d["v"])] + ([P(d["a"]), P(d["b"]), None] if form == "ab" else [None, None, P(d["beta"])]) + [P(d["gk"]), P(h0)]
        o, ht, stream = torch.empty_like(d["v"]), torch.empty_like(h0), _lib.current_stream(DEV)
        if pass_ == _lib.PASS_FWD:
            rc = lib.hdla_chunk_fwd_b(ctypes.byref(dims), *head, P(o), P(ht), None, 0, P(ws), ws.numel(), stream)
        elif pass_ == _lib.PASS_FWD_KEEP:
            rc = lib.hdla_chunk_fwd_keep(ctypes.byref(dims), *head, P(o), P(ht), P(ws), ws.numel(), stream)
        else:
            g = [torch.empty_like(d[n]) for n in ("q", "k", "v", "a", "b", "beta", "gk")] + [torch.empty_like(h0)]
            out = [P(t) for t in g]
            rc = lib.hdla_chunk_bwd_b(ctypes.byref(dims), *head, P(d["do"]), None, *out, None, 0, P(ws), ws.numel(), stream)
        assert rc == 0
        torch.cuda.synchronize()
        got.append(G.pair_tiles(ws, L["KGT"], BF, H, L["nch"], K // 16, stride=L["SA_STRIDE"]))
    assert torch.isfinite(got[0]).all() and torch.equal(got[0], got[1])


def test_passes_that_have_none():
    for dtype, pass_ in ((BF, _lib.PASS_FWD), (BF, _lib.PASS_BWD_KEPT), (torch.float32, _lib.PASS_BWD), (torch.float32, _lib.PASS_FWD_KEEP)):
        L = _lib.workspace_layout(_lib.make_dims(1, 64, 2, 128, 128, 2, 1, dtype, dtype, 1.0, None), pass_)
        assert L["AAK"] == L["AAK_STRIDE"] == L["SUM"] == 0
