"""The fused route's record (what the forward pass leaves for the backward pass): a backward pass that reads it gives the
gradients of one that forms it itself first, and both those of the classic route."""
import ctypes

import pytest
import torch

from hdla_hip import _lib
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _call(x, cu, segments, route, with_record, beta):
    lib, P = _lib.load(), _lib.ptr
    B, T, H, K = x["q"].shape
    V, N = x["v"].shape[-1], x["h0"].shape[0]
    dims = _lib.make_dims(B, T, H, K, V, 2, N, torch.bfloat16, x["gk"].dtype, 0.7, cu, route=route, segments=segments)
    s = _lib.current_stream(torch.device(DEV))
    rec = _lib.record(dims, DEV) if with_record else None
    assert not with_record or rec is not None
    nrec = 0 if rec is None else rec.numel()
    a, b, bt = (None, None, x["beta"]) if beta else (x["a"], x["b"], None)
    o, ht = torch.zeros_like(x["v"]), torch.empty_like(x["h0"])
    ws = _lib.workspace(dims, 0, DEV)
    _lib.check(lib.hdla_chunk_fwd_b(ctypes.byref(dims), P(x["q"]), P(x["k"]), P(x["v"]), P(a), P(b), P(bt), P(x["gk"]), P(x["h0"]), P(o),
                                    P(ht), P(rec), nrec, P(ws), ws.numel(), s), "fwd")
    g = {n: torch.zeros_like(x[n]) for n in (("q", "k", "v", "beta", "gk") if beta else ("q", "k", "v", "a", "b", "gk"))}
    g["h0"] = torch.empty_like(x["h0"])
    ws = _lib.workspace(dims, 1, DEV)
    _lib.check(lib.hdla_chunk_bwd_b(ctypes.byref(dims), P(x["q"]), P(x["k"]), P(x["v"]), P(a), P(b), P(bt), P(x["gk"]), P(x["h0"]),
                                    P(x["do"]), P(x["dht"]), P(g["q"]), P(g["k"]), P(g["v"]), P(g.get("a")), P(g.get("b")),
                                    P(g.get("beta")), P(g["gk"]), P(g["h0"]), P(rec), nrec, P(ws), ws.numel(), s), "bwd")
    torch.cuda.synchronize()
    return {"o": o, "ht": ht, **g}


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("gk_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,H,cu,segments,gk_div", [
    (1, 5, 2, None, 1, 2.0), (2, 16, 1, None, 1, 2.0), (1, 129, 3, None, 1, 2.0), (2, 203, 2, None, 2, 8.0), (1, 1000, 2, None, 8, 8.0),
    (1, 300, 2, (0, 37, 37, 200, 300), 3, 8.0), (1, 150, 2, None, 2, 0.05)])
def test_backward_pass_from_the_record(B, T, H, cu, segments, gk_div, gk_dtype, beta):
    n_states = B if cu is None else len(cu) - 1
    inp = make_inputs(31, B, T, H, 64, 64, gk_div=gk_div, n_states=n_states)
    x = {n: getattr(inp, n).to(DEV).to(torch.bfloat16 if n not in ("h0", "dht", "gk") else gk_dtype if n == "gk" else torch.float32)
         for n in ("q", "k", "v", "a", "b", "gk", "h0", "do", "dht")}
    if beta:
        x["k"] = torch.nn.functional.normalize(x["k"].float(), dim=-1).bfloat16()
        x["beta"] = torch.rand(B, T, H, generator=torch.Generator().manual_seed(3)).bfloat16().to(DEV)
    cud = None if cu is None else torch.tensor(cu, dtype=torch.int64, device=DEV)
    kept = _call(x, cud, segments, _lib.ROUTE_FUSED, True, beta)
    formed = _call(x, cud, segments, _lib.ROUTE_FUSED, False, beta)
    classic = _call(x, cud, 0, _lib.ROUTE_CLASSIC, False, beta)
    for n in kept:
        print(n, f"{O.rel_l2(kept[n], formed[n]):.1e} {O.rel_l2(kept[n], classic[n]):.1e}", flush=True)
        assert torch.isfinite(kept[n].float()).all(), n
        assert O.rel_l2(kept[n], formed[n]) <= 1e-3, n
        assert O.rel_l2(kept[n], classic[n]) <= (6e-3 if segments > 1 else 2e-3), n


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("form", ["ab", "beta", "layer"])
def test_the_environment_may_change_between_the_passes(form, native, monkeypatch):
    """The record is laid out by the forward pass's route and segments: the backward pass runs with these, not with what the
    environment asks for by then."""
    from hdla_hip import chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
    from hdla_hip.layer import HDLA_Custom
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    x = make_inputs(46, 1, 600, 2, 64, 64)
    t = [y.bfloat16().to(DEV).requires_grad_() for y in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    do = x.do.bfloat16().to(DEV)
    if form == "layer":
        torch.manual_seed(1)
        m = HDLA_Custom(128, 2, token_mixer_init_type=2, rescale_type=0).to(DEV).bfloat16().train()
        leaves = [torch.randn(1, 600, 128, device=DEV).bfloat16().requires_grad_(), *m.parameters()]
        do, run = torch.randn(1, 600, 128, device=DEV).bfloat16(), lambda: m(leaves[0])[0]
    elif form == "ab":
        leaves, run = t, lambda: chunk_hrdplr_delta_rule(*t, 2, scale=0.7)[0]
    else:
        leaves = [*t[:3], torch.rand(1, 600, 2, 1, device=DEV).bfloat16().requires_grad_(), t[5]]
        run = lambda: chunk_hdla_delta_rule(*leaves, scale=0.7)[0]
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", "4")
    ref = torch.autograd.grad(run(), leaves, do)
    for env in ({"HDLA_HIP_SEGMENTS": "2"}, {"HDLA_HIP_SEGMENTS": "8"}, {"HDLA_HIP_ROUTE": "classic"}):
        with monkeypatch.context() as c:
            y = run()
            for name, value in env.items():
                c.setenv(name, value)
            assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, leaves, do), ref)), env


@pytest.mark.parametrize("T,segments,cu", [(5, 1, None), (600, 4, None), (500, 3, [0, 100, 100, 411, 500])])
def test_the_scratch_beside_a_record_is_enough(T, segments, cu):
    """hdla_record_workspace_bytes bytes and not one more are touched, and the gradients are those on a whole workspace."""
    x = make_inputs(47, 1, T, 2, 64, 64, n_states=None if cu is None else len(cu) - 1)
    t = [y.bfloat16().to(DEV) for y in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    do, h0, dht = x.do.bfloat16().to(DEV), x.h0.to(DEV), x.dht.to(DEV)
    table = None if cu is None else torch.tensor(cu, device=DEV)
    lib, P, plan = _lib.load(), _lib.ptr, (_lib.ROUTE_FUSED, segments)
    dims = _lib.make_dims(1, T, 2, 64, 64, 2, h0.shape[0], torch.bfloat16, torch.bfloat16, 0.7, table, *plan)
    rec = _lib.record(dims, DEV)
    s, o, ws = _lib.current_stream(torch.device(DEV)), torch.empty_like(t[2]), _lib.workspace(dims, 0, DEV)
    _lib.check(lib.hdla_chunk_fwd_b(ctypes.byref(dims), *[P(y) for y in t[:5]], None, P(t[5]), P(h0), P(o), None, P(rec), rec.numel(), P(ws),
                                    ws.numel(), s), "fwd")
    res = []
    small = lib.hdla_record_workspace_bytes(ctypes.byref(dims))
    for n in (lib.hdla_workspace_bytes(ctypes.byref(dims), 1), small):
        ws = torch.full((n + 4096,), 0xa5, dtype=torch.uint8, device=DEV)
        g = [torch.empty_like(y) for y in t] + [torch.empty_like(h0)]
        run = lambda have: lib.hdla_chunk_bwd_b(ctypes.byref(dims), *[P(y) for y in t[:5]], None, P(t[5]), P(h0), P(do), P(dht),
                                                *[P(y) for y in g[:5]], None, P(g[5]), P(g[6]), P(rec), rec.numel(), P(ws), have, s)
        _lib.check(run(n), "bwd")
        assert bool((ws[n:] == 0xa5).all())
        res.append(g)
    assert run(small - 256) == -5
    assert all(torch.equal(a, b) for a, b in zip(*res))
