"""Buffers that are there to be looked at belong to callers who name the classic route: the plans that the library makes for itself, and the plain
route, have the classic one's kernels and bits without them."""
import ctypes

import pytest
import torch

import hdla_hip.chunk as CK
from hdla_hip import _lib, chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

DEV = "cuda"
SHAPES = [(64, 64), (128, 128), (64, 128), (128, 64)]


def _dims(T, H, K, V, route, segments=0, gk=torch.bfloat16):
    return _lib.make_dims(1, T, H, K, V, 2, 1, torch.bfloat16, gk, 1.0, None, route=route, segments=segments)


def _size(d):
    return _lib.load().hdla_workspace_bytes(ctypes.byref(d), _lib.PASS_BWD)


@pytest.mark.parametrize("K,V", SHAPES)
def test_workspaces(K, V):
    up = lambda n: -(-n // 256) * 256
    for T, H in ((16, 1), (256, 2), (1537, 16)):
        slots = H * -(-T // 16)
        for gk, shown in ((torch.bfloat16, up(slots * 32 * V * 2) + up(slots * 16 * V * 2)), (torch.float32, up(slots * 16 * V * 2))):
            classic, plain = _dims(T, H, K, V, _lib.ROUTE_CLASSIC, gk=gk), _dims(T, H, K, V, _lib.ROUTE_PLAIN, gk=gk)
            assert _size(classic) - _size(plain) == shown
            assert _lib.workspace_layout(plain, 1)["VTT"] == 0 < _lib.workspace_layout(classic, 1)["VTT"]
        plain = _dims(T, H, K, V, _lib.ROUTE_PLAIN)
        assert _lib.load().hdla_record_bytes(ctypes.byref(plain)) == 0 and _lib.keep_plan(plain)[1:] == (1, 1)


@pytest.mark.parametrize("T,H,K,V", [(256, 2, 64, 64), (1537, 16, 128, 128), (640, 16, 64, 128)])
def test_the_plan_of_a_backward_pass_without_a_kept_workspace(T, H, K, V, monkeypatch):
    monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    monkeypatch.setattr(_lib._native, "kept_room", lambda like, n: None, raising=False)
    x = [torch.empty(1, T, H, d, dtype=torch.bfloat16, device="meta") for d in (K, V, K)]
    _, plan, room = CK.keep_plan(*x, 1.0, None)
    assert room is False and plan[1] == 1
    assert _size(_dims(T, H, K, V, *plan)) == _size(_dims(T, H, K, V, _lib.ROUTE_PLAIN)) < _size(_dims(T, H, K, V, _lib.ROUTE_CLASSIC))


def _step(x, do, dht, form):
    leaves = [t.detach().requires_grad_() for t in x]
    op = (lambda *a, **kw: chunk_hrdplr_delta_rule(*a, 2, **kw)) if form == "ab" else chunk_hdla_delta_rule
    o, ht = op(*leaves[:-1], scale=0.7, initial_state=leaves[-1], output_final_state=True)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_stats()["requested_bytes.all.current"]
    g = torch.autograd.grad([o, ht], leaves, [do, dht])
    return [o.detach(), ht.detach(), *g], torch.cuda.memory_stats()["requested_bytes.all.peak"] - held


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("T,H,K,V", [(256, 2, 64, 64), (300, 12, 128, 128), (200, 16, 64, 128), (170, 9, 128, 64)])
def test_bits_and_memory(T, H, K, V, form, native, monkeypatch):
    """A call that finds no room to keep its forward pass (here: under saved-tensor hooks) takes for its backward pass what the plain route takes."""
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    inp = make_inputs(31, 1, T, H, K, V, gk_div=4.0)
    beta = 2.0 * torch.rand(1, T, H, 1, generator=torch.Generator().manual_seed(5))
    k = torch.nn.functional.normalize(inp.k, dim=-1)
    x = [inp.q, k, inp.v] + ([inp.a, inp.b] if form == "ab" else [beta]) + [inp.gk]
    x = [t.bfloat16().to(DEV) for t in x] + [inp.h0.to(DEV)]
    do, dht = inp.do.bfloat16().to(DEV), inp.dht.to(DEV)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        hooked, peak = _step(x, do, dht, form)
    results = {}
    for route in ("plain", "classic"):
        monkeypatch.setenv("HDLA_HIP_ROUTE", route)
        monkeypatch.setenv("HDLA_HIP_KEEP_FORWARD", "0")
        results[route] = _step(x, do, dht, form)
    assert peak == results["plain"][1] < results["classic"][1]
    for got, _ in results.values():
        assert all(torch.equal(a, b) for a, b in zip(got, hooked))
