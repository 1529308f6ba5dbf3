"""Training calls whose forward pass leaves the states that enter the chunks (hdla_states_plan): where that is chosen (on the CPU), and that the backward
pass on them, with one scan, is the one that recomputes them with two, bit for bit."""
import ctypes

import pytest
import torch

from hdla_hip import _lib, chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs

DEV = "cuda"


def _plan(B, T, H, K, V, N=None, dtype=torch.bfloat16, gk=torch.bfloat16, **kw):
    d = _lib.make_dims(B, T, H, K, V, 2, N or B, dtype, gk if dtype == torch.bfloat16 else dtype, 1.0, None, **kw)
    if N:
        d.cu_seqlens = 256                                      # never read on the host
    fwd, bwd = ctypes.c_size_t(0), ctypes.c_size_t(0)
    f = _lib.load().hdla_states_plan
    f.restype = ctypes.c_size_t
    return f(ctypes.byref(d), ctypes.byref(fwd), ctypes.byref(bwd)), fwd.value, bwd.value


def test_where_it_is_chosen():
    up = lambda n: -(-n // 256) * 256
    # the scan block without q's part, the reverse scan's, (I - A_ab)^-1, A_ak, the sums, the flags and the states; q's part; what the reverse scan leaves
    n, fwd, bwd = _plan(4, 1000, 16, 128, 128)
    slots = 4 * 16 * 63
    assert n == sum(up(slots * b) for b in (21504, 5120, 2048, 1024, 64, 4, 32768))
    assert fwd == up(slots * 5120) and bwd == up(slots * 32768) + up(slots * 8192)
    assert 0 < _plan(1, 16384, 16, 128, 128, N=4)[0] <= 1 << 30
    # where both scans in workgroups of one column block are more workgroups than the device has compute units
    for K, V, lanes in ((128, 128, 16), (64, 128, 16), (128, 64, 32), (64, 64, 32)):
        assert _plan(1, 300, lanes, K, V)[0] == 0 < _plan(1, 300, lanes + 1, K, V)[0]
    assert _plan(1, 32768, 16, 128, 128, N=4)[0] == 0            # more than a gibibyte
    assert _plan(4, 1000, 16, 64, 64)[0] == 0                    # the fused route
    assert _plan(4, 1000, 16, 128, 128, dtype=torch.float32)[0] == 0
    assert _plan(4, 1000, 16, 128, 128, segments=2)[0] == 0 and _plan(4, 0, 16, 128, 128)[0] == 0 and _plan(4, 1000, 16, 96, 128)[0] == 0
    for route in (_lib.ROUTE_CLASSIC, _lib.ROUTE_PLAIN):
        assert _plan(4, 1000, 16, 128, 128, route=route)[0] == 0


def _leaves(form, B, T, H, K, V, N, gk, gk_div):
    inp = make_inputs(7, B, T, H, K, V, gk_div=gk_div)
    k = torch.nn.functional.normalize(inp.k, dim=-1)
    beta = 2.0 * torch.rand(B, T, H, 1, generator=torch.Generator().manual_seed(5))
    x = [inp.q, k, inp.v] + ([inp.a, inp.b] if form == "ab" else [beta])
    h0 = torch.randn(N, H, K, V, generator=torch.Generator().manual_seed(6)) * 0.1
    x = [t.bfloat16() for t in x] + [inp.gk.to(gk), h0]
    dht = torch.randn(N, H, K, V, generator=torch.Generator().manual_seed(8))
    return [t.to(DEV).requires_grad_() for t in x], inp.do.bfloat16().to(DEV), dht.to(DEV)


# lengths of whole chunks and of a token more or less; several widths of the scans' workgroups; packed: sequences without a chunk, rows of no sequence
@pytest.mark.gpu
@pytest.mark.parametrize("form,gk_div", [("ab", 64.0), ("beta", 1.0)])
@pytest.mark.parametrize("B,T,H,K,V,cu,gk", [
    (3, 47, 16, 128, 128, None, torch.bfloat16), (4, 16, 16, 128, 128, None, torch.bfloat16), (5, 1, 9, 128, 128, None, torch.bfloat16), (1, 33, 17, 128, 128, None, torch.bfloat16), (3, 250, 16, 64, 64, None, torch.bfloat16),
    (4, 129, 32, 128, 128, None, torch.float32), (8, 100, 12, 64, 128, None, torch.bfloat16), (4, 65, 24, 128, 64, None, torch.bfloat16),
    (1, 700, 16, 128, 128, (0, 300, 337, 337, 640, 700), torch.bfloat16), (1, 500, 32, 128, 64, (3, 200, 201, 330, 490), torch.bfloat16),
    (1, 1400, 3, 128, 128, tuple(range(0, 1401, 35)), torch.bfloat16), (1, 900, 24, 64, 128, (0, 16, 500, 620, 700, 900), torch.float32)])
def test_one_scan_and_two(B, T, H, K, V, cu, gk, form, gk_div):
    """Nothing is left under saved-tensor hooks."""
    N = B if cu is None else len(cu) - 1
    all_, fwd, _ = _plan(B, T, H, K, V, N=None if cu is None else N, gk=gk)
    assert all_ > 0
    x, do, dht = _leaves(form, B, T, H, K, V, N, gk, gk_div)
    table = None if cu is None else torch.tensor(cu, device=DEV)
    op = (lambda *a, **kw: chunk_hrdplr_delta_rule(*a, 2, **kw)) if form == "ab" else chunk_hdla_delta_rule
    run = lambda: op(*x[:-1], scale=0.7, initial_state=x[-1], output_final_state=True, cu_seqlens=table)
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()["requested_bytes.all.current"]
    o, ht = run()
    held = torch.cuda.memory_stats()["requested_bytes.all.current"] - before
    assert all_ <= held < all_ + fwd + o.numel() * 2 + ht.numel() * 4
    got = [o, ht, *torch.autograd.grad([o, ht], x, [do, dht], retain_graph=True)]
    twice = torch.autograd.grad([o, ht], x, [do, dht])           # on the same buffer
    with torch.no_grad():
        plain = run()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        o2, ht2 = run()
        want = [o2, ht2, *torch.autograd.grad([o2, ht2], x, [do, dht])]
    names = ["o", "ht", "dq", "dk", "dv", "da", "db", "dgk", "dh0"] if form == "ab" else ["o", "ht", "dq", "dk", "dv", "dbeta", "dgk", "dh0"]
    for name, a, b in zip(names, got, want):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b), name
    assert all(torch.equal(a, b) for a, b in zip(got[2:], twice)) and all(torch.equal(a, b) for a, b in zip(got, plain))
