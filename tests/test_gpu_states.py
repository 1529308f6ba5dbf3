"""Training calls whose forward pass leaves the states that enter the chunks (hdla_states_plan): where there is such a plan (on the CPU), that the backward pass on them, with one scan, is
the one that recomputes them with two, bit for bit, and which calls of a device have which buffer."""
import ctypes
import gc

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


def test_where_there_is_a_plan():
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


# lengths of whole chunks and of a token more or less; several widths of the scans' workgroups; packed: sequences without a chunk, rows of no sequence, more than 64 of them
@pytest.mark.gpu
@pytest.mark.parametrize("form,gk_div", [("ab", 64.0), ("beta", 1.0)])
@pytest.mark.parametrize("B,T,H,K,V,cu,gk", [
    (3, 47, 16, 128, 128, None, torch.bfloat16), (4, 16, 16, 128, 128, None, torch.bfloat16), (5, 1, 9, 128, 128, None, torch.bfloat16), (1, 33, 17, 128, 128, None, torch.bfloat16), (3, 250, 16, 64, 64, None, torch.bfloat16),
    (4, 129, 32, 128, 128, None, torch.float32), (8, 100, 12, 64, 128, None, torch.bfloat16), (4, 65, 24, 128, 64, None, torch.bfloat16),
    (1, 700, 16, 128, 128, (0, 300, 337, 337, 640, 700), torch.bfloat16), (1, 500, 32, 128, 64, (3, 200, 201, 330, 490), torch.bfloat16),
    (1, 1400, 3, 128, 128, tuple(range(0, 1401, 35)), torch.bfloat16), (1, 900, 24, 64, 128, (0, 16, 500, 620, 700, 900), torch.float32), (1, 1700, 2, 128, 128, tuple(range(0, 1701, 25)) + (1700, 1700), torch.bfloat16)])
def test_one_scan_and_two(B, T, H, K, V, cu, gk, form, gk_div):
    """The two entry points on buffers of the sizes that the plan says, and the operator, which keeps nothing of calls under saved-tensor hooks."""
    N = B if cu is None else len(cu) - 1
    x, do, dht = _leaves(form, B, T, H, K, V, N, gk, gk_div)
    table = None if cu is None else torch.tensor(cu, device=DEV)
    dims = _lib.make_dims(B, T, H, K, V, 2, N, torch.bfloat16, gk, 0.7, table)
    sizes = _plan(B, T, H, K, V, N=None if cu is None else N, gk=gk)
    assert all(sizes)
    kept, ws_fwd, ws_bwd = (torch.empty(n, dtype=torch.uint8, device=DEV) for n in sizes)
    P, lib = _lib.ptr, _lib.load()
    size, stream, of = ctypes.c_size_t, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.byref(dims)
    d = [t.detach() for t in x]
    ins = [P(t) for t in d[:3]] + ([P(d[3]), P(d[4]), None] if form == "ab" else [None, None, P(d[3])]) + [P(d[-2]), P(d[-1])]
    o, ht = torch.empty_like(d[2]), torch.empty_like(d[-1])
    fwd, bwd = lib.hdla_chunk_fwd_states, lib.hdla_chunk_bwd_states
    _lib.check(fwd(of, *ins, P(o), P(ht), P(kept), size(sizes[0]), P(ws_fwd), size(sizes[1]), stream), "hdla_chunk_fwd_states")
    grads = []
    for _ in range(2):                                           # on the same buffer
        g = [torch.full_like(t, float("nan")) for t in d]
        outs = [P(t) for t in g[:3]] + ([P(g[3]), P(g[4]), None] if form == "ab" else [None, None, P(g[3])]) + [P(g[-2]), P(g[-1])]
        _lib.check(bwd(of, *ins, P(do), P(dht), *outs, P(kept), size(sizes[0]), P(ws_bwd), size(sizes[2]), stream), "hdla_chunk_bwd_states")
        grads.append(g)
    op = (lambda *a, **kw: chunk_hrdplr_delta_rule(*a, 2, **kw)) if form == "ab" else chunk_hdla_delta_rule
    run = lambda: op(*x[:-1], scale=0.7, initial_state=x[-1], output_final_state=True, cu_seqlens=table)
    with torch.no_grad():
        plain = run()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        o2, ht2 = run()
        want = [o2, ht2, *torch.autograd.grad([o2, ht2], x, [do, dht])]
    names = ["o", "ht", "dq", "dk", "dv", "da", "db", "dgk", "dh0"] if form == "ab" else ["o", "ht", "dq", "dk", "dv", "dbeta", "dgk", "dh0"]
    for g in grads:
        for name, a, b in zip(names, [o, ht] + g, want):
            assert torch.isfinite(a.float()).all() and torch.equal(a, b), name
    assert torch.equal(o, plain[0]) and torch.equal(ht, plain[1])


class _Call:
    """A training call of the operator: what it holds between its passes, and that its gradients are those of a call that keeps its inputs."""
    def __init__(self, B, T, H, K, V):
        self.x, self.do, _ = _leaves("ab", B, T, H, K, V, B, torch.bfloat16, 64.0)
        self.run = lambda: chunk_hrdplr_delta_rule(*self.x[:-1], 2, scale=0.7, initial_state=self.x[-1])[0]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
            self.want = torch.autograd.grad(self.run(), self.x, self.do)
        self.states = _plan(B, T, H, K, V)[0]
        self.plain = _lib.keep_plan(_lib.make_dims(B, T, H, K, V, 2, B, torch.bfloat16, torch.bfloat16, 1.0, None))[0]

    def forward(self):
        gc.collect()
        torch.cuda.synchronize()
        at = torch.cuda.memory_stats()["requested_bytes.all.current"]
        self.o = self.run()
        return torch.cuda.memory_stats()["requested_bytes.all.current"] - at - self.o.numel() * 2

    def check(self):
        assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(self.o, self.x, self.do), self.want))
        del self.o


@pytest.mark.gpu
def test_calls_that_may_keep_the_chunks_operands_keep_no_states():
    """The gibibyte of a device holds more calls of these, each of which gains more by a byte of it."""
    call = _Call(4, 1000, 16, 128, 128)
    assert 0 < call.plain < call.states
    slack = 4 << 20                                               # (final states and the like)
    assert call.plain <= call.forward() < call.plain + slack
    call.check()


@pytest.mark.gpu
def test_who_finds_room():
    """Calls too large for the operands alone (256 MiB) hold the states, two of these; the third and what is next to them take what is left, and give and get the same bits."""
    large, mid, small = [_Call(4, 2048, 16, 128, 128) for _ in range(3)], _Call(4, 1000, 16, 128, 128), _Call(2, 300, 16, 128, 128)
    n = large[0].states
    assert large[0].plain == 0 and 2 * n <= 1 << 30 < 3 * n and 0 < small.plain <= (1 << 30) - 2 * n < mid.plain
    slack = 4 << 20
    assert all(n <= c.forward() < n + slack for c in large[:2])
    assert large[2].forward() < slack and mid.forward() < slack   # no room: the inputs
    assert small.plain <= small.forward() < small.plain + slack
    for c in large + [mid, small]:
        c.check()
    assert n <= large[2].forward() < n + slack                    # given back
    large[2].check()


@pytest.mark.gpu
@pytest.mark.parametrize("missing", ["buffer", "scratch"])
def test_where_the_states_cannot_be_had(missing):
    """A limit of torch's allocator between what the call needs and what it would keep, or between that and what it needs beside it."""
    gc.collect()
    torch.cuda.empty_cache()                                      # (or the inputs may lie in a block that has room for the buffer too)
    call = _Call(4, 2048, 16, 128, 128)
    d = _lib.make_dims(4, 2048, 16, 128, 128, 2, 4, torch.bfloat16, torch.bfloat16, 1.0, None)
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    blocks = 24 << 20                                             # (the allocator's blocks of 2 and 20 MiB)
    room = _lib.load().hdla_workspace_bytes(ctypes.byref(d), _lib.PASS_FWD) + call.do.numel() * 2 + blocks
    assert room < call.states and blocks < _plan(4, 2048, 16, 128, 128)[1]
    if missing == "scratch":
        room = call.states + call.do.numel() * 2 + blocks
    limit = lambda more: torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + more) / torch.cuda.get_device_properties(0).total_memory)
    gaps = []                                                     # what is free in the blocks of what is held
    try:
        limit(0)
        for size in (64 << 20, 16 << 20, 2 << 20):
            try:
                while True:
                    gaps.append(torch.empty(size, dtype=torch.uint8, device=DEV))
            except torch.OutOfMemoryError:
                pass
        limit(room)
        held = call.forward()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert held < 4 << 20
    call.check()
