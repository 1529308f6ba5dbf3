"""What a training call keeps of its forward pass where nothing is said about it (hdla_keep_plan): where the library suggests it (on the CPU), and
that a backward pass on it is the one that recomputes in as many time segments, bit for bit."""
import ctypes
import gc
import time

import pytest
import torch

import hdla_hip.chunk as CK
from hdla_hip import _lib, chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.layer import HDLA_Custom
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

DEV = "cuda"


def _plan(T, lanes, K=128, V=128, dtype=torch.bfloat16, cu=None, **kw):
    d = _lib.make_dims(1, T, lanes, K, V, 2, 1, dtype, dtype, 1.0, None, **kw)
    if cu:
        d.N, d.cu_seqlens = cu, 256                             # never read on the host
    return _lib.keep_plan(d)


def test_where_it_is_suggested():
    n, fwd, bwd = _plan(1537, 16)
    assert 0 < n <= 256 << 20 and (fwd, bwd) == (1, 1)
    assert _plan(16384, 16)[0] == 0                             # more than 256 MiB
    assert _plan(2048, 64, K=64, V=64)[0] == 0                  # the fused route has its record
    assert _plan(256, 2, K=64, V=64)[1:] == (1, 1)              # few short sequences: the classic kernels
    assert _plan(96, 2, K=64, V=64)[0] == 0                     # (their backward pass only)
    assert _plan(0, 4)[0] == 0 and _plan(64, 4, K=96)[0] == 0
    # as many segments as were asked for in both passes; none on the classic route
    assert _plan(600, 4, segments=3)[1:] == (3, 3) and _plan(600, 4, route=_lib.ROUTE_CLASSIC)[1:] == (1, 1)
    d = _lib.make_dims(1, 600, 4, 128, 128, 2, 1, torch.bfloat16, torch.bfloat16, 1.0, None, segments=3)
    size = lambda p: _lib.load().hdla_workspace_bytes(ctypes.byref(d), p)
    assert _lib.keep_plan(d)[0] == size(_lib.PASS_FWD_KEEP)
    d.segments = 1
    assert size(_lib.PASS_FWD_KEEP) < _plan(600, 4, segments=3)[0]


# the forward pass's segments, and the faster of these and one for the backward pass
@pytest.mark.parametrize("K,V,lanes,chunks,dtype,want", [
    (128, 128, 1, 313, torch.bfloat16, (16, 16)), (128, 128, 8, 128, torch.bfloat16, (8, 8)), (128, 128, 16, 16, torch.bfloat16, (1, 1)),
    (128, 128, 16, 200, torch.bfloat16, (4, 4)), (64, 128, 2, 200, torch.bfloat16, (16, 16)), (64, 64, 16, 63, torch.float32, (8, 8)),
    (128, 128, 16, 8, torch.float32, (1, 1)), (64, 64, 1, 8, torch.float32, (1, 1))])
def test_segments(K, V, lanes, chunks, dtype, want):
    assert _plan(16 * chunks, lanes, K, V, dtype)[1:] == want


def test_the_forward_pass_runs_in_the_segments_it_has_without_gradients():
    """Read off the workspace, which holds the segments' records."""
    for dtype in (torch.bfloat16, torch.float32):
        for K, V in ((64, 64), (64, 128), (128, 64), (128, 128)):
            for lanes in (1, 2, 3, 5, 8, 12, 16, 33, 64, 200):
                for chunks in (1, 4, 8, 12, 15, 16, 31, 64, 97, 128, 200, 313, 500):
                    for cu in (None, 2):
                        n, fwd, bwd = _plan(16 * chunks * (cu or 1), lanes, K, V, dtype, cu)
                        if not n:
                            continue
                        assert bwd in (1, fwd)
                        if dtype == torch.bfloat16 and K == V == 64:
                            assert fwd == 1                     # (asked for, segments are the fused route's)
                            continue
                        d = _lib.make_dims(1, 16 * chunks * (cu or 1), lanes, K, V, 2, cu or 1, dtype, dtype, 1.0, None)
                        d.cu_seqlens = 256 if cu else None
                        size = lambda: _lib.load().hdla_workspace_bytes(ctypes.byref(d), _lib.PASS_FWD)
                        own, d.segments = size(), fwd
                        assert size() == own, (dtype, K, V, lanes, chunks, cu)


CASES = [(2, 100, 2, 64, 64, None), (1, 70, 3, 128, 128, None), (1, 300, 2, 64, 128, (0, 37, 37, 200, 300)), (1, 330, 2, 128, 64, None),
         (1, 260, 3, 128, 128, (0, 5, 101, 117, 260))]


def _leaves(form, B, T, H, K, V, cu, dtype, gk_div=4.0):
    inp = make_inputs(2100 + T, B, T, H, K, V, gk_div=gk_div, n_states=B if cu is None else len(cu) - 1)
    k = torch.nn.functional.normalize(inp.k, dim=-1)
    beta = 2.0 * torch.rand(B, T, H, 1, generator=torch.Generator().manual_seed(5))
    x = [inp.q, k, inp.v] + ([inp.a, inp.b] if form == "ab" else [beta]) + [inp.gk]
    return [t.to(dtype) for t in x] + [inp.h0], inp.do.to(dtype), inp.dht


def _grads(form, leaves, do, dht, cu, keep):
    op = (lambda *a, **kw: chunk_hrdplr_delta_rule(*a, 2, **kw)) if form == "ab" else chunk_hdla_delta_rule
    o, ht = op(*leaves[:-1], scale=0.7, initial_state=leaves[-1], output_final_state=True, cu_seqlens=cu, keep_forward=keep)
    return [o.detach(), ht.detach(), *torch.autograd.grad([o, ht], leaves, [do, dht])]


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,H,K,V,cu", CASES)
@pytest.mark.parametrize("segments", [1, 2, 3, 5])
def test_the_gradients_of_a_pass_that_recomputes(B, T, H, K, V, cu, dtype, form, native, segments, monkeypatch):
    if K == V == 64 and dtype == torch.bfloat16:
        if segments > 1:
            pytest.skip("the fused route's")
        T = 256                                                 # few short sequences
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    x, do, dht = _leaves(form, B, T, H, K, V, cu, dtype)
    x, do, dht = [t.to(DEV).requires_grad_() for t in x], do.to(DEV), dht.to(DEV)
    table = None if cu is None else torch.tensor(cu, device=DEV)
    if segments > 1 or dtype == torch.float32 or K != 64 or V != 64:
        monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(segments))
    got, again = _grads(form, x, do, dht, table, None), _grads(form, x, do, dht, table, False)
    for i, (a, b) in enumerate(zip(got, again)):
        assert torch.equal(a, b), (i, O.rel_l2(a, b))
    if segments == 3 and native:                                # against the float64 recurrence
        ref = [t.detach().cpu().double().requires_grad_() for t in x]
        ab = list(O.parameterize_a_b(ref[3], ref[1], ref[4])) if form == "beta" else ref[3:5]
        o, ht = O.recurrence(*ref[:3], *ab, ref[-2], 0.7, ref[-1], cu_seqlens=None if cu is None else torch.tensor(cu))
        want = [o.detach(), ht.detach(), *torch.autograd.grad([o, ht], ref, [do.cpu().double(), dht.cpu().double()])]
        errs = [O.rel_l2(a, b) for a, b in zip(got, want)]
        assert max(errs) <= (1e-2 if dtype == torch.bfloat16 else 1e-5), errs


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("T,H,K,V,cu,dtype", [(3200, 16, 128, 128, None, torch.bfloat16), (3200, 1, 128, 128, None, torch.bfloat16),
                                              (2048, 4, 64, 128, None, torch.bfloat16), (3300, 3, 128, 64, (0, 1900, 1917, 3300), torch.bfloat16),
                                              (128, 16, 128, 128, None, torch.float32), (250, 2, 128, 64, None, torch.float32)])
def test_outputs_with_and_without_gradients(T, H, K, V, cu, dtype, native, monkeypatch):
    """The same bits, as a recomputation that replaces a pass without gradients expects them."""
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    x, _, _ = _leaves("ab", 1, T, H, K, V, cu, dtype, gk_div=64.0)      # (so little decay that every segment hears of the first)
    x = [t.to(DEV) for t in x]
    table = None if cu is None else torch.tensor(cu, device=DEV)
    run = lambda: chunk_hrdplr_delta_rule(*x[:-1], 2, scale=0.7, initial_state=x[-1], output_final_state=True, cu_seqlens=table)
    plain = run()
    x[0].requires_grad_()
    assert all(torch.equal(a, b) for a, b in zip(run(), plain))


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_it_is_kept_and_given_back(native, monkeypatch):
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    x, do, dht = _leaves("ab", 1, 400, 4, 128, 128, None, torch.bfloat16)
    x, do = [t.to(DEV).requires_grad_() for t in x], do.to(DEV)
    run = lambda keep=None: chunk_hrdplr_delta_rule(*x[:-1], 2, scale=0.7, initial_state=x[-1], keep_forward=keep)[0]

    def becomes(want, what):                                    # (the engine's thread lets go of its last tensors a moment after the call has returned)
        for _ in range(1000):
            if what() == want:
                return True
            time.sleep(1e-3)
        return False

    def held(keep=None):
        torch.cuda.synchronize()
        at = torch.cuda.memory_allocated()
        o = run(keep)
        n = torch.cuda.memory_allocated() - at - o.numel() * 2
        torch.autograd.grad(o, x, do, retain_graph=True)
        assert becomes(n, lambda: torch.cuda.memory_allocated() - at - o.numel() * 2)
        del o
        assert becomes(at, torch.cuda.memory_allocated)
        return n

    want = _plan(400, 4)[0]
    assert want <= held() <= want + (1 << 16)
    assert held(False) < 1 << 16
    for name, value in (("HDLA_HIP_INPUTS_ONLY", "1"), ("HDLA_HIP_KEEP_FORWARD", "0")):
        with monkeypatch.context() as c:
            c.setenv(name, value)
            assert held() < 1 << 16
    # the plan is the forward pass's, whatever the environment says by the backward pass
    monkeypatch.setenv("HDLA_HIP_SEGMENTS", "4")
    ref = torch.autograd.grad(run(), x, do)
    for env in ({"HDLA_HIP_SEGMENTS": "2"}, {"HDLA_HIP_ROUTE": "classic"}, {"HDLA_HIP_INPUTS_ONLY": "1"}, {"HDLA_HIP_KEEP_FORWARD": "0"}):
        o = run()
        with monkeypatch.context() as c:
            for name, value in env.items():
                c.setenv(name, value)
            assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, x, do), ref)), env


def test_the_account_of_the_python_code(monkeypatch):
    """On the CPU: what a call holds is on it until its backward pass is through, also behind torch's saved tensors."""
    monkeypatch.setattr(_lib, "KEPT_MOST", 1000)
    acc, like = _lib._NoNative(), torch.empty(1)

    class Keep(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, n):
            room = acc.kept_room(like, n)
            ctx.got = room is not None
            ctx.save_for_backward(x, room)
            return x * 2

        @staticmethod
        def backward(ctx, g):
            ctx.saved_tensors
            return g * 2, None

    x = torch.ones(3, requires_grad=True)
    got = lambda y: y.grad_fn.got
    a, b, c = Keep.apply(x, 400), Keep.apply(x, 600), Keep.apply(x, 1)
    gc.collect()
    d = Keep.apply(x, 1)
    assert [got(y) for y in (a, b, c, d)] == [True, True, False, False]
    torch.autograd.grad(a.sum(), x)                              # (the graph's end lets go of its saved tensors)
    e, f = Keep.apply(x, 300), Keep.apply(x, 200)
    assert got(e) and not got(f)
    del b, e
    fresh = lambda: [got(Keep.apply(x, 1000)) for _ in range(2)]
    assert fresh() == [True, True]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert fresh() == [False, False]
    assert fresh() == [True, True]
    many = [Keep.apply(x, 1) for _ in range(_lib.KEPT_CALLS + 1)]
    assert [got(y) for y in many] == [True] * _lib.KEPT_CALLS + [False]
    del many
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: (_ for _ in ()).throw(torch.OutOfMemoryError()))
    assert acc.kept_room(like, 900) is None and acc._coming == {None: 0}


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_calls_whose_backward_pass_is_to_come_hold_a_gibibyte_at_most(native, monkeypatch):
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    T, H, D = 5008, 16, 128
    each = _plan(T, H)[0]
    most = (1 << 30) // each
    assert 2 < most < 8
    x, do, _ = _leaves("ab", 1, T, H, D, D, None, torch.bfloat16, gk_div=64.0)
    x, do = [t.to(DEV).requires_grad_() for t in x], do.to(DEV)
    run = lambda: chunk_hrdplr_delta_rule(*x[:-1], 2, scale=0.7, initial_state=x[-1])[0]
    gc.collect()
    torch.cuda.synchronize()
    held, outs = [], []
    for _ in range(most + 2):
        at = torch.cuda.memory_allocated()
        outs.append(run())
        held.append(torch.cuda.memory_allocated() - at - outs[-1].numel() * 2 >= each)
    assert held == [True] * most + [False] * 2
    first = torch.autograd.grad(outs[0], x, do)
    for o in outs[1:]:                                           # kept or not: the same bits
        assert torch.equal(o, outs[0]) and all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, x, do), first))
    del o, outs
    for _ in range(1000):
        at = torch.cuda.memory_allocated()
        o = run()
        if torch.cuda.memory_allocated() - at >= each:
            return
        del o
        time.sleep(1e-3)
    assert False, "nothing was given back"


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("full", ["first", "again"])
def test_a_checkpointed_call_saves_the_same_when_it_is_run_again(full, native, monkeypatch):
    """With the room taken by other calls in one of its two forward passes."""
    from torch.utils.checkpoint import checkpoint
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    T, H, D = 5008, 16, 128
    x, do, _ = _leaves("ab", 1, T, H, D, D, None, torch.bfloat16)
    x, do = [t.to(DEV).requires_grad_() for t in x], do.to(DEV)
    run = lambda *x: chunk_hrdplr_delta_rule(*x[:-1], 2, scale=0.7, initial_state=x[-1])[0]
    want = torch.autograd.grad(run(*x), x, do)
    fill = lambda: [run(*x) for _ in range((1 << 30) // _plan(T, H)[0] + 1)]
    others = fill() if full == "first" else None
    o = checkpoint(run, *x, use_reentrant=False)
    others = fill() if full == "again" else None
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, x, do), want))
    del others


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("T,H,K,V,cu,dtype,plan", [
    (1024, 4, 128, 64, None, torch.bfloat16, (8, 1)), (2048, 8, 128, 128, None, torch.bfloat16, (8, 8)), (700, 12, 128, 128, None, torch.bfloat16, (1, 1)),
    (3000, 2, 128, 64, (0, 1700, 3000), torch.bfloat16, (8, 8)), (256, 2, 64, 64, None, torch.bfloat16, (1, 1)),
    (500, 6, 64, 64, None, torch.float32, (8, 8)), (250, 16, 128, 128, None, torch.float32, (4, 4)), (200, 16, 128, 128, None, torch.float32, (1, 1))])
def test_the_librarys_own_plan_kept_and_not(T, H, K, V, cu, dtype, plan, form, native, monkeypatch):
    """Nothing is kept under saved-tensor hooks: what is computed is the same, whichever segments the library chooses."""
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    assert _plan(T, H, K, V, dtype, None if cu is None else len(cu) - 1)[1:] == plan
    x, do, dht = _leaves(form, 1, T, H, K, V, cu, dtype, gk_div=64.0)
    x, do, dht = [t.to(DEV).requires_grad_() for t in x], do.to(DEV), dht.to(DEV)
    table = None if cu is None else torch.tensor(cu, device=DEV)
    got, saved = _grads(form, x, do, dht, table, None), []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: saved.append(t.dtype) or t, lambda t: t):
        again = _grads(form, x, do, dht, table, None)
    assert torch.uint8 not in saved and all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_where_the_buffer_cannot_be_had(native, monkeypatch):
    """A limit of torch's allocator between what the call needs and what it would keep: it runs, and so does its backward pass later."""
    if not native:
        monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    # (decays in 32 bits, beside which u is kept: with those of 16 the buffer, 38 KB a chunk and head, is less than what the call needs anyway, 32 KB, its
    # output's 4 KB and the allocator's blocks)
    T, H, D = 5008, 16, 128
    d = _lib.make_dims(1, T, H, D, D, 2, 1, torch.bfloat16, torch.float32, 1.0, None)
    each = _lib.keep_plan(d)[0]
    x, do, _ = _leaves("ab", 1, T, H, D, D, None, torch.bfloat16, gk_div=64.0)
    x[-2] = x[-2].float()
    x, do = [t.to(DEV).requires_grad_() for t in x], do.to(DEV)
    run = lambda: chunk_hrdplr_delta_rule(*x[:-1], 2, scale=0.7, initial_state=x[-1])[0]
    want = torch.autograd.grad(run(), x, do)
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    need = _lib.load().hdla_workspace_bytes(ctypes.byref(d), _lib.PASS_FWD) + 2 * T * H * D
    room = need + (24 << 20)                                     # (the allocator's blocks of 2 and 20 MiB)
    assert room < each
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / torch.cuda.get_device_properties(0).total_memory)
        o = run()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, x, do), want))


@pytest.mark.gpu
@pytest.mark.parametrize("segments", [1, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["ab", "beta"])
def test_rows_of_no_sequence(form, dtype, segments):
    """A packed batch padded at both ends: the kept pass clears the gradients' rows that no sequence has, whatever they held."""
    T, H, K, V = 170, 2, 128, 64
    cu, plan, P = torch.tensor([3, 40, 150], device=DEV), (_lib.ROUTE_AUTO, segments), _lib.ptr
    x, do, dht = _leaves(form, 1, T, H, K, V, (0, 85, 170), dtype)
    x, do, dht = [t.to(DEV) for t in x], do.to(DEV), dht.to(DEV)
    q, k, v, gk, h0 = x[0], x[1], x[2], x[-2], x[-1]
    a, b, beta = (*x[3:5], None) if form == "ab" else (None, None, x[3])
    kept = CK.chunk_hrdplr_fwd(q, k, v, a, b, gk, 0.7, h0, True, cu, keep=True, beta=beta, plan=plan)[2]
    dims = CK._dims(q, v, gk, 0.7, cu, 2, plan)
    ws = _lib.workspace(dims, _lib.PASS_BWD_KEPT, q.device)
    da, db, dbeta = [None if t is None else torch.full_like(t, float("nan")) for t in (a, b, beta)]
    dq, dk, dv, dgk, dh0 = [torch.full_like(t, float("nan")) for t in (q, k, v, gk, h0)]
    assert _lib.load().hdla_chunk_bwd_kept(ctypes.byref(dims), P(q), P(k), P(v), P(a), P(b), P(beta), P(gk), P(h0), P(do), P(dht), P(dq), P(dk), P(dv),
                                           P(da), P(db), P(dbeta), P(dgk), P(dh0), P(kept), kept.numel(), P(ws), ws.numel(),
                                           _lib.current_stream(q.device)) == 0
    for i, g in enumerate(t for t in (dq, dk, dv, dgk, da, db, dbeta) if t is not None):
        r = g.shape[1] // T
        assert torch.isfinite(g.float()).all() and not g[:, :3 * r].any() and not g[:, 150 * r:].any() and g[:, 3 * r:150 * r].any(), i
    assert torch.isfinite(dh0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("d,H,T", [(256, 4, 256), (512, 4, 300)])
def test_the_layer(d, H, T, monkeypatch):
    torch.manual_seed(3)
    m = HDLA_Custom(d, H, token_mixer_init_type=2, rescale_type=0).to(DEV).bfloat16().train()
    x, do = torch.randn(1, T, d, device=DEV).bfloat16().requires_grad_(), torch.randn(1, T, d, device=DEV).bfloat16()
    run = lambda: torch.autograd.grad(m(x)[0], [x, *m.parameters()], do)
    got = run()
    monkeypatch.setenv("HDLA_HIP_INPUTS_ONLY", "1")
    assert all(torch.equal(a, b) for a, b in zip(got, run()))


@pytest.mark.gpu
def test_a_buffer_of_another_plan_is_refused():
    x, do, dht = [t if isinstance(t, list) else t.to(DEV) for t in _leaves("ab", 1, 200, 2, 128, 128, None, torch.float32)]
    q, k, v, a, b, gk, h0 = [t.to(DEV) for t in x]
    plan = lambda n: (_lib.ROUTE_AUTO, n)
    kept = {n: CK.chunk_hrdplr_fwd(q, k, v, a, b, gk, 0.7, h0, True, keep=True, plan=plan(n))[2] for n in (1, 4, 8)}
    bwd = lambda n, buffer: CK.chunk_hrdplr_bwd_kept(q, k, v, a, b, gk, 0.7, h0, do, dht, buffer, plan=plan(n))
    # too few records, too many, and a longer buffer that may be either; one segment reads none of them
    for n, buffer in ((4, kept[1]), (8, kept[4]), (4, kept[8]), (4, torch.cat([kept[4], kept[4]]))):
        with pytest.raises(_lib.HdlaError, match="-5"):
            bwd(n, buffer)
    for n in (4, 8):
        bwd(n, kept[n])
        assert all(torch.equal(s, t) for s, t in zip(bwd(1, kept[n]), bwd(1, kept[1])))
