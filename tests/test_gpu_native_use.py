"""The native host path in the surroundings a training program puts it in: autocast, activation checkpointing, hooks, parameters at
any address, more than one stream, more than one thread."""
import sys
import threading
import time

import pytest
import torch
import torch.nn as nn

from hdla_hip import _lib, chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.layer import HDLA_Custom, RecurrentCache
from hdla_hip.normalize import normalize_fn
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(d=256, H=4, **kw):
    torch.manual_seed(3)
    return HDLA_Custom(d, H, token_mixer_init_type=2, rescale_type=0, **kw).to(DEV).bfloat16().train()


def _x(B, T, d=256, seed=4, grad=True):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(B, T, d, generator=g).bfloat16().to(DEV).requires_grad_(grad), torch.randn(B, T, d, generator=g).bfloat16().to(DEV)


def _operands(T=70, H=2, K=64, seed=41):
    x = make_inputs(seed, 1, T, H, K, K)
    return [t.bfloat16().to(DEV).requires_grad_() for t in (x.q, x.k, x.v, x.a, x.b, x.gk)], x.do.bfloat16().to(DEV)


# ---- autocast -------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("what", ["layer", "operator", "norm"])
def test_backward_inside_an_autocast_region(what, dtype):
    """A forward pass outside autocast (or in a region that switches it off) and backward() inside one, whose products torch
    would run in that region's type: the gradients are those of a backward pass outside."""
    if what == "layer":
        m, (x, do) = _layer(), _x(2, 40)
        leaves, run = [x] + list(m.parameters()), lambda: m(x)[0]
    elif what == "operator":
        leaves, do = _operands()
        run = lambda: chunk_hrdplr_delta_rule(*leaves, 2, scale=0.5)[0]
    else:
        (x, do), (gate, _) = _x(2, 40), _x(2, 40, seed=5)
        w = torch.ones(256, device=DEV, requires_grad=True)
        leaves, run = [x, gate, w], lambda: normalize_fn(x, w, gate=gate, gate_pos="pre", c=16.0, eps=1e-5)
    ref = torch.autograd.grad(run(), leaves, do)
    with torch.autocast("cuda", dtype=dtype):
        with torch.autocast("cuda", enabled=False):
            y = run()
        got = torch.autograd.grad(y, leaves, do)
    for a, b in zip(ref, got):
        assert a.dtype == b.dtype and torch.equal(a, b)


# ---- parameters and inputs at any address -----------------------------------------------------------------------------
def _shifted(t):
    """The same values, contiguous, eight bytes behind a multiple of 16."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    assert flat.data_ptr() % 16 == 0
    return flat[4:4 + t.numel()].view(t.shape).copy_(t.detach())


@pytest.mark.parametrize("B,T", [(2, 3), (2, 40)])                 # few rows (kernels of this library), more (BLAS)
@pytest.mark.parametrize("which", ["q_proj", "f_proj.0", "f_proj.1", "output_gate.1", "o_proj", "x"])
def test_layer_tensors_off_the_16_byte_grid(which, B, T):
    m, (x, do) = _layer(), _x(B, T)
    params = dict(m.named_parameters())

    def both(x):
        y = m(x)[0]
        g = torch.autograd.grad(y, [x] + list(m.parameters()), do)
        m.eval()
        with torch.no_grad():
            e = m(x, past_key_values=RecurrentCache(), use_cache=True)[0]
        m.train()
        return [y.detach(), e, *g]

    ref = both(x)
    if which == "x":
        x = _shifted(x).requires_grad_()
    else:
        mod = m.get_submodule(which)
        mod.weight = nn.Parameter(_shifted(params[which + ".weight"]))
        assert mod.weight.data_ptr() % 16 == 8
    # (the same products by other kernels: their results may round to another bf16 value, and so on down the layer)
    for a, b in zip(ref, both(x)):
        assert O.rel_l2(b, a) <= 2e-2


# ---- activation checkpointing, saved-tensor hooks, hooks on the layer -------------------------------------------------
@pytest.mark.parametrize("reentrant", [False, True])
def test_layer_and_operator_under_activation_checkpointing(reentrant):
    from torch.utils.checkpoint import checkpoint
    m, (x, do) = _layer(), _x(2, 40)
    leaves = [x] + list(m.parameters())
    ref = torch.autograd.grad(m(x)[0], leaves, do)
    for p in leaves:
        p.grad = None
    checkpoint(lambda t: m(t)[0], x, use_reentrant=reentrant).backward(do)
    assert all(torch.equal(p.grad, g) for p, g in zip(leaves, ref))
    ops, do = _operands()
    ref = torch.autograd.grad(chunk_hrdplr_delta_rule(*ops, 2)[0], ops, do)
    checkpoint(lambda *t: chunk_hrdplr_delta_rule(*t, 2)[0], *ops, use_reentrant=reentrant).backward(do)
    assert all(torch.equal(p.grad, g) for p, g in zip(ops, ref))


def test_saved_tensors_on_the_host():
    m, (x, do) = _layer(), _x(2, 40)
    leaves = [x] + list(m.parameters())
    ref = torch.autograd.grad(m(x)[0], leaves, do)
    with torch.autograd.graph.save_on_cpu():
        y = m(x)[0]
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, leaves, do), ref))


def test_hooks_on_the_layer_and_on_its_gradients():
    m, (x, do) = _layer(), _x(2, 40)
    ref = torch.autograd.grad(m(x)[0], [x, m.o_proj.weight], do)
    seen = []
    m.register_forward_hook(lambda mod, a, out: (out[0] * 2, out[1]))
    m.register_full_backward_hook(lambda mod, gi, go: seen.append(len(gi)))
    m.o_proj.weight.register_hook(lambda g: g * 4)
    got = torch.autograd.grad(m(x)[0], [x, m.o_proj.weight], do)
    assert seen == [1] and torch.equal(got[0], 2 * ref[0]) and torch.equal(got[1], 8 * ref[1])


# ---- streams and threads ----------------------------------------------------------------------------------------------
def _step(m, x, do, n=3):
    """n training steps and cached decode steps on the current stream; what they give."""
    out = []
    for _ in range(n):
        y = m(x)[0]
        out += [y.detach(), *torch.autograd.grad(y, [x] + list(m.parameters()), do)]
    m.eval()
    with torch.no_grad():
        cache = RecurrentCache()
        for i in range(n):
            out.append(m(x[:, 20 * i:20 * i + 20 if i == 0 else 20 * i + 1], past_key_values=cache, use_cache=True)[0])
    m.train()
    return out


def test_calls_on_a_second_stream():
    """Whole steps on a stream that is not the default one, with the default stream allocating and writing at the same time."""
    m, (x, do) = _layer(), _x(2, 70)
    ref = _step(m, x, do)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = _step(m, x, do)
    for _ in range(20):
        torch.full((1 << 22,), float("nan"), device=DEV)
    torch.cuda.current_stream().wait_stream(s)
    assert all(torch.equal(a, b) for a, b in zip(ref, got))


def test_threads_with_a_stream_each():
    n = 4
    ms, xs = [_layer() for _ in range(n)], [_x(2, 70, seed=10 + i) for i in range(n)]
    refs = [_step(m, *x) for m, x in zip(ms, xs)]
    torch.cuda.synchronize()
    got, errors = [None] * n, []

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                got[i] = _step(ms[i], *xs[i])
            s.synchronize()
        except Exception as e:                                     # reported by the main thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    for r, g in zip(refs, got):
        assert all(torch.equal(a, b) for a, b in zip(r, g))


@pytest.mark.parametrize("call", ["chunk", "chunk_grad", "chunk_hdla", "recurrent", "normalize", "layer"])
def test_other_threads_run_during_a_call(call):
    """A native call gives the interpreter lock back while it allocates and launches, as torch's own operators do."""
    x = make_inputs(42, 1, 64, 2, 64, 64)
    t = [y.bfloat16().to(DEV) for y in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    g = [y.clone().requires_grad_() for y in t]
    beta = torch.rand(1, 64, 2, 1, device=DEV).bfloat16()
    m, (lx, _) = _layer(), _x(2, 8, grad=False)
    n, row = _lib.native(), torch.randn(8, 64, device=DEV).bfloat16()
    one = {
        "chunk": lambda: n.chunk(*t, 2, None, None, False, False, 16, None, False),
        "chunk_grad": lambda: n.chunk(*g, 2, None, None, False, False, 16, None, False),
        "chunk_hdla": lambda: n.chunk_hdla(t[0], t[1], t[2], beta, t[5], None, None, False, None, False),
        "recurrent": lambda: n.recurrent(*t, 2, None, None, False, False, None, False),
        "normalize": lambda: n.normalize(row, None, None, None, None, "sigmoid", "pre", 1.0, 1e-5, False, 1, False),
        "layer": lambda: m._forward_native(lx, None, False),
    }[call]
    assert one() is not None
    count, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            count[0] += 1
            time.sleep(0)

    th = threading.Thread(target=other)
    old = sys.getswitchinterval()
    sys.setswitchinterval(30.0)              # from here on a thread runs Python only when another one lets go of the lock itself
    try:
        th.start()
        before = count[0]
        for _ in range(5000):
            one()
            if count[0] != before:
                break
        ran = count[0] - before
    finally:
        stop.set()
        th.join()
        sys.setswitchinterval(old)
    assert ran > 0


def test_an_exception_of_a_saved_tensor_hook_comes_through():
    ops, _ = _operands()

    def refuse(t):
        raise KeyError("not today")

    with pytest.raises(KeyError, match="not today"):
        with torch.autograd.graph.saved_tensors_hooks(refuse, lambda t: t):
            chunk_hrdplr_delta_rule(*ops, 2)
    assert torch.isfinite(chunk_hrdplr_delta_rule(*ops, 2)[0].float()).all()


def test_operators_and_layer_without_the_native_host_path(monkeypatch):
    ops, do = _operands()
    m, (x, ldo) = _layer(), _x(2, 40)
    run = lambda: torch.autograd.grad(chunk_hrdplr_delta_rule(*ops, 2)[0], ops, do)
    ref, lref = run(), torch.autograd.grad(m(x)[0], [x, m.o_proj.weight], ldo)
    monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    assert all(torch.equal(a, b) for a, b in zip(ref, run()))
    for a, b in zip(lref, torch.autograd.grad(m(x)[0], [x, m.o_proj.weight], ldo)):
        assert O.rel_l2(a, b) <= 2e-2                                  # (the layer's steps round to bf16 in between)
