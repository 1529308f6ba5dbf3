"""The layer's decode step between the projections in one launch (csrc/layer_step.hip) against the three kernels that it stands
for, run one after the other."""
import ctypes

import pytest
import torch

from hdla_hip import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


P = _lib.ptr


def _rn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)


def _rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N,T,H,norm_q,norm_v,gate_pos,weight,state", [
    (1, 1, 2, True, False, 1, "bf16", True), (3, 1, 6, True, True, 2, "fp32", True), (2, 2, 4, False, True, 1, None, False),
    (2, 8, 16, True, False, 2, "bf16", True), (40, 1, 8, False, False, 1, "fp32", False)])
def test_layer_step(D, N, T, H, norm_q, norm_v, gate_pos, weight, state):
    lib, st, ref = _lib.load(), _lib.current_stream(DEV), ctypes.byref
    rows, d = N * T, H * D
    f0, ld = (3 * d + H + 1 + 7) // 8 * 8, (3 * d + H + 1 + 7) // 8 * 8 + 2 * D + 8
    y = _rn(1, rows, ld).bfloat16()
    y[0, d:d + D] = 0.                                          # a head of k of length nought, values at the ends of the activations
    y[0, 0:4] = torch.tensor([80., -80., 3e4, -3e4])
    wf, wg = (_rn(6, d, D) * .2).bfloat16(), (_rn(7, d, D) * .2).bfloat16()
    w = None if weight is None else (1. + .1 * _rn(4, d)).to(torch.bfloat16 if weight == "bf16" else torch.float32)
    h0 = _rn(5, N, H, D, D) if state else None
    pre = _lib.HdlaPreDims(rows, H, D, _lib.dtype_code(torch.bfloat16), ld, 2 * d, d, 0, 3 * d + 1, norm_q, 1, norm_v, 2.0, 1e-5, 0)   # v, k, q: any columns
    up = _lib.HdlaUpDims(rows, d, D, ld, f0, f0 + D)
    nd = _lib.HdlaNormDims(rows, H, D, _lib.dtype_code(torch.bfloat16), _lib.dtype_code(torch.float32) if weight == "fp32" else _lib.dtype_code(torch.bfloat16), gate_pos, D ** .5, 1e-5)

    # the kernels that it stands for
    new = lambda *s: torch.empty(*s, device=DEV, dtype=torch.bfloat16)
    q, k, v, log_f, gate, ro, rn = (new(rows, H, D) for _ in range(7))
    beta, rht = new(rows, H), torch.empty(N, H, D, D, device=DEV)
    assert lib.hdla_layer_up_fwd(ref(up), P(y), P(wf), P(wg), None, P(log_f), P(gate), st) == 0
    assert lib.hdla_layer_pre_fwd(ref(pre), P(y), P(q), P(k), P(v), P(beta), st) == 0
    cd = _lib.make_dims(N, T, H, D, D, 2, N, torch.bfloat16, torch.bfloat16, 1.0, None)
    assert lib.hdla_param_recurrent_fwd(ref(cd), P(q), P(k), P(v), P(beta), P(log_f), 0, P(h0), P(ro), P(rht), st) == 0
    assert lib.hdla_normalize_fwd(ref(nd), P(ro), P(w), P(gate), P(rn), st) == 0
    # Sums over a head run in another order, 2^-24 each; where that moves one of the values that are rounded to bf16 across the middle
    # between two of its numbers (one in 2^10, sums of 128 terms), it moves by 2^-8 of itself.  Not more than a hundredth of all does.
    tol = 2 ** -8 * .1

    def run(norm, with_up, want_ht=True):
        o, ht, g = torch.full((rows + 1, H, D), 7., device=DEV, dtype=torch.bfloat16), torch.empty_like(rht), new(rows, H, D)
        assert lib.hdla_layer_step(ref(pre), ref(up) if with_up else None, ref(nd) if norm else None, T, P(y), P(wf) if with_up else None,
                                   P(wg) if with_up else None, None if with_up else P(log_f), P(g) if with_up else P(gate), P(w) if norm else None,
                                   P(h0), P(o), None, P(ht) if want_ht else None, st) == 0
        assert bool((o[rows:] == 7.).all())
        assert _rel(o[:rows], rn if norm else ro) <= tol
        assert not want_ht or _rel(ht, rht) <= tol
        assert not with_up or _rel(g, gate) <= tol
        return o

    first = run(True, False)
    assert torch.equal(first, run(True, False, False))          # with no final state asked for
    run(False, False)
    if T == 1:
        run(True, True)
        run(False, True)
    bad = lambda pre, up, nd, T, y=P(y): lib.hdla_layer_step(pre, up, nd, T, y, P(wf), P(wg), P(log_f), P(gate), None, None, P(ro), None, None, st)
    assert bad(ref(pre), None, None, 0) == -2 and bad(ref(pre), None, None, rows + 1) == -2 and bad(ref(pre), ref(up), None, 2) == -2
    assert bad(ref(pre), None, ref(_lib.HdlaNormDims(rows, 2 * H, D // 2, _lib.dtype_code(torch.bfloat16), _lib.dtype_code(torch.bfloat16), 1, 1., 1e-5)), T) == -2
    assert bad(ref(pre), None, None, T, None) != 0 and bad(ref(pre), None, None, T, ctypes.c_void_p(y.data_ptr() + 2)) != 0


@pytest.mark.parametrize("gate_pos", [1, 2])
@pytest.mark.parametrize("D,rows,T,H,N,weight", [(64, 1, 1, 2, 20, "bf16"), (64, 16, 1, 9, 200, "fp32"), (128, 5, 1, 16, 2048, "bf16"), (64, 14, 7, 4, 16, None),
                                                (128, 16, 2, 4, 100, "bf16")])
def test_norm_left_to_the_projection(D, rows, T, H, N, weight, gate_pos):
    """hdla_layer_step with `gated`, then hdla_rows_gemm_norm, against step, norm and product."""
    lib, st, ref = _lib.load(), _lib.current_stream(DEV), ctypes.byref
    d = H * D
    ld = (3 * d + H + 7) // 8 * 8
    y, log_f, gate, w = _rn(1, rows, ld).bfloat16(), -_rn(2, rows, d).abs().bfloat16(), _rn(3, rows, d).bfloat16(), _rn(4, N, d).bfloat16()
    wn = None if weight is None else (1. + .1 * _rn(5, d)).to(torch.bfloat16 if weight == "bf16" else torch.float32)
    h0 = _rn(6, rows // T, H, D, D)
    bf = _lib.dtype_code(torch.bfloat16)
    pre = _lib.HdlaPreDims(rows, H, D, bf, ld, 0, d, 2 * d, 3 * d, 0, 1, 0, 1.0, 1e-5, 0)
    nd = _lib.HdlaNormDims(rows, 1, d, bf, _lib.dtype_code(torch.float32 if weight == "fp32" else torch.bfloat16), gate_pos, d ** .5, 1e-5)
    o, n = torch.empty(rows, d, device=DEV, dtype=torch.bfloat16), torch.empty(rows, d, device=DEV, dtype=torch.bfloat16)
    step = lambda norm, out, gated: lib.hdla_layer_step(ref(pre), None, norm, T, P(y), None, None, P(log_f), P(gate), None, P(h0), out, gated, None, st)
    assert step(None, P(o), None) == 0
    assert lib.hdla_normalize_fwd(ref(nd), P(o), P(wn), P(gate), P(n), st) == 0
    want = n.double() @ w.double().t()
    gated = torch.full((rows * (d + H) + 4,), 7., device=DEV)
    assert step(ref(nd), None, P(gated)) == 0
    assert bool((gated[rows * (d + H):] == 7.).all())
    out = torch.full((rows + 1, N + 4), 7., device=DEV, dtype=torch.bfloat16)
    run = lambda M, K=d, nd=nd: lib.hdla_rows_gemm_norm(M, N, K, P(gated), H, ref(nd), P(wn), P(w), d, P(out), N + 4, st)
    assert run(rows) == 0
    # one rounding of the result: at most 2^-8 of each (a third of that in the mean of many, but N = 20 are few)
    assert _rel(out[:rows, :N], want) <= 2 ** -8
    assert bool((out[rows:] == 7.).all() and (out[:, N:] == 7.).all())
    assert run(17) == -2 and run(rows, d - 32) == -2 and step(None, None, P(gated)) != 0


@pytest.mark.parametrize("norm", ["rmsnorm", "grouprmsnorm"])
@pytest.mark.parametrize("B,T,H", [(3, 1, 4), (17, 1, 4), (65, 1, 2), (2, 8, 4), (3, 8, 4), (2, 9, 4), (2, 1, 34)])
def test_layer_routes(B, T, H, norm):
    """Both sides of the lines that the native call chooses by (tokens, rows, the norm's groups) next to the layer's Python
    code, and replays of a captured step."""
    from hdla_hip.layer import HDLA_Custom, RecurrentCache
    torch.manual_seed(3)
    with torch.device("cuda"):
        m = HDLA_Custom(64 * H, H, token_mixer_init_type=2, rescale_type=0, token_mixer_norm_type=norm).to(torch.bfloat16).eval()
    x, s0 = _rn(9, B, T, 64 * H).bfloat16(), _rn(10, B, H, 64, 64)

    def step():
        cache = RecurrentCache()
        cache.update(recurrent_state=[s0], layer_idx=0, offset=T)
        o, cache = m(x, past_key_values=cache, use_cache=True)
        return o, cache[0]["recurrent_state"][0]

    with torch.no_grad():
        a, sa = step()
        m._forward_native = lambda *_: None
        b, sb = step()
        del m._forward_native
        # Both are rounded to bf16 nine times on the way (y, q, k, v, f, the decay, the gate, o, the norm's output), each time by up to
        # 2^-9, 2^-9 / sqrt(3) in the mean, and in part at other places: sqrt(2 * 9) of that
        assert _rel(a, b) <= 5e-3 and _rel(sa, sb) <= 5e-3
        g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        with torch.cuda.graph(g):
            c, sc = step()
        for i in range(3):
            s0.mul_(.5)
            x.neg_()
            want, ws = step()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, want) and torch.equal(sc, ws)


@pytest.mark.parametrize("norm", ["rmsnorm", "grouprmsnorm"])
@pytest.mark.parametrize("B,T,H,few", [(192, 1, 32, (True, True)), (192, 2, 16, (True, True)), (193, 2, 16, (True, False)),
                                       (192, 8, 4, (True, True)), (193, 8, 4, (True, False)), (192, 8, 8, (True, False)), (193, 8, 8, (False, False))])
def test_several_tokens_of_many_sequences(B, T, H, few, norm):
    """Both sides of the line by which the native call takes several tokens of many sequences in few launches or as steps (few: with the norm
    in the same launch, in one of its own): which of the two runs shows in the tensors it holds, and both agree with the Python code."""
    from hdla_hip.layer import HDLA_Custom, RecurrentCache
    torch.manual_seed(4)
    d = 64 * H
    with torch.device("cuda"):
        m = HDLA_Custom(d, H, token_mixer_init_type=2, rescale_type=0, token_mixer_norm_type=norm).to(torch.bfloat16).eval()
    x, s0 = _rn(9, B, T, d).bfloat16(), _rn(10, B, H, 64, 64)

    def step():
        cache = RecurrentCache()
        cache.update(recurrent_state=[s0], layer_idx=0, offset=T)
        return m(x, past_key_values=cache, use_cache=True)[0], cache[0]["recurrent_state"][0]

    with torch.no_grad():
        step()                                                  # (the weights gathered, the BLAS library's workspace there)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        at = torch.cuda.memory_allocated()
        a, sa = step()
        # beside the new state: y (three d and up to one more) and the output both ways; the steps hold q, k, v, the decay, the gate, o and the
        # norm's result at once, the few launches the gate, o and the decay at the most
        held = (torch.cuda.max_memory_allocated() - at - sa.numel() * 4) / (B * T * d * 2)
        assert (held < 10.) == few[norm == "rmsnorm"], held
        m._forward_native = lambda *_: None
        b, sb = step()
        assert _rel(a, b) <= 5e-3 and _rel(sa, sb) <= 5e-3      # (as above)


# ---- against float64, without the library's other kernels ----------------------------------------------------------------
def _exact(y, wf, wg, w, h0, N, T, H, D, cols, norm_q, norm_v, gate_pos, groups, log_f=None, gate=None):
    """What lies between the projections, in float64 and rounded nowhere: (o as the norm leaves it, final state)."""
    from oracle import hrdplr_oracle as O
    from oracle import normalize_oracle as NO
    y = y.double()
    take = lambda c, n: y[:, c:c + n]
    head = lambda t: t.reshape(N, T, H, D)
    silu = lambda x: x * torch.sigmoid(x)
    q, k, v = (head(silu(take(cols[i], H * D))) for i in "qkv")
    q, k, v = NO.l2_norm(q) if norm_q else q, NO.l2_norm(k), NO.l2_norm(v) if norm_v else v
    beta = 2.0 * torch.sigmoid(take(cols["b"], H)).reshape(N, T, H, 1)
    if log_f is None:
        log_f, gate = torch.nn.functional.logsigmoid(take(cols["f"], D) @ wf.double().t()), take(cols["g"], D) @ wg.double().t()
    log_f, gate = head(log_f.double()), gate.double().reshape(N, T, H * D)
    a, b = O.parameterize_a_b(beta, k, log_f)
    o, S = O.recurrence(q, k, v, a, b, log_f, 1.0, h0.double())
    pos = "pre" if gate_pos == 1 else "post"
    return NO.normalize(o.reshape(N, T, H * D), w, gate, gate_pos=pos, c=(H * D // groups) ** .5, eps=1e-5, num_groups=groups), S


def _operands(seed, N, T, H, D):
    rows, d = N * T, H * D
    cols = dict(q=0, k=d, v=2 * d, f=3 * d, g=3 * d + D, b=3 * d + 2 * D)
    y = _rn(seed, rows, (cols["b"] + H + 7) // 8 * 8).bfloat16()
    wf, wg = (_rn(seed + 1, d, D) * .2).bfloat16(), (_rn(seed + 2, d, D) * .2).bfloat16()
    w, h0 = 1. + .1 * _rn(seed + 3, d), _rn(seed + 4, N, H, D, D)
    log_f, gate = -_rn(seed + 5, rows, d).abs().bfloat16(), _rn(seed + 6, rows, d).bfloat16()
    return cols, y, wf, wg, w, h0, log_f, gate


def _step(cols, y, wf, wg, w, h0, log_f, gate, N, T, H, D, norm_q, norm_v, gate_pos, groups, later=False):
    """The launch (T = 1: with the low-rank products), and the norm of its own where that is over all channels, or (later) the projection that
    forms it, with the identity for its weight."""
    lib, st, ref, bf, rows, d = _lib.load(), _lib.current_stream(DEV), ctypes.byref, _lib.dtype_code(torch.bfloat16), N * T, H * D
    pre = _lib.HdlaPreDims(rows, H, D, bf, y.shape[1], cols["q"], cols["k"], cols["v"], cols["b"], norm_q, 1, norm_v, 2.0, 1e-5, 0)
    up = _lib.HdlaUpDims(rows, d, D, y.shape[1], cols["f"], cols["g"]) if T == 1 else None
    nd = _lib.HdlaNormDims(rows, groups, d // groups, bf, _lib.dtype_code(torch.float32), gate_pos, (d // groups) ** .5, 1e-5)
    o, n, ht = torch.empty(rows, d, device=DEV, dtype=torch.bfloat16), torch.empty(rows, d, device=DEV, dtype=torch.bfloat16), torch.empty_like(h0)
    g = torch.empty_like(gate) if T == 1 else gate
    here = groups == H
    if later:
        gated, eye = torch.empty(rows * (d + H), device=DEV), torch.eye(d, device=DEV).bfloat16()
        assert lib.hdla_layer_step(ref(pre), ref(up) if up else None, ref(nd), T, P(y), P(wf) if up else None, P(wg) if up else None,
                                   None if up else P(log_f), P(g), None, P(h0), None, P(gated), P(ht), st) == 0
        assert lib.hdla_rows_gemm_norm(rows, d, d, P(gated), H, ref(nd), P(w), P(eye), d, P(n), d, st) == 0
        return n, ht
    assert lib.hdla_layer_step(ref(pre), ref(up) if up else None, ref(nd) if here else None, T, P(y), P(wf) if up else None, P(wg) if up else None,
                               None if up else P(log_f), P(g), P(w) if here else None, P(h0), P(o), None, P(ht), st) == 0
    if here:
        return o, ht
    assert lib.hdla_normalize_fwd(ref(nd), P(o), P(w), P(g), P(n), st) == 0
    return n, ht


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N,T,H,norm_q,norm_v,gate_pos,all_channels", [(1, 1, 2, True, False, 1, False), (5, 1, 4, False, True, 2, True), (3, 2, 3, True, True, 2, False),
                                                                      (2, 8, 4, True, False, 1, True)])
def test_layer_step_against_float64(D, N, T, H, norm_q, norm_v, gate_pos, all_channels):
    ops, groups = _operands(50 + T, N, T, H, D), 1 if all_channels else H
    cols, y, wf, wg, w, h0, log_f, gate = ops
    more = {} if T == 1 else dict(log_f=log_f, gate=gate)
    o_r, ht_r = _exact(y.cpu(), wf.cpu(), wg.cpu(), w.cpu(), h0.cpu(), N, T, H, D, cols, norm_q, norm_v, gate_pos, groups, **{k: t.cpu() for k, t in more.items()})
    # On the way to o: q, k, v, beta, f, its logarithm, the gate, the two rank terms, o and the result are rounded to 8 bits, 2^-9 / sqrt(3) of
    # each in the mean: sqrt(11) of that; the state sees the first nine.  Twice it for sums in which parts of the terms cancel
    rms = 2 ** -9 / 3 ** .5
    for later in ([False, True] if all_channels else [False]):
        o, ht = _step(*ops, N, T, H, D, norm_q, norm_v, gate_pos, groups, later)
        assert _rel(o.view(N, T, -1).cpu(), o_r) <= 2 * 11 ** .5 * rms and _rel(ht.cpu(), ht_r) <= 2 * 3 * rms


LOWEST = -3.3895313892515355e38                              # of bf16


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [1, 3])
@pytest.mark.parametrize("norm", ["head", "all channels", "later"])
@pytest.mark.parametrize("where,value", [("q", float("nan")), ("k", float("nan")), ("v", float("nan")), ("b", float("nan")), ("f", float("nan")), ("g", float("nan")),
                                         ("S", float("nan")), ("v", float("inf")), ("S", float("inf")), ("S", -float("inf")), ("b", float("inf")), ("b", -float("inf")),
                                         ("b", LOWEST), ("q", LOWEST), ("k", LOWEST), ("f", LOWEST), ("g", LOWEST), ("g", float("inf"))])
def test_layer_step_on_values_that_are_none(D, T, norm, where, value):
    """A NaN, an infinity or the lowest number in one head (or one token's inner activations) of one sequence: what it reaches in float64
    arithmetic is what it reaches here, and nothing else; the other sequences keep their bits."""
    N, H = 3, 4
    groups, later = H if norm == "head" else 1, norm == "later"
    cols, y, wf, wg, w, h0, log_f, gate = _operands(70, N, T, H, D)
    clean = _step(cols, y, wf, wg, w, h0, log_f, gate, N, T, H, D, True, False, 1, groups, later)
    row = T                                                  # the first token of the second sequence
    if where == "S":
        h0[1, 2, 5, 7] = value
    elif T > 1 and where in "fg":                            # formed before this launch
        (log_f if where == "f" else gate)[row, 2 * D + 9] = value
    else:
        y[row, cols[where] + (2 if where == "b" else 9 if where in "fg" else 2 * D + 9)] = value
    o, ht = _step(cols, y, wf, wg, w, h0, log_f, gate, N, T, H, D, True, False, 1, groups, later)
    more = {} if T == 1 else dict(log_f=log_f.cpu(), gate=gate.cpu())
    o_r, ht_r = _exact(y.cpu(), wf.cpu(), wg.cpu(), w.cpu(), h0.cpu(), N, T, H, D, cols, True, False, 1, groups, **more)
    if later:
        o_r = o_r @ torch.eye(H * D, dtype=torch.float64)
    o, o_0 = (t.view(N, T, -1).cpu() for t in (o, clean[0]))
    for other in (0, 2):
        assert torch.equal(o[other], o_0[other]) and torch.equal(ht[other], clean[1][other])
    for got, want in ((o[1], o_r[1]), (ht[1].cpu(), ht_r[1])):
        ok = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), ok)
        assert not ok.any() or _rel(got[ok], want[ok]) <= 2e-2
