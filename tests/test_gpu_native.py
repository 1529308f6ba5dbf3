"""The operators' native host path (csrc/native.cpp): what it takes gives the bits of the Python autograd functions it
stands in front of, and what is not its case it leaves alone."""
import pytest
import torch

from hdla_hip import (ChunkDPLRDeltaRuleFunction, ChunkHDLAFunction, _lib, chunk_hdla_delta_rule, chunk_hrdplr_delta_rule,
                      fused_recurrent_dplr_delta_rule)
from hdla_hip.synthetic import make_inputs

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,K,V,cu,state", [(1, 64, 64, None, True), (40, 64, 64, None, False), (33, 128, 64, [0, 5, 5, 33], True)])
def test_chunked_operators_against_the_python_functions(form, dtype, T, K, V, cu, state):
    x = make_inputs(41, 1, T, 2, K, V, n_states=None if cu is None else len(cu) - 1)
    beta = 2 * torch.rand(1, T, 2, 1, generator=torch.Generator().manual_seed(1))
    names = (x.q, x.k, x.v, x.a, x.b, x.gk) if form == "ab" else (x.q, x.k, x.v, beta, x.gk)
    # q as a strided view: the native path makes it contiguous itself
    leaves = [t.to(dtype).to(DEV) for t in names]
    leaves[0] = torch.stack([leaves[0], leaves[0]], dim=-1)[..., 0]
    leaves = [t.detach().requires_grad_() for t in leaves]
    h0 = x.h0.to(DEV).requires_grad_() if state else None
    cu = None if cu is None else torch.tensor(cu, device=DEV)
    fn, op, pos = ((ChunkDPLRDeltaRuleFunction, chunk_hrdplr_delta_rule, (2,)) if form == "ab"
                   else (ChunkHDLAFunction, chunk_hdla_delta_rule, ()))
    args = (0.5, h0, state) + ((2, False, 16, cu, False) if form == "ab" else (cu, False))
    if form == "beta":
        leaves_py = leaves[:3] + [leaves[3].reshape(1, T, 2)] + leaves[4:]
    else:
        leaves_py = leaves
    ref = fn.apply(*leaves_py, *args)
    got = op(*leaves, *pos, scale=0.5, initial_state=h0, output_final_state=state, cu_seqlens=cu, keep_forward=False)
    gos = [x.do.to(dtype).to(DEV)] + ([x.dht.to(DEV)] if state else [])
    wrt = leaves + ([h0] if state else [])
    g_ref = torch.autograd.grad([t for t in ref if t is not None], wrt, gos)
    g_got = torch.autograd.grad([t for t in got if t is not None], wrt, gos)
    for a, b in zip(list(ref) + list(g_ref), list(got) + list(g_got)):
        assert (a is None and b is None) or torch.equal(a, b)


@pytest.mark.gpu
def test_outputs_that_no_loss_uses_and_calls_that_are_left_to_python():
    x = make_inputs(42, 1, 20, 2, 64, 64)
    leaves = [t.bfloat16().to(DEV).requires_grad_() for t in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    o, ht = chunk_hrdplr_delta_rule(*leaves, 2, output_final_state=True)
    only_ht = torch.autograd.grad(ht, leaves, x.dht.to(DEV))                   # no gradient of o: taken as zeros
    assert all(torch.isfinite(g.float()).all() for g in only_ht) and float(only_ht[1].float().abs().sum()) > 0
    n = _lib.native()
    t = [y.detach() for y in leaves]
    assert n.recurrent(*leaves, 2, None, None, False, False, None, False) is None      # gradients wanted
    assert n.recurrent(*t, 1, None, None, False, False, None, False) is None           # a and b of one rank
    assert n.recurrent(*[y.half() for y in t], 2, None, None, False, False, None, False) is None
    assert n.chunk(*t, 2, None, x.h0, False, False, 16, None, None) is None            # state on the CPU
    assert n.chunk(*t, 2, None, None, False, False, 16, None, True) is None            # kept forward pass
    assert torch.equal(fused_recurrent_dplr_delta_rule(*t, 2)[0], n.recurrent(*t, 2, None, None, False, False, None, False)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,d,H,kw", [
    (1, 1023, 256, 4, {}),                                          # rows of y padded to 16 bytes only (H = 4: not by themselves)
    (2, 512, 256, 4, {"gate_pos": "post", "norm_q": True}),         # from 1024 rows on: padded to whole GEMM tiles
    (4, 2048, 256, 2, {"token_mixer_norm_type": "grouprmsnorm"}),   # the output projection's weight gradient in four row ranges
])
def test_layer_as_one_call_against_its_steps(B, T, d, H, kw):
    """The layer's one native call against the same module run step by step (_common switched off), training and decode.
    The two differ where the steps round to bf16 in between (H = 4: the elementwise stage in torch's operators)."""
    from hdla_hip.layer import HDLA_Custom, RecurrentCache
    from oracle import hrdplr_oracle as O
    torch.manual_seed(3)
    m = HDLA_Custom(d, H, token_mixer_init_type=2, rescale_type=0, **kw).to(DEV).bfloat16().train()
    g = torch.Generator().manual_seed(4)
    x = torch.randn(B, T, d, generator=g).bfloat16().to(DEV).requires_grad_()
    do = torch.randn(B, T, d, generator=g).bfloat16().to(DEV)
    ps = list(m.parameters())
    res = []
    for common in (True, False):
        m._common = common
        y, _ = m(x)
        res.append([y.detach()] + list(torch.autograd.grad(y, [x] + ps, do)))
    assert res[0][0].grad_fn is None
    errs = [O.rel_l2(a, b) for a, b in zip(*res)]
    print([f"{e:.1e}" for e in errs], flush=True)
    assert errs[0] <= 1e-2 and max(errs) <= 2e-2
    m.eval()
    outs = []
    with torch.no_grad():
        for common in (True, False):
            m._common = common
            cache = RecurrentCache()
            _, cache = m(x[:, :20], past_key_values=cache, use_cache=True)
            y = [m(x[:, 20 + i:21 + i], past_key_values=cache, use_cache=True)[0] for i in range(2)]
            m.q_proj.weight.mul_(-1.0)                              # the kept concatenation has to notice
            y.append(m(x[:, 22:23], past_key_values=cache, use_cache=True)[0])
            m.q_proj.weight.mul_(-1.0)
            outs.append(y + [cache[0]["recurrent_state"][0]])
    for a, b in zip(*outs):
        assert O.rel_l2(a, b) <= 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 128])
def test_rows_of_no_sequence_are_zeros(K):
    """A table that comes unchecked from the device and leaves rows out (gaps at both ends and between, where it falls):
    outputs and gradients read zero there, and the covered rows are those of the same sequences by themselves."""
    T, H = 60, 2
    cu = torch.tensor([3, 20, 14, 14, 30, 41], device=DEV)          # sequences 3..20, 14..14, 14..30 (overlapping), 30..41
    x = make_inputs(43, 1, T, H, K, K, n_states=5)
    leaves = [t.bfloat16().to(DEV).requires_grad_() for t in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    junk = [torch.full((1 << 22,), float("nan"), device=DEV) for _ in range(8)]         # what recycled memory may hold
    del junk
    o, _ = chunk_hrdplr_delta_rule(*leaves, 2, cu_seqlens=cu)
    g = torch.autograd.grad(o, leaves, x.do.bfloat16().to(DEV))
    inside = torch.zeros(T, dtype=torch.bool, device=DEV)
    inside[3:41] = True
    for t in (o, *g):
        r = 2 if t.shape[1] == 2 * T else 1
        rows = inside.repeat_interleave(r)
        assert bool((t[0, ~rows] == 0).all()) and torch.isfinite(t.float()).all()
    alone, _ = chunk_hrdplr_delta_rule(*[t[:, 30 * (t.shape[1] // T):41 * (t.shape[1] // T)] for t in leaves], 2)
    assert torch.equal(alone, o[:, 30:41])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,K,V,segments", [(torch.bfloat16, 128, 128, 4), (torch.bfloat16, 128, 64, 7), (torch.bfloat16, 64, 128, 2),
                                                (torch.float32, 64, 64, 4), (torch.float32, 128, 128, 3), (torch.float32, 64, 128, 5)])
@pytest.mark.parametrize("T,cu", [(145, None), (150, [0, 33, 33, 40, 150])])
def test_time_segments_of_the_stand_alone_scans(dtype, K, V, segments, T, cu, monkeypatch):
    """The scans cut into time segments (ragged last chunks, segments without chunks, an empty sequence, segments longer and
    shorter than the scans' rings) against whole sequences."""
    from oracle import hrdplr_oracle as O
    x = make_inputs(44, 1, T, 2, K, V, gk_div=4.0, n_states=None if cu is None else len(cu) - 1)
    leaves = [t.to(dtype).to(DEV).requires_grad_() for t in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    h0 = x.h0.to(DEV).requires_grad_()
    cu = None if cu is None else torch.tensor(cu, device=DEV)
    res = []
    for n in (segments, 1):
        monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(n))
        o, ht = chunk_hrdplr_delta_rule(*leaves, 2, scale=0.7, initial_state=h0, output_final_state=True, cu_seqlens=cu)
        res.append([o.detach(), ht.detach()] + list(torch.autograd.grad([o, ht], leaves + [h0], [x.do.to(dtype).to(DEV), x.dht.to(DEV)])))
    errs = [O.rel_l2(a, b) for a, b in zip(*res)]
    print([f"{e:.1e}" for e in errs], flush=True)
    assert max(errs) <= (6e-3 if dtype == torch.bfloat16 else 3e-6)


@pytest.mark.gpu
def test_fp32_segments_are_as_precise_as_whole_sequences(monkeypatch):
    """Errors against float64 under slow decay, where the chained states carry everything.  The two share all roundings but those of
    the states entering the segments; over inputs like these their ratio is 1.0002 with a spread of 0.001 a run (chained in fp32 it
    was 1.010 to 1.016)."""
    from oracle import hrdplr_oracle as O
    x = make_inputs(45, 1, 1008, 4, 64, 64, gk_div=16.0)
    cpu = [t.double().requires_grad_() for t in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    o_ref, _ = O.chunk_naive(*cpu, 0.7, dtype=torch.float64)
    ref = [o_ref.detach(), *torch.autograd.grad(o_ref, cpu, x.do.double())]
    leaves = [t.float().to(DEV).requires_grad_() for t in (x.q, x.k, x.v, x.a, x.b, x.gk)]
    errs = []
    for n in (8, 1):
        monkeypatch.setenv("HDLA_HIP_SEGMENTS", str(n))
        o, _ = chunk_hrdplr_delta_rule(*leaves, 2, scale=0.7)
        got = [o.detach(), *torch.autograd.grad(o, leaves, x.do.float().to(DEV))]
        errs.append([O.rel_l2(a, b) for a, b in zip(got, ref)])
    print([f"{e:.4e} {e / f:.4f}" for e, f in zip(*errs)], flush=True)
    assert max(errs[1]) <= 1e-6
    assert all(e <= 1.005 * f for e, f in zip(*errs))


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["chunk", "recurrent", "norm", "layer"])
@pytest.mark.parametrize("transform", ["dual", "vmap"])
def test_forward_mode_and_transforms_are_refused(call, transform):
    """The operators have no forward-mode rule: a tangent on an input that needs no gradient is refused, not dropped."""
    import torch.autograd.forward_ad as fwad
    from hdla_hip.layer import HDLA_Custom
    from hdla_hip.normalize import normalize_fn
    g = torch.Generator(device="cuda").manual_seed(2)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    q, a = rn(2, 1, 32, 2, 64), rn(1, 64, 2, 64)
    layer = HDLA_Custom(256, 4, token_mixer_init_type=2, rescale_type=0).cuda().bfloat16().eval().requires_grad_(False)
    w = torch.ones(64, device="cuda")

    def run(x):
        if call == "chunk":
            return chunk_hrdplr_delta_rule(x, q[0], q[0], a, a, -q[0].abs(), 2, scale=1.0)[0]
        if call == "recurrent":
            return fused_recurrent_dplr_delta_rule(x, q[0], q[0], a, a, -q[0].abs(), 2, scale=1.0)[0]
        if call == "norm":
            return normalize_fn(x, w, gate=q[0], gate_pos="pre", c=8.0, eps=1e-5)
        return layer(x)[0]

    x = rn(2, 2, 32, 256) if call == "layer" else q
    run(x[0])                                                 # accepted as it is
    with pytest.raises((RuntimeError, NotImplementedError)):
        if transform == "vmap":
            torch.func.vmap(run)(x)
        else:
            with fwad.dual_level():
                run(fwad.make_dual(x[0], torch.ones_like(x[0])))
