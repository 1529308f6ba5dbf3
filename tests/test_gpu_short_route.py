"""bf16, K = V = 64, few short sequences: the classic kernels are the library's choice there.  Where the line lies (on the CPU),
and that what goes over it comes out as on the fused route."""
import pytest
import torch

from hdla_hip import _lib, chunk_hdla_delta_rule, chunk_hrdplr_delta_rule
from hdla_hip.synthetic import make_inputs
from oracle import hrdplr_oracle as O

DEV = "cuda"


def _record(B, T, H, N=None, cu=None, **kw):
    import ctypes
    d = _lib.make_dims(B, T, H, 64, 64, 2, N or B, torch.bfloat16, torch.bfloat16, 1.0, None, **kw)
    if cu:
        d.cu_seqlens = 256                                # never read on the host
    return _lib.load().hdla_record_bytes(ctypes.byref(d))


@pytest.mark.parametrize("T,lanes,short", [(80, 2, False), (96, 2, True), (496, 2, True), (512, 2, False), (256, 64, True), (256, 65, False)])
def test_where_the_line_lies(T, lanes, short):
    assert (_record(1, T, lanes) == 0) == short
    assert _record(1, T, lanes, route=_lib.ROUTE_FUSED) > 0 and _record(1, T, lanes, segments=2) > 0
    # packed: the average length counts
    assert (_record(1, 3 * T, lanes, N=3, cu=True) == 0) == (short and 3 * lanes <= 64)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("gk_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,H,cu,states,gk_div", [
    (1, 81, 2, None, True, 2.0), (2, 129, 3, None, False, 8.0), (1, 300, 1, (0, 37, 37, 200, 300), True, 8.0), (1, 495, 5, None, True, 0.05),
    (4, 240, 16, None, False, 16.0)])
def test_the_same_results_as_on_the_fused_route(form, gk_dtype, B, T, H, cu, states, gk_div, monkeypatch):
    inp = make_inputs(900 + T, B, T, H, 64, 64, gk_div=gk_div, n_states=B if cu is None else len(cu) - 1)
    table = None if cu is None else torch.tensor(cu)
    k = torch.nn.functional.normalize(inp.k, dim=-1)
    beta = 2.0 * torch.rand(B, T, H, 1, generator=torch.Generator().manual_seed(5))
    mid = [inp.a, inp.b] if form == "ab" else [beta]
    leaves = [t.bfloat16().to(DEV).requires_grad_() for t in [inp.q, k, inp.v, *mid]] + [inp.gk.to(gk_dtype).to(DEV).requires_grad_()]
    if states:
        leaves.append(inp.h0.to(DEV).requires_grad_())
    do, dht = inp.do.bfloat16().to(DEV), inp.dht.to(DEV)

    def run():
        h0 = leaves[-1] if states else None
        if form == "ab":
            o, ht = chunk_hrdplr_delta_rule(*leaves[:6], 2, scale=0.7, initial_state=h0, output_final_state=True, cu_seqlens=table)
        else:
            o, ht = chunk_hdla_delta_rule(*leaves[:5], scale=0.7, initial_state=h0, output_final_state=True, cu_seqlens=table)
        return [o.detach(), ht.detach(), *torch.autograd.grad([o, ht], leaves, [do, dht])]

    got = run()
    monkeypatch.setenv("HDLA_HIP_ROUTE", "fused")
    for i, (x, y) in enumerate(zip(got, run())):
        assert x.dtype == y.dtype and torch.isfinite(x.float()).all(), i
        # both are within 5e-3 (outputs) and 1e-2 (gradients) of exact arithmetic, and share most of their roundings
        assert O.rel_l2(x, y) <= 6e-3, (i, O.rel_l2(x, y))


@pytest.mark.gpu
@pytest.mark.parametrize("B,H", [(1, 3), (4, 16)])
@pytest.mark.parametrize("T,route", [(16, "fused"), (33, "fused"), (80, "fused"), (240, "fused"), (241, "classic"), (496, "classic"), (497, "fused")])
def test_the_forward_pass_alone(B, H, T, route, monkeypatch):
    """Which route a forward pass is on shows in its bits; below 16 chunks they are also those of the prompt in pieces."""
    inp = make_inputs(970 + T, B, T, H, 64, 64, gk_div=4.0)
    leaves = [t.bfloat16().to(DEV) for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)]

    def run(h0, first=0, last=T):
        part = [t[:, first * (t.shape[1] // T):last * (t.shape[1] // T)].contiguous() for t in leaves]      # (a, b: two rows a token)
        return chunk_hrdplr_delta_rule(*part, 2, scale=0.7, initial_state=h0, output_final_state=True)

    with torch.no_grad():
        o, ht = run(inp.h0.to(DEV))
        if 16 < T <= 240:
            o_1, h = run(inp.h0.to(DEV), 0, 16)
            o_2, h = run(h, 16)
            assert torch.equal(o, torch.cat([o_1, o_2], 1)) and torch.equal(ht, h)
        monkeypatch.setenv("HDLA_HIP_ROUTE", route)
        o_r, ht_r = run(inp.h0.to(DEV))
    assert torch.equal(o, o_r) and torch.equal(ht, ht_r)
