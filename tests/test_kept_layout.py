"""What a call holds from forward to backward holds nothing that no kernel reads, but u for whoever names the classic route: behind everything else."""
import ctypes

import pytest
import torch

import gpu_util as G
from hdla_hip import _lib
from hdla_hip.synthetic import make_inputs
from oracle import chunk_stages as CS
from oracle import hrdplr_oracle as O

DEV = "cuda"
SHAPES = [(64, 64), (128, 128), (64, 128), (128, 64)]


def _dims(B, T, H, K, V, route, gk=torch.bfloat16, segments=0):
    return _lib.make_dims(B, T, H, K, V, 2, B, torch.bfloat16, gk, 0.7, None, route=route, segments=segments)


def _size(d, pass_=_lib.PASS_FWD_KEEP):
    return _lib.load().hdla_workspace_bytes(ctypes.byref(d), pass_)


@pytest.mark.parametrize("K,V", SHAPES)
@pytest.mark.parametrize("T,H", [(16, 1), (100, 3), (1537, 16)])
def test_u_is_kept_beside_fp32_decays_only(T, H, K, V):
    """With decays of the inputs' 16 bits the scans and chunk_grad form u themselves."""
    slots, up = H * 2 * -(-T // 16), lambda n: -(-n // 256) * 256
    for route in (_lib.ROUTE_AUTO, _lib.ROUTE_PLAIN):
        narrow, wide = (_dims(2, T, H, K, V, route, gk) for gk in (torch.bfloat16, torch.float32))
        assert _size(wide) - _size(narrow) == up(slots * 2 * V * 16 * 2)
        assert _lib.workspace_layout(wide, 2)["UT"] > 0 == _lib.workspace_layout(narrow, 2)["UT"]
    plain, named = (_lib.workspace_layout(_dims(2, T, H, K, V, r), 2) for r in (_lib.ROUTE_PLAIN, _lib.ROUTE_CLASSIC))
    assert named["UT"] == plain["total"] and named["total"] - plain["total"] == up(slots * 2 * V * 16 * 2)
    assert all(named[n] == plain[n] for n in plain if n not in ("UT", "total"))
    # with segments, of which the classic route has none
    assert _lib.workspace_layout(_dims(2, T, H, K, V, _lib.ROUTE_AUTO, segments=4), 2)["UT"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("K,V", SHAPES)
def test_kept_on_one_route_and_read_on_the_other(K, V):
    B, T, H = 2, 90, 3
    inp = make_inputs(17, B, T, H, K, V, gk_div=2.0)
    x = [t.bfloat16().to(DEV) for t in (inp.q, inp.k, inp.v, inp.a, inp.b, inp.gk)]
    h0, do, dht, P = inp.h0.to(DEV), inp.do.bfloat16().to(DEV), inp.dht.to(DEV), _lib.ptr
    lib, stream = _lib.load(), _lib.current_stream(DEV)
    results, kept = [], {}
    for fwd in (_lib.ROUTE_PLAIN, _lib.ROUTE_CLASSIC):
        d = _dims(B, T, H, K, V, fwd)
        kept[fwd] = torch.zeros(_size(d), dtype=torch.uint8, device=DEV)
        o, ht = torch.empty_like(x[2]), torch.empty_like(h0)
        assert lib.hdla_chunk_fwd_keep(ctypes.byref(d), *map(P, x[:5]), None, P(x[5]), P(h0), P(o), P(ht), P(kept[fwd]), kept[fwd].numel(), stream) == 0
        for bwd in (_lib.ROUTE_PLAIN, _lib.ROUTE_CLASSIC):
            d = _dims(B, T, H, K, V, bwd)
            ws = torch.empty(_size(d, _lib.PASS_BWD_KEPT), dtype=torch.uint8, device=DEV)
            g = [torch.empty_like(t) for t in x[:5]] + [None, torch.empty_like(x[5]), torch.empty_like(h0)]
            assert lib.hdla_chunk_bwd_kept(ctypes.byref(d), *map(P, x[:5]), None, P(x[5]), P(h0), P(do), P(dht), *map(P, g), P(kept[fwd]), kept[fwd].numel(),
                                           P(ws), ws.numel(), stream) == 0
            results.append([o, ht] + [t for t in g if t is not None])
    torch.cuda.synchronize()
    for r in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(r, results[0]))
    # u in the buffer that the classic route was named for, in the tiles of hdla_ws_layout
    L = _lib.workspace_layout(_dims(B, T, H, K, V, _lib.ROUTE_CLASSIC), 2)
    got = G.cat_tiles(G.pair_tiles(kept[_lib.ROUTE_CLASSIC], L["UT"], torch.bfloat16, H, L["nch"], V // 16, 2).transpose(2, 3), 3, transpose=True)
    u = CS.forward(*(t.cpu().double() for t in x), 0.7, inp.h0.double())[2]["u"]
    want = u.permute(1, 0, 2, *range(3, u.dim())).reshape(H, L["nch"], *u.shape[3:])
    assert O.rel_l2(got, want) <= 1e-2
