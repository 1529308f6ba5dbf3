"""Packed batches whose table leaves rows to no sequence (a batch padded at its end to a fixed length, for one): those rows of the
outputs and gradients are zeros, and clearing them costs what writing them costs."""
import ctypes

import pytest
import torch

from hdla_hip import _lib, chunk_hdla_delta_rule
from hdla_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype,gk_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("form", ["ab", "beta"])
@pytest.mark.parametrize("H,K,V", [(1, 64, 64), (3, 128, 64)])
@pytest.mark.parametrize("T,cu", [(1, [0, 0]), (33, [0, 20, 33]), (33, [5, 20, 31]), (33, [0, 32]), (600, [7, 7, 40, 300]), (600, [600, 600]),
                                  (600, [40, 100, 90, 600]), (60, [-4, 20, 99])])
def test_outputs_start_as_garbage(dtype, gk_dtype, form, H, K, V, T, cu):
    """Every entry of every output is written: zeros outside the sequences, finite values inside.  Tables: a partition, gaps at
    either end or both, nothing covered, one that decreases (everything is cleared first), entries outside [0, T]."""
    x = make_inputs(43, 1, T, H, K, V, n_states=len(cu) - 1)
    lib, P = _lib.load(), _lib.ptr
    t = {n: getattr(x, n).to(dtype).to(DEV) for n in ("q", "k", "v", "a", "b", "do")}
    t["gk"] = x.gk.to(gk_dtype).to(DEV)
    t["beta"] = torch.rand(1, T, H, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    a, b, bt = (t["a"], t["b"], None) if form == "ab" else (None, None, t["beta"])
    table = torch.tensor(cu, device=DEV)
    dims = _lib.make_dims(1, T, H, K, V, 2, len(cu) - 1, dtype, gk_dtype, 0.7, table)
    # outputs one row behind the front of NaN buffers that go on behind them: what lies around them must stay
    room, out = {}, {}
    for n in ("o", "q", "k", "v", "a", "b", "gk", "beta"):
        like = t["v"] if n == "o" else t[n]
        pad = 128
        room[n] = torch.full((like.numel() + 2 * pad,), float("nan"), dtype=like.dtype, device=DEV)
        out[n] = room[n][pad:pad + like.numel()].view(like.shape)
    s = _lib.current_stream(torch.device(DEV))
    ws = _lib.workspace(dims, 0, DEV)
    _lib.check(lib.hdla_chunk_fwd_b(ctypes.byref(dims), P(t["q"]), P(t["k"]), P(t["v"]), P(a), P(b), P(bt), P(t["gk"]), None, P(out["o"]), None,
                                    None, 0, P(ws), ws.numel(), s), "fwd")
    ws = _lib.workspace(dims, 1, DEV)
    ab = form == "ab"
    _lib.check(lib.hdla_chunk_bwd_b(ctypes.byref(dims), P(t["q"]), P(t["k"]), P(t["v"]), P(a), P(b), P(bt), P(t["gk"]), None, P(t["do"]), None,
                                    P(out["q"]), P(out["k"]), P(out["v"]), P(out["a"]) if ab else None, P(out["b"]) if ab else None,
                                    None if ab else P(out["beta"]), P(out["gk"]), None, None, 0, P(ws), ws.numel(), s), "bwd")
    torch.cuda.synchronize()
    inside = torch.zeros(T, dtype=torch.bool)
    for i, e in zip(cu, cu[1:]):
        inside[max(i, 0):max(min(e, T), 0)] = True
    inside = inside.to(DEV)
    for n in out:
        if n in (("beta",) if ab else ("a", "b")):
            continue
        y = out[n]
        rows = inside.repeat_interleave(y.shape[1] // T)
        assert bool((y[0, ~rows] == 0).all()), n
        assert bool(torch.isfinite(y.float()).all()), n
        assert bool(torch.isnan(room[n][:128]).all()) and bool(torch.isnan(room[n][-128:]).all()), n


def test_a_batch_padded_at_its_end_costs_what_a_full_one_does():
    """16384 tokens of 16 heads: 537 MB of outputs.  Written 2 bytes a lane by one workgroup they take 20 ms;
    the bound leaves room for them at a tenth of the rate a copy reaches."""
    T, H, K = 16384, 16, 128
    g = torch.Generator(device=DEV).manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    unit = lambda: torch.nn.functional.normalize(rn(1, T, H, K).float(), dim=-1).bfloat16()
    leaves = [x.requires_grad_() for x in (unit(), unit(), rn(1, T, H, K), 2 * torch.rand(1, T, H, 1, generator=g, device=DEV).bfloat16(),
                                           torch.nn.functional.logsigmoid(rn(1, T, H, K)) / 16)]
    do = rn(1, T, H, K)

    def once(cu):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        o, _ = chunk_hdla_delta_rule(*leaves, scale=1.0, cu_seqlens=cu)
        torch.autograd.grad(o, leaves, do)
        e[1].record()
        e[1].synchronize()
        return e[0].elapsed_time(e[1])

    tables = [torch.tensor([0, 2048, 6144, 10240, end], device=DEV) for end in (T, T - 200)]
    best = [min(once(cu) for _ in range(5)) for cu in tables]
    print(f"{best[0]:.3f} ms, padded {best[1]:.3f} ms", flush=True)
    assert best[1] <= best[0] + 1.2
