"""The chunk table of packed batches around the number of sequences up to which it is made in registers, one sequence a lane: by prep_kernel's last
workgroups (classic route) or by a launch of its own (fused route)."""
import ctypes
import random

import pytest
import torch

from hdla_hip import _lib
from hdla_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _table(T, cu):
    """Chunk offsets, each chunk's sequence and the sequences from the one with the most chunks down, ties as they come."""
    bounds = [(min(max(s, 0), T), min(max(e, min(max(s, 0), T)), T)) for s, e in zip(cu, cu[1:])]
    counts = [-(-(e - s) // 16) for s, e in bounds]
    off = [sum(counts[:n]) for n in range(len(counts) + 1)]
    return off, [n for n, c in enumerate(counts) for _ in range(c)], sorted(range(len(counts)), key=lambda n: -counts[n])


@pytest.mark.parametrize("route,K,V", [(_lib.ROUTE_CLASSIC, 64, 64), (_lib.ROUTE_CLASSIC, 128, 64), (_lib.ROUTE_CLASSIC, 128, 128), (_lib.ROUTE_FUSED, 64, 64)])
@pytest.mark.parametrize("N", [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 300])
@pytest.mark.parametrize("kind", ["ragged", "one long", "outside"])
def test_the_table(route, K, V, N, kind):
    rng = random.Random(100 * N + K)
    lens = [rng.choice([0, 1, 15, 16, 17, 33, 48]) for _ in range(N)]
    if kind == "one long":
        lens[rng.randrange(N)] = 3000                        # more chunks than a workgroup has threads
    lens[N // 2] = max(lens[N // 2], 5)
    cu = [sum(lens[:n]) for n in range(N + 1)]
    T = cu[-1]
    if kind == "outside":                                    # entries outside [0, T]
        cu[0], cu[-1] = -7, T + 40
    H = 3
    x = make_inputs(11, 1, T, H, K, V, n_states=N)
    t = [getattr(x, n).bfloat16().to(DEV) for n in ("q", "k", "v", "a", "b", "gk")]
    table = torch.tensor(cu, device=DEV)
    dims = _lib.make_dims(1, T, H, K, V, 2, N, torch.bfloat16, torch.bfloat16, 1.0, table, route=route)
    lib, P = _lib.load(), _lib.ptr
    o = torch.empty_like(t[2])
    ws = _lib.workspace(dims, 0, DEV)
    ws.zero_()
    _lib.check(lib.hdla_chunk_fwd(ctypes.byref(dims), *[P(a) for a in t], None, P(o), None, P(ws), ws.numel(), _lib.current_stream(torch.device(DEV))), "fwd")
    at = _lib.workspace_layout(dims, 0)
    ints = lambda first, n: ws[first:first + 4 * n].view(torch.int32).cpu()
    off, seq, order = _table(T, cu)
    assert ints(at["CHUNK_OFF"], N + 1).tolist() == off
    assert ints(at["CHUNK_SEQ"], len(seq)).tolist() == seq
    assert (ints(at["CHUNK_OFF"] + 4 * (N + 1), N) & 0x0FFFFFFF).tolist() == order
