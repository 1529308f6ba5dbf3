"""The operators under HIP graph capture: the library only launches kernels on the caller's stream (no allocation, no
memset, no synchronisation), so a captured call must replay to exactly what the eager call gives.  Every graph is
replayed several times on fresh input contents, with eager work and synchronisations in between, and every replay is
compared bit for bit with the eager result on the same inputs."""
import pytest
import torch

from hdla_hip import chunk_hdla_delta_rule, chunk_hrdplr_delta_rule, fused_recurrent_hdla_delta_rule, normalize_fn
from hdla_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _capture(fn, warmup=2):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(warmup):
            fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _replay_and_compare(g, static_in, static_out, eager, fresh, n=4):
    for i in range(n):
        new = fresh(i)
        for s, t in zip(static_in, new):
            s.copy_(t)
        g.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in static_out]
        ref = eager(*new)                                     # eager work between replays
        torch.cuda.synchronize()
        for a, b in zip(got, ref):
            assert torch.equal(a, b), f"replay {i} differs from the eager call"


def test_chunked_forward_and_backward_replay():
    B, T, H, K, V = 2, 200, 3, 64, 64
    def fresh(i):
        x = make_inputs(100 + i, B, T, H, K, V)
        return [t.bfloat16().to(DEV) for t in (x.q, x.k, x.v, x.a, x.b, x.gk)] + [x.h0.to(DEV), x.do.bfloat16().to(DEV), x.dht.to(DEV)]

    def run(q, k, v, a, b, gk, h0, do, dht):
        leaves = [t.detach().requires_grad_() for t in (q, k, v, a, b, gk, h0)]
        o, ht = chunk_hrdplr_delta_rule(*leaves[:6], 2, scale=1.0, initial_state=leaves[6], output_final_state=True)
        return [o.detach(), ht.detach()] + list(torch.autograd.grad([o, ht], leaves, [do, dht]))

    static_in = fresh(99)
    g, static_out = _capture(lambda: run(*static_in))
    _replay_and_compare(g, static_in, static_out, run, fresh)


def test_parameterised_operator_and_norm_replay():
    B, T, H, K, V = 1, 130, 4, 128, 128
    def fresh(i):
        x = make_inputs(200 + i, B, T, H, K, V)
        beta = 2 * torch.rand(B, T, H, 1, generator=torch.Generator().manual_seed(i))
        return [t.bfloat16().to(DEV) for t in (x.q, x.k, x.v, beta, x.gk, x.do)]

    w = torch.ones(H * V, device=DEV)

    def run(q, k, v, beta, lf, do):
        leaves = [t.detach().requires_grad_() for t in (q, k, v, beta, lf)]
        wl = w.detach().requires_grad_()
        o, _ = chunk_hdla_delta_rule(*leaves, scale=1.0)
        y = normalize_fn(o.flatten(2), wl, gate=leaves[2].flatten(2), c=(H * V) ** 0.5, eps=1e-5)
        return [y.detach()] + list(torch.autograd.grad(y, leaves + [wl], do.flatten(2)))

    static_in = fresh(99)
    g, static_out = _capture(lambda: run(*static_in))
    _replay_and_compare(g, static_in, static_out, run, fresh)


def test_decode_step_replay_carries_the_state():
    B, H, K, V = 8, 4, 128, 128
    def fresh(i):
        x = make_inputs(300 + i, B, 1, H, K, V)
        beta = 2 * torch.rand(B, 1, H, 1, generator=torch.Generator().manual_seed(i))
        return [t.bfloat16().to(DEV) for t in (x.q, x.k, x.v, beta, x.gk)]

    S = torch.zeros(B, H, K, V, device=DEV)                   # the graph updates its state in place

    def step(q, k, v, beta, lf):
        o, S_new = fused_recurrent_hdla_delta_rule(q, k, v, beta, lf, scale=1.0, initial_state=S, output_final_state=True)
        S.copy_(S_new)
        return [o]

    static_in = fresh(99)
    g, static_out = _capture(lambda: step(*static_in), warmup=1)
    S.zero_()
    S_ref = torch.zeros_like(S)
    for i in range(5):
        new = fresh(i)
        for s, t in zip(static_in, new):
            s.copy_(t)
        g.replay()
        torch.cuda.synchronize()
        o_ref, S_ref = fused_recurrent_hdla_delta_rule(*new, scale=1.0, initial_state=S_ref, output_final_state=True)
        assert torch.equal(static_out[0], o_ref) and torch.equal(S, S_ref), f"decode replay {i}"


def test_layer_decode_replay_between_long_prefills():
    """A captured decode step of the layer reads the concatenated weight that evaluation mode keeps: long calls in between, which
    use a padded one, must leave it where it is."""
    from hdla_hip.layer import HDLA_Custom, RecurrentCache
    torch.manual_seed(5)
    m = HDLA_Custom(256, 4, token_mixer_init_type=2, rescale_type=0).to(DEV).bfloat16().eval()
    x = torch.randn(3, 1, 256, device=DEV).bfloat16()
    prompt = torch.randn(1, 1100, 256, device=DEV).bfloat16()
    state = torch.randn(3, 4, 64, 64, device=DEV)

    def step(x, state):
        cache = RecurrentCache()
        cache.update(recurrent_state=[state])
        y, cache = m(x, past_key_values=cache, use_cache=True)
        return [y, cache[0]["recurrent_state"][0]]

    with torch.no_grad():
        g, static_out = _capture(lambda: step(x, state))
        for i in range(4):
            m(prompt, past_key_values=RecurrentCache(), use_cache=True)
            junk = [torch.full((1 << 20,), float("nan"), device=DEV) for _ in range(8)]
            x.copy_(torch.randn(3, 1, 256, generator=torch.Generator().manual_seed(i)))
            g.replay()
            torch.cuda.synchronize()
            got = [t.clone() for t in static_out]
            del junk
            assert all(torch.equal(a, b) for a, b in zip(got, step(x, state))), f"replay {i}"


@pytest.mark.parametrize("common", [True, False])                 # one native call, the steps
def test_layer_first_called_under_capture(common):
    """What evaluation mode keeps must not come from a capture: it is not there before the graph is replayed."""
    from hdla_hip.layer import HDLA_Custom
    torch.manual_seed(6)
    ms = [HDLA_Custom(256, 4, token_mixer_init_type=2, rescale_type=0).to(DEV).bfloat16().eval() for _ in range(2)]
    ms[1].load_state_dict(ms[0].state_dict())
    x = torch.randn(3, 1, 256, device=DEV).bfloat16()
    for m in ms:
        m._common = common
    with torch.no_grad():
        ref = ms[0](x)[0]
        g, out = _capture(lambda: ms[1](x)[0], warmup=0)
        assert torch.equal(ms[1](x)[0], ref)
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref) and torch.equal(ms[1](x)[0], ref)
