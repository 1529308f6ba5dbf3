"""The concatenated projection weight that HDLA_Custom keeps in evaluation mode: calls on other streams than the one that forms
it, and captured graphs that read it."""
import copy
import io

import pytest
import torch

from hdla_hip.layer import HDLA_Custom

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(common, **kw):
    torch.manual_seed(3)
    m = HDLA_Custom(256, 4, token_mixer_init_type=2, rescale_type=0, **kw).to(DEV).bfloat16().eval()
    m._common = common and m._common
    return m


def _x(seed, B=3):
    return torch.randn(B, 1, 256, generator=torch.Generator().manual_seed(seed)).bfloat16().to(DEV)


def _held(m):
    """The kept weight, wherever it is."""
    return m._native_cache[1] if m._native_cache[1] is not None else m._kept.w


def _junk(n=16):
    """Fills what the allocator would hand out next."""
    return [torch.full((1 << k,), float("nan"), device=DEV, dtype=torch.bfloat16) for k in range(10, 21) for _ in range(n)]


def _capture(m, x):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = m(x)[0]
    return g, y


both = pytest.mark.parametrize("common", [True, False])           # one native call, the steps


@both
def test_a_second_stream_waits_for_the_weight(common):
    m, x = _layer(common), _x(1)
    with torch.no_grad():
        ref = m(x)[0]
        m.reset_cache()
        a, b = torch.cuda.Stream(), torch.cuda.Stream()
        for s in (a, b):
            s.wait_stream(torch.cuda.current_stream())
        for r in range(3):
            with torch.cuda.stream(a):
                torch.cuda._sleep(20_000_000)                     # the weight is formed behind this
                m(x)
            with torch.cuda.stream(b):
                y = m(x)[0]
            torch.cuda.synchronize()
            assert torch.equal(y, ref), r
            m.reset_cache()


@both
def test_the_weight_outlives_the_calls_of_other_streams(common):
    m, x = _layer(common), _x(1)
    with torch.no_grad():
        ref = m(x)[0]
        torch.cuda.synchronize()
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            torch.cuda._sleep(20_000_000)
            y = m(x)[0]                                           # reads the weight of the default stream
        m.reset_cache()
        junk = _junk()                                            # on the default stream: nothing to wait for
        torch.cuda.synchronize()
        assert torch.equal(y, ref) and junk


@both
def test_what_a_captured_graph_reads_stays(common):
    m, x = _layer(common), _x(1)
    with torch.no_grad():
        m(x)
        g, y = _capture(m, x)
        at = _held(m).data_ptr()
        for i, change in enumerate([m.eval, lambda: m.train().eval(), lambda: m.to(DEV),
                                    lambda: m.load_state_dict({k: v.clone() for k, v in m.state_dict().items()}),
                                    lambda: m.q_proj.weight.mul_(0.5), lambda: m.v_proj.weight.data.mul_(0.5)]):
            change()
            if i == 5:
                m.eval()                                          # (an untracked write)
            junk = _junk()
            x.copy_(_x(10 + i))
            if i < 4:                                             # no parameter has another value: replays go on as they are
                g.replay()
                torch.cuda.synchronize()
                first = y.clone()
            want = m(x)[0]                                        # forms it anew, in its place
            assert _held(m).data_ptr() == at, i
            assert i >= 4 or torch.equal(first, want), i
            for _ in range(2):
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, want), i
            del junk
            # and a graph captured from here on reads it too
            g2, y2 = _capture(m, x)
            g2.replay()
            torch.cuda.synchronize()
            assert torch.equal(y2, want) and _held(m).data_ptr() == at
        del g, g2
        m.reset_cache()
        assert torch.equal(m(x)[0], want)


@both
def test_a_capture_takes_no_weight_that_is_not_there(common):
    """Formed on a stream that is still busy, or out of date: the graph forms its own."""
    m, x = _layer(common), _x(1)
    with torch.no_grad():
        ref, side = m(x)[0], torch.cuda.Stream()
        torch.cuda.synchronize()
        for stale in (False, True):
            m.reset_cache()
            if stale:
                m(x)
                _capture(m, x)
                m.eval()
            else:
                with torch.cuda.stream(side):
                    m(x)                                          # (complete or not: either is right)
            g, y = _capture(m, x)
            m.reset_cache()
            if stale:
                junk = _junk()
            for _ in range(2):
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, ref)


@both
def test_memory_is_given_back(common):
    m, x = _layer(common), _x(1)
    with torch.no_grad():
        at = torch.cuda.memory_allocated()
        m(x)
        assert torch.cuda.memory_allocated() > at
        m.train()
        assert torch.cuda.memory_allocated() == at
        m.eval()
        m(x)
        g, y = _capture(m, x)
        w = _held(m)
        m.train()
        assert _held(m) is w
        del g, y, w
        m.reset_cache()
        assert m._native_cache == [None] * 4 and getattr(m, "_kept", None) is None


@both
@pytest.mark.parametrize("bias", [False, True])
def test_copies_form_their_own(common, bias):
    m, x = _layer(common, bias=bias), _x(1)
    with torch.no_grad():
        ref = m(x)[0]
        g, y = _capture(m, x)
        buf = io.BytesIO()
        torch.save(m, buf)
        buf.seek(0)
        for other in (copy.deepcopy(m), torch.load(buf, weights_only=False)):       # written right here
            assert other._native_cache == [None] * 4 and "_kept" not in other.__dict__
            assert torch.equal(other(x)[0], ref)
            other.q_proj.weight.mul_(2.0)
            other(x)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
