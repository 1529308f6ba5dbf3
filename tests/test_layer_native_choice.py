"""When HDLA_Custom runs as one native call: not where something that the call would pass by has been replaced, overridden or
hooked.  The native function is a recorder here, so this runs without a GPU."""
import pytest
import torch
import torch.nn as nn

from hdla_hip import layer as L


class _Recorder:
    def __init__(self):
        self.calls = []

    def layer(self, *args):
        self.calls.append(args)
        return "output", "state"


@pytest.fixture
def native(monkeypatch):
    r = _Recorder()
    monkeypatch.setattr(L._lib, "native", lambda: r)
    return r


def _layer(cls=L.HDLA_Custom, **kw):
    return cls(128, 2, token_mixer_init_type=2, rescale_type=0, **kw)


def _taken(m, native):
    n = len(native.calls)
    out = m._forward_native(torch.zeros(1, 4, 128), None, False)
    assert (out is not None) == (len(native.calls) > n)
    return out is not None


class _Plain(L.HDLA_Custom):
    def extra_repr(self):
        return "another layer"


class _OwnProject(L.HDLA_Custom):
    def project(self, *args, **kw):
        return super().project(*args, **kw)


class _OwnUp(L.HDLA_Custom):
    def _up(self, lin, x0):
        return lin(x0)


@pytest.mark.parametrize("cls,kw,want", [(L.HDLA_Custom, {}, True), (L.HDLA_Custom, {"token_mixer_norm_type": "grouprmsnorm"}, True),
                                         (_Plain, {}, True), (_OwnProject, {}, False), (_OwnUp, {}, False)])
def test_classes(cls, kw, want, native):
    assert _taken(_layer(cls, **kw), native) is want


@pytest.mark.parametrize("which", ["norm", "o_proj", "q_proj", "f_proj.1"])
@pytest.mark.parametrize("how", ["forward", "forward_hook", "forward_pre_hook", "full_backward_hook", "full_backward_pre_hook", "weight", "bias"])
def test_submodules(which, how, native):
    m = _layer()
    assert _taken(m, native)
    s = m.get_submodule(which)
    if how == "forward":
        old = s.forward
        s.forward = lambda *a: 2 * old(*a)
    elif how == "weight":                                          # no parameter any more
        w = s.weight.detach()
        del s.weight
        s.weight = w
    elif how == "bias":
        s.register_parameter("bias", nn.Parameter(torch.zeros(128)))
    else:
        getattr(s, "register_" + how)(lambda *a: None)
    assert not _taken(m, native)


@pytest.mark.parametrize("how", ["forward_hook", "forward_pre_hook", "full_backward_hook", "full_backward_pre_hook"])
def test_hooks_on_all_modules(how, native):
    m = _layer()
    h = getattr(nn.modules.module, "register_module_" + how)(lambda *a: None)
    try:
        assert not _taken(m, native)
    finally:
        h.remove()
    assert _taken(m, native)


@pytest.mark.parametrize("what", ["project", "_up", "use_beta", "use_output_gate", "use_offset", "num_blocks", "gate_act", "gate_pos", "norm",
                                  "no norm", "output_gate", "f_proj"])
def test_attributes_of_an_instance(what, native):
    m = _layer()
    if what in ("project", "_up"):
        setattr(m, what, lambda *a, **k: None)
    elif what in ("use_beta", "use_output_gate"):
        setattr(m, what, False)
    elif what in ("use_offset", "num_blocks"):
        setattr(m, what, 2)
    elif what in ("gate_act", "gate_pos"):
        setattr(m.norm, what, "other")
    elif what == "norm":
        m.norm = nn.RMSNorm(128)
    elif what == "no norm":
        m.norm = None
    else:
        setattr(m, what, nn.Sequential(*getattr(m, what), nn.Identity()))
    assert not _taken(m, native)


@pytest.mark.parametrize("cls,name", [(L.HDLA_Custom, "project"), (nn.Linear, "forward"), (L.RMSNormFusedGate, "forward"), (nn.Module, "__call__")])
def test_patched_classes(cls, name, native, monkeypatch):
    m = _layer()
    old = getattr(cls, name)
    monkeypatch.setattr(cls, name, lambda *a, **k: old(*a, **k))
    assert not _taken(m, native)


def test_the_scale_of_the_norm_is_its_own(native):
    for kw, c in (({}, 128 ** 0.5), ({"token_mixer_norm_type": "grouprmsnorm"}, 8.0)):
        m = _layer(**kw)
        assert _taken(m, native) and native.calls[-1][11] == c


def test_a_module_pickled_before_there_was_a_native_call(native):
    import io
    m = _layer()
    for n in ("_common", "_native_cache"):
        del m.__dict__[n]
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    old = torch.load(buf, weights_only=False)                      # written right here
    assert not old._common and old._native_cache is None
    with pytest.raises(AttributeError, match="normalize"):         # the steps (the recorder has nothing but the layer's call)
        old(torch.zeros(1, 4, 128))
    assert not native.calls
    old.eval()
    assert len(old._native_cache) == 4
