"""The HDLA token mixer built on this library's operators: the drop-in for ``HDLA_Custom``, HRDPLR/hdla_custom.py:45-350.

Same constructor arguments, parameter names (so a reference ``state_dict`` loads), forward signature and return value
``(output, past_key_values)``.  What runs on the GPU:

* projections: the BLAS library through torch, as in the reference (hdla_custom.py:206-213), but with everything
  that multiplies x gathered into one GEMM
* activations, head split, per-head l2 normalisation of q, k, v, beta and the log decay: two kernels each way
  (``hdla_hip.layer_pre``; hdla_custom.py:214-251) in the default configuration (silu activations, one block);
  otherwise, or with ``fuse_pre=False``, torch's elementwise operators and ``hdla_hip.normalize.l2_norm``
* the gated RMS norm after the operator: ``hdla_hip.normalize`` (hdla_custom.py:341-345)
* the recurrence: ``chunk_hdla_delta_rule`` / ``fused_recurrent_hdla_delta_rule``, which form a and b from
  (beta, k, log_f) inside the kernels; the reference calls ``parameterize_a_b`` first (hdla_custom.py:290, a function
  that as shipped returns nothing) and hands a, b to the plain operators (:296-323).  ``fuse_ab=False`` takes that
  route with the working helper.

Which operator runs: the reference uses the chunked one when training or when ``use_cache`` is set and the token-serial
one otherwise (hdla_custom.py:295,310); ``dispatch="reference"`` keeps that.  The default ``dispatch="auto"`` uses the
chunked operator when gradients are needed or the call carries more than 8 tokens and the token-serial one for shorter
calls (decode steps, short bursts), which is where each is the faster (at 8 tokens they take the same time from
B=1, H=16 to B=256, H=32; at 1 token the token-serial one is 1.5-2.3x faster, at 64 tokens the chunked one 3x); both
compute the same function.

``past_key_values`` is duck-typed on the three calls the reference makes (hdla_custom.py:254-257, 332-337):
``len(cache)``, ``cache[layer_idx]["recurrent_state"][0]``, ``cache.get_seq_length(layer_idx)`` and
``cache.update(recurrent_state=[S], layer_idx=i, offset=n)``; ``RecurrentCache`` below is a minimal one.
"""
import math
from typing import Callable, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib
from .chunk import chunk_hrdplr_delta_rule
from . import layer_pre as _pre
from .hdla import chunk_hdla_delta_rule, fused_recurrent_hdla_delta_rule, parameterize_a_b
from .normalize import GroupRMSNormFusedGate, RMSNormFusedGate, get_norm_fn, l2_norm
from .recurrent import fused_recurrent_dplr_delta_rule

EMBED_DIM_BASE = 256                 # HRDPLR/normalizations/normalization_utils.py:14
RECURRENT_BELOW = 9                  # dispatch="auto": calls shorter than this run token by token (measured crossover: 8)


def get_activation_fn(activation: str) -> Callable[[torch.Tensor], torch.Tensor]:
    """HRDPLR/activations.py:10-58."""
    table = {
        "gelu": F.gelu, "relu": F.relu, "elu": F.elu, "sigmoid": torch.sigmoid, "exp": torch.exp, "leak": F.leaky_relu,
        "relu2": lambda x: F.relu(x) ** 2, "1+elu": lambda x: 1 + F.elu(x), "2+elu": lambda x: 2 + F.elu(x),
        "swish": F.silu, "silu": F.silu, "softmax_1": lambda x: F.softmax(x, dim=-1),
        "softmax_2": lambda x: F.softmax(x, dim=-2),
    }
    return table.get(activation, lambda x: x)


class RecurrentCache:
    """The part of fla's ``Cache`` the layer touches: one state list and a token count per layer."""

    def __init__(self):
        self.states, self.seen = [], []

    def __len__(self):
        return len(self.states)

    def __getitem__(self, layer_idx):
        return self.states[layer_idx]

    def get_seq_length(self, layer_idx: int = 0) -> int:
        return self.seen[layer_idx] if layer_idx < len(self.seen) else 0

    def update(self, recurrent_state=None, layer_idx: int = 0, offset: int = 1, **kwargs):
        while len(self.states) <= layer_idx:
            self.states.append({"recurrent_state": [None]})
            self.seen.append(0)
        self.states[layer_idx] = {"recurrent_state": recurrent_state}
        self.seen[layer_idx] += offset
        return self.states[layer_idx]


class _Kept:
    """A concatenated weight (and bias) that evaluation mode keeps: what it was formed from, where, and whether a captured graph reads it."""

    def __init__(self, key, w, b, captured=False):
        self.key, self.w, self.b, self.captured = key, w, b, captured
        self.made = self.ready = None

    def formed_on(self, stream):
        self.made, self.ready = stream, torch.cuda.Event()
        self.ready.record(stream)
        self.used_on(stream)

    def used_on(self, stream):
        """Memory of another stream's is not given back before what is on this one has run."""
        for t in (self.w, self.b):
            if t is not None:
                t.record_stream(stream)

    def wait_for(self, stream, capturing) -> bool:
        """Makes `stream` wait for the weight.  Under capture it has to be there: what the replay waits for is not known here."""
        if self.ready is None or (stream == self.made and not capturing):
            return True
        if _lib.native().passed(self.ready.cuda_event):
            self.ready = None
        elif not capturing:
            stream.wait_event(self.ready)
        return self.ready is None or not capturing


class HDLA_Custom(nn.Module):
    """S[t] = (I - beta k k^T) Diag(f) (I - beta k k^T) S[t-1] + k v^T,  o[t] = S[t]^T q[t]   (hdla_custom.py:46-62,270-288)."""

    # what a module that was pickled whole before there was a native call does not bring along: it runs as steps
    _common, _native_cache = False, None

    def __init__(
        self,
        embed_dim: int,
        num_heads: int,
        bias: bool = False,
        layer_idx: int = 0,
        use_output_gate: bool = True,
        token_mixer_norm_type: str = "rmsnorm",
        q_activation: str = "silu",
        k_activation: str = "silu",
        v_activation: str = "silu",
        use_beta: bool = True,
        beta_activation: str = "neg",
        qkv_norm_type: int = 2,
        norm_q: bool = False,
        norm_v: bool = False,
        causal: bool = True,
        max_position_embeddings: int = 1024,
        token_mixer_init_type: int = 4,
        rescale_type: int = 2,
        num_hidden_layers: int = 12,
        init_std: float = 0.02,
        gain: float = 0.01,
        gate_act: str = "sigmoid",
        gate_pos: str = "pre",
        threshold: float = 0.99,
        use_offset: bool = False,
        num_blocks: int = 1,
        fuse_ab: bool = True,
        dispatch: str = "auto",
        fuse_pre: bool = True,
        **kwargs,
    ):
        super().__init__()
        assert causal, f"Only causal={causal} is supported"
        assert dispatch in ("auto", "reference")
        self.layer_idx, self.causal, self.use_output_gate = layer_idx, causal, use_output_gate
        self.q_proj = nn.Linear(embed_dim, embed_dim, bias=bias)
        self.k_proj = nn.Linear(embed_dim, embed_dim, bias=bias)
        self.v_proj = nn.Linear(embed_dim, embed_dim, bias=bias)
        self.head_dim = embed_dim // num_heads
        self.f_proj = nn.Sequential(nn.Linear(embed_dim, self.head_dim, bias=bias),
                                    nn.Linear(self.head_dim, embed_dim, bias=bias))
        self.use_beta = use_beta
        if use_beta:
            self.bet_proj = nn.Linear(embed_dim, num_heads, bias=bias)
        self.o_proj = nn.Linear(embed_dim, embed_dim, bias=bias)
        self.q_act, self.k_act, self.v_act = (get_activation_fn(a) for a in (q_activation, k_activation, v_activation))
        self.beta_activation = beta_activation
        norm_type = f"{token_mixer_norm_type}_fused_gate" if use_output_gate else token_mixer_norm_type
        self.norm = get_norm_fn(norm_type)(embed_dim, bias=bias, gate_act=gate_act, gate_pos=gate_pos,
                                           num_groups=num_heads)
        if use_output_gate:
            self.output_gate = nn.Sequential(nn.Linear(embed_dim, self.head_dim, bias=bias),
                                             nn.Linear(self.head_dim, embed_dim, bias=bias))
        self.embed_dim, self.num_heads = embed_dim, num_heads
        self.use_offset, self.threshold = use_offset, threshold
        self.qkv_norm_type, self.norm_q, self.norm_v = qkv_norm_type, norm_q, norm_v
        self.token_mixer_init_type, self.rescale_type = token_mixer_init_type, rescale_type
        self.num_hidden_layers, self.init_std, self.gain = num_hidden_layers, init_std, gain
        self.num_blocks = num_blocks
        self.fuse_ab, self.dispatch, self.fuse_pre = fuse_ab, dispatch, fuse_pre
        self._all_silu = all(a in ("silu", "swish") for a in (q_activation, k_activation, v_activation))
        # the form the native host path runs as one call, as far as the constructor decides it
        self._common = (self._all_silu and use_beta and use_output_gate and not bias and num_blocks == 1 and not use_offset
                        and gate_act == "sigmoid" and gate_pos in ("pre", "post"))
        self._native_cache = [None] * 4
        self._init_weights()

    # ---- initialisation: hdla_custom.py:159-187 and normalization_utils.py:115-211 (the branches a module of this
    # layer can reach: Linear weights, the decay offset, the rescaling of o_proj) ------------------------------------
    def _init_weights(self):
        self.setup_decay()
        self.apply(self._initialize_weights)

    def setup_decay(self):
        if not self.use_offset:
            return
        a = self.threshold                                   # sigmoid(offset) = threshold at f_proj(x) = 0
        offset = torch.ones(self.embed_dim) * math.log(a / (1 - a))
        if hasattr(self, "offset"):
            self.offset.data.copy_(offset)
        else:
            self.offset = nn.Parameter(offset, requires_grad=True)

    def _initialize_weights(self, module):
        if getattr(module, "_is_hf_initialized", False):
            return
        if self.token_mixer_init_type in (1, 2, 3, 4):
            gain = {1: 2 ** -2.5, 2: 2 ** -0.5, 3: self.init_std / ((self.embed_dim / EMBED_DIM_BASE) ** 0.5),
                    4: self.gain}[self.token_mixer_init_type]
            if isinstance(module, nn.Linear):
                nn.init.xavier_uniform_(module.weight, gain=gain)
                if module.bias is not None:
                    nn.init.zeros_(module.bias)
        for name, p in module.named_parameters():
            if name in ("o_proj.weight", "out_proj.weight"):
                with torch.no_grad():
                    if self.rescale_type == 1:
                        p /= math.sqrt(2 * self.num_hidden_layers)
                    elif self.rescale_type == 2:
                        p *= 0
        module._is_hf_initialized = True

    def extra_repr(self):
        return (f"embed_dim={self.embed_dim}, num_heads={self.num_heads}, num_blocks={self.num_blocks}, "
                f"fuse_ab={self.fuse_ab}, dispatch={self.dispatch}")

    def _gathered(self, heads):
        """Weights (and biases) of the projections of x, concatenated.  With gradients, or in training mode, the
        concatenation is rebuilt per call (and is part of the graph).  In evaluation mode without gradients it is built
        once and reused: it is rebuilt when a parameter is replaced or modified in place (tracked by its version
        counter), on ``.train()`` / ``.eval()``, ``.to()`` and ``load_state_dict``, and by ``reset_cache()`` -- which
        is what code that writes through ``param.data`` (untracked) has to call.

        Calls on another stream than the one that built it wait for it.  A captured graph that reads it keeps reading the same
        memory: rebuilt, by the next call outside a capture, it is rebuilt in its place, and only ``reset_cache()`` or the end of the module
        gives it back."""
        ps = [m.weight for m in heads] + ([m.bias for m in heads] if heads[0].bias is not None else [])
        if self.training or (torch.is_grad_enabled() and any(p.requires_grad for p in ps)):
            w = torch.cat([m.weight for m in heads], dim=0)
            return w, (torch.cat([m.bias for m in heads], dim=0) if heads[0].bias is not None else None)
        key, kept = tuple((p.data_ptr(), p._version, p.dtype, p.device) for p in ps), getattr(self, "_kept", None)
        if not ps[0].is_cuda:
            if kept is None or kept.key != key:
                kept = self._kept = _Kept(key, *self._concatenated(heads))
            return kept.w, kept.b
        with torch.cuda.device(ps[0].device):
            capturing, here = torch.cuda.is_current_stream_capturing(), torch.cuda.current_stream()
            if kept is not None and kept.key == key and kept.wait_for(here, capturing):
                kept.captured = kept.captured or capturing
                if not capturing:
                    kept.used_on(here)
                return kept.w, kept.b
            if capturing:                                                      # not there before the graph is replayed
                return self._concatenated(heads)
            like = lambda x, m: x is None or (x.dtype, x.device) == (m.dtype, m.device)
            if kept is not None and kept.captured and like(kept.w, ps[0]) and like(kept.b, ps[-1]):
                kept.wait_for(here, False)                                     # formed anew in its place
                kept.used_on(here)
                with torch.inference_mode(kept.w.is_inference()):
                    self._concatenated(heads, kept.w, kept.b)
                new = _Kept(key, kept.w, kept.b, True)
            else:
                new = _Kept(key, *self._concatenated(heads))
            new.formed_on(here)
            self._kept = new
        return new.w, new.b

    @staticmethod
    def _concatenated(heads, w=None, b=None):
        with torch.no_grad():
            w = torch.cat([m.weight for m in heads], dim=0, out=w)
            if heads[0].bias is not None:
                b = torch.cat([m.bias for m in heads], dim=0, out=b)
        return w, b

    def reset_cache(self):
        """Forget the concatenated projection weight of evaluation mode, also where a captured graph reads it: that must be captured
        anew."""
        self._kept, self._native_cache = None, [None] * 4

    def _form_anew(self):
        """The next call forms the concatenated weight of evaluation mode anew: where a captured graph reads it, in its place."""
        kept, native = getattr(self, "_kept", None), self._native_cache
        if kept is not None:
            if kept.captured:
                kept.key = None
            else:
                self._kept = None
        self._native_cache = [None] * 4 if native is None or native == [None] * 4 else _lib.native().forget(native)

    def __getstate__(self):
        """A copy forms its own weight."""
        state = self.__dict__.copy()
        state.pop("_kept", None)
        if state.get("_native_cache") is not None:
            state["_native_cache"] = [None] * 4
        return state

    def train(self, mode: bool = True):
        self._form_anew()
        return super().train(mode)

    def _apply(self, fn, *args, **kwargs):
        self._form_anew()
        return super()._apply(fn, *args, **kwargs)

    def _load_from_state_dict(self, *args, **kwargs):
        self._form_anew()
        return super()._load_from_state_dict(*args, **kwargs)

    def _up(self, lin: nn.Linear, x0: torch.Tensor) -> torch.Tensor:
        """Second half of a low-rank projection (head_dim -> embed_dim)."""
        if self.fuse_pre and lin.bias is None and x0.is_cuda and x0.dtype == torch.bfloat16 == lin.weight.dtype:
            return _pre.low_rank_up(x0, lin.weight)
        return lin(x0)

    # ---- the part of forward() before the recurrence (hdla_custom.py:202-267) --------------------------------------
    def project(self, x, attention_mask=None, q_offset=0, lower_bound=None):
        """x [b, n, d] -> q, k, v [b, n, H, D], beta [b, n, H, 1], log_f [b, n, H, D] with H = num_heads * num_blocks,
        and the inner activations of the output gate [b, n, head_dim] (None without a gate)."""
        b, n, d = x.shape
        # every projection of x in one GEMM (q, k, v, beta, the first halves of the decay and gate projections): one
        # read of x forward, one GEMM each for dx and dW backward instead of six and their sums
        heads = [self.q_proj, self.k_proj, self.v_proj]
        if self.use_beta:
            heads.append(self.bet_proj)
        heads.append(self.f_proj[0])
        if self.use_output_gate:
            heads.append(self.output_gate[0])
        w, bias = self._gathered(heads)
        y = F.linear(x, w, bias)
        ldy, hd = y.shape[-1], self.head_dim
        if (self.fuse_pre and self._all_silu and self.num_blocks == 1 and lower_bound is None and x.is_cuda
                and _pre.supported(y.dtype, hd, ldy, (d, 2 * d, 3 * d))):
            # activations, head split, l2 normalisation and beta in one kernel each way; its backward pass writes the
            # gradient of y in place
            col_tail = 3 * d + (self.num_heads if self.use_beta else 0)
            q, k, v, beta, f0, *rest = _pre.layer_pre(
                y.reshape(b * n, ldy), self.num_heads, hd, 0, d, 2 * d, 3 * d if self.use_beta else -1, col_tail,
                (hd, hd) if self.use_output_gate else (hd,), self.norm_q, True, self.norm_v,
                2.0 if self.beta_activation == "neg" else 1.0)
            q, k, v = (t.view(b, n, self.num_heads, hd) for t in (q, k, v))
            beta = beta.view(b, n, self.num_heads, 1) if self.use_beta else x.new_full((b, n, self.num_heads, 1), 2.0)
            f = self._up(self.f_proj[1], f0).view(b, n, d)
            if self.use_offset:
                f = f + self.offset
            log_f = _pre.logsigmoid(f).view(b, n, self.num_heads, hd)
            gate0 = rest[0].view(b, n, hd) if self.use_output_gate else None
            if attention_mask is not None and not attention_mask.all() and n > 1:        # left padding
                keep = attention_mask[:, q_offset:].unsqueeze(-1).unsqueeze(-1) != 0
                k = k.masked_fill(~keep, 0)
                log_f = log_f.masked_fill(~keep, 0)
            return q, k, v, beta, log_f, gate0
        parts = dict(zip([id(m) for m in heads], y.split([m.out_features for m in heads], dim=-1)))
        q, k, v, f0 = (parts[id(m)] for m in (self.q_proj, self.k_proj, self.v_proj, self.f_proj[0]))
        gate0 = parts[id(self.output_gate[0])] if self.use_output_gate else None
        f = self.f_proj[1](f0)
        if self.use_offset:
            f = f + self.offset
        if lower_bound is not None:
            log_f = torch.log(lower_bound + (1 - lower_bound) * torch.sigmoid(f))
        else:
            log_f = F.logsigmoid(f)
        if self.use_beta:
            beta = torch.sigmoid(parts[id(self.bet_proj)]).unsqueeze(-1)
            if self.beta_activation == "neg":
                beta = beta * 2
        else:
            beta = x.new_full((b, n, self.num_heads, 1), 2.0)
        q, k, v = self.q_act(q), self.k_act(k), self.v_act(v)
        q, k, v, log_f = (t.unflatten(-1, (-1, self.head_dim)) for t in (q, k, v, log_f))
        if self.num_blocks > 1:
            nb = self.num_blocks
            q, k, log_f = (t.unflatten(-1, (nb, -1)).flatten(2, 3) for t in (q, k, log_f))     # b n (h k) d
            v = v.repeat_interleave(nb, dim=2)
            beta = beta.repeat_interleave(nb, dim=2)
        if self.norm_q:
            q = l2_norm(q)
        k = l2_norm(k)
        if self.norm_v:
            v = l2_norm(v)
        if attention_mask is not None and not attention_mask.all() and n > 1:        # left padding
            keep = attention_mask[:, q_offset:].unsqueeze(-1).unsqueeze(-1) != 0
            k = k.masked_fill(~keep, 0)
            log_f = log_f.masked_fill(~keep, 0)
        return q, k, v, beta, log_f, gate0

    def _native_params(self):
        """Parameters for the native call, or None where something that it stands in for has been replaced or carries hooks."""
        own, cls = self.__dict__, type(self)
        if (cls.project is not _PROJECT or cls._up is not _UP or cls._gathered is not _GATHERED or "project" in own or "_up" in own
                or "_gathered" in own or nn.Linear.forward is not _LINEAR or nn.Module.__call__ is not _MODULE_CALL):
            return None
        if not own["use_beta"] or not own["use_output_gate"] or own["use_offset"] or own["num_blocks"] != 1 or any(_GLOBAL_HOOKS):
            return None
        mods = own["_modules"]
        f, g, norm = mods.get("f_proj"), mods.get("output_gate"), mods.get("norm")
        if type(f) is not nn.Sequential or type(g) is not nn.Sequential or len(f._modules) != 2 or len(g._modules) != 2:
            return None
        if type(norm) not in _NORMS or type(norm).forward is not _NORMS[type(norm)]:
            return None
        if norm.gate_act != "sigmoid" or norm.gate_pos not in ("pre", "post"):
            return None
        (f0, f1), (g0, g1), out = f._modules.values(), g._modules.values(), []
        for m in (mods.get("q_proj"), mods.get("k_proj"), mods.get("v_proj"), f0, g0, mods.get("bet_proj"), f1, g1, norm,
                  mods.get("o_proj")):
            if type(m) is not nn.Linear and m is not norm:
                return None
            d = m.__dict__
            if "forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"]:
                return None
            p = d["_parameters"]
            w = p.get("weight")
            if w is None or p.get("bias") is not None:
                return None
            out.append(w)
        return tuple(out)

    def _forward_native(self, x, state, use_cache):
        """The whole layer as one native call in its common form (csrc/native.cpp); None where this call is not of it."""
        params = self._native_params()
        if params is None:
            return None
        norm = self.norm
        groups, width = (norm.num_groups, norm.num_channels) if type(norm) is GroupRMSNormFusedGate else (1, norm.dim)
        mode = 0 if self.dispatch == "auto" else (1 if self.training or use_cache else 2)
        return _lib.native().layer(
            x, params, state, bool(use_cache), mode, None if self.training else self._native_cache, self.num_heads, groups,
            bool(self.norm_q), bool(self.norm_v), 2.0 if self.beta_activation == "neg" else 1.0,
            (width // groups) ** 0.5, norm.eps, 1 if norm.gate_pos == "pre" else 2)

    def forward(self, x, attention_mask: Optional[torch.Tensor] = None, past_key_values=None,
                use_cache: Optional[bool] = False, lower_bound: Optional[torch.Tensor] = None, **kwargs):
        b, n, d = x.shape
        recurrent_state, q_offset = None, 0
        if past_key_values is not None and len(past_key_values) > self.layer_idx:
            recurrent_state = past_key_values[self.layer_idx]["recurrent_state"][0]
            q_offset = past_key_values.get_seq_length(self.layer_idx)
        if self._common and self.fuse_ab and self.fuse_pre and attention_mask is None and lower_bound is None:
            out = self._forward_native(x, recurrent_state, use_cache)
            if out is not None:
                if past_key_values is not None:
                    past_key_values.update(recurrent_state=[out[1]], layer_idx=self.layer_idx, offset=n)
                return out[0], past_key_values
        q, k, v, beta, log_f, gate0 = self.project(x, attention_mask, q_offset, lower_bound)
        dtype = q.dtype
        k, v, beta, log_f = k.to(dtype), v.to(dtype), beta.to(dtype), log_f.to(dtype)

        if self.dispatch == "reference":
            chunked = bool(self.training or use_cache)
        else:
            chunked = (torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v, beta, log_f))) \
                or n >= RECURRENT_BELOW
        # output_final_state: the reference asks for it iff use_cache (hdla_custom.py:306,320)
        if self.fuse_ab:
            op = chunk_hdla_delta_rule if chunked else fused_recurrent_hdla_delta_rule
            output, recurrent_state = op(q, k, v, beta, log_f, scale=1.0, initial_state=recurrent_state,
                                         output_final_state=bool(use_cache))
        else:
            a, bb = parameterize_a_b(beta=beta.float(), k=k.float(), log_f=log_f.float())
            if chunked:
                output, recurrent_state = chunk_hrdplr_delta_rule(
                    q=q, k=k, v=v, a=a.to(dtype), b=bb.to(dtype), gk=log_f, RANK_AB=2, initial_state=recurrent_state,
                    output_final_state=bool(use_cache), scale=1.0, head_first=False, chunk_size=16)
            else:
                output, recurrent_state = fused_recurrent_dplr_delta_rule(
                    q=q, k=k, v=v, a=a.to(dtype), b=bb.to(dtype), gk=log_f, rank_ab=2, initial_state=recurrent_state,
                    output_final_state=bool(use_cache), scale=1.0, head_first=False)

        if self.num_blocks > 1:
            output = output.unflatten(2, (-1, self.num_blocks)).sum(dim=-2)
        if past_key_values is not None:
            past_key_values.update(recurrent_state=[recurrent_state], layer_idx=self.layer_idx, offset=n)
        output = output.flatten(2, 3)
        if self.use_output_gate:
            output = self.norm(output, self._up(self.output_gate[1], gate0))
        else:
            output = self.norm(output)
        return self.o_proj(output), past_key_values


# What the native call stands in for, as written here and in torch: it steps back where any of it is another function by now (a
# subclass or an instance that overrides a step, a module whose forward has been replaced, a patched class).
_PROJECT, _UP, _GATHERED = HDLA_Custom.project, HDLA_Custom._up, HDLA_Custom._gathered
_NORMS = {t: t.forward for t in (RMSNormFusedGate, GroupRMSNormFusedGate)}
_LINEAR, _MODULE_CALL = nn.Linear.forward, nn.Module.__call__
_GLOBAL_HOOKS = [getattr(nn.modules.module, n, {}) for n in ("_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks",
                                                            "_global_backward_pre_hooks")]
