"""The work that a user of this library has it do, as cases that can be timed: the operators and the layer through their
public entry points, from a single decoded token to the largest training step of the repository's own configurations.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)` one more of the same ranges, `prepare` makes
what a program has in hand before the call (on the GPU, from a seed), `run` is one pass, `work` and `tolerance` say what a
pass cannot do without and how far two correct implementations may be apart.

Kinds of cases ("kind"):
  decode        one call of a token-serial operator that takes a state and gives the next one, T tokens per sequence
  prefill       one forward pass of a chunked operator without gradients, state in and state out
  train         forward and backward pass of a chunked operator, every gradient
  layer_train   forward and backward pass of the HDLA layer, gradients of its input and of every parameter
  layer_decode  one cached decode step of the HDLA layer, state carried in the cache
  norm          forward and backward pass of the fused gated RMS norm

"form" says how the state transition is given: "ab" by the tensors a and b (the plain operators), "beta" by beta, k and the
log-decay (the operators as the layer calls them).  Distributions are those of hdla_hip/synthetic.py, drawn on the GPU.
"""
import math
import os
import sys

# the package lives below a folder whose name is no identifier, relative to the root the process works in
_PKG = os.path.join(os.getcwd(), "hdla-impl_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import torch
import torch.nn.functional as F

import hdla_hip
from hdla_hip.layer import HDLA_Custom, RecurrentCache
from hdla_hip.normalize import normalize_fn

_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
_ES = {"bf16": 2, "fp32": 4}


def _op(kind, name=None, *, B, T, H, K, V, form="ab", dtype="bf16", lens="", state=True, decay_div=16.0):
    """A case of one of the operators.  `lens`: lengths of packed sequences ("" = B sequences of T tokens).  `state`: an
    initial state is given (in training: and a gradient into the final one).  `decay_div`: the log-decay is
    logsigmoid(N(0,1)) / decay_div."""
    c = dict(kind=kind, B=B, T=T, H=H, K=K, V=V, form=form, dtype=dtype, lens=lens, state=state, decay_div=decay_div)
    return dict(c, name=name) if name else c


def listed():
    return [
        # interactive generation: one token of one sequence, where the call itself is the cost
        _op("decode", "decode_one", B=1, T=1, H=16, K=64, V=64),
        # a serving batch: one token each for 256 sequences, the state streams through (the repository's configuration 4)
        _op("decode", "decode_batch", B=256, T=1, H=32, K=128, V=128),
        # prefill of a batch of prompts (configuration 1's shape, with the states handed on)
        _op("prefill", "prefill", B=4, T=2048, H=16, K=64, V=64),
        # prompts of unequal, odd lengths packed into one batch, at the larger head size, as the layer calls the operator
        _op("prefill", "prefill_packed", B=1, T=5003, H=16, K=128, V=128, form="beta", lens="1731,37,2204,1031", decay_div=1.0),
        # a short training step, as in tests, fine-tuning on short texts and debugging (configuration 0's shape)
        _op("train", "train_short", B=1, T=256, H=2, K=64, V=64, state=False),
        # the training step of the repository's headline (configuration 2)
        _op("train", "train", B=4, T=2048, H=16, K=64, V=64),
        # long packed documents at the larger head size (configuration 3)
        _op("train", "train_packed", B=1, T=16384, H=16, K=128, V=128, lens="2048,4096,4096,6144"),
        # full precision, a length that fills no chunk: numerics work and checks against fp32
        _op("train", "train_fp32", B=2, T=1003, H=8, K=64, V=64, dtype="fp32"),
        # the operator as a layer of wider heads trains it: few sequences, odd length, decays undivided, no states given
        _op("train", "train_beta_128", B=2, T=1537, H=8, K=128, V=128, form="beta", state=False, decay_div=1.0),
        # a training step of the whole layer (bench.py's layer workload)
        dict(name="layer_train", kind="layer_train", B=4, T=2048, d=1024, H=16),
        # a cached decode step of the whole layer for a small serving batch
        dict(name="layer_decode", kind="layer_decode", B=16, d=2048, H=16),
        # the normalisation behind the operator, at the shape of the layer above
        dict(name="norm", kind="norm", rows=8192, D=1024, gate="pre", dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _split(rng, total, n):
    """n lengths (at least one token each) that add up to total, none of them in any order."""
    cuts = sorted(rng.sample(range(1, total), n - 1))
    return ",".join(str(b - a) for a, b in zip([0] + cuts, cuts + [total]))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "train", "train", "train", "layer_train", "layer_decode", "norm"])
    if kind == "layer_train":
        D, H = rng.choice([64, 64, 128]), rng.choice([4, 8, 16])
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, T=_log(rng, 64, 8192 // B), d=D * H, H=H)
    if kind == "layer_decode":
        D, H = rng.choice([64, 128]), rng.choice([8, 16, 32])
        return dict(kind=kind, B=_log(rng, 1, 256), d=D * H, H=H)
    if kind == "norm":
        return dict(kind=kind, rows=_log(rng, 100, 65536), D=rng.choice([512, 1024, 2048, 4096]), gate=rng.choice(["pre", "pre", "post"]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    form = rng.choice(["ab", "beta"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    K = rng.choice([64, 64, 128])
    V = K if rng.random() < 0.75 else 192 - K
    H = rng.choice([2, 4, 8, 12, 16, 32])
    div = rng.choice([16.0, 4.0, 1.0])
    if kind == "decode":
        # mostly one token per call, now and then a short burst; the states of the largest listed batch bound the size
        most = 256 * 32 * 128 * 128 // (H * K * V)
        return _op(kind, B=_log(rng, 1, min(256, most)), T=rng.choice([1, 1, 1, rng.randint(2, 8)]), H=H, K=K, V=V, form=form, dtype=dtype,
                   decay_div=div)
    # as many token x head x channel as the largest listed training step at most (an eighth of it in fp32), 16384 tokens at most
    most = 16384 * 16 * 256 // (H * (K + V)) // (8 if dtype == "fp32" else 1)
    total = _log(rng, 50, min(32768, most))
    state = rng.random() < 0.6
    if rng.random() < 0.4 and total <= 16384:
        n = min(rng.randint(2, 12), total // 8)
        return _op(kind, B=1, T=total, H=H, K=K, V=V, form=form, dtype=dtype, lens=_split(rng, total, n), state=state, decay_div=div)
    B = max(rng.choice([1, 1, 2, 3, 4, 8]), -(-total // 16384))
    return _op(kind, B=B, T=max(1, total // B), H=H, K=K, V=V, form=form, dtype=dtype, state=state, decay_div=div)


# ---- inputs --------------------------------------------------------------------------------------------------------
def _op_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    B, T, H, K, V, dt = c["B"], c["T"], c["H"], c["K"], c["V"], _DT[c["dtype"]]
    lens = [int(x) for x in c["lens"].split(",")] if c["lens"] else []
    N = len(lens) if lens else B
    s = {"c": c, "train": c["kind"] == "train"}
    unit = lambda: F.normalize(rn(B, T, H, K), dim=-1)
    q, k, v = unit(), unit(), rn(B, T, H, V)
    if c["form"] == "ab":
        a, b = [], []
        for _ in range(2):
            u, beta = unit(), 2.0 * torch.rand(B, T, H, 1, generator=g, device="cuda")
            a.append(-beta * u)
            b.append(u)
        more = [torch.stack(x, dim=2).reshape(B, 2 * T, H, K) for x in (a, b)]
    else:
        more = [2.0 * torch.rand(B, T, H, 1, generator=g, device="cuda")]
    gk = F.logsigmoid(rn(B, T, H, K)) / c["decay_div"]
    s["x"] = [t.to(dt).requires_grad_(s["train"]) for t in [q, k, v] + more + [gk]]
    s["h0"] = (0.1 * rn(N, H, K, V)).requires_grad_(s["train"]) if c["state"] else None
    s["cu"] = torch.tensor([sum(lens[:i]) for i in range(N + 1)], device="cuda") if lens else None
    if s["train"]:
        s["do"], s["dht"] = rn(B, T, H, V).to(dt), rn(N, H, K, V) if c["state"] else None
    return s


def _layer(c, seed):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        return HDLA_Custom(c["d"], c["H"], token_mixer_init_type=2, rescale_type=0).to(torch.bfloat16)


def prepare(case, seed):
    c = case
    if c["kind"] in ("decode", "prefill", "train"):
        return _op_inputs(c, seed)
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    if c["kind"] == "layer_train":
        m = _layer(c, seed).train()
        return {"c": c, "m": m, "params": list(m.parameters()), "x": rn(c["B"], c["T"], c["d"]).bfloat16().requires_grad_(),
                "do": rn(c["B"], c["T"], c["d"]).bfloat16()}
    if c["kind"] == "layer_decode":
        m, cache = _layer(c, seed).eval(), RecurrentCache()
        with torch.no_grad():                                 # the prompt: its states are in the cache when decoding begins
            _, cache = m(rn(c["B"], 16, c["d"]).bfloat16(), past_key_values=cache, use_cache=True)
        return {"c": c, "m": m, "cache": cache, "x": rn(c["B"], 1, c["d"]).bfloat16()}
    dt = _DT[c["dtype"]]
    return {"c": c, "x": rn(c["rows"], c["D"]).to(dt).requires_grad_(), "gate": rn(c["rows"], c["D"]).to(dt).requires_grad_(),
            "w": (1.0 + 0.1 * rn(c["D"])).requires_grad_(), "do": rn(c["rows"], c["D"]).to(dt)}


# ---- one pass ------------------------------------------------------------------------------------------------------
def run(state):
    s, c = state, state["c"]
    kind = c["kind"]
    if kind == "decode":
        with torch.no_grad():
            if c["form"] == "ab":
                return hdla_hip.fused_recurrent_dplr_delta_rule(*s["x"], 2, scale=1.0, initial_state=s["h0"], output_final_state=True)
            return hdla_hip.fused_recurrent_hdla_delta_rule(*s["x"], scale=1.0, initial_state=s["h0"], output_final_state=True)
    if kind == "prefill":
        with torch.no_grad():
            return _chunked(s, True)
    if kind == "train":
        o, ht = _chunked(s, s["h0"] is not None)
        leaves = s["x"] + ([s["h0"]] if s["h0"] is not None else [])
        outs, gos = ([o, ht], [s["do"], s["dht"]]) if s["h0"] is not None else ([o], [s["do"]])
        return [t.detach() for t in outs] + list(torch.autograd.grad(outs, leaves, gos))
    if kind == "layer_train":
        y, _ = s["m"](s["x"])
        return [y.detach()] + list(torch.autograd.grad(y, [s["x"]] + s["params"], s["do"]))
    if kind == "layer_decode":
        with torch.no_grad():
            y, s["cache"] = s["m"](s["x"], past_key_values=s["cache"], use_cache=True)
        return y, s["cache"][0]["recurrent_state"][0]
    y = normalize_fn(s["x"], s["w"], gate=s["gate"], gate_pos=c["gate"], c=c["D"] ** 0.5, eps=1e-5)
    return [y.detach()] + list(torch.autograd.grad(y, [s["x"], s["gate"], s["w"]], s["do"]))


def _chunked(s, want_state):
    if s["c"]["form"] == "ab":
        return hdla_hip.chunk_hrdplr_delta_rule(*s["x"], 2, scale=1.0, initial_state=s["h0"], output_final_state=want_state, chunk_size=16,
                                                cu_seqlens=s["cu"])
    return hdla_hip.chunk_hdla_delta_rule(*s["x"], scale=1.0, initial_state=s["h0"], output_final_state=want_state, cu_seqlens=s["cu"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def work(case):
    """Bytes: every input once, every output once.  Operations: those of the recurrence itself (13 K V per token and head
    forward, three times that with the backward pass, whatever the chunk length), and 2 per weight and token for each
    projection of the layer (three times that in training)."""
    c = case
    if c["kind"] == "norm":
        es, n = _ES[c["dtype"]], c["rows"] * c["D"]
        return {"bytes": 6 * n * es + 2 * c["D"] * 4, "flops": 30 * n}         # x, gate, do; o, dx, dgate; weight and its gradient
    if c["kind"] in ("layer_train", "layer_decode"):
        d, H, D = c["d"], c["H"], c["d"] // c["H"]
        weights = 4 * d * d + 4 * d * D + d * H + d
        if c["kind"] == "layer_decode":
            return {"bytes": 2 * weights + 2 * c["B"] * H * D * D * 4 + 2 * c["B"] * d * 2,
                    "flops": c["B"] * (2 * weights + 13 * H * D * D)}
        n = c["B"] * c["T"]
        return {"bytes": 2 * 2 * weights + 4 * n * d * 2, "flops": n * (6 * weights + 39 * H * D * D)}
    es, K, V, rows = _ES[c["dtype"]], c["K"], c["V"], c["B"] * c["T"] * c["H"]
    N = len(c["lens"].split(",")) if c["lens"] else c["B"]
    ins = (7 * K if c["form"] == "ab" else 3 * K + 1) + V                      # q, k, gk, (a, b | beta), v
    st = N * c["H"] * K * V * 4
    if c["kind"] == "train":
        # inputs, do; o, the inputs' gradients; with states: h0, dht, the final state and dh0
        return {"bytes": rows * (2 * ins + 2 * V) * es + (4 * st if c["state"] else 0), "flops": 39 * K * V * rows}
    return {"bytes": rows * (ins + V) * es + (2 if c["state"] else 1) * st, "flops": 13 * K * V * rows}


def tolerance(case):
    """Relative 2-norm of the difference: 32-bit sums where the inputs are 32-bit; for bf16 inputs what their rounding and
    that of the operands of the products leave (the operators stay within 5e-3 forward and 1e-2 backward of exact
    arithmetic), twice that for the layer, where every stage rounds its result to bf16."""
    if case["kind"] in ("layer_train", "layer_decode"):
        return {"rel": 2e-2}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1e-5}
