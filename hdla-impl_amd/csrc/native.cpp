// Host path of the Python operators: argument checks, allocations, autograd nodes and calls of the C ABI in native code.
//
// A call on a few tokens costs the GPU 4 to 30 microseconds; what it cost the host in Python (shape checks, ctypes
// marshalling, autograd.Function with its decorators, one tensor allocation at a time) was 25 to 250.  Every operator of
// the package therefore asks here first.  A function of this module takes the arguments of the public operator as they
// are, and either runs the whole call or, for anything that is not its case (another dtype or head size, tensors on the
// CPU, shapes that do not fit, ...), returns None without having touched anything: the Python code of the operator then
// converts, pads or raises as it always did.  So this file holds no error messages of its own; it only recognises what
// needs none.
//
// The kernels stay behind the C ABI of libhdla_hip.so: `bind` receives the handle of the library the package loaded and
// looks the entry points up in it.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/hdla_hip.h"
#include "host_path.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- the C ABI -------------------------------------------------------------------------------------------------------
struct Api {
#define HDLA_FN(name) decltype(&hdla_##name) name
    HDLA_FN(strerror); HDLA_FN(workspace_bytes); HDLA_FN(record_bytes); HDLA_FN(record_workspace_bytes); HDLA_FN(chunk_fwd_b); HDLA_FN(chunk_bwd_b);
    HDLA_FN(keep_plan); HDLA_FN(chunk_fwd_keep); HDLA_FN(chunk_bwd_kept); HDLA_FN(states_plan); HDLA_FN(chunk_fwd_states); HDLA_FN(chunk_bwd_states);
    HDLA_FN(tile_gemm); HDLA_FN(layer_pre_bwd_to);
    HDLA_FN(recurrent_fwd); HDLA_FN(param_recurrent_fwd); HDLA_FN(normalize_fwd); HDLA_FN(normalize_bwd_as);
    HDLA_FN(normalize_workspace_bytes); HDLA_FN(layer_pre_fwd); HDLA_FN(layer_pre_bwd); HDLA_FN(layer_up_fwd); HDLA_FN(layer_down);
    HDLA_FN(layer_up_wgrad); HDLA_FN(layer_up_wgrad_workspace_bytes); HDLA_FN(rows_gemm); HDLA_FN(sum_partials); HDLA_FN(stack_rows);
    HDLA_FN(weight_grad); HDLA_FN(weight_grad_workspace_bytes); HDLA_FN(weight_grad_pair); HDLA_FN(weight_grad_pair_workspace_bytes);
    HDLA_FN(normalize_bwd_later); HDLA_FN(layer_up_wgrad_later); HDLA_FN(run_sums);
    HDLA_FN(layer_step); HDLA_FN(rows_gemm_norm);
#undef HDLA_FN
} api;
PyObject* error_class = nullptr;                 // _lib.HdlaError
PyObject* memory_error = nullptr;                // torch.OutOfMemoryError

// what _lib.check raises: "<entry point> failed with code <rc>: <text>"
struct AbiError : std::runtime_error { using std::runtime_error::runtime_error; };
void check(int rc, const char* what) {
    if (rc) throw AbiError(std::string(what) + " failed with code " + std::to_string(rc) + ": " + api.strerror(rc));
}

// The same on a thread of the autograd engine: the Python exception is set here and carried by the engine to the caller.
template <typename F> auto in_backward(F fn) {
    try {
        return fn();
    } catch (const AbiError& e) {
        const PyGILState_STATE gil = PyGILState_Ensure();
        PyErr_SetString(error_class ? error_class : PyExc_RuntimeError, e.what());
        python_error err;
        err.persist();
        PyGILState_Release(gil);
        throw err;
    }
}

// an autograd function takes defined tensors, or std::optional
using Maybe = std::optional<Tensor>;
inline Maybe maybe(const Tensor& t) { return t.defined() ? Maybe(t) : Maybe(); }
inline Tensor value(const Maybe& t) { return t ? *t : Tensor(); }

inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
inline int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? HDLA_BF16 : HDLA_FP32; }
inline bool native_dtype(at::ScalarType t) { return t == at::kBFloat16 || t == at::kFloat; }
inline Tensor bytes_like(const Tensor& t, size_t n) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }

// The package's environment switches, read on every call like the Python code does, and once: while the interpreter lock is held, under
// which os.environ writes them.
const char* env(const char* name) {
    if (!PyGILState_Check()) throw std::logic_error("the environment is read with the interpreter lock held");
    return getenv(name);
}
bool env_is(const char* name, std::initializer_list<const char*> values, bool unset) {
    const char* v = env(name);
    if (!v) return unset;
    for (const char* x : values) if (!strcmp(v, x)) return true;
    return false;
}
bool keep_forward_default() { return !env_is("HDLA_HIP_KEEP_FORWARD", {"", "0", "false", "False"}, true); }
bool keep_forward_unsaid() { return env("HDLA_HIP_KEEP_FORWARD") == nullptr; }
// launch plan of a chunked call, and what its backward pass may be given: the record, and where the route has none the forward pass's workspace
// (keep: KEEP_STATES with the states that enter the chunks)
enum Keep : int32_t { KEEP_NOTHING, KEEP_FORWARD, KEEP_STATES };
struct Plan { int32_t route, segments; bool record; Keep keep; };
// false: the Python code has to look at it (another spelling, a number that is none)
bool read_plan(Plan& p) {
    const char* r = env("HDLA_HIP_ROUTE");
    if (!r || !*r || !strcmp(r, "auto")) p.route = HDLA_ROUTE_AUTO;
    else if (!strcmp(r, "classic")) p.route = HDLA_ROUTE_CLASSIC;
    else if (!strcmp(r, "plain")) p.route = HDLA_ROUTE_PLAIN;
    else if (!strcmp(r, "fused")) p.route = HDLA_ROUTE_FUSED;
    else return false;
    p.record = env_is("HDLA_HIP_INPUTS_ONLY", {"", "0", "false", "False"}, true);
    p.keep = KEEP_NOTHING;
    p.segments = 0;
    const char* s = env("HDLA_HIP_SEGMENTS");
    if (!s) return true;
    char* end = nullptr;
    p.segments = (int32_t)strtol(s, &end, 10);
    return *s && !*end;
}

// ---- the chunked operators -------------------------------------------------------------------------------------------
// a and b, or beta (the other undefined)
struct ChunkIn {
    Tensor q, k, v, a, b, beta, gk, h0, cu;
};

void chunk_dims(const ChunkIn& x, double scale, const Plan& p, hdla_dims& d) {
    d = hdla_dims{};
    d.route = p.route; d.segments = p.segments;
    d.B = (int32_t)x.q.size(0); d.T = (int32_t)x.q.size(1); d.H = (int32_t)x.q.size(2); d.K = (int32_t)x.q.size(3);
    d.V = (int32_t)x.v.size(3); d.R = 2;
    d.N = x.cu.defined() ? (int32_t)(x.cu.numel() - 1) : d.B;
    d.in_dtype = dtype_code(x.q.scalar_type());
    d.gk_dtype = dtype_code(x.gk.scalar_type());
    d.scale = (float)scale;
    d.cu_seqlens = x.cu.defined() ? x.cu.data_ptr<int64_t>() : nullptr;
}

// The launch plan of a backward pass is that of its forward pass, whatever the environment says by then: what that left is laid out by it.
void save_plan(AutogradContext* ctx, const Plan& p) { ctx->saved_data["plan"] = std::vector<int64_t>{p.route, p.segments, p.keep}; }
Plan saved_plan(AutogradContext* ctx) {
    const auto p = ctx->saved_data["plan"].toIntVector();
    return {(int32_t)p[0], (int32_t)p[1], false, (Keep)p[2]};
}

// with_record: of a backward pass that is given the forward pass's record
Tensor workspace(const hdla_dims& d, int pass, const Tensor& like, bool with_record = false) {
    const size_t n = with_record ? api.record_workspace_bytes(&d) : api.workspace_bytes(&d, pass);
    if (!n) throw AbiError("hdla_workspace_bytes rejected the dimensions (B=" + std::to_string(d.B) + ",T=" + std::to_string(d.T) +
                           ",H=" + std::to_string(d.H) + ",K=" + std::to_string(d.K) + ",V=" + std::to_string(d.V) +
                           ",R=" + std::to_string(d.R) + ",N=" + std::to_string(d.N) + ")");
    return bytes_like(like, n);
}

// Forward workspaces that calls hold for their backward passes because the library suggests it (hdla_keep_plan, hdla_states_plan), and nobody asked: as much as KEPT_MOST
// a device over all calls whose backward pass is still to come, 0.4 % of its memory, so that a stack of layers that trains within the device's memory
// without them does so with them, and that of KEPT_CALLS calls, a microsecond to look through.  A call that finds no room, there or with the allocator,
// keeps its inputs and recomputes, the same bits.  So does one under saved-tensor hooks: what these see of a call must not depend on the room that
// others leave (a checkpointed part that is run again has to save what it saved the first time), nor grow what they move or count.  us a training step with room / without / with keep_forward=False: fp32, 2 x 1003 tokens, 8 heads,
// K = V = 64 181 / 218 / 224; 2 x 1537 tokens, 8 heads, K = V = 128 195 / 212 / 215; 4 x 1000, 16 heads 379 / 408 / 410.
constexpr int64_t KEPT_MOST = (int64_t)1 << 30;
constexpr size_t KEPT_CALLS = 256;
struct KeptRoom {
    std::mutex lock;
    int64_t coming = 0;                                   // of calls that are allocating theirs
    std::vector<std::pair<c10::weak_intrusive_ptr<c10::StorageImpl>, int64_t>> held;
    bool take(int64_t n) {
        const std::lock_guard<std::mutex> g(lock);
        held.erase(std::remove_if(held.begin(), held.end(), [](const auto& h) { return h.first.expired(); }), held.end());
        int64_t sum = coming + n;
        for (const auto& h : held) sum += h.second;
        if (sum > KEPT_MOST || held.size() >= KEPT_CALLS) return false;
        coming += n;
        return true;
    }
    void settle(int64_t n, const Tensor& t) {
        const std::lock_guard<std::mutex> g(lock);
        coming -= n;
        if (t.defined()) held.emplace_back(t.storage().getWeakStorageImpl(), n);
    }
};
constexpr int KEPT_DEVICES = 64;
// undefined: no room
Tensor kept_room(const Tensor& like, int64_t n) {
    static KeptRoom* const rooms = new KeptRoom[KEPT_DEVICES];    // (never destroyed: tensors may outlive this library's statics)
    const int dev = like.device().index();
    if (dev < 0 || dev >= KEPT_DEVICES || !at::SavedTensorDefaultHooks::get_tls_state().stack.empty() || !rooms[dev].take(n)) return Tensor();
    Tensor t;
    try {
        t = bytes_like(like, (size_t)n);
    } catch (const c10::OutOfMemoryError&) {
    } catch (...) {
        rooms[dev].settle(n, Tensor());
        throw;
    }
    rooms[dev].settle(n, t);
    return t;
}

// left: what the backward pass is given (undefined: the inputs are all); plan: the one that pass is to run with
void chunk_forward(const ChunkIn& x, const hdla_dims& d, bool want_ht, Plan* plan, Tensor& o, Tensor& ht, Tensor& left) {
    const auto f32 = x.q.options().dtype(at::kFloat);
    o = at::empty_like(x.v);
    if (want_ht) ht = at::empty({d.N, d.H, d.K, d.V}, f32);
    const size_t nb = plan && plan->record ? api.record_bytes(&d) : 0;
    if (plan && plan->keep) {
        hdla_dims k = d;
        int32_t for_bwd = 0;
        const bool may = plan->record && !nb;
        const size_t n = may ? api.keep_plan(&d, &k.segments, &for_bwd) : 0;
        if (n) {                                          // one plan for the backward pass, kept or not
            plan->segments = for_bwd;
            if (for_bwd == 1) plan->route = HDLA_ROUTE_PLAIN;   // (one segment, also where a number asked for would be the fused route's)
            left = kept_room(x.q, (int64_t)n);
        } else if (may) {
            // Too large for that (KEEP_MOST, api.hip): with the states, 490 to 980 MiB that save 80 to 210 us.  Not where the smaller buffer is to be had: with them the gibibyte holds half
            // as many calls, and one that finds no room loses more than the others gain.  us a step of several calls of 4 x 1000 tokens, 16 heads, K = V = 128, with states first / without: 1
            // 350 / 363, 4 1399 / 1389, 8 2923 / 2841; 8 of 2 x 2048 3339 / 3276; 16 of 4 x 500 2937 / 2875.  Large ones, states / nothing: 1 and 3 of 16384 packed tokens 1424 / 1630,
            // 4675 / 4877 (the first has the room), 4 of 4 x 2048, beta form 2621 / 2846; seven of the first behind a packed one 4063 / 4073.
            size_t ws_fwd = 0, ws_bwd = 0;
            const size_t all = api.states_plan(&d, &ws_fwd, &ws_bwd);
            if (all) left = kept_room(x.q, (int64_t)all);
            Tensor ws;
            if (left.defined()) {
                try {
                    ws = bytes_like(x.q, ws_fwd);
                } catch (const c10::OutOfMemoryError&) {
                    left = Tensor();                      // (a call without the buffer needs less)
                }
            }
            if (left.defined()) {
                plan->keep = KEEP_STATES;
                check(api.chunk_fwd_states(&d, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.a), ptr(x.b), ptr(x.beta), ptr(x.gk), fptr(x.h0), ptr(o), fptr(ht),
                                           ptr(left), all, ptr(ws), ws_fwd, stream_of(x.q)), "hdla_chunk_fwd_states");
                return;
            }
        }
        plan->keep = left.defined() ? KEEP_FORWARD : KEEP_NOTHING;
        if (plan->keep) {
            check(api.chunk_fwd_keep(&k, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.a), ptr(x.b), ptr(x.beta), ptr(x.gk), fptr(x.h0), ptr(o), fptr(ht),
                                     ptr(left), n, stream_of(x.q)), "hdla_chunk_fwd_keep");
            return;
        }
    }
    if (nb) left = bytes_like(x.q, nb);
    const Tensor ws = workspace(d, HDLA_PASS_FWD, x.q);
    check(api.chunk_fwd_b(&d, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.a), ptr(x.b), ptr(x.beta), ptr(x.gk), fptr(x.h0), ptr(o), fptr(ht),
                          ptr(left), nb, ptr(ws), (size_t)ws.numel(), stream_of(x.q)), "hdla_chunk_fwd_b");
}

struct ChunkGrads { Tensor q, k, v, a, b, beta, gk, h0; };      // of what is defined
Tensor backward_workspace(const hdla_dims& d, const Plan& plan, const Tensor& like, const Tensor& left) {
    if (plan.keep == KEEP_STATES) {
        size_t fwd = 0, bwd = 0;
        if (!api.states_plan(&d, &fwd, &bwd)) throw AbiError("hdla_states_plan: not the forward pass's dimensions");
        return bytes_like(like, bwd);
    }
    return plan.keep ? workspace(d, HDLA_PASS_BWD_KEPT, like) : workspace(d, HDLA_PASS_BWD, like, left.defined());
}
void chunk_backward(const ChunkIn& x, const hdla_dims& d, const Plan& plan, const Tensor& d_o, const Tensor& dht, const Tensor& left, const Tensor& ws,
                    const ChunkGrads& g) {
    if (plan.keep) {
        const bool states = plan.keep == KEEP_STATES;
        check((states ? api.chunk_bwd_states : api.chunk_bwd_kept)(
                  &d, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.a), ptr(x.b), ptr(x.beta), ptr(x.gk), fptr(x.h0), ptr(d_o), fptr(dht),
                  ptr(g.q), ptr(g.k), ptr(g.v), ptr(g.a), ptr(g.b), ptr(g.beta), ptr(g.gk), fptr(g.h0), ptr(left),
                  (size_t)left.numel(), ptr(ws), (size_t)ws.numel(), stream_of(x.q)), states ? "hdla_chunk_bwd_states" : "hdla_chunk_bwd_kept");
        return;
    }
    check(api.chunk_bwd_b(&d, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.a), ptr(x.b), ptr(x.beta), ptr(x.gk), fptr(x.h0), ptr(d_o), fptr(dht),
                          ptr(g.q), ptr(g.k), ptr(g.v), ptr(g.a), ptr(g.b), ptr(g.beta), ptr(g.gk), fptr(g.h0), ptr(left),
                          left.defined() ? (size_t)left.numel() : 0, ptr(ws), (size_t)ws.numel(), stream_of(x.q)), "hdla_chunk_bwd_b");
}

// The autograd node: the contract of ChunkDPLRDeltaRuleFunction and ChunkHDLAFunction (the inputs and, where the route
// has one, the record for the backward pass are saved; everything else is recomputed).
struct ChunkFn : torch::autograd::Function<ChunkFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Maybe& a, const Maybe& b,
                                 const Maybe& beta, const Tensor& gk, const Maybe& h0, const Maybe& cu, double scale, bool want_ht,
                                 Plan plan) {
        ChunkIn x{q, k, v, value(a), value(b), value(beta), gk, value(h0), value(cu)};
        if (h0) x.h0 = h0->to(at::kFloat).contiguous();
        hdla_dims d;
        chunk_dims(x, scale, plan, d);
        Tensor o, ht, left;
        chunk_forward(x, d, want_ht, &plan, o, ht, left);
        save_plan(ctx, plan);
        ctx->save_for_backward({q, k, v, x.a, x.b, x.beta, gk, value(h0), x.cu, left});
        ctx->saved_data["scale"] = scale;
        ctx->set_materialize_grads(false);
        return want_ht ? variable_list{o, ht} : variable_list{o};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return in_backward([&] { return gradients(ctx, grads); });
    }
    static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
        const auto s = ctx->get_saved_variables();
        ChunkIn x{s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8]};
        const at::DeviceGuard guard(x.q.device());
        if (x.h0.defined()) x.h0 = x.h0.to(at::kFloat).contiguous();
        const Plan plan = saved_plan(ctx);
        hdla_dims d;
        chunk_dims(x, ctx->saved_data["scale"].toDouble(), plan, d);
        const Tensor d_o = grads[0].defined() ? grads[0].to(x.v.scalar_type()).contiguous() : at::zeros_like(x.v);
        Tensor dht;
        if (grads.size() > 1 && grads[1].defined()) dht = grads[1].to(at::kFloat).contiguous();
        const Tensor ws = backward_workspace(d, plan, x.q, s[9]);
        ChunkGrads r;
        r.q = at::empty_like(x.q); r.k = at::empty_like(x.k); r.v = at::empty_like(x.v); r.gk = at::empty_like(x.gk);
        if (x.beta.defined()) r.beta = at::empty_like(x.beta);
        else { r.a = at::empty_like(x.a); r.b = at::empty_like(x.b); }
        if (x.h0.defined()) r.h0 = at::empty_like(x.h0);
        chunk_backward(x, d, plan, d_o, dht, s[9], ws, r);
        if (r.h0.defined()) r.h0 = r.h0.to(s[7].scalar_type());
        return {r.q, r.k, r.v, r.a, r.b, r.beta, r.gk, r.h0, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ---- reading the Python arguments ------------------------------------------------------------------------------------
// a plain tensor (or parameter): no subclass, nothing that overrides torch functions
inline bool is_tensor(PyObject* o) { return THPVariable_CheckExact(o); }
inline const Tensor& unpack(PyObject* o) { return THPVariable_Unpack(o); }
inline bool truth(PyObject* o, bool& out) {
    const int r = PyObject_IsTrue(o);
    if (r < 0) PyErr_Clear();
    out = r > 0;
    return r >= 0;
}
inline bool number(PyObject* o, double& out) {
    out = PyFloat_AsDouble(o);
    if (out == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}
// (a tensor that carries a forward-mode tangent or is the wrapper of a function transform goes to the Python code, whose autograd
// functions refuse it: here a call without gradients would drop the tangent)
inline bool gpu_like(const Tensor& t, const at::Device& dev) {
    return t.device() == dev && t.layout() == at::kStrided && !t.is_complex() && t.has_storage() && !t._fw_grad(/*level=*/0).defined();
}
inline bool off_grid(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0; }
inline bool same_sizes(const Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s); }

// What the chunked and the token-serial operators have in common: q, k, v, gk, the states and the sequence table.
// False: not a case of this file.
bool read_operands(PyObject* pq, PyObject* pk, PyObject* pv, PyObject* pgk, PyObject* ph0, PyObject* pcu, bool serial, ChunkIn& x) {
    if (!api.strerror || !is_tensor(pq) || !is_tensor(pk) || !is_tensor(pv) || !is_tensor(pgk)) return false;
    const Tensor &q = unpack(pq), &k = unpack(pk), &v = unpack(pv), &gk = unpack(pgk);
    const auto dt = q.scalar_type();
    const at::Device dev = q.device();
    if (!dev.is_cuda() || !native_dtype(dt) || k.scalar_type() != dt || v.scalar_type() != dt) return false;
    if (gk.scalar_type() != dt && gk.scalar_type() != at::kFloat) return false;
    if (q.dim() != 4 || v.dim() != 4 || k.sizes() != q.sizes() || gk.sizes() != q.sizes()) return false;
    if (!gpu_like(q, dev) || !gpu_like(k, dev) || !gpu_like(v, dev) || !gpu_like(gk, dev)) return false;
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), K = q.size(3), V = v.size(3);
    const auto native = [&](int64_t d) { return d == 64 || d == 128 || (serial && d == 256); };
    if (!native(K) || !native(V) || v.size(0) != B || v.size(1) != T || v.size(2) != H || B < 1 || T < 1 || H < 1) return false;
    if (B > INT32_MAX || T > INT32_MAX / 4 || H > 65535) return false;
    int64_t N = B;
    if (pcu != Py_None) {
        if (!is_tensor(pcu)) return false;
        const Tensor& cu = unpack(pcu);
        if (cu.device() != dev || cu.scalar_type() != at::kLong || cu.dim() != 1 || cu.numel() < 2 || B != 1) return false;
        N = cu.numel() - 1;
        x.cu = cu.contiguous();
    }
    if (ph0 != Py_None) {
        if (!is_tensor(ph0)) return false;
        const Tensor& h0 = unpack(ph0);
        if (!gpu_like(h0, dev) || !same_sizes(h0, {N, H, K, V}) || !h0.is_floating_point()) return false;
        x.h0 = h0;
    }
    x.q = q; x.k = k; x.v = v; x.gk = gk;
    return true;
}
bool read_ab(PyObject* pa, PyObject* pb, ChunkIn& x) {
    if (!is_tensor(pa) || !is_tensor(pb)) return false;
    const Tensor &a = unpack(pa), &b = unpack(pb);
    const auto s = x.q.sizes();
    if (a.scalar_type() != x.q.scalar_type() || b.scalar_type() != x.q.scalar_type() || !gpu_like(a, x.q.device()) || !gpu_like(b, x.q.device()))
        return false;
    if (!same_sizes(a, {s[0], 2 * s[1], s[2], s[3]}) || !same_sizes(b, {s[0], 2 * s[1], s[2], s[3]})) return false;
    x.a = a; x.b = b;
    return true;
}
// beta [B,T,H] or [B,T,H,1]; keeps the tensor as given
bool read_beta(PyObject* p, ChunkIn& x) {
    if (!is_tensor(p)) return false;
    const Tensor& t = unpack(p);
    const auto s = x.q.sizes();
    if (t.scalar_type() != x.q.scalar_type() || !gpu_like(t, x.q.device())) return false;
    if (!same_sizes(t, {s[0], s[1], s[2], 1}) && !same_sizes(t, {s[0], s[1], s[2]})) return false;
    x.beta = t;
    return true;
}
inline bool wants_grad(const Tensor& t) { return t.defined() && t.requires_grad(); }
bool any_grad(const ChunkIn& x) {
    return c10::GradMode::is_enabled() && (wants_grad(x.q) || wants_grad(x.k) || wants_grad(x.v) || wants_grad(x.a) || wants_grad(x.b) ||
                                           wants_grad(x.beta) || wants_grad(x.gk) || wants_grad(x.h0));
}
void make_contiguous(ChunkIn& x) {
    x.q = x.q.contiguous(); x.k = x.k.contiguous(); x.v = x.v.contiguous(); x.gk = x.gk.contiguous();
    if (x.a.defined()) { x.a = x.a.contiguous(); x.b = x.b.contiguous(); }
    if (x.beta.defined()) x.beta = x.beta.contiguous();
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap_or_none(const Tensor& t) { return t.defined() ? THPVariable_Wrap(t) : none(); }
PyObject* pair(const Tensor& a, const Tensor& b) {
    PyObject* r = PyTuple_New(2);
    if (!r) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(a));
    PyTuple_SET_ITEM(r, 1, wrap_or_none(b));
    return r;
}

// The interpreter lock is given back while a call allocates and launches, as torch's own operators do: nothing in between touches
// a Python object (what does, such as a saved-tensor hook, takes the lock itself).
struct Unlocked {
    PyThreadState* const state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    Unlocked& operator=(const Unlocked&) = delete;
};
template <typename F> auto unlocked(F fn) {
    const Unlocked u;
    return fn();
}

// runs fn, turning C++ exceptions into Python ones
template <typename F> PyObject* guarded(F fn) {
    try {
        return fn();
    } catch (const AbiError& e) {
        PyErr_SetString(error_class ? error_class : PyExc_RuntimeError, e.what());
    } catch (const c10::OutOfMemoryError& e) {
        PyErr_SetString(memory_error ? memory_error : PyExc_MemoryError, e.what_without_backtrace());
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (python_error& e) {                           // raised by Python code on the way (a saved-tensor hook)
        e.restore();
    } catch (const std::exception& e) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

PyObject* run_chunk(ChunkIn& x, PyObject* pscale, PyObject* pwant, PyObject* pkeep) {
    bool want = false, keep = false;
    double scale = 0;
    if (!truth(pwant, want)) return none();
    if (pkeep == Py_None ? keep_forward_default() : (!truth(pkeep, keep) || keep)) return none();
    if (pscale == Py_None) scale = std::pow((double)x.q.size(3), -0.5);
    else if (!number(pscale, scale)) return none();
    Plan plan;
    if (!read_plan(plan)) return none();
    plan.keep = pkeep == Py_None && keep_forward_unsaid() ? KEEP_FORWARD : KEEP_NOTHING;
    return guarded([&]() -> PyObject* {
        hdla_dims d;
        chunk_dims(x, scale, plan, d);
        Tensor o, ht;
        unlocked([&] {
            const at::DeviceGuard guard(x.q.device());
            make_contiguous(x);
            if (any_grad(x)) {
                const auto r = ChunkFn::apply(x.q, x.k, x.v, maybe(x.a), maybe(x.b), maybe(x.beta), x.gk, maybe(x.h0), maybe(x.cu), scale, want,
                                              plan);
                o = r[0];
                if (want) ht = r[1];
                return;
            }
            if (x.h0.defined()) x.h0 = x.h0.to(at::kFloat).contiguous();
            Tensor left;
            chunk_forward(x, d, want, nullptr, o, ht, left);
        });
        return pair(o, ht);
    });
}

// chunk(q, k, v, a, b, gk, RANK_AB, scale, initial_state, output_final_state, head_first, chunk_size, cu_seqlens, keep_forward)
PyObject* py_chunk(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 14) return none();
    ChunkIn x;
    bool head_first = false;
    if (!PyLong_CheckExact(a[6]) || PyLong_AsLong(a[6]) != 2 || !PyLong_CheckExact(a[11]) || PyLong_AsLong(a[11]) < 1) { PyErr_Clear(); return none(); }
    if (!truth(a[10], head_first) || head_first) return none();
    if (!read_operands(a[0], a[1], a[2], a[5], a[8], a[12], false, x) || !read_ab(a[3], a[4], x)) return none();
    return run_chunk(x, a[7], a[9], a[13]);
}

// chunk_hdla(q, k, v, beta, log_f, scale, initial_state, output_final_state, cu_seqlens, keep_forward)
PyObject* py_chunk_hdla(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 10) return none();
    ChunkIn x;
    if (!read_operands(a[0], a[1], a[2], a[4], a[6], a[8], false, x) || !read_beta(a[3], x)) return none();
    return run_chunk(x, a[5], a[7], a[9]);
}

// ---- the token-serial operators: no gradients ------------------------------------------------------------------------
PyObject* run_recurrent(ChunkIn& x, PyObject* pscale, PyObject* pwant, PyObject* preverse) {
    bool want = false, reverse = false;
    double scale = 0;
    if (any_grad(x) || !truth(pwant, want) || !truth(preverse, reverse)) return none();
    if (pscale == Py_None) scale = std::pow((double)x.q.size(3), -0.5);
    else if (!number(pscale, scale)) return none();
    Plan plan;
    if (!read_plan(plan)) return none();
    return guarded([&]() -> PyObject* {
        hdla_dims d;
        chunk_dims(x, scale, plan, d);
        Tensor o, ht;
        unlocked([&] {
            const at::DeviceGuard guard(x.q.device());
            make_contiguous(x);
            if (x.h0.defined()) x.h0 = x.h0.to(at::kFloat).contiguous();
            o = x.cu.defined() ? at::zeros_like(x.v) : at::empty_like(x.v);      // rows of no sequence stay zero
            if (want) ht = at::empty({d.N, d.H, d.K, d.V}, x.q.options().dtype(at::kFloat));
            if (x.beta.defined())
                check(api.param_recurrent_fwd(&d, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.beta), ptr(x.gk), reverse, fptr(x.h0), ptr(o), fptr(ht),
                                              stream_of(x.q)), "hdla_param_recurrent_fwd");
            else
                check(api.recurrent_fwd(&d, ptr(x.q), ptr(x.k), ptr(x.v), ptr(x.a), ptr(x.b), ptr(x.gk), reverse, fptr(x.h0), ptr(o), fptr(ht),
                                        stream_of(x.q)), "hdla_recurrent_fwd");
        });
        return pair(o, ht);
    });
}

// recurrent(q, k, v, a, b, gk, rank_ab, scale, initial_state, output_final_state, reverse, cu_seqlens, head_first)
PyObject* py_recurrent(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 13) return none();
    ChunkIn x;
    bool head_first = false;
    if (!PyLong_CheckExact(a[6]) || PyLong_AsLong(a[6]) != 2) { PyErr_Clear(); return none(); }
    if (!truth(a[12], head_first) || head_first) return none();
    if (!read_operands(a[0], a[1], a[2], a[5], a[8], a[11], true, x) || !read_ab(a[3], a[4], x)) return none();
    return run_recurrent(x, a[7], a[9], a[10]);
}

// recurrent_hdla(q, k, v, beta, log_f, scale, initial_state, output_final_state, reverse, cu_seqlens)
PyObject* py_recurrent_hdla(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 10) return none();
    ChunkIn x;
    if (!read_operands(a[0], a[1], a[2], a[4], a[6], a[9], true, x) || !read_beta(a[3], x)) return none();
    return run_recurrent(x, a[5], a[7], a[8]);
}

// ---- the fused normalisation -----------------------------------------------------------------------------------------
hdla_norm_dims norm_dims(const Tensor& x, const Tensor& w, int gate_pos, double c, double eps, int64_t groups) {
    hdla_norm_dims d{};
    const int64_t D = x.size(-1);
    d.rows = D ? x.numel() / D : 0;
    d.G = (int32_t)groups; d.E = (int32_t)(D / groups);
    d.dtype = dtype_code(x.scalar_type());
    d.weight_dtype = w.defined() ? dtype_code(w.scalar_type()) : HDLA_FP32;
    d.gate_pos = gate_pos; d.c = (float)c; d.eps = (float)eps;
    return d;
}
Tensor norm_forward(const Tensor& x, const Tensor& w, const Tensor& gate, const hdla_norm_dims& d) {
    Tensor o = at::empty_like(x);
    check(api.normalize_fwd(&d, ptr(x), ptr(w), ptr(gate), ptr(o), stream_of(x)), "hdla_normalize_fwd");
    return o;
}
struct NormFn : torch::autograd::Function<NormFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Maybe& weight, const Maybe& g, int64_t gate_pos, double c, double eps,
                          int64_t groups) {
        const Tensor w = value(weight), gate = value(g);
        ctx->save_for_backward({x, w, gate});
        ctx->saved_data["p"] = gate_pos; ctx->saved_data["c"] = c; ctx->saved_data["e"] = eps; ctx->saved_data["g"] = groups;
        return norm_forward(x, w, gate, norm_dims(x, w, (int)gate_pos, c, eps, groups));
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return in_backward([&] { return gradients(ctx, grads); });
    }
    static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &w = s[1], &gate = s[2];
        const at::DeviceGuard guard(x.device());
        const hdla_norm_dims d = norm_dims(x, w, (int)ctx->saved_data["p"].toInt(), ctx->saved_data["c"].toDouble(),
                                           ctx->saved_data["e"].toDouble(), ctx->saved_data["g"].toInt());
        const Tensor d_o = grads[0].to(x.scalar_type()).contiguous();
        const Tensor dx = at::empty_like(x);
        Tensor dgate, dw, ws;
        if (gate.defined()) dgate = at::empty_like(x);
        size_t nws = 0;
        if (w.defined()) {
            dw = at::empty(w.sizes(), w.options());
            nws = api.normalize_workspace_bytes(&d);
            ws = bytes_like(x, nws < 16 ? 16 : nws);
        }
        check(api.normalize_bwd_as(&d, ptr(x), ptr(w), ptr(gate), ptr(d_o), ptr(dx), ptr(dgate), ptr(dw), ptr(ws), nws, stream_of(x)),
              "hdla_normalize_bwd_as");
        return {dx, dw, dgate, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// normalize(x, weight, bias, residual, gate, gate_act, gate_pos, c, eps, use_mean, num_groups, return_residual)
PyObject* py_normalize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 12 || !api.strerror || !is_tensor(a[0]) || a[2] != Py_None || a[3] != Py_None || a[9] != Py_False || a[11] != Py_False) return none();
    Tensor x = unpack(a[0]), w, gate;
    const at::Device dev = x.device();
    if (!dev.is_cuda() || !native_dtype(x.scalar_type()) || !gpu_like(x, dev) || x.dim() < 1) return none();
    const int64_t D = x.size(-1);
    if (!PyLong_CheckExact(a[10])) return none();
    const int64_t groups = PyLong_AsLongLong(a[10]);
    if (groups < 1 || D < 1 || D % groups) { PyErr_Clear(); return none(); }
    if (a[1] != Py_None) {
        if (!is_tensor(a[1])) return none();
        w = unpack(a[1]);
        if (!gpu_like(w, dev) || !native_dtype(w.scalar_type()) || w.numel() != D) return none();
    }
    int64_t pos = 0;
    if (a[4] != Py_None) {
        if (!is_tensor(a[4]) || !PyUnicode_Check(a[5]) || PyUnicode_CompareWithASCIIString(a[5], "sigmoid") || !PyUnicode_Check(a[6])) return none();
        gate = unpack(a[4]);
        pos = !PyUnicode_CompareWithASCIIString(a[6], "pre") ? 1 : !PyUnicode_CompareWithASCIIString(a[6], "post") ? 2 : 0;
        if (!pos || !gpu_like(gate, dev) || gate.sizes() != x.sizes() || gate.scalar_type() != x.scalar_type()) return none();
    }
    double c = 0, eps = 0;
    if (!number(a[7], c) || !number(a[8], eps)) return none();
    return guarded([&]() -> PyObject* {
        return THPVariable_Wrap(unlocked([&] {
            const at::DeviceGuard guard(dev);
            x = x.contiguous();
            if (w.defined()) w = w.contiguous();
            if (gate.defined()) gate = gate.contiguous();
            if (c10::GradMode::is_enabled() && (wants_grad(x) || wants_grad(w) || wants_grad(gate)))
                return NormFn::apply(x, maybe(w), maybe(gate), pos, c, eps, groups);
            return norm_forward(x, w, gate, norm_dims(x, w, (int)pos, c, eps, groups));
        }));
    });
}

// ---- the layer -------------------------------------------------------------------------------------------------------
// HDLA_Custom.forward in its common form (bf16, silu activations, one block, beta, output gate, no biases; layer.py checks
// that) as one call and one autograd node.  What one node buys over one per step: the GEMMs read the inner activations of
// the low-rank projections where they lie in y and write their gradients where they belong in dy (no copies), the rows of
// the concatenated weight can be padded to what the GEMMs like, and the host is out of the way (200 us of Python
// around a decode step's kernels of 4-10 us each).
struct LayerCfg {
    int64_t H, groups;
    bool norm_q, norm_v;
    double beta_scale, c, eps;
    int gate_pos;
};
constexpr int RECURRENT_BELOW = 9;               // see layer.py
constexpr double PRE_EPS = 1e-5;                 // l2_norm's

// Columns of y: q, k, v (d each), the inner activations of decay and gate (D each), beta (H), padding.
struct LayerCols {
    int64_t d, D, H, f0, g0, beta, used, ld;
    LayerCols(int64_t d_, int64_t H_, bool padded) : d(d_), D(d_ / H_), H(H_) {
        f0 = 3 * d; g0 = f0 + D; beta = g0 + D; used = beta + H;
        // The GEMM on x runs at its best on output widths that are whole tiles of 256 (8192 x 3216 x 1024: 82 us, with
        // 3328 columns 50; its input gradient 60 -> 55, its weight gradient 86 -> 80).  Short calls read the weight once and are
        // bound by that: there only up to the 16 bytes that rows are aligned to.
        ld = padded ? (used + 255) / 256 * 256 : (used + 7) / 8 * 8;
    }
};
constexpr int64_t PAD_FROM_ROWS = 1024;
// Rows of the weight in training, and columns of y's gradient: where that makes the weight's gradient one of the library's own (own_weight_grad), up to whole tiles of its kernel: a
// BLAS call less, and both weight gradients in one launch.  (y itself is as wide as without gradients, and so the same call's, bit for bit: a part of a model that is checkpointed runs
// once without them.)  us a training step (all of these are bound by the host): 4 x 121 tokens, 256 channels 239 -> 218, 1 x 64, 512 246 -> 222,
// 2 x 500, 512 275 -> 248, 1 x 512, 1024 271 -> 245, 1 x 1000, 1024 273 -> 246.  Wider layers, whose gradient has more tiles, stay as they are (1 x 900, 2048 384 and 379).
int64_t training_rows(const LayerCols& L, int64_t rows) {
    const int64_t tiles = (L.used + 127) / 128;
    return rows < PAD_FROM_ROWS && L.d % 128 == 0 && tiles * (L.d / 128) <= 256 ? 128 * tiles : L.ld;
}

// the concatenated projection weight [n, d], in `out` if there is one; rows behind the last projection are zero
Tensor gather_weights(const Tensor* w, const LayerCols& L, int64_t n, Tensor out = Tensor()) {       // wq, wk, wv, wf0, wg0, wbeta
    if (!out.defined()) out = at::empty({n, L.d}, w[0].options());
    const void* parts[6];
    int64_t rows[6];
    std::vector<Tensor> whole(6);                                  // (a parameter may be a view at any address)
    for (int i = 0; i < 6; ++i) {
        whole[i] = off_grid(w[i]) ? w[i].detach().clone() : w[i];
        parts[i] = whole[i].data_ptr();
        rows[i] = whole[i].size(0);
    }
    check(api.stack_rows(parts, rows, 6, L.d, ptr(out), n, stream_of(out)), "hdla_stack_rows");
    return out;
}
hdla_pre_dims pre_dims(const LayerCols& L, const LayerCfg& f, int64_t rows) {
    hdla_pre_dims p{};
    p.rows = rows; p.H = (int32_t)L.H; p.D = (int32_t)L.D; p.dtype = HDLA_BF16; p.ldy = (int32_t)L.ld;
    p.col_q = 0; p.col_k = (int32_t)L.d; p.col_v = (int32_t)(2 * L.d); p.col_beta = (int32_t)L.beta;
    p.norm_q = f.norm_q; p.norm_k = 1; p.norm_v = f.norm_v;
    p.beta_scale = (float)f.beta_scale; p.eps = (float)PRE_EPS;
    p.zero_from = (int32_t)L.used;
    return p;
}
hdla_up_dims up_dims(const LayerCols& L, int64_t rows, int64_t ld) {
    hdla_up_dims u{};
    u.rows = rows; u.d = (int32_t)L.d; u.D = (int32_t)L.D; u.ld = ld; u.col_f = (int32_t)L.f0; u.col_g = (int32_t)L.g0;
    return u;
}
// Products of some hundred rows by hdla_tile_gemm: what is one round of its workgroups on the device (figures there).  us a call, BLAS -> this: a decode step
// of 100 sequences, 1024 channels 58 -> 37, of 256, 512 57 -> 30; training steps, bound by the host, 4 x 121 tokens, 256 channels 334 -> 261, 1 x 512, 1024 333 -> 285,
// 4 x 1000, 512 320 -> 317; 2 x 1024, 2048 channels, one product of four, 579 -> 565.
Tensor tile_gemm(const Tensor& x, const Tensor& w, bool turned) {
    const int64_t M = x.size(0), K = x.size(1), N = w.size(turned ? 1 : 0);
    if ((M + 63) / 64 * ((N + 63) / 64) > 256 || K < 8 || K % 8 || N < 8 || N % (turned ? 64 : 8) || x.stride(1) != 1 || w.stride(1) != 1 || x.stride(0) % 8 ||
        w.stride(0) % 8 || x.stride(0) < K || w.stride(0) < w.size(1) || off_grid(x) || off_grid(w)) return at::mm(x, turned ? w : w.t());
    const Tensor y = at::empty({M, N}, x.options());
    check(api.tile_gemm((int32_t)M, (int32_t)N, (int32_t)K, ptr(x), x.stride(0), ptr(w), w.stride(0), turned, ptr(y), N, stream_of(x)), "hdla_tile_gemm");
    return y;
}
// x w^T.  For the few rows of a decode step by hdla_rows_gemm, which is a launch where the BLAS call is 19 us of host time.
// GPU time alone (us, here / there, weights from HBM): 16 x 6416 x 2048 9.0/13.0,
// 64 x 6416 x 2048 12.1/13.5, 64 x 4096 x 4096 14.6/15.0, 16 x 12576 x 4096 24.4/27.0; with more than 16 rows of x, which every
// workgroup reads, the BLAS kernels' larger tiles win from there on: 32 x 12576 x 4096 29.3/25.1, 64 rows 35.4/26.6.
constexpr int64_t FEW_ROWS = 64;
Tensor project(const Tensor& x, const Tensor& w) {
    const int64_t M = x.size(0), most = (M <= 16 ? int64_t(64) : int64_t(16)) << 20;
    if (M > FEW_ROWS) return tile_gemm(x, w, false);
    if (w.numel() > most) return at::mm(x, w.t());
    const Tensor y = at::empty({x.size(0), w.size(0)}, x.options());
    check(api.rows_gemm((int32_t)x.size(0), (int32_t)w.size(0), (int32_t)w.size(1), ptr(x), x.stride(0), ptr(w), w.stride(0), ptr(y), y.stride(0),
                        stream_of(x)), "hdla_rows_gemm");
    return y;
}
// everything between x and the output; what the backward pass needs of it
struct LayerFwd { Tensor x, w, y, f, g, o, n, out, ht, left; ChunkIn op; hdla_dims dims; };

// A few tokens: what is between the projections in one to three launches, without the tensors that the steps would hand on (see
// in_few_launches).  One token after a cached state, us a
// call, as six launches and eleven tensors -> as this (batch x channels, heads): 1 x 512, 8 37.8 -> 19.7, 16 x 2048, 16 36.9 -> 24.3,
// 25 x 4096, 32 67.7 -> 54.5, 256 x 1024, 16 71 -> 57, 256 x 4096, 32 281 -> 249.  The low-rank products in the same launch or in
// one before it (and the norm in one of its own): 23.9 / 26.8, 25.2 / 27.0, 54.5 / 55.9, 57 / 60, 249 / 252; the other way round only at 256 x 2048, 32: 85.3 / 84.5.
void layer_step(const Tensor* P, const LayerCfg& f, const LayerCols& L, const hdla_pre_dims& pd, int64_t T, const Tensor& h0, bool want_ht,
                LayerFwd& r) {
    const int64_t rows = pd.rows, N = rows / T;
    void* const s = stream_of(r.x);
    const auto opt = r.x.options();
    const bool in_step = T == 1, norm_in_step = f.groups == L.H;
    // A norm over all channels of at most 16 rows: formed where the projection reads it, by every workgroup of the projection for itself.
    // A launch less, which the host is glad of, but what the workgroups read grows with the square of the channels.  us a call, in a launch
    // of its own / here: 1 x 512 24.1 / 19.7, 16 x 1024 24.9 / 19.7, 3 x 2048 24.5 / 21.9, 16 x 2048 25.2 / 24.3; wider ones on the
    // device: 3 x 2560, 40 23.4 / 24.6 (the host 25.3 / 24.7), 3 x 3072, 48 26.6 / 28.6, 3 x 3584, 28 33.1 / 35.3, 1 x 4096, 32 39.2 / 41.8.
    const bool later = !norm_in_step && f.groups == 1 && rows <= 16 && L.d <= 2048, own_norm = !norm_in_step && !later;
    if (!later) r.n = at::empty({rows, L.d}, opt);
    const hdla_up_dims ud = up_dims(L, rows, L.ld);
    const hdla_norm_dims nd = norm_dims(r.x, P[8], f.gate_pos, f.c, f.eps, f.groups);
    // gate, o, log_f and the gated o (fp32) with its sums, as far as they are handed on
    const int64_t one = rows * L.d, parts = (own_norm ? 2 : 0) + (in_step ? 0 : own_norm ? 1 : 2);
    Tensor between;
    if (parts || later) between = at::empty({parts * one + (later ? 2 * (one + rows * L.H) : 0)}, opt);
    char* room = static_cast<char*>(ptr(between));
    void *gate = nullptr, *o = ptr(r.n), *log_f = nullptr;
    const auto take = [&] { void* const p = room; room += one * 2; return p; };
    if (own_norm) o = take();
    if (own_norm || !in_step) gate = take();
    if (!in_step) {
        log_f = take();
        check(api.layer_up_fwd(&ud, ptr(r.y), ptr(P[6]), ptr(P[7]), nullptr, log_f, gate, s), "hdla_layer_up_fwd");
    }
    Tensor state;
    if (h0.defined()) state = h0.to(at::kFloat).contiguous();
    if (want_ht) r.ht = at::empty({N, L.H, L.D, L.D}, opt.dtype(at::kFloat));
    float* const gated = later ? reinterpret_cast<float*>(room) : nullptr;
    check(api.layer_step(&pd, in_step ? &ud : nullptr, own_norm ? nullptr : &nd, (int32_t)T, ptr(r.y), in_step ? ptr(P[6]) : nullptr,
                         in_step ? ptr(P[7]) : nullptr, log_f, gate, norm_in_step ? ptr(P[8]) : nullptr, fptr(state), o, gated, fptr(r.ht), s),
          "hdla_layer_step");
    if (later) {
        const Tensor &w = P[9];
        r.out = at::empty({rows, L.d}, opt);
        check(api.rows_gemm_norm((int32_t)rows, (int32_t)L.d, (int32_t)L.d, gated, (int32_t)L.H, &nd, ptr(P[8]), ptr(w), w.stride(0), ptr(r.out),
                                 r.out.stride(0), s), "hdla_rows_gemm_norm");
        return;
    }
    if (own_norm) check(api.normalize_fwd(&nd, o, ptr(P[8]), gate, ptr(r.n), s), "hdla_normalize_fwd");
    r.out = project(r.n, P[9]);
}

// Whether layer_step takes the tokens of a token-serial call.  It works a head's tokens off one after the other; with several tokens of
// many sequences the steps are the faster, which do what does not depend on the state for all tokens at once.  One token: always.  us on the device, steps / here
// (sequences x tokens, channels, heads).  With the norm in layer_step's launch: 256 x 2 4096, 32 304/300; 48 x 8 1024, 16 56/52; 128 x 6 74.7/72.7;
// 128 x 8 84/84; 256 x 8 134/139; 64 x 3 2048, 16 74/71; 48 x 8 95/101; 256 x 8 315/371; 24 x 8 4096, 32 127/128; 64 x 8 217/232; 256 x 8 698/815.  With it in a
// launch of its own: 64 x 3 1024, 16 44.7/41.7; 48 x 8 56.7/57.8 (the host 72/61); 128 x 8 84/89; 24 x 8 2048, 32 63.0/64.4; 64 x 8 95/99; 16 x 8 4096, 32 96/97;
// 64 x 8 217/240; 256 x 8 695/809; 256 x 2 2048, 16 150/155.
bool in_few_launches(int64_t rows, int64_t T, int64_t d, bool norm_in_step) {
    if (T == 1 || (T == 2 && norm_in_step)) return true;
    return rows * d <= (norm_in_step ? 3 << 18 : 3 << 17);
}

// params: wq, wk, wv, wf0, wg0, wbeta, wf1, wg1, wnorm, wo; r.w gathered; keep: a backward pass follows (which plan is for then)
void layer_forward(const Tensor& x3, const Tensor* P, const LayerCfg& f, Plan& plan, const Tensor& h0, bool want_ht, bool chunked, bool keep,
                   LayerFwd& r) {
    const int64_t B = x3.size(0), T = x3.size(1), d = x3.size(2), rows = B * T;
    const LayerCols L(d, f.H, rows >= PAD_FROM_ROWS);
    const auto opt = x3.options();
    r.x = x3.contiguous().view({rows, d});
    r.y = project(r.x, r.w.size(0) == L.ld ? r.w : r.w.narrow(0, 0, L.ld));
    const hdla_pre_dims pd = pre_dims(L, f, rows);
    if (!chunked && T < RECURRENT_BELOW && in_few_launches(rows, T, d, f.groups == f.H)) {
        layer_step(P, f, L, pd, T, h0, want_ht, r);
        r.out = r.out.view({B, T, d});
        return;
    }
    ChunkIn& in = r.op;
    in.q = at::empty({B, T, L.H, L.D}, opt); in.k = at::empty({B, T, L.H, L.D}, opt); in.v = at::empty({B, T, L.H, L.D}, opt);
    in.beta = at::empty({B, T, L.H, 1}, opt);
    void* const s = stream_of(x3);
    check(api.layer_pre_fwd(&pd, ptr(r.y), ptr(in.q), ptr(in.k), ptr(in.v), ptr(in.beta), s), "hdla_layer_pre_fwd");
    const hdla_up_dims ud = up_dims(L, rows, L.ld);
    if (keep) r.f = at::empty({rows, d}, opt);
    in.gk = at::empty({B, T, L.H, L.D}, opt);
    r.g = at::empty({rows, d}, opt);
    check(api.layer_up_fwd(&ud, ptr(r.y), ptr(P[6]), ptr(P[7]), ptr(r.f), ptr(in.gk), ptr(r.g), s), "hdla_layer_up_fwd");
    if (h0.defined()) in.h0 = h0.to(at::kFloat).contiguous();
    hdla_dims& cd = r.dims;
    chunk_dims(in, 1.0, plan, cd);
    if (chunked) {
        chunk_forward(in, cd, want_ht, keep ? &plan : nullptr, r.o, r.ht, r.left);
    } else {
        r.o = at::empty_like(in.v);
        if (want_ht) r.ht = at::empty({cd.N, cd.H, cd.K, cd.V}, opt.dtype(at::kFloat));
        check(api.param_recurrent_fwd(&cd, ptr(in.q), ptr(in.k), ptr(in.v), ptr(in.beta), ptr(in.gk), 0, fptr(in.h0), ptr(r.o), fptr(r.ht), s),
              "hdla_param_recurrent_fwd");
    }
    const Tensor o2 = r.o.view({rows, d});
    r.n = norm_forward(o2, P[8], r.g, norm_dims(o2, P[8], f.gate_pos, f.c, f.eps, f.groups));
    r.out = project(r.n, P[9]).view({B, T, d});
}

// dW [n, k] = dY [rows, n]^T X [rows, k].  Up to one round of whole 128 x 128 tiles on the device by the library's own kernel (us
// within a training step: 8192 rows, 3328 x 1024 102 -> 82, 1024 x 1024 33 -> 30; 4000 rows, 2048 x 2048 56 -> 44; 1500 rows, 3328 x 1024 30 -> 17; but
// 4000 rows, 6656 x 2048, 832 tiles: 128 and 147).  The line: one call behind the other, 16 to 8192 rows, 2 to 256 tiles are all faster (4096 rows, 256 tiles
// 44 -> 38), but a second round of workgroups for a few tiles costs what it gains: 288 tiles, 1000 / 2048 / 4096 / 8192 rows 27 -> 23, 33 -> 35, 59 -> 62,
// 114 -> 115; 512 tiles 29 -> 30, 39 -> 43, 68 -> 75, 130 -> 135.  Others: an output of few tiles would leave most of the chip idle (1024 x 1024 over 8192 rows: 54 us), so the rows are split over a batch
// of products whose fp32 results one kernel adds (28 + 4 us).
bool own_weight_grad(const Tensor& dy, const Tensor& x) {
    const int64_t rows = dy.size(0), n = dy.size(1), k = x.size(1);
    return rows > 0 && rows <= 0x7fff0000 && n > 0 && k > 0 && n % 128 == 0 && k % 128 == 0 && n / 128 * (k / 128) <= 256 && dy.stride(1) == 1 &&
           x.stride(1) == 1 && dy.stride(0) >= n && x.stride(0) >= k && dy.stride(0) % 8 == 0 && x.stride(0) % 8 == 0 && !off_grid(dy) && !off_grid(x);
}
Tensor weight_grad(const Tensor& dy, const Tensor& x) {
    const int64_t rows = dy.size(0), n = dy.size(1), k = x.size(1);
    if (own_weight_grad(dy, x)) {
        const Tensor dw = at::empty({n, k}, dy.options());
        const size_t nws = api.weight_grad_workspace_bytes(rows, (int32_t)n, (int32_t)k);
        const Tensor ws = nws ? bytes_like(x, nws) : Tensor();
        check(api.weight_grad(rows, (int32_t)n, (int32_t)k, ptr(dy), dy.stride(0), ptr(x), x.stride(0), ptr(dw), ptr(ws), nws, stream_of(dy)),
              "hdla_weight_grad");
        return dw;
    }
    const int64_t tiles = ((n + 127) / 128) * ((k + 127) / 128);
    int64_t S = 1;
    while (S < 8 && tiles * S * 2 <= 256 && rows % (S * 2) == 0 && rows / (S * 2) >= 1024) S *= 2;
    if (S == 1 || dy.stride(0) != n || x.stride(0) != k || n * k % 8) return at::mm(dy.t(), x);
    const Tensor part = at::bmm(dy.view({S, rows / S, n}).transpose(1, 2), x.view({S, rows / S, k}), at::kFloat);
    const Tensor dw = at::empty({n, k}, dy.options());
    check(api.sum_partials(fptr(part), (int32_t)S, n * k, ptr(dw), stream_of(dy)), "hdla_sum_partials");
    return dw;
}
// Sums over partial results that a backward pass leaves for its end, and what they are read from
struct Sums {
    hdla_sum of[4] = {};
    Tensor room[3];
};
// Two of them over the same rows: in one launch where each is the library's own (figures in wgrad.hip).
void weight_grads(const Tensor (&dy)[2], const Tensor (&x)[2], Tensor (&dw)[2], hdla_sum& sum, Tensor& ws) {
    if (!own_weight_grad(dy[0], x[0]) || !own_weight_grad(dy[1], x[1])) {
        for (int i = 0; i < 2; ++i) dw[i] = weight_grad(dy[i], x[i]);
        return;
    }
    int32_t n[2], k[2];
    int64_t ldy[2], ldx[2];
    const void *pdy[2], *px[2];
    void* pdw[2];
    for (int i = 0; i < 2; ++i) {
        n[i] = (int32_t)dy[i].size(1);
        k[i] = (int32_t)x[i].size(1);
        dw[i] = at::empty({n[i], k[i]}, dy[i].options());
        ldy[i] = dy[i].stride(0);
        ldx[i] = x[i].stride(0);
        pdy[i] = ptr(dy[i]);
        px[i] = ptr(x[i]);
        pdw[i] = ptr(dw[i]);
    }
    const size_t nws = api.weight_grad_pair_workspace_bytes(dy[0].size(0), n, k);
    if (nws) ws = bytes_like(x[0], nws);
    check(api.weight_grad_pair(dy[0].size(0), n, k, pdy, ldy, px, ldx, pdw, ptr(ws), nws, &sum, stream_of(dy[0])), "hdla_weight_grad_pair");
}
struct LayerFn : torch::autograd::Function<LayerFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& wq, const Tensor& wk, const Tensor& wv, const Tensor& wf0,
                                 const Tensor& wg0, const Tensor& wbeta, const Tensor& wf1, const Tensor& wg1, const Tensor& wnorm,
                                 const Tensor& wo, const Maybe& h0, const LayerCfg& f, bool want_ht, Plan plan) {
        const Tensor P[10] = {wq, wk, wv, wf0, wg0, wbeta, wf1, wg1, wnorm, wo};
        LayerFwd r;
        const int64_t rows = x.size(0) * x.size(1);
        const LayerCols L(x.size(2), f.H, rows >= PAD_FROM_ROWS);
        r.w = gather_weights(P, L, training_rows(L, rows));
        layer_forward(x, P, f, plan, value(h0), want_ht, true, true, r);
        save_plan(ctx, plan);
        ctx->save_for_backward({r.x, r.w, r.y, r.f, r.g, r.o, r.n, r.left, r.op.q, r.op.k, r.op.v, r.op.beta, r.op.gk, value(h0), wf1, wg1,
                                wnorm, wo});
        ctx->saved_data["c"] = std::vector<double>{f.beta_scale, f.c, f.eps};
        ctx->saved_data["i"] = std::vector<int64_t>{f.H, f.groups, f.norm_q, f.norm_v, f.gate_pos, x.size(0), x.size(1)};
        ctx->set_materialize_grads(false);
        return want_ht ? variable_list{r.out, r.ht} : variable_list{r.out};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return in_backward([&] { return gradients(ctx, grads); });
    }
    static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
        // backward() may be called inside an autocast region although the forward pass ran outside one.  The engine carries that
        // state to this thread, and torch's products below would come out in the region's type where kernels read bf16.
        const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::DispatchKey::AutocastCUDA);
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &w = s[1], &y = s[2], &f = s[3], &g = s[4], &o = s[5], &n = s[6], &left = s[7];
        const Tensor &q = s[8], &k = s[9], &v = s[10], &beta = s[11], &gk = s[12], &h0 = s[13], &wf1 = s[14], &wg1 = s[15], &wnorm = s[16],
                     &wo = s[17];
        const at::DeviceGuard guard(x.device());
        const auto cc = ctx->saved_data["c"].toDoubleVector();
        const auto ci = ctx->saved_data["i"].toIntVector();
        const LayerCfg cfg{ci[0], ci[1], ci[2] != 0, ci[3] != 0, cc[0], cc[1], cc[2], (int)ci[4]};
        const int64_t B = ci[5], T = ci[6], rows = x.size(0), d = x.size(1);
        const LayerCols L(d, cfg.H, rows >= PAD_FROM_ROWS);
        void* const stream = stream_of(x);
        const auto opt = x.options();
        const auto need = [&](size_t i) { return ctx->needs_input_grad(i); };
        variable_list out(15);
        Sums sums;

        // output projection and gated norm
        const Tensor dout = grads[0].defined() ? grads[0].to(at::kBFloat16).contiguous().view({rows, d}) : at::zeros({rows, d}, opt);
        const bool projections = need(1) || need(2) || need(3) || need(4) || need(5) || need(6);
        if (need(10) && !projections) out[10] = weight_grad(dout, n);     // (else with theirs)
        const Tensor dn = tile_gemm(dout, wo, true);
        const Tensor o2 = o.view({rows, d}), d_o = at::empty({rows, d}, opt), dgate = at::empty({rows, d}, opt);
        const Tensor dwn = at::empty(wnorm.sizes(), wnorm.options());
        {
            const hdla_norm_dims nd = norm_dims(o2, wnorm, cfg.gate_pos, cfg.c, cfg.eps, cfg.groups);
            const size_t nws = api.normalize_workspace_bytes(&nd);
            sums.room[0] = bytes_like(x, nws < 16 ? 16 : nws);
            check(api.normalize_bwd_later(&nd, ptr(o2), ptr(wnorm), ptr(g), ptr(dn), ptr(d_o), ptr(dgate), ptr(dwn), ptr(sums.room[0]), nws, &sums.of[0], stream),
                  "hdla_normalize_bwd_later");
        }
        if (need(9)) out[9] = dwn;

        // the operator
        Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), dbeta = at::empty_like(beta), dgk = at::empty_like(gk), dh0;
        {
            ChunkIn in{q, k, v, Tensor(), Tensor(), beta, gk, h0, Tensor()};
            if (h0.defined()) { in.h0 = h0.to(at::kFloat).contiguous(); dh0 = at::empty_like(in.h0); }
            Tensor dht;
            if (grads.size() > 1 && grads[1].defined()) dht = grads[1].to(at::kFloat).contiguous();
            hdla_dims cd;
            const Plan plan = saved_plan(ctx);
            chunk_dims(in, 1.0, plan, cd);
            chunk_backward(in, cd, plan, d_o, dht, left, backward_workspace(cd, plan, x, left), ChunkGrads{dq, dk, dv, Tensor(), Tensor(), dbeta, dgk, dh0});
            if (dh0.defined()) out[11] = dh0.to(h0.scalar_type());
        }

        // gradient of y, each part written where it belongs
        const Tensor dy = at::empty({rows, w.size(0)}, opt);
        const hdla_pre_dims pd = pre_dims(L, cfg, rows);
        check(api.layer_pre_bwd_to(&pd, ptr(y), ptr(dq), ptr(dk), ptr(dv), ptr(dbeta), ptr(dy), (int32_t)w.size(0), stream), "hdla_layer_pre_bwd_to");
        const hdla_up_dims ud = up_dims(L, rows, L.ld), down = up_dims(L, rows, w.size(0));
        check(api.layer_down(&down, ptr(wf1), ptr(wg1), ptr(f), ptr(dgk), ptr(dgate), ptr(dy), stream), "hdla_layer_down");
        if (need(7) || need(8)) {
            out[7] = at::empty_like(wf1);
            out[8] = at::empty_like(wg1);
            const size_t nws = api.layer_up_wgrad_workspace_bytes(&ud);
            sums.room[1] = bytes_like(x, nws);
            check(api.layer_up_wgrad_later(&ud, ptr(y), ptr(f), ptr(dgk), ptr(dgate), ptr(out[7]), ptr(out[8]), ptr(sums.room[1]), nws, &sums.of[1], stream),
                  "hdla_layer_up_wgrad_later");
        }

        // the projections of x
        if (projections) {
            Tensor dw;
            if (need(10)) {
                Tensor both[2];
                weight_grads({dy, dout}, {x, n}, both, sums.of[3], sums.room[2]);
                dw = both[0];
                out[10] = both[1];
            } else {
                dw = weight_grad(dy, x);
            }
            const int64_t at_row[7] = {0, d, 2 * d, L.f0, L.g0, L.beta, L.used};
            for (int i = 0; i < 6; ++i) out[1 + i] = dw.narrow(0, at_row[i], at_row[i + 1] - at_row[i]);
        }
        check(api.run_sums(sums.of, 4, stream), "hdla_run_sums");
        if (need(0)) out[0] = tile_gemm(dy, w, true).view({B, T, d});
        return out;
    }
};

// What evaluation mode knows of a concatenated weight that it keeps between calls without gradients.
struct Kept {
    struct Part { const void* p; uint64_t v; } of[7];              // the parameters it was formed from, and its width
    c10::Event ready;                                              // behind the launch that formed it
    c10::Stream made, home;                                        // the stream of that launch, and the one the memory is from
    bool complete = false;                                         // `ready` is known to have passed
    bool captured = false;                                         // a captured graph reads it: it stays where it is
    bool stale = false;                                            // to be formed anew all the same
};
constexpr const char* KEPT = "hdla_hip.kept";
Kept* kept_at(PyObject* list, Py_ssize_t slot) {
    PyObject* const o = PyList_GET_ITEM(list, slot);
    return PyCapsule_IsValid(o, KEPT) ? static_cast<Kept*>(PyCapsule_GetPointer(o, KEPT)) : nullptr;
}
PyObject* kept_capsule(Kept&& k) {
    Kept* const p = new Kept(std::move(k));
    PyObject* const o = PyCapsule_New(p, KEPT, [](PyObject* c) { delete static_cast<Kept*>(PyCapsule_GetPointer(c, KEPT)); });
    if (!o) delete p;
    return o;
}
// of the current device
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }
// an event that a capture has no part in may be asked for while one is under way, if the thread says that it knows
bool has_passed(const c10::Event& e) {
    const c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
    return e.query();
}
// Makes the stream `here` read or write behind the launch that formed the weight.  A graph under capture can only take one that is
// complete: what the replay waits for is not known here.
bool wait_for(Kept& k, const c10::Stream& here, bool under_capture) {
    if (k.complete || (here == k.made && !under_capture)) return true;
    k.complete = has_passed(k.ready);
    if (!k.complete && !under_capture) k.ready.block(here);
    return k.complete || !under_capture;
}

// forget(cache) -> the cache to go on with: what a captured graph reads stays there, to be formed anew in its place by the next call
PyObject* py_forget(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 1 || !PyList_CheckExact(a[0]) || PyList_GET_SIZE(a[0]) != 4) { PyErr_SetString(PyExc_TypeError, "forget(cache)"); return nullptr; }
    PyObject* const out = PyList_New(4);
    if (!out) return nullptr;
    for (Py_ssize_t i = 0; i < 4; ++i) { Py_INCREF(Py_None); PyList_SET_ITEM(out, i, Py_None); }
    for (Py_ssize_t slot = 0; slot < 4; slot += 2) {
        Kept* const k = kept_at(a[0], slot);
        if (!k || !k->captured) continue;
        k->stale = true;
        for (Py_ssize_t i = slot; i < slot + 2; ++i) {
            PyObject* const o = PyList_GET_ITEM(a[0], i);
            Py_INCREF(o);
            PyList_SetItem(out, i, o);
        }
    }
    return out;
}
// passed(event handle) -> whether a torch event has passed; also while a capture is under way
// kept_room(like, bytes): for the Python code of the chunked operators, on the same account; None: no room
PyObject* py_kept_room(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2 || !is_tensor(a[0])) return none();
    const int64_t bytes = PyLong_AsLongLong(a[1]);
    if (bytes < 0) { PyErr_Clear(); return none(); }
    return guarded([&] {
        const Tensor& like = unpack(a[0]);
        return wrap_or_none(unlocked([&] { return kept_room(like, bytes); }));
    });
}

PyObject* py_passed(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 1) { PyErr_SetString(PyExc_TypeError, "passed(event)"); return nullptr; }
    void* const e = PyLong_AsVoidPtr(a[0]);
    if (PyErr_Occurred()) return nullptr;
    return guarded([&]() -> PyObject* {
        const c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
        const hipError_t rc = hipEventQuery(static_cast<hipEvent_t>(e));
        if (rc != hipSuccess) (void)hipGetLastError();
        return PyBool_FromLong(rc == hipSuccess);
    });
}

// layer(x, (wq, wk, wv, wf0, wg0, wbeta, wf1, wg1, wnorm, wo), initial_state, want_state, mode, cache,
//       H, groups, norm_q, norm_v, beta_scale, c, eps, gate_pos) -> (output, state) or None
// mode: 0 chunked with gradients and from RECURRENT_BELOW tokens on, else token-serial; 1 chunked; 2 token-serial
// cache: a list [Kept, weight] x 2 that keeps the concatenated weight, narrow and padded, between calls without gradients, or None
PyObject* py_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 14 || !api.strerror || !is_tensor(a[0]) || !PyTuple_CheckExact(a[1]) || PyTuple_GET_SIZE(a[1]) != 10) return none();
    const Tensor& x = unpack(a[0]);
    const at::Device dev = x.device();
    if (!dev.is_cuda() || x.scalar_type() != at::kBFloat16 || !gpu_like(x, dev) || x.dim() != 3 || x.numel() == 0) return none();
    if (at::autocast::is_autocast_enabled(at::kCUDA)) return none();
    LayerCfg f{};
    f.H = PyLong_AsLongLong(a[6]); f.groups = PyLong_AsLongLong(a[7]);
    f.norm_q = a[8] == Py_True; f.norm_v = a[9] == Py_True;
    const int mode = (int)PyLong_AsLong(a[4]);
    f.gate_pos = (int)PyLong_AsLong(a[13]);
    bool want = false;
    if (!number(a[10], f.beta_scale) || !number(a[11], f.c) || !number(a[12], f.eps) || !truth(a[3], want) || PyErr_Occurred()) { PyErr_Clear(); return none(); }
    const int64_t B = x.size(0), T = x.size(1), d = x.size(2);
    if (f.H < 1 || d % f.H || d % 128 || f.groups < 1 || d % f.groups || B * T > INT32_MAX / 4) return none();
    const int64_t D = d / f.H;
    if (D != 64 && D != 128) return none();
    const int64_t shapes[10][2] = {{d, d}, {d, d}, {d, d}, {D, d}, {D, d}, {f.H, d}, {d, D}, {d, D}, {d, 0}, {d, d}};
    Tensor P[10];
    bool op_grad = wants_grad(x), any = op_grad;
    for (int i = 0; i < 10; ++i) {
        PyObject* o = PyTuple_GET_ITEM(a[1], i);
        if (!is_tensor(o)) return none();
        P[i] = unpack(o);
        if (!gpu_like(P[i], dev) || !P[i].is_contiguous()) return none();
        if (i == 8 ? (P[i].dim() != 1 || P[i].size(0) != d || !native_dtype(P[i].scalar_type()))
                   : (P[i].scalar_type() != at::kBFloat16 || !same_sizes(P[i], {shapes[i][0], shapes[i][1]}))) return none();
        any = any || wants_grad(P[i]);
        op_grad = op_grad || ((i < 4 || i == 5 || i == 6) && wants_grad(P[i]));
    }
    // Kernels of this library read these 16 bytes at a time; the BLAS calls of the Python code take them at any address.  (The
    // weights that multiply x are copied together anyway, gather_weights.)
    const bool few = B * T <= FEW_ROWS;
    if (off_grid(P[6]) || off_grid(P[7]) || (few && (off_grid(P[9]) || (x.is_contiguous() && off_grid(x))))) return none();
    Tensor h0;
    if (a[2] != Py_None) {
        if (!is_tensor(a[2])) return none();
        h0 = unpack(a[2]);
        if (!gpu_like(h0, dev) || !same_sizes(h0, {B, f.H, D, D}) || !h0.is_floating_point()) return none();
        any = any || wants_grad(h0);
    }
    const bool grad = c10::GradMode::is_enabled() && any;
    const bool chunked = mode == 1 || (mode == 0 && ((c10::GradMode::is_enabled() && op_grad) || T >= RECURRENT_BELOW));
    if (grad && !chunked) return none();                         // gradients behind the token-serial operator: as the Python code has it
    if (keep_forward_default() && grad) return none();
    Plan plan;
    if (!read_plan(plan)) return none();
    plan.keep = keep_forward_unsaid() ? KEEP_FORWARD : KEEP_NOTHING;
    return guarded([&]() -> PyObject* {
        Tensor out, ht;
        if (grad) {
            unlocked([&] {
                const at::DeviceGuard guard(dev);
                const auto r = LayerFn::apply(x, P[0], P[1], P[2], P[3], P[4], P[5], P[6], P[7], P[8], P[9], maybe(h0), f, want, plan);
                out = r[0];
                if (want) ht = r[1];
            });
            return pair(out, ht);
        }
        LayerFwd r;
        const LayerCols L(d, f.H, B * T >= PAD_FROM_ROWS);
        const at::DeviceGuard guard(dev);
        // the weight of the last call, as long as the parameters are the ones it was built from, unmodified
        // (each width has its own place: a captured graph of decode steps goes on reading the one while long calls use the other)
        const bool cached = PyList_CheckExact(a[5]) && PyList_GET_SIZE(a[5]) == 4;
        const Py_ssize_t slot = B * T >= PAD_FROM_ROWS ? 2 : 0;
        Kept::Part of[7];
        const c10::Stream here = c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getStream(dev);
        bool built = true, fill = false;                          // fill: in the place that a captured graph reads
        if (cached) {
            for (int i = 0; i < 6; ++i) of[i] = {P[i].data_ptr(), (uint64_t)P[i]._version()};
            of[6] = {nullptr, (uint64_t)L.ld};
            Kept* const k = kept_at(a[5], slot);
            PyObject* const old = PyList_GET_ITEM(a[5], slot + 1);
            if (k && is_tensor(old)) {
                const Tensor& w = unpack(old);
                const bool under_capture = (!k->complete || !k->captured) && capturing();
                if (!k->stale && !memcmp(k->of, of, sizeof of)) {
                    built = !wait_for(*k, here, under_capture);
                    if (!built) {
                        k->captured = k->captured || under_capture;
                        if (here != k->home && !under_capture) w.record_stream(here);
                        r.w = w;
                    }
                } else if (k->captured && w.device() == dev && same_sizes(w, {L.ld, L.d}) && !capturing()) {
                    fill = wait_for(*k, here, false);            // (one launch that forms it behind the other)
                    if (here != k->home) w.record_stream(here);
                    r.w = w;
                }
            }
        }
        std::optional<c10::Event> ready;
        unlocked([&] {
            if (built) {
                r.w = gather_weights(P, L, L.ld, r.w);
                // (one gathered under capture is not there before the graph is replayed, and belongs to it)
                if (cached && !capturing()) {
                    ready.emplace(c10::DeviceType::CUDA);
                    ready->record(here);
                }
            }
            layer_forward(x, P, f, plan, h0, want, chunked, false, r);
        });
        if (ready && PyList_GET_SIZE(a[5]) == 4) {
            // (key and weight one behind the other, with the lock held: another thread sees both or neither)
            const Kept* const now = kept_at(a[5], slot);
            const bool taken = now && now->captured && is_tensor(PyList_GET_ITEM(a[5], slot + 1));
            if (taken && !fill && unpack(PyList_GET_ITEM(a[5], slot + 1)).device() == dev) return pair(r.out, r.ht);    // captured meanwhile
            Kept k{{}, std::move(*ready), here, fill && taken ? now->home : here};
            memcpy(k.of, of, sizeof of);
            k.captured = fill;
            PyObject* const key = kept_capsule(std::move(k));
            if (!key) return nullptr;
            PyObject* const w = THPVariable_Wrap(r.w);
            if (!w) { Py_DECREF(key); return nullptr; }
            PyList_SetItem(a[5], slot, key);
            PyList_SetItem(a[5], slot + 1, w);
        }
        return pair(r.out, r.ht);
    });
}

// ---- module ----------------------------------------------------------------------------------------------------------
// bind(handle of libhdla_hip.so, HdlaError, torch.OutOfMemoryError)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 3) { PyErr_SetString(PyExc_TypeError, "bind(handle, error, memory_error)"); return nullptr; }
    void* h = PyLong_AsVoidPtr(a[0]);
    if (!h) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no library"); return nullptr; }
    Api x{};
#define HDLA_FN(name)                                                                                              \
    if (!(x.name = reinterpret_cast<decltype(x.name)>(dlsym(h, "hdla_" #name)))) {                                 \
        PyErr_SetString(a[1], "the library does not export hdla_" #name);                                          \
        return nullptr;                                                                                            \
    }
    HDLA_FN(strerror) HDLA_FN(workspace_bytes) HDLA_FN(record_bytes) HDLA_FN(record_workspace_bytes) HDLA_FN(chunk_fwd_b) HDLA_FN(chunk_bwd_b)
    HDLA_FN(keep_plan) HDLA_FN(chunk_fwd_keep) HDLA_FN(chunk_bwd_kept) HDLA_FN(states_plan) HDLA_FN(chunk_fwd_states) HDLA_FN(chunk_bwd_states) HDLA_FN(tile_gemm)
    HDLA_FN(layer_pre_bwd_to)
    HDLA_FN(recurrent_fwd) HDLA_FN(param_recurrent_fwd) HDLA_FN(normalize_fwd) HDLA_FN(normalize_bwd_as)
    HDLA_FN(normalize_workspace_bytes) HDLA_FN(layer_pre_fwd) HDLA_FN(layer_pre_bwd) HDLA_FN(layer_up_fwd) HDLA_FN(layer_down)
    HDLA_FN(layer_up_wgrad) HDLA_FN(layer_up_wgrad_workspace_bytes) HDLA_FN(rows_gemm) HDLA_FN(sum_partials) HDLA_FN(stack_rows) HDLA_FN(layer_step)
    HDLA_FN(weight_grad) HDLA_FN(weight_grad_workspace_bytes) HDLA_FN(weight_grad_pair) HDLA_FN(weight_grad_pair_workspace_bytes)
    HDLA_FN(normalize_bwd_later) HDLA_FN(layer_up_wgrad_later) HDLA_FN(run_sums)
    HDLA_FN(rows_gemm_norm)
#undef HDLA_FN
    Py_INCREF(a[1]);
    Py_XDECREF(error_class);
    error_class = a[1];
    Py_INCREF(a[2]);
    Py_XDECREF(memory_error);
    memory_error = a[2];
    api = x;
    return none();
}

#define HDLA_DEF(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    HDLA_DEF("bind", py_bind), HDLA_DEF("chunk", py_chunk), HDLA_DEF("chunk_hdla", py_chunk_hdla), HDLA_DEF("recurrent", py_recurrent),
    HDLA_DEF("recurrent_hdla", py_recurrent_hdla), HDLA_DEF("normalize", py_normalize), HDLA_DEF("layer", py_layer), HDLA_DEF("forget", py_forget), HDLA_DEF("passed", py_passed),
    HDLA_DEF("kept_room", py_kept_room), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
