"""ctypes binding of libhdla_hip.so (the C ABI declared in include/hdla_hip.h).

The library is the only compute path: if it cannot be loaded every operator raises, there is no fallback.
"""
import ctypes
import os
import threading
import warnings
import weakref
from typing import Optional, Tuple

import torch

HDLA_BF16, HDLA_FP32 = 0, 1
HDLA_VERSION = 211          # the header this binding was written against (struct layouts, entry points)
ROUTE_AUTO, ROUTE_CLASSIC, ROUTE_FUSED, ROUTE_PLAIN = 0, 1, 2, 4
_ROUTES = {"": ROUTE_AUTO, "auto": ROUTE_AUTO, "classic": ROUTE_CLASSIC, "plain": ROUTE_PLAIN, "fused": ROUTE_FUSED}
_HERE = os.path.dirname(os.path.abspath(__file__))
_LIB_NAME = "libhdla_hip.so"
_lib = None
_native = None


class HdlaDims(ctypes.Structure):
    _fields_ = [
        ("B", ctypes.c_int32), ("T", ctypes.c_int32), ("H", ctypes.c_int32), ("K", ctypes.c_int32),
        ("V", ctypes.c_int32), ("R", ctypes.c_int32), ("N", ctypes.c_int32),
        ("in_dtype", ctypes.c_int32), ("gk_dtype", ctypes.c_int32), ("scale", ctypes.c_float),
        ("cu_seqlens", ctypes.c_void_p), ("route", ctypes.c_int32), ("segments", ctypes.c_int32),
    ]


class HdlaWsLayout(ctypes.Structure):
    _names = ["nch", "W", "UT", "KGT", "BGT", "VTT", "EGL", "QG", "AQK", "AQB", "AQBT", "QGT", "TM",
              "HC", "DHC", "DVN", "STRONG", "SA_STRIDE", "SB_STRIDE", "CHUNK_OFF", "CHUNK_SEQ", "total", "ERR", "AAK", "AAK_STRIDE", "SUM"]
    _fields_ = [(n, ctypes.c_int64) for n in _names]


class HdlaNormDims(ctypes.Structure):
    """struct hdla_norm_dims of include/hdla_hip.h."""
    _fields_ = [("rows", ctypes.c_int64), ("G", ctypes.c_int32), ("E", ctypes.c_int32), ("dtype", ctypes.c_int32),
                ("weight_dtype", ctypes.c_int32), ("gate_pos", ctypes.c_int32), ("c", ctypes.c_float),
                ("eps", ctypes.c_float)]


class HdlaPreDims(ctypes.Structure):
    """struct hdla_pre_dims of include/hdla_hip.h."""
    _fields_ = [("rows", ctypes.c_int64)] + [(n, ctypes.c_int32) for n in (
        "H", "D", "dtype", "ldy", "col_q", "col_k", "col_v", "col_beta", "norm_q", "norm_k", "norm_v")] + [
        ("beta_scale", ctypes.c_float), ("eps", ctypes.c_float), ("zero_from", ctypes.c_int32)]


class HdlaUpDims(ctypes.Structure):
    """struct hdla_up_dims of include/hdla_hip.h."""
    _fields_ = [("rows", ctypes.c_int64), ("d", ctypes.c_int32), ("D", ctypes.c_int32), ("ld", ctypes.c_int64),
                ("col_f", ctypes.c_int32), ("col_g", ctypes.c_int32)]


class HdlaError(RuntimeError):
    pass


def lib_path() -> str:
    return os.environ.get("HDLA_HIP_LIB", os.path.join(_HERE, _LIB_NAME))


def load():
    """Load the shared library once; raise if it is missing (build it with __graft_entry__.build() or
    `make -C hdla-impl_amd/csrc`)."""
    global _lib
    if _lib is not None:
        return _lib
    path = lib_path()
    if not os.path.exists(path):
        raise HdlaError(f"{path} not found: build the HIP library first (make -C hdla-impl_amd/csrc); "
                        "there is no CPU or PyTorch fallback for these operators")
    lib = ctypes.CDLL(path)
    P, F = ctypes.c_void_p, ctypes.POINTER(HdlaDims)
    lib.hdla_version.restype = ctypes.c_int
    lib.hdla_version.argtypes = []
    if lib.hdla_version() != HDLA_VERSION:
        raise HdlaError(f"{path} is version {lib.hdla_version()} of the C ABI, this binding needs {HDLA_VERSION}: "
                        "rebuild the library (make -C hdla-impl_amd/csrc)")
    lib.hdla_strerror.restype = ctypes.c_char_p
    lib.hdla_strerror.argtypes = [ctypes.c_int]
    lib.hdla_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_workspace_bytes.argtypes = [F, ctypes.c_int]
    lib.hdla_workspace_layout.restype = ctypes.c_int
    lib.hdla_workspace_layout.argtypes = [F, ctypes.c_int, ctypes.POINTER(HdlaWsLayout)]
    lib.hdla_chunk_fwd.restype = ctypes.c_int
    lib.hdla_chunk_fwd.argtypes = [F] + [P] * 9 + [P, ctypes.c_size_t, P]
    lib.hdla_chunk_fwd_static.restype = ctypes.c_int
    lib.hdla_chunk_fwd_static.argtypes = [F] + [P] * 9 + [P]
    lib.hdla_chunk_bwd.restype = ctypes.c_int
    lib.hdla_chunk_bwd.argtypes = [F] + [P] * 16 + [P, ctypes.c_size_t, P]
    lib.hdla_param_chunk_fwd.restype = ctypes.c_int
    lib.hdla_param_chunk_fwd.argtypes = [F] + [P] * 8 + [P, ctypes.c_size_t, P]
    lib.hdla_param_chunk_bwd.restype = ctypes.c_int
    lib.hdla_param_chunk_bwd.argtypes = [F] + [P] * 14 + [P, ctypes.c_size_t, P]
    lib.hdla_boundary_bytes.restype = ctypes.c_size_t
    lib.hdla_boundary_bytes.argtypes = [F]
    lib.hdla_record_bytes.restype = ctypes.c_size_t
    lib.hdla_record_bytes.argtypes = [F]
    lib.hdla_record_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_record_workspace_bytes.argtypes = [F]
    lib.hdla_chunk_fwd_b.restype = ctypes.c_int
    lib.hdla_chunk_fwd_b.argtypes = [F] + [P] * 10 + [P, ctypes.c_size_t, P, ctypes.c_size_t, P]
    lib.hdla_chunk_bwd_b.restype = ctypes.c_int
    lib.hdla_chunk_bwd_b.argtypes = [F] + [P] * 18 + [P, ctypes.c_size_t, P, ctypes.c_size_t, P]
    lib.hdla_keep_plan.restype = ctypes.c_size_t
    lib.hdla_keep_plan.argtypes = [F, ctypes.POINTER(ctypes.c_int32), ctypes.POINTER(ctypes.c_int32)]
    lib.hdla_chunk_fwd_keep.restype = ctypes.c_int
    lib.hdla_chunk_fwd_keep.argtypes = [F] + [P] * 10 + [P, ctypes.c_size_t, P]
    lib.hdla_chunk_bwd_kept.restype = ctypes.c_int
    lib.hdla_chunk_bwd_kept.argtypes = [F] + [P] * 18 + [P, ctypes.c_size_t, P, ctypes.c_size_t, P]
    lib.hdla_chunk_stages.restype = ctypes.c_int
    lib.hdla_chunk_stages.argtypes = [F, ctypes.c_int, ctypes.c_int] + [P] * 18 + [P, ctypes.c_size_t, P]
    lib.hdla_calib_stream.restype = ctypes.c_int
    lib.hdla_calib_stream.argtypes = [ctypes.POINTER(P), ctypes.c_int, ctypes.POINTER(P), ctypes.c_int, ctypes.c_size_t, P]
    lib.hdla_recurrent_fwd.restype = ctypes.c_int
    lib.hdla_recurrent_fwd.argtypes = [F] + [P] * 6 + [ctypes.c_int] + [P] * 4
    lib.hdla_param_recurrent_fwd.restype = ctypes.c_int
    lib.hdla_param_recurrent_fwd.argtypes = [F] + [P] * 5 + [ctypes.c_int] + [P] * 4
    NF = ctypes.POINTER(HdlaNormDims)
    lib.hdla_normalize_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_normalize_workspace_bytes.argtypes = [NF]
    lib.hdla_normalize_fwd.restype = ctypes.c_int
    lib.hdla_normalize_fwd.argtypes = [NF] + [P] * 5
    lib.hdla_normalize_bwd.restype = ctypes.c_int
    lib.hdla_normalize_bwd.argtypes = [NF] + [P] * 8 + [ctypes.c_size_t, P]
    lib.hdla_normalize_bwd_as.restype = ctypes.c_int
    lib.hdla_normalize_bwd_as.argtypes = [NF] + [P] * 8 + [ctypes.c_size_t, P]
    PF = ctypes.POINTER(HdlaPreDims)
    lib.hdla_layer_pre_fwd.restype = ctypes.c_int
    lib.hdla_layer_pre_fwd.argtypes = [PF] + [P] * 6
    lib.hdla_layer_pre_bwd.restype = ctypes.c_int
    lib.hdla_layer_pre_bwd.argtypes = [PF] + [P] * 7
    lib.hdla_logsigmoid_fwd.restype = ctypes.c_int
    lib.hdla_logsigmoid_fwd.argtypes = [ctypes.c_int, ctypes.c_int64, P, P, P]
    lib.hdla_logsigmoid_bwd.restype = ctypes.c_int
    lib.hdla_logsigmoid_bwd.argtypes = [ctypes.c_int, ctypes.c_int64, P, P, P, P]
    lib.hdla_skinny_wgrad.restype = ctypes.c_int
    lib.hdla_skinny_wgrad.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int32, ctypes.c_int32, P, ctypes.c_int64, P,
                                      ctypes.c_int64, P, P, ctypes.c_size_t, P]
    lib.hdla_skinny_wgrad_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_skinny_wgrad_workspace_bytes.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int32, ctypes.c_int32]
    UF = ctypes.POINTER(HdlaUpDims)
    lib.hdla_layer_up_fwd.restype = ctypes.c_int
    lib.hdla_layer_up_fwd.argtypes = [UF] + [P] * 7
    lib.hdla_layer_down.restype = ctypes.c_int
    lib.hdla_layer_down.argtypes = [UF] + [P] * 7
    lib.hdla_layer_up_wgrad.restype = ctypes.c_int
    lib.hdla_layer_up_wgrad.argtypes = [UF] + [P] * 7 + [ctypes.c_size_t, P]
    lib.hdla_layer_up_wgrad_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_layer_up_wgrad_workspace_bytes.argtypes = [UF]
    lib.hdla_layer_step.restype = ctypes.c_int
    lib.hdla_layer_step.argtypes = [PF, UF, NF, ctypes.c_int32] + [P] * 11
    lib.hdla_rows_gemm_norm.restype = ctypes.c_int
    lib.hdla_rows_gemm_norm.argtypes = [ctypes.c_int32] * 3 + [P, ctypes.c_int32, NF, P, P, ctypes.c_int64, P, ctypes.c_int64, P]
    lib.hdla_rows_gemm.restype = ctypes.c_int
    lib.hdla_rows_gemm.argtypes = [ctypes.c_int32] * 3 + [P, ctypes.c_int64, P, ctypes.c_int64, P, ctypes.c_int64, P]
    lib.hdla_sum_partials.restype = ctypes.c_int
    lib.hdla_sum_partials.argtypes = [P, ctypes.c_int32, ctypes.c_int64, P, P]
    lib.hdla_weight_grad_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_weight_grad_workspace_bytes.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int32]
    lib.hdla_weight_grad.restype = ctypes.c_int
    lib.hdla_weight_grad.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int32, P, ctypes.c_int64, P, ctypes.c_int64, P, P, ctypes.c_size_t, P]
    lib.hdla_weight_grad_pair_workspace_bytes.restype = ctypes.c_size_t
    lib.hdla_weight_grad_pair_workspace_bytes.argtypes = [ctypes.c_int64, P, P]
    lib.hdla_weight_grad_pair.restype = ctypes.c_int
    lib.hdla_weight_grad_pair.argtypes = [ctypes.c_int64, P, P, P, P, P, P, P, P, ctypes.c_size_t, P, P]
    lib.hdla_stack_rows.restype = ctypes.c_int
    lib.hdla_stack_rows.argtypes = [P, P, ctypes.c_int32, ctypes.c_int64, P, ctypes.c_int64, P]
    _lib = lib
    return lib


KEPT_MOST, KEPT_CALLS = 1 << 30, 256             # as in csrc/native.cpp


class _NoNative:
    """What stands in for the native host path where that cannot be loaded: nothing is its case."""

    def _not_mine(self, *args):
        return None

    chunk = chunk_hdla = recurrent = recurrent_hdla = normalize = layer = passed = _not_mine

    def forget(self, cache):
        return [None] * 4

    def __init__(self):
        self._held, self._coming, self._lock = {}, {}, threading.Lock()

    def kept_room(self, like, n):
        """Room for a forward workspace that a call holds for its backward pass unasked, or None: KEPT_MOST bytes a device and KEPT_CALLS calls
        over all whose backward pass is still to come, and what the allocator has; none under saved-tensor hooks (csrc/native.cpp,
        kept_room)."""
        dev, t = like.device.index, None
        if torch._C._autograd._top_saved_tensors_default_hooks(False) is not None:
            return None
        with self._lock:
            held = self._held[dev] = [h for h in self._held.get(dev, ()) if h[0]() is not None]
            if sum(h[1] for h in held) + self._coming.get(dev, 0) + n > KEPT_MOST or len(held) >= KEPT_CALLS:
                return None
            self._coming[dev] = self._coming.get(dev, 0) + n
        try:
            t = torch.empty(n, dtype=torch.uint8, device=like.device)
        except torch.OutOfMemoryError:
            pass
        finally:
            with self._lock:
                self._coming[dev] -= n
                if t is not None:
                    self._held[dev].append((weakref.ref(t), n))
        return t


def native():
    """The operators' native host path (csrc/native.cpp), bound to the loaded library.  Its functions take the arguments
    of the public operators; they return None, having done nothing, for a call that is not theirs.  It is built against one
    torch's C++ headers: where it cannot be loaded, a warning says so once and every call takes the Python code behind it,
    which runs the same kernels with more host time."""
    global _native
    if _native is None:
        lib = load()
        try:
            from . import _native as module
        except ImportError as e:
            warnings.warn(f"hdla_hip: the native host path could not be loaded ({e}); calls go through the slower Python host code. "
                          "Build it for this torch with: make -C hdla-impl_amd/csrc", RuntimeWarning, stacklevel=2)
            _native = _NoNative()
        else:
            module.bind(lib._handle, HdlaError, torch.OutOfMemoryError)
            _native = module
    return _native


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = load().hdla_strerror(rc).decode()
        raise HdlaError(f"{what} failed with code {rc}: {msg}")


def ptr(t: Optional[torch.Tensor]):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def dtype_code(dt: torch.dtype) -> int:
    if dt == torch.bfloat16:
        return HDLA_BF16
    if dt == torch.float32:
        return HDLA_FP32
    raise HdlaError(f"unsupported dtype {dt}")


def default_route() -> int:
    """Launch plan of the chunked operators when the caller does not say: environment variable HDLA_HIP_ROUTE =
    auto (the library chooses: the fused kernels where they are built), classic, plain (the same without the buffers that are
    there to be looked at) or fused."""
    name = os.environ.get("HDLA_HIP_ROUTE", "auto").lower()
    if name not in _ROUTES:
        raise HdlaError(f"HDLA_HIP_ROUTE must be one of auto, classic, plain, fused (got {name!r})")
    return _ROUTES[name]


def default_segments() -> int:
    """Time segments per sequence, of the fused kernels and of the stand-alone scans: environment variable HDLA_HIP_SEGMENTS,
    0 = the library chooses."""
    return int(os.environ.get("HDLA_HIP_SEGMENTS", "0"))


def make_dims(B, T, H, K, V, R, N, in_dtype, gk_dtype, scale, cu_seqlens: Optional[torch.Tensor],
              route: Optional[int] = None, segments: Optional[int] = None) -> HdlaDims:
    return HdlaDims(B, T, H, K, V, R, N, dtype_code(in_dtype), dtype_code(gk_dtype), float(scale),
                    None if cu_seqlens is None else cu_seqlens.data_ptr(),
                    default_route() if route is None else route, default_segments() if segments is None else segments)


def keep_boundaries_default() -> bool:
    """Whether the forward pass of the chunked operators hands its record (fused route: the states at the time-segment
    boundaries and what the chunks' score tiles come to, 37 % of the inputs' bytes) to the backward pass, which otherwise
    re-derives it from the inputs with one more pass.  On by default; HDLA_HIP_INPUTS_ONLY=1 keeps strictly the inputs
    between the passes."""
    return os.environ.get("HDLA_HIP_INPUTS_ONLY", "0") in ("", "0", "false", "False")


def boundary(dims: HdlaDims, device) -> Optional[torch.Tensor]:
    """Room for the states at the segment boundaries for these dimensions, or None where the route has none."""
    n = load().hdla_boundary_bytes(ctypes.byref(dims))
    return torch.empty(n, dtype=torch.uint8, device=device) if n else None


def record(dims: HdlaDims, device) -> Optional[torch.Tensor]:
    """Room for the forward pass's record (boundary states included), or None where the route has none."""
    n = load().hdla_record_bytes(ctypes.byref(dims))
    return torch.empty(n, dtype=torch.uint8, device=device) if n else None


def keep_plan(dims: HdlaDims) -> Tuple[int, int, int]:
    """What the library suggests a training call keep of its forward pass where the route has no record: bytes (0: nothing), and the
    segments for hdla_chunk_fwd_keep and hdla_chunk_bwd_kept."""
    fwd, bwd = ctypes.c_int32(0), ctypes.c_int32(0)
    n = load().hdla_keep_plan(ctypes.byref(dims), ctypes.byref(fwd), ctypes.byref(bwd))
    return n, fwd.value, bwd.value


def check_cu_seqlens(cu_seqlens: torch.Tensor, T: int) -> None:
    """Validate a packed-sequence table that is still on the CPU (free: no device synchronisation): it must start at
    0, end at T and never decrease.  A table that already lives on the GPU is not read back; the kernels force its
    entries into [0, T], so a bad one cannot cause an access outside the tensors, but rows that belong to no sequence
    are then zeros in the outputs."""
    if cu_seqlens.dim() != 1 or cu_seqlens.numel() < 2:
        raise ValueError(f"cu_seqlens must be a 1-d tensor of N+1 >= 2 entries, got shape {tuple(cu_seqlens.shape)}")
    if cu_seqlens.is_cuda:
        return
    cu = cu_seqlens.to(torch.int64)
    if int(cu[0]) != 0 or int(cu[-1]) != T or bool((cu[1:] < cu[:-1]).any()):
        raise ValueError(f"cu_seqlens must start at 0, end at the number of tokens ({T}) and never decrease, "
                         f"got {cu.tolist()}")


PASS_FWD, PASS_BWD, PASS_FWD_KEEP, PASS_BWD_KEPT = 0, 1, 2, 3


def keep_forward_default() -> Optional[bool]:
    """Whether the chunked operators keep the forward pass's per-chunk intermediates for the backward pass when the
    caller does not say (``keep_forward=None``): environment variable HDLA_HIP_KEEP_FORWARD=1 or 0.  Where that does not say
    either (None), the library keeps them where they are small (``keep_plan``) and there is room (``kept_room``), unless
    HDLA_HIP_INPUTS_ONLY=1."""
    v = os.environ.get("HDLA_HIP_KEEP_FORWARD")
    return None if v is None else v not in ("", "0", "false", "False")


def current_stream(device) -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def workspace(dims: HdlaDims, pass_: int, device, with_record: bool = False) -> torch.Tensor:
    """Scratch of a pass; ``with_record``: of a backward pass that is given the forward pass's record."""
    lib = load()
    n = lib.hdla_record_workspace_bytes(ctypes.byref(dims)) if with_record else lib.hdla_workspace_bytes(ctypes.byref(dims), pass_)
    if n == 0:
        raise HdlaError("hdla_workspace_bytes rejected the dimensions "
                        f"(B={dims.B},T={dims.T},H={dims.H},K={dims.K},V={dims.V},R={dims.R},N={dims.N})")
    return torch.empty(n, dtype=torch.uint8, device=device)


def workspace_layout(dims: HdlaDims, pass_: int) -> dict:
    out = HdlaWsLayout()
    check(load().hdla_workspace_layout(ctypes.byref(dims), pass_, ctypes.byref(out)), "hdla_workspace_layout")
    return {n: getattr(out, n) for n in HdlaWsLayout._names}
