"""ctypes binding of liboal_amd.so (the C ABI declared in include/oal_amd.h).

PyTorch supplies device memory and the current HIP stream; every byte of the
operator's arithmetic runs in the HIP kernels behind this library. There is no
fallback: if the library is missing or the tensors are not on a ROCm device,
the call raises.

While a profiler runs, each call sits in a ``torch.profiler.record_function``
range ("oal_amd::forward", "oal_amd::backward"), and the library brackets its own
launches with roctx ranges, as the reference brackets its stages
(``oal_attention/hd_block_gemm_profiling.py:195-226``).
"""

from __future__ import annotations

import contextlib
import ctypes
import os
import threading

import torch

_LIB_NAME = "liboal_amd.so"
_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), _LIB_NAME)
_LOCK = threading.Lock()
_LIB = None

DTYPE_F32 = 0
DTYPE_BF16 = 1
PRECISION_FP32 = 0
PRECISION_BF16 = 1
HEAD_DIM = 64

_vp = ctypes.c_void_p
_i = ctypes.c_int
_f = ctypes.c_float
_sz = ctypes.c_size_t

_SIGNATURES = {
    "oal_abi_version": ([], _i),
    "oal_last_error": ([], ctypes.c_char_p),
    "oal_profile_enable": ([_i], _i),
    "oal_profile_collect": ([ctypes.c_char_p, _sz], _i),
    "oal_feature_count": ([], _i),
    "oal_feature_stride": ([], _i),
    "oal_chunk_size": ([], _i),
    "oal_forward_saved_bytes": ([_i, _i, _i, _i, _i, _i, _i], _sz),
    "oal_backward_workspace_bytes": ([_i, _i, _i, _i, _i, _i, _i], _sz),
    "oal_forward": (
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _f, _f, _vp, _vp, _vp, _vp, _vp],
        _i,
    ),
    "oal_backward": (
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _f, _f, _vp, _vp, _vp, _vp, _vp, _vp,
         _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp],
        _i,
    ),
    "oal_backward_noalloc": (
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _f, _f, _vp, _vp, _vp, _vp, _vp, _vp,
         _vp, _vp, _vp, _vp, _vp, _vp, _vp],
        _i,
    ),
    "oal_selftest": ([_vp, _vp], _i),
    "oal_forward_f64": (
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, ctypes.c_double, _vp, _vp, _vp, _vp],
        _i,
    ),
    "oal_backward_f64_workspace_bytes": ([_i, _i, _i, _i, _i], _sz),
    "oal_backward_f64": (
        [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, ctypes.c_double, _vp, _vp, _vp, _vp, _vp, _vp,
         _vp, _vp, _vp, _vp, _vp, _vp, _vp],
        _i,
    ),
    "oal_expand_factor": ([_vp, _i, _i, _i, _i, ctypes.c_double, _vp, _vp, _vp, _vp], _i),
    "oal_expand_factor_backward": ([_vp, _i, _i, _i, _i, _vp, _vp, _vp, _vp, _vp], _i),
    "oal_expand_pairs": ([_vp, _vp, _i, _i, _vp, _vp, _vp, _vp], _i),
    "oal_expand_pairs_backward": ([_vp, _i, _i, _vp, _vp], _i),
    "oal_rotary_heads": ([_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp], _i),
    "oal_check_labels": ([_vp, _i, _i, _i, _i, _i, _vp, _vp, _vp], _i),
    "oal_check_outputs": ([_i, _i, _vp, _vp, _vp, _sz, _i, _i, _i, _vp, _vp], _i),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)


def library_path() -> str:
    return _LIB_PATH


def load_library(path: str | None = None) -> ctypes.CDLL:
    """Load liboal_amd.so once; raise if it has not been built."""
    global _LIB
    with _LOCK:
        if _LIB is not None and path is None:
            return _LIB
        target = path or _LIB_PATH
        if not os.path.exists(target):
            raise RuntimeError(
                f"{_LIB_NAME} is not built ({target}); run __graft_entry__.build() "
                "(hipcc --offload-arch=gfx950) before using oal_amd"
            )
        lib = ctypes.CDLL(target)
        for name, (args, res) in _SIGNATURES.items():
            fn = getattr(lib, name)
            fn.argtypes = args
            fn.restype = res
        if lib.oal_abi_version() != 2:
            raise RuntimeError("liboal_amd.so ABI version mismatch")
        if path is None:
            _LIB = lib
        return lib


def load_hd_cublas_compat(manifest_path=None, runtime_probe_path=None, device=None, *, identity_policy=None):
    """Setup hook with the signature of the reference's bf16 loader
    (``oal_attention/hd_cublas_compat.py:688-799``): loads liboal_amd.so and
    checks that ``device`` is a ROCm device. The manifest and probe paths of
    the cuBLAS artifact have no meaning here and are ignored.
    """
    lib = load_library()
    if device is not None:
        dev = torch.device(device)
        if dev.type != "cuda" or torch.version.hip is None:
            raise RuntimeError("oal_amd runs only on a ROCm (HIP) device; got " + str(dev))
    return lib


def _check(rc: int, lib: ctypes.CDLL, what: str) -> None:
    if rc != 0:
        msg = lib.oal_last_error().decode("utf-8", "replace")
        raise RuntimeError(f"{what} failed: {msg}")


def _ptr(t: torch.Tensor | None):
    """The address as an int (None: a null pointer); the argument types make it a pointer."""
    return None if t is None else t.data_ptr()


_NOTHING = contextlib.nullcontext()


def _scope(device: torch.device, name: str | None = None):
    """``device`` made current and, while a profiler runs, the range ``name``. A call's
    host time is most of a short one (at N = 128 a prepared forward took 96 us with
    both always entered, pointers boxed and every check spelled out, 74 without),
    so nothing is entered that has no effect."""
    here = device.type == "cuda" and torch.cuda.current_device() == device.index
    traced = name is not None and torch._C._autograd._profiler_enabled()
    if not traced:
        return _NOTHING if here else torch.cuda.device(device)
    stack = contextlib.ExitStack()
    if not here:
        stack.enter_context(torch.cuda.device(device))
    stack.enter_context(torch.profiler.record_function(name))
    return stack


_C = torch._C
_PLAIN_TYPES = (torch.Tensor, torch.nn.Parameter)
_TRACERS = tuple(getattr(_C._TorchDispatchModeKey, name) for name in ("FAKE", "PROXY", "FUNCTIONAL"))


def ordinary(*tensors: torch.Tensor) -> bool:
    """Whether a kernel may stand in for a few torch operations on these tensors:
    plain ROCm tensors in an eager call. Whatever has to see the operations -- a
    compiler or tracer, fake tensors, a tensor subclass, functorch's transforms,
    forward-mode derivatives -- gets them. (Under 1 us: it is asked in every call.)"""
    for t in tensors:
        if type(t) not in _PLAIN_TYPES or not t.is_cuda:
            return False
    if (torch.compiler.is_compiling() or _C._is_tracing() or _C._are_functorch_transforms_active()
            or torch.autograd.forward_ad._current_level >= 0):
        return False
    tracing = _C._len_torch_dispatch_stack() and any(_C._get_dispatch_mode(key) is not None for key in _TRACERS)
    return torch.version.hip is not None and not tracing


def _aligned(t: torch.Tensor | None) -> torch.Tensor | None:
    """t, or a fresh copy when its data pointer is not 16-byte aligned (the
    kernels move rows with 16-byte accesses; a view with an odd storage offset
    would otherwise be rejected by the library)."""
    if t is None or t.data_ptr() % 16 == 0:
        return t
    return t.clone(memory_format=torch.contiguous_format)


def _dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return DTYPE_F32
    if dtype == torch.bfloat16:
        return DTYPE_BF16
    raise RuntimeError("q, k and v must be float32 or bfloat16 for the HIP kernels")


# ---------------------------------------------------------------------------
# Argument checks. Every tensor is checked for type, dtype, shape, layout and
# device before any pointer crosses the C ABI, as the reference's native op
# checks its operands (oal_attention/csrc/hd_cublas_compat.cpp:47-61, 104-148):
# the kernels trust the sizes they are given, so a short or mis-shaped buffer
# would otherwise be read or written out of bounds on the device. Failures are
# RuntimeError (the reference's TORCH_CHECK) and leave nothing enqueued.
# ---------------------------------------------------------------------------
def _check_tensor(t, name: str, *, dtype: torch.dtype, shape: tuple, device: torch.device | None = None) -> None:
    if (isinstance(t, torch.Tensor) and t.dtype == dtype and t.shape == shape and t.layout == torch.strided
            and t.is_contiguous() and (device is None or t.device == device)):
        return
    if not isinstance(t, torch.Tensor):
        raise RuntimeError(f"{name} must be a torch.Tensor")
    if t.layout != torch.strided:
        raise RuntimeError(f"{name} must be strided")
    if t.dtype != dtype:
        raise RuntimeError(f"{name} must be {str(dtype).replace('torch.', '')}, got {str(t.dtype).replace('torch.', '')}")
    if tuple(t.shape) != tuple(shape):
        raise RuntimeError(f"{name} must have shape {list(shape)}, got {list(t.shape)}")
    if not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")
    if device is not None and t.device != device:
        raise RuntimeError(f"{name} must be on the same device as q ({device}), got {t.device}")


def _check_bytes(t, name: str, nbytes: int, device: torch.device) -> None:
    if not isinstance(t, torch.Tensor):
        raise RuntimeError(f"{name} must be a torch.Tensor")
    if t.dtype != torch.uint8 or t.ndim != 1 or not t.is_contiguous():
        raise RuntimeError(f"{name} must be a contiguous 1-D uint8 tensor")
    if t.numel() < nbytes:
        raise RuntimeError(f"{name} holds {t.numel()} bytes; {nbytes} are needed")
    if t.device != device:
        raise RuntimeError(f"{name} must be on the same device as q ({device}), got {t.device}")


def _span(t: torch.Tensor) -> tuple[int, int]:
    start = t.data_ptr()
    return start, start + t.numel() * t.element_size()


def _check_no_overlap(out: torch.Tensor, name: str, others: dict) -> None:
    lo, hi = _span(out)
    for other_name, t in others.items():
        if t is None or t.device != out.device:
            continue
        a, b = _span(t)
        if a < hi and lo < b:
            raise RuntimeError(f"{name} must not overlap {other_name}")


def check_forward_args(q, k, v, labels, c0, lam, gam) -> tuple[int, int, int, int, int]:
    """Validate the forward operands; returns (B, Hq, Hkv, N, groups)."""
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not isinstance(t, torch.Tensor):
            raise RuntimeError(f"{name} must be a torch.Tensor")
        if t.ndim != 4:
            raise RuntimeError(f"{name} must be rank 4 [B, H, N, {HEAD_DIM}]")
    b, hq, n, d = q.shape
    hkv = k.shape[1]
    if min(b, hq, hkv, n) <= 0:
        raise RuntimeError("batch, head counts and sequence length must be positive")
    if hq % hkv != 0:
        raise RuntimeError("query head count must be divisible by KV head count")
    if d != HEAD_DIM:
        raise RuntimeError(f"q, k and v must be padded to {HEAD_DIM} features")
    _dtype_code(q.dtype)
    dev = q.device
    _check_tensor(q, "q", dtype=q.dtype, shape=(b, hq, n, HEAD_DIM))
    _check_tensor(k, "k", dtype=q.dtype, shape=(b, hkv, n, HEAD_DIM), device=dev)
    _check_tensor(v, "v", dtype=q.dtype, shape=(b, hkv, n, HEAD_DIM), device=dev)
    if not isinstance(lam, torch.Tensor) or lam.ndim != 2:
        raise RuntimeError("lam must be a [Hq, G] tensor")
    groups = lam.shape[1]
    if not 1 <= groups <= 64:
        raise RuntimeError("the group count must be in [1, 64]")
    _check_tensor(labels, "labels", dtype=torch.int32, shape=(hq, HEAD_DIM), device=dev)
    _check_tensor(c0, "c0", dtype=torch.float32, shape=(hq,), device=dev)
    _check_tensor(lam, "lam", dtype=torch.float32, shape=(hq, groups), device=dev)
    _check_tensor(gam, "gam", dtype=torch.float32, shape=(hq, groups, groups), device=dev)
    return b, hq, hkv, n, groups


def check_backward_args(q, k, v, labels, c0, lam, gam, num, den, saved, dout, dnum, dden):
    """Validate the VJP operands (dout, dnum and dden in the kernels' dtypes);
    returns (B, Hq, Hkv, N, groups)."""
    b, hq, hkv, n, groups = check_forward_args(q, k, v, labels, c0, lam, gam)
    dev = q.device
    _check_tensor(num, "num", dtype=torch.float32, shape=(b, hq, n, HEAD_DIM), device=dev)
    _check_tensor(den, "den", dtype=torch.float32, shape=(b, hq, n, 1), device=dev)
    if not isinstance(saved, torch.Tensor) or saved.dtype != torch.uint8 or saved.ndim != 1:
        raise RuntimeError("saved must be the 1-D uint8 tensor the forward returned")
    if dout is not None:
        _check_tensor(dout, "dout", dtype=q.dtype, shape=(b, hq, n, HEAD_DIM), device=dev)
    if dnum is not None:
        _check_tensor(dnum, "dnum", dtype=torch.float32, shape=(b, hq, n, HEAD_DIM), device=dev)
    if dden is not None:
        _check_tensor(dden, "dden", dtype=torch.float32, shape=(b, hq, n, 1), device=dev)
    return b, hq, hkv, n, groups


def _require_device(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if t is None:
            continue
        if t.device.type != "cuda" or torch.version.hip is None:
            raise RuntimeError("oal_amd runs only on a ROCm (HIP) device; got a tensor on " + str(t.device))


def _stream(device: torch.device) -> int:
    return torch._C._cuda_getCurrentRawStream(device.index)


def profile_enable(enable: bool) -> None:
    load_library().oal_profile_enable(1 if enable else 0)


def profile_collect() -> dict[str, tuple[int, float]]:
    """{kernel: (launches, total_ms)} for launches since the last collect."""
    lib = load_library()
    buf = ctypes.create_string_buffer(1 << 16)
    _check(lib.oal_profile_collect(buf, len(buf)), lib, "oal_profile_collect")
    result = {}
    for line in buf.value.decode().splitlines():
        name, count, total = line.split()
        result[name] = (int(count), float(total))
    return result


def chunk_size() -> int:
    return load_library().oal_chunk_size()


def _precision_code(precision: str) -> int:
    if precision == "fp32":
        return PRECISION_FP32
    if precision == "bf16":
        return PRECISION_BF16
    raise ValueError("precision must be 'fp32' or 'bf16'")


def selftest() -> int:
    """Run the matrix-core layout self-test on the current device; returns mismatches."""
    lib = load_library()
    dev = torch.device("cuda", torch.cuda.current_device())
    errors = torch.zeros(1, dtype=torch.int32, device=dev)
    _check(lib.oal_selftest(_ptr(errors), _stream(dev)), lib, "oal_selftest")
    return int(errors.item())


def forward(q, k, v, labels, c0, lam, gam, *, scale: float, floor: float, precision: str = "fp32",
            zero_saved: bool = False):
    """Run the HIP forward. q [B,Hq,N,64], k/v [B,Hkv,N,64] contiguous, same dtype;
    labels int32 [Hq,64]; c0 [Hq], lam [Hq,G], gam [Hq,G,G] float32.

    Returns (out [dtype], num f32, den f32 [B,Hq,N,1], saved uint8). The kernels
    leave the saved state's alignment gaps and padding tails unwritten;
    ``zero_saved`` allocates it zero-filled, so that every byte is defined (the
    registered operator's output, which tracing compares bytewise).
    """
    lib = load_library()
    b, hq, hkv, n, groups = check_forward_args(q, k, v, labels, c0, lam, gam)
    pcode = _precision_code(precision)
    _require_device(q)
    q, k, v = (_aligned(t) for t in (q, k, v))
    code = _dtype_code(q.dtype)
    dev = q.device
    with _scope(dev, "oal_amd::forward"):
        nbytes = lib.oal_forward_saved_bytes(b, hq, hkv, n, groups, code, pcode)
        if nbytes == 0:
            _check(1, lib, "oal_forward_saved_bytes")
        out = torch.empty((b, hq, n, HEAD_DIM), dtype=q.dtype, device=dev)
        num = torch.empty((b, hq, n, HEAD_DIM), dtype=torch.float32, device=dev)
        den = torch.empty((b, hq, n, 1), dtype=torch.float32, device=dev)
        saved = (torch.zeros if zero_saved else torch.empty)((nbytes,), dtype=torch.uint8, device=dev)
        rc = lib.oal_forward(
            _ptr(q), _ptr(k), _ptr(v), _ptr(labels), _ptr(c0), _ptr(lam), _ptr(gam), groups,
            b, hq, hkv, n, code, pcode, float(scale), float(floor),
            _ptr(out), _ptr(num), _ptr(den), _ptr(saved), _stream(dev),
        )
        _check(rc, lib, "oal_forward")
    return out, num, den, saved


def backward(q, k, v, labels, c0, lam, gam, num, den, saved, dout, dnum, dden, *, scale: float, floor: float,
             need_q: bool, need_k: bool, need_v: bool, need_coef: bool, precision: str = "fp32",
             workspace: torch.Tensor | None = None):
    """Run the HIP VJP; returns (dq, dk, dv, dc0, dlam, dgam) with None where not requested.

    dout is cast to q's dtype and dnum, dden to float32 (the kernels' operand
    types) before the checks; every operand is then validated.
    """
    lib = load_library()
    if isinstance(q, torch.Tensor):
        if dout is not None:
            dout = dout.to(q.dtype).contiguous()
        if dnum is not None:
            dnum = dnum.to(torch.float32).contiguous()
        if dden is not None:
            dden = dden.to(torch.float32)
            dden = (dden.unsqueeze(-1) if dden.ndim == 3 else dden).contiguous()
    b, hq, hkv, n, groups = check_backward_args(q, k, v, labels, c0, lam, gam, num, den, saved, dout, dnum, dden)
    pcode = _precision_code(precision)
    _require_device(q)
    code = _dtype_code(q.dtype)
    dev = q.device
    with _scope(dev, "oal_amd::backward"):
        sbytes = lib.oal_forward_saved_bytes(b, hq, hkv, n, groups, code, pcode)
        wbytes = lib.oal_backward_workspace_bytes(b, hq, hkv, n, groups, code, pcode)
        if sbytes == 0 or wbytes == 0:
            _check(1, lib, "oal_backward_workspace_bytes")
        _check_bytes(saved, "saved", sbytes, dev)
        if workspace is not None:
            _check_bytes(workspace, "workspace", wbytes, dev)
            _check_no_overlap(workspace, "workspace", {"q": q, "k": k, "v": v, "num": num, "den": den,
                                                       "saved": saved, "dout": dout, "dnum": dnum, "dden": dden})
        work = workspace if workspace is not None else torch.empty((wbytes,), dtype=torch.uint8, device=dev)
        dq = torch.empty_like(q) if need_q else None
        # the key-side kernels produce dk and dv together
        dk = torch.empty_like(k) if need_k or need_v else None
        dv = torch.empty_like(v) if need_k or need_v else None
        if need_coef:
            dc0 = torch.empty_like(c0)
            dlam = torch.empty_like(lam)
            dgam = torch.empty_like(gam)
        else:
            dc0 = dlam = dgam = None
        q, k, v, num, den, saved, dout, dnum, dden = (
            _aligned(t) for t in (q, k, v, num, den, saved, dout, dnum, dden))
        rc = lib.oal_backward(
            _ptr(q), _ptr(k), _ptr(v), _ptr(labels), _ptr(c0), _ptr(lam), _ptr(gam), groups,
            b, hq, hkv, n, code, pcode, float(scale), float(floor),
            _ptr(num), _ptr(den), _ptr(saved), _ptr(dout), _ptr(dnum), _ptr(dden),
            _ptr(dq), _ptr(dk), _ptr(dv), _ptr(dc0), _ptr(dlam), _ptr(dgam), _ptr(work), _stream(dev),
        )
        _check(rc, lib, "oal_backward")
    return dq, dk if need_k else None, dv if need_v else None, dc0, dlam, dgam


# ---------------------------------------------------------------------------
# FP64 route (oal_forward_f64 / oal_backward_f64): every tensor float64.
# ---------------------------------------------------------------------------
def check_forward_args_f64(q, k, v, labels, c0, lam, gam) -> tuple[int, int, int, int, int]:
    """Validate the FP64 operands; returns (B, Hq, Hkv, N, groups)."""
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not isinstance(t, torch.Tensor):
            raise RuntimeError(f"{name} must be a torch.Tensor")
        if t.ndim != 4:
            raise RuntimeError(f"{name} must be rank 4 [B, H, N, {HEAD_DIM}]")
    b, hq, n, d = q.shape
    hkv = k.shape[1]
    if min(b, hq, hkv, n) <= 0:
        raise RuntimeError("batch, head counts and sequence length must be positive")
    if hq % hkv != 0:
        raise RuntimeError("query head count must be divisible by KV head count")
    if d != HEAD_DIM:
        raise RuntimeError(f"q, k and v must be padded to {HEAD_DIM} features")
    dev = q.device
    f64 = torch.float64
    _check_tensor(q, "q", dtype=f64, shape=(b, hq, n, HEAD_DIM))
    _check_tensor(k, "k", dtype=f64, shape=(b, hkv, n, HEAD_DIM), device=dev)
    _check_tensor(v, "v", dtype=f64, shape=(b, hkv, n, HEAD_DIM), device=dev)
    if not isinstance(lam, torch.Tensor) or lam.ndim != 2:
        raise RuntimeError("lam must be a [Hq, G] tensor")
    groups = lam.shape[1]
    if not 1 <= groups <= 64:
        raise RuntimeError("the group count must be in [1, 64]")
    _check_tensor(labels, "labels", dtype=torch.int32, shape=(hq, HEAD_DIM), device=dev)
    _check_tensor(c0, "c0", dtype=f64, shape=(hq,), device=dev)
    _check_tensor(lam, "lam", dtype=f64, shape=(hq, groups), device=dev)
    _check_tensor(gam, "gam", dtype=f64, shape=(hq, groups, groups), device=dev)
    return b, hq, hkv, n, groups


def forward_f64(q, k, v, labels, c0, lam, gam, *, scale: float):
    """FP64 forward: q [B,Hq,N,64], k/v [B,Hkv,N,64], c0/lam/gam float64, labels
    int32 [Hq,64]. Returns (out, num [B,Hq,N,64], den [B,Hq,N,1]), all float64."""
    lib = load_library()
    b, hq, hkv, n, groups = check_forward_args_f64(q, k, v, labels, c0, lam, gam)
    _require_device(q)
    q, k, v = (_aligned(t) for t in (q, k, v))
    dev = q.device
    with _scope(dev, "oal_amd::forward_f64"):
        out = torch.empty((b, hq, n, HEAD_DIM), dtype=torch.float64, device=dev)
        num = torch.empty((b, hq, n, HEAD_DIM), dtype=torch.float64, device=dev)
        den = torch.empty((b, hq, n, 1), dtype=torch.float64, device=dev)
        rc = lib.oal_forward_f64(
            _ptr(q), _ptr(k), _ptr(v), _ptr(labels), _ptr(c0), _ptr(lam), _ptr(gam), groups,
            b, hq, hkv, n, float(scale), _ptr(out), _ptr(num), _ptr(den), _stream(dev),
        )
        _check(rc, lib, "oal_forward_f64")
    return out, num, den


def backward_f64(q, k, v, labels, c0, lam, gam, num, den, dout, dnum, dden, *, scale: float, need_q: bool,
                 need_kv: bool, need_coef: bool):
    """FP64 VJP; returns (dq, dk, dv, dc0, dlam, dgam) with None where not requested."""
    lib = load_library()
    f64 = torch.float64
    if dout is not None:
        dout = dout.to(f64).contiguous()
    if dnum is not None:
        dnum = dnum.to(f64).contiguous()
    if dden is not None:
        dden = dden.to(f64)
        dden = (dden.unsqueeze(-1) if dden.ndim == 3 else dden).contiguous()
    b, hq, hkv, n, groups = check_forward_args_f64(q, k, v, labels, c0, lam, gam)
    dev = q.device
    _check_tensor(num, "num", dtype=f64, shape=(b, hq, n, HEAD_DIM), device=dev)
    _check_tensor(den, "den", dtype=f64, shape=(b, hq, n, 1), device=dev)
    if dout is not None:
        _check_tensor(dout, "dout", dtype=f64, shape=(b, hq, n, HEAD_DIM), device=dev)
    if dnum is not None:
        _check_tensor(dnum, "dnum", dtype=f64, shape=(b, hq, n, HEAD_DIM), device=dev)
    if dden is not None:
        _check_tensor(dden, "dden", dtype=f64, shape=(b, hq, n, 1), device=dev)
    _require_device(q)
    with _scope(dev, "oal_amd::backward_f64"):
        wbytes = lib.oal_backward_f64_workspace_bytes(b, hq, hkv, n, groups)
        if wbytes == 0:
            _check(1, lib, "oal_backward_f64_workspace_bytes")
        work = torch.empty((wbytes,), dtype=torch.uint8, device=dev)
        dq = torch.empty_like(q) if need_q else None
        dk = torch.empty_like(k) if need_kv else None
        dv = torch.empty_like(v) if need_kv else None
        if need_coef:
            dc0, dlam, dgam = torch.empty_like(c0), torch.empty_like(lam), torch.empty_like(gam)
        else:
            dc0 = dlam = dgam = None
        q, k, v, num, den, dout, dnum, dden = (_aligned(t) for t in (q, k, v, num, den, dout, dnum, dden))
        rc = lib.oal_backward_f64(
            _ptr(q), _ptr(k), _ptr(v), _ptr(labels), _ptr(c0), _ptr(lam), _ptr(gam), groups,
            b, hq, hkv, n, float(scale), _ptr(num), _ptr(den), _ptr(dout), _ptr(dnum), _ptr(dden),
            _ptr(dq), _ptr(dk), _ptr(dv), _ptr(dc0), _ptr(dlam), _ptr(dgam), _ptr(work), _stream(dev),
        )
        _check(rc, lib, "oal_backward_f64")
    return dq, dk, dv, dc0, dlam, dgam


# ---------------------------------------------------------------------------
# Adapter entry points: factor expansion and its VJP, checks of labels and outputs.
# ---------------------------------------------------------------------------
_OUT_KINDS = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2, torch.float64: 3}


def expand_factor(factor: torch.Tensor, query_heads: int, groups: int, eps: float):
    """(c0 [Hq], lam [Hq, G], gam [Hq, G, G]) of a contiguous float32 or float64
    packed factor [P] or [Hq, P] on a ROCm device, in its dtype."""
    lib = load_library()
    _require_device(factor)
    side = groups + 1
    shape = (side * (side + 1) // 2,) if factor.ndim == 1 else (query_heads, side * (side + 1) // 2)
    if factor.dtype not in (torch.float32, torch.float64):
        raise RuntimeError("factor must be float32 or float64")
    _check_tensor(factor, "factor", dtype=factor.dtype, shape=shape)
    with _scope(factor.device):
        c0, lam, gam = (factor.new_empty(s) for s in ((query_heads,), (query_heads, groups),
                                                      (query_heads, groups, groups)))
        rc = lib.oal_expand_factor(_ptr(factor), int(factor.dtype == torch.float64), int(factor.ndim == 2), query_heads,
                                   groups, float(eps), _ptr(c0), _ptr(lam), _ptr(gam), _stream(factor.device))
        _check(rc, lib, "oal_expand_factor")
    return c0, lam, gam


def expand_factor_backward(factor: torch.Tensor, query_heads: int, groups: int, dc0, dlam, dgam) -> torch.Tensor:
    """The VJP of :func:`expand_factor`; a gradient given as None counts as zero."""
    lib = load_library()
    _require_device(factor)
    shapes = ((query_heads,), (query_heads, groups), (query_heads, groups, groups))
    grads = []
    for name, t, shape in zip(("dc0", "dlam", "dgam"), (dc0, dlam, dgam), shapes):
        if t is not None:
            t = t.to(factor.dtype).contiguous()
            _check_tensor(t, name, dtype=factor.dtype, shape=shape, device=factor.device)
        grads.append(t)
    with _scope(factor.device):
        dfactor = torch.empty_like(factor)
        rc = lib.oal_expand_factor_backward(_ptr(factor), int(factor.dtype == torch.float64), int(factor.ndim == 2),
                                            query_heads, groups, *(_ptr(t) for t in grads), _ptr(dfactor),
                                            _stream(factor.device))
        _check(rc, lib, "oal_expand_factor_backward")
    return dfactor


def expand_pairs(b: torch.Tensor, c: torch.Tensor):
    """(lam [Hq, 64], gam [Hq, 64, 64], labels [Hq, 64]) of contiguous float32
    b [Hq, D] and c [Hq, D(D+1)/2]: one group per dimension, zero past D."""
    lib = load_library()
    _require_device(b, c)
    hq, d = b.shape
    _check_tensor(b, "b", dtype=torch.float32, shape=(hq, d))
    _check_tensor(c, "c", dtype=torch.float32, shape=(hq, d * (d + 1) // 2), device=b.device)
    with _scope(b.device):
        lam, gam = b.new_empty((hq, HEAD_DIM)), b.new_empty((hq, HEAD_DIM, HEAD_DIM))
        labels = torch.empty((hq, HEAD_DIM), dtype=torch.int32, device=b.device)
        rc = lib.oal_expand_pairs(_ptr(b), _ptr(c), hq, d, _ptr(lam), _ptr(gam), _ptr(labels), _stream(b.device))
        _check(rc, lib, "oal_expand_pairs")
    return lam, gam, labels


def expand_pairs_backward(dgam: torch.Tensor, head_dim: int) -> torch.Tensor:
    """dc [Hq, D(D+1)/2] of the contiguous float32 gradient of :func:`expand_pairs`'s gam."""
    lib = load_library()
    _require_device(dgam)
    hq = dgam.shape[0]
    _check_tensor(dgam, "dgam", dtype=torch.float32, shape=(hq, HEAD_DIM, HEAD_DIM))
    with _scope(dgam.device):
        dc = dgam.new_empty((hq, head_dim * (head_dim + 1) // 2))
        rc = lib.oal_expand_pairs_backward(_ptr(dgam), hq, head_dim, _ptr(dc), _stream(dgam.device))
        _check(rc, lib, "oal_expand_pairs_backward")
    return dc


def rotary_heads(tensors, cos: torch.Tensor, sin: torch.Tensor, q_heads: int, kv_heads: int, *, back: bool):
    """q, k, v projections [B, N, heads * 64] -> head-first [B, heads, N, 64], q
    and k rotated by cos, sin [N, 64]; or, with ``back``, head-first gradients ->
    projection gradients. A tensor given as None comes back as None."""
    lib = load_library()
    given = next(t for t in tensors if t is not None)
    _require_device(given)
    code, dev = _dtype_code(given.dtype), given.device
    b, n = given.shape[0], cos.shape[0]
    _check_tensor(cos, "cos", dtype=given.dtype, shape=(n, HEAD_DIM), device=dev)
    _check_tensor(sin, "sin", dtype=given.dtype, shape=(n, HEAD_DIM), device=dev)
    cos, sin = _aligned(cos), _aligned(sin)
    source, result = [], []
    with _scope(dev):
        for name, t, heads in zip("qkv", tensors, (q_heads, kv_heads, kv_heads)):
            if t is None:
                source.append(None)
                result.append(None)
                continue
            flat, split = (b, n, heads * HEAD_DIM), (b, heads, n, HEAD_DIM)
            _check_tensor(t, name, dtype=given.dtype, shape=split if back else flat, device=dev)
            source.append(_aligned(t))
            result.append(t.new_empty(flat if back else split))
        proj, head = (result, source) if back else (source, result)
        rc = lib.oal_rotary_heads(*map(_ptr, proj), *map(_ptr, head), _ptr(cos), _ptr(sin), int(back), b, q_heads,
                                  kv_heads, n, code, _stream(dev))
        _check(rc, lib, "oal_rotary_heads")
    return tuple(result)


class Verdict:
    """Host-mapped words that checks enqueued on the current stream of a device
    set bits in; :meth:`read` synchronizes that stream. One per call: the words
    live until the kernels that may write them are done."""

    _pending = False

    def __init__(self, device: torch.device):
        # on the host whatever the caller's default device is
        self._words = torch.zeros(2, dtype=torch.int32, device="cpu", pin_memory=True)
        self._stream = torch.cuda.current_stream(device)
        self._device = device

    def check_labels(self, labels: torch.Tensor, query_heads: int, groups: int) -> torch.Tensor:
        """Enqueue the check of [D] or [Hq, D] int32 or int64 labels (D <= 64);
        returns the int32 [Hq, 64] table that the kernels read."""
        lib = load_library()
        labels = labels.contiguous()
        with _scope(self._device):
            table = torch.empty((query_heads, HEAD_DIM), dtype=torch.int32, device=self._device)
            self._pending = True
            rc = lib.oal_check_labels(_ptr(labels), int(labels.dtype == torch.int64), int(labels.ndim == 2),
                                      labels.shape[-1], query_heads, groups, _ptr(table), self._words.data_ptr(),
                                      self._stream.cuda_stream)
            _check(rc, lib, "oal_check_labels")
        return table

    def check_outputs(self, num, den: torch.Tensor, out) -> None:
        """Enqueue the check of den and, where given, of num and out ([..., DV])."""
        lib = load_library()
        width, strides = 1, []
        tensors = []
        for t in (num, out):
            if t is not None:
                t = t.detach()
                width = t.shape[-1]
                # rows one stride apart: contiguous, or a slice of wider rows
                row = t.stride(-2) if t.ndim > 1 else width
                regular = t.stride(-1) == 1 and all(
                    t.stride(i) == t.stride(i + 1) * t.shape[i + 1] for i in range(t.ndim - 2))
                if not regular:
                    t, row = t.contiguous(), width
                strides.append(row)
            else:
                strides.append(0)
            tensors.append(t)
        den = den.detach().contiguous()
        kind = 0 if out is None else _OUT_KINDS[out.dtype]
        with _scope(self._device):
            self._pending = True
            rc = lib.oal_check_outputs(int(den.dtype == torch.float64), kind, _ptr(tensors[0]), _ptr(den),
                                       _ptr(tensors[1]), den.numel(), width, strides[0], strides[1],
                                       self._words.data_ptr() + 4, self._stream.cuda_stream)
            _check(rc, lib, "oal_check_outputs")

    def __del__(self):
        # an abandoned check (an error in between) may still write its words
        if self._pending:
            self._stream.synchronize()

    def read(self) -> tuple[int, int]:
        """(label bits, output bits) of the checks enqueued so far."""
        if self._pending:
            self._stream.synchronize()
            self._pending = False
        labels, outputs = self._words.tolist()
        return labels, outputs
