"""Python-facing Stream-K GEMM entry points over the C ABI.

Mirrors the reference's operator surface:
  * `streamk_fp16(A, B)` / `streamk_fp32(A, B)`: what running streamk_fp16.py / streamk_fp32.py
    computes (C = A @ B.T for the fp16 NT script, C = A @ B for the fp32 NN script);
  * `tl_matmul_streamk(M, N, K, ...)` returns a callable `kernel(A, B, C)` that writes C in place,
    the shape of the reference's `tl_mod = TL.Profiler(...)`; `tl_mod(A, B, b_c)`
    (streamk_fp16.py:382-387), including `do_bench`.

Every GEMM is registered with the PyTorch dispatcher as a custom operator of the `streamk` namespace
(`torch.ops.streamk.gemm_f16`, `gemm_bf16`, `gemm_f32`, `gemm_q4`, `gemm_f8`, `gemm_i8`, each with an
`_out` twin that writes a caller's C, plus `dequant_q4`): a HIP implementation that hands data
pointers and the current stream to the C ABI (native for ordinary calls, csrc/torch_ops.cpp, which passes every other
one on to the implementations here, registered as `<name>_general`), and a fake (meta) implementation that gives shape and
dtype of the result, so that `torch.compile`, FakeTensor tracing and graph capture see an ordinary
operator.  This is the role of the reference's `@jit(out_idx=[2])` wrapper, which turns the kernel
into `f(A, B) -> C` (autotune/streamk_fp16_autotune.py:93-94).  The functions below are thin argument
adapters over those operators.  torch is used for device memory, streams and the dispatcher only;
all arithmetic happens in libstreamk.so.
"""
import ctypes
import itertools
import weakref

import torch

from . import _lib
from . import plan as _plan_mod
from .plan import make_plan

_workspaces = {}


def _stream_ptr():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _workspace(nbytes, device):
    """One self-cleaning workspace per (device, stream), grown on demand and zeroed once."""
    if nbytes == 0:
        return None
    key = (device.index if device.index is not None else torch.cuda.current_device(),
           torch.cuda.current_stream().cuda_stream)
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < nbytes:
        if ws is not None:  # the library must not take a later allocation at this address for this workspace
            _lib.tell_native_operators("sk_torch_set_workspace", *key, None, 0)
            _lib.lib().sk_workspace_release(ws.data_ptr())
        ws = torch.empty(max(nbytes, 1 << 20), dtype=torch.uint8, device=device)
        _lib.check(_lib.lib().sk_workspace_init(ws.data_ptr(), ws.numel(), _stream_ptr()),
                   "sk_workspace_init")
        _workspaces[key] = ws
        _lib.tell_native_operators("sk_torch_set_workspace", *key, ws.data_ptr(), ws.numel())
    return ws


def _ws_args(plan, device):
    ws = _workspace(plan.workspace_bytes, device)
    return (ctypes.byref(plan), ws.data_ptr() if ws is not None else None, ws.numel() if ws is not None else 0,
            _stream_ptr())


def reset_workspaces():
    """Drops cached workspaces.  Needed after workspace_status() (or a launch) has raised StreamKError
    with status SK_ERR_TIMEOUT: the library refuses a workspace on which a fix-up wait gave up until it
    has been initialised again, which the next call on a fresh workspace does."""
    for key, ws in _workspaces.items():
        _lib.tell_native_operators("sk_torch_set_workspace", *key, None, 0)
        _lib.lib().sk_workspace_release(ws.data_ptr())
    _workspaces.clear()


def workspace_status():
    """Synchronises the current stream and raises StreamKError(SK_ERR_TIMEOUT) if a fix-up wait on its
    workspace gave up (the tile it was waiting for is then incomplete in C).  The launches themselves
    only enqueue work, so this is where a timeout surfaces: call it wherever the caller synchronises
    anyway (bench_ms, StreamKKernel.do_bench and the autotuner do)."""
    for (dev, stream), ws in _workspaces.items():
        if stream == torch.cuda.current_stream().cuda_stream:
            _lib.check(_lib.lib().sk_workspace_status(ws.data_ptr(), _stream_ptr()), "sk_workspace_status")


def _check_matrix(t, name, dtype):
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise TypeError(f"{name} must be a CUDA/HIP tensor")
    if t.dtype != dtype:
        raise TypeError(f"{name} must be {dtype}, got {t.dtype}")
    if t.dim() != 2 or t.stride(1) != 1:
        raise ValueError(f"{name} must be 2-D with unit stride along its last dimension")


def _epilogue(bias, N, dtype, device, activation=None):
    """sk_epilogue for a bias vector (N values of C's type on C's device) and / or an activation
    ('relu', 'gelu_tanh', 'silu'), or None when there is neither."""
    if activation not in _lib.ACTIVATIONS:
        raise ValueError(f"activation must be one of {sorted(k for k in _lib.ACTIVATIONS if k)} or None")
    act = _lib.ACTIVATIONS[activation]
    if bias is None:
        return _lib.SkEpilogue(bias=None, activation=act) if act else None
    if not isinstance(bias, torch.Tensor) or bias.dtype != dtype or bias.dim() != 1 or bias.shape[0] != N \
            or not bias.is_contiguous() or bias.device != device:
        raise ValueError(f"bias must be a contiguous {dtype} vector of {N} elements on {device}")
    return _lib.SkEpilogue(bias=bias.data_ptr(), activation=act)


# ---------------------------------------------------------------------------------------------
# Plans behind the operators.  An operator's schema carries tensors, numbers and strings only, so a
# configuration travels as a string: "" (tuned cache, else the library's heuristic), "k=v;k=v" for
# make_config keys, or "#n" for a plan object the caller made itself (kept in a registry here).
# ---------------------------------------------------------------------------------------------
# (weak: a plan object lives as long as its caller keeps it -- the autotuner makes hundreds per shape)
_plan_registry = weakref.WeakValueDictionary()
_plan_serial = itertools.count(1)
_plan_cache = {}


def _plan_handle(plan):
    h = getattr(plan, "_sk_handle", None)
    if h is None:
        h = plan._sk_handle = f"#{next(_plan_serial)}"
        _plan_registry[h] = plan
    return h


def _config_string(plan, config, kw):
    if plan is None and not config and not kw:
        return ""
    if plan is not None:
        return _plan_handle(plan)
    d = dict(config or {})
    d.update({k: v for k, v in kw.items() if v is not None})
    return ";".join(f"{k}={d[k]}" for k in sorted(d))


def _parse_config(text):
    out = {}
    for item in text.split(";"):
        k, v = item.split("=", 1)
        out[k] = int(v) if v.lstrip("-").isdigit() else v
    return out


def _takes_rows(plan, pitch_a, pitch_b):
    """Whether the plan's tiles take rows of A and of the weights that are so many bytes apart (the library refuses a tile
    whose rows span 2 GiB)."""
    return plan.bm * pitch_a < 1 << 31 and plan.bn * pitch_b < 1 << 31


# configuration of a call that names none and whose rows are too far apart for the plan of "": see operator_config (no string, so that
# no caller's is taken for it)
_LONG_ROWS = ("long rows",)


def _plan_of(config, M, N, K, dtype, layout):
    """The plan of a configuration string for this shape (made once per (shape, type, layout, configuration))."""
    # (a plan depends on the tuned cache it was made from and on the device it was made for)
    generation, device = _plan_mod.tuned_generation(), torch.cuda.current_device() if torch.cuda.is_available() else -1
    key = (M, N, K, dtype, layout, config, generation, device)
    plan = _plan_cache.get(key)
    if plan is None:
        named = config not in ("", _LONG_ROWS)
        plan = make_plan(M, N, K, dtype, layout,
                         _parse_config(config) if named else _plan_mod.operator_config(M, N, K, dtype, layout, config == _LONG_ROWS))
        if len(_plan_cache) < 4096:
            _plan_cache[key] = plan
            if config == "":   # from now on the native implementation answers calls of this shape
                with _plan_mod.tuned_lock:
                    if generation == _plan_mod.tuned_generation():
                        _lib.tell_native_operators("sk_torch_add_plan", ctypes.byref(plan), device)
    return plan


def _plan_for(config, M, N, K, dtype, layout, pitch_a=0, pitch_b=0):
    """The plan an operator call runs: the registered plan object, or the one of the configuration string.  Where rows of A or of
    the weights (pitch_a, pitch_b bytes apart) are too long for the tile that a call without a configuration takes, the kernel
    that it takes otherwise, whose tile may have fewer rows."""
    if config.startswith("#"):
        plan = _plan_registry.get(config)
        if plan is None:
            raise ValueError(f"unknown plan handle {config!r}")
        return plan
    plan = _plan_of(config, M, N, K, dtype, layout)
    if config == "" and not _takes_rows(plan, pitch_a, pitch_b):
        plan = _plan_of(_LONG_ROWS, M, N, K, dtype, layout)
    return plan


def _nk_of(B, layout):
    if layout not in ("nt", "nn"):
        raise ValueError("layout must be 'nt' (B is [N,K]) or 'nn' (B is [K,N])")
    return tuple(B.shape) if layout == "nt" else (B.shape[1], B.shape[0])


def _check_out(C, M, N, dtype):
    _check_matrix(C, "out", dtype)
    if tuple(C.shape) != (M, N):
        raise ValueError("out has the wrong shape")


def _act(activation):
    return None if activation in (None, "none", "") else activation


def _aligned_rows(A):
    """A as the kernels can read it: unit stride along K, rows 16 bytes apart or more in multiples of 16, first
    element 16-byte aligned.  Views that are not (a column slice, an odd storage offset) are copied."""
    if isinstance(A, torch.Tensor) and A.dim() == 2 and A.is_cuda and A.shape[0] > 0 and (
            A.stride(1) != 1 or (A.shape[0] > 1 and A.stride(0) * A.element_size() % 16) or A.data_ptr() % 16):
        return A.clone(memory_format=torch.contiguous_format)
    return A


# ---- HIP implementations (write `C`) ----
def _run_16bit(A, B, C, layout, config, bias, activation, tdtype, name):
    A = _aligned_rows(A)
    _check_matrix(A, "A", tdtype)
    _check_matrix(B, "B", tdtype)
    M, K = A.shape
    N, Kb = _nk_of(B, layout)
    if K != Kb:
        raise ValueError(f"K mismatch: A is {tuple(A.shape)}, B is {tuple(B.shape)}")
    _check_out(C, M, N, tdtype)
    plan = _plan_for(config, M, N, K, name, layout, 2 * A.stride(0), 2 * B.stride(0) if layout == "nt" else 0)
    epi = _epilogue(bias, N, tdtype, A.device, _act(activation))
    args = (A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0), C.stride(0),
            *_ws_args(plan, A.device))
    L = _lib.lib()
    plain, ex = (L.sk_gemm_f16, L.sk_gemm_f16_ex) if tdtype == torch.float16 else (L.sk_gemm_bf16, L.sk_gemm_bf16_ex)
    rc = plain(*args) if epi is None else ex(*args, ctypes.byref(epi))
    _lib.check(rc, "sk_gemm_f16" if tdtype == torch.float16 else "sk_gemm_bf16")


def _run_f32(A, B, C, layout, config):
    _check_matrix(A, "A", torch.float32)
    _check_matrix(B, "B", torch.float32)
    M, K = A.shape
    N, Kb = _nk_of(B, layout)
    if K != Kb:
        raise ValueError(f"K mismatch: A is {tuple(A.shape)}, B is {tuple(B.shape)}")
    _check_out(C, M, N, torch.float32)
    plan = _plan_for(config, M, N, K, "float32", layout)
    rc = _lib.lib().sk_gemm_f32(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0),
                                C.stride(0), *_ws_args(plan, A.device))
    _lib.check(rc, "sk_gemm_f32")


_F8_KINDS = {getattr(torch, "float8_e4m3fn", None): "e4m3", getattr(torch, "float8_e5m2", None): "e5m2"}


def _f8_format(A, B, fmt):
    fmt = fmt or None
    for t, name in ((A, "A"), (B, "B")):
        if not isinstance(t, torch.Tensor) or (t.dtype != torch.uint8 and t.dtype not in _F8_KINDS):
            raise TypeError(f"{name} must be a float8_e4m3fn / float8_e5m2 (or uint8) tensor")
        if t.dtype != torch.uint8:
            if fmt not in (None, _F8_KINDS[t.dtype]):
                raise TypeError("A and B must be in the same fp8 format")
            fmt = _F8_KINDS[t.dtype]
    fmt = fmt or "e4m3"
    if fmt not in ("e4m3", "e5m2"):
        raise ValueError("fmt must be 'e4m3' or 'e5m2'")
    return fmt


def _run_f8(A, B, C, alpha, fmt, config, bias, activation):
    fmt = _f8_format(A, B, fmt)
    _check_matrix(A, "A", A.dtype)
    _check_matrix(B, "B", B.dtype)
    M, K = A.shape
    N, Kb = B.shape
    if K != Kb:
        raise ValueError(f"K mismatch: A is {tuple(A.shape)}, B is {tuple(B.shape)}")
    _check_out(C, M, N, torch.float16)
    plan = _plan_for(config, M, N, K, "float8_" + fmt, "nt", A.stride(0), B.stride(0))
    if plan.dtype != (_lib.SK_F8E5M2 if fmt == "e5m2" else _lib.SK_F8E4M3):
        raise ValueError("the plan was made for the other fp8 format")
    epi = _epilogue(bias, N, torch.float16, A.device, _act(activation))
    args = (A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0), C.stride(0), float(alpha),
            *_ws_args(plan, A.device))
    rc = _lib.lib().sk_gemm_f8(*args) if epi is None else _lib.lib().sk_gemm_f8_ex(*args, ctypes.byref(epi))
    _lib.check(rc, "sk_gemm_f8")


def _run_i8(A, B, C, config):
    _check_matrix(A, "A", torch.int8)
    _check_matrix(B, "B", torch.int8)
    M, K = A.shape
    N, Kb = B.shape
    if K != Kb:
        raise ValueError(f"K mismatch: A is {tuple(A.shape)}, B is {tuple(B.shape)}")
    _check_out(C, M, N, torch.int32)
    plan = _plan_for(config, M, N, K, "int8", "nt", A.stride(0), B.stride(0))
    rc = _lib.lib().sk_gemm_i8(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0),
                               C.stride(0), *_ws_args(plan, A.device))
    _lib.check(rc, "sk_gemm_i8")


Q4_MAX_M = 64  # rows of A the weight-streaming Q4 kernels take in one launch
Q4_FUSED_MAX_M = 1024  # up to here the Q4 tile kernels (dequantisation inside the GEMM) beat dequantise-then-GEMM
_stagings = {}


def _staging(nbytes, device):
    """Scratch for dequantised weights: one buffer per (device, stream), grown on demand, never freed."""
    key = (device.index if device.index is not None else torch.cuda.current_device(),
           torch.cuda.current_stream().cuda_stream)
    buf = _stagings.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = _stagings[key] = torch.empty(nbytes, dtype=torch.uint8, device=device)
    return buf


def _zero_points(zeros, scales):
    """Per-group zero points as the library takes them: fp16 [N, K/group] holding integers 0..15.  Integer
    tensors are converted (an allocation per call: keep them as fp16 to avoid it)."""
    if zeros.dtype != torch.float16:
        zeros = zeros.to(torch.float16)
    _check_matrix(zeros, "zeros", torch.float16)
    if tuple(zeros.shape) != tuple(scales.shape) or not zeros.is_contiguous():
        raise ValueError(f"zeros must be contiguous and shaped like scales; got {tuple(zeros.shape)}")
    return zeros


_without_plan = set()   # (configuration, shape, type, generation of the tuned cache) that no kernel runs at once


def _has_plan(config, M, N, K, dtype, pitch_a, pitch_b):
    """Whether some kernel runs the configuration, on rows so far apart, for all the rows at once.  (Asked on every call, and a plan
    that the library refuses is an exception: where the configuration names none, status -4, is remembered.)"""
    generation = _plan_mod.tuned_generation()
    key = (config, M, N, K, dtype, generation)
    if key in _without_plan:
        return False
    try:
        plan = _plan_of(config, M, N, K, dtype, "nt")
    except _lib.StreamKError as e:
        if e.status == -4 and len(_without_plan) < 4096:
            _without_plan.add(key)
        return False
    return _takes_rows(plan, pitch_a, pitch_b)


def _dequantises(M, N, K, zero_points):
    """Whether a call on row-major Q4 weights without a configuration dequantises them first (prefill-sized calls): beyond 1024
    rows, and with per-group zero points, whose kernels for many rows have 64 x 64 tiles, beyond 256 rows from three rounds of them
    on, beyond 512 from two (512 x 8192 x 8192 97 us against 103, 768 x 4096 x 11008 93 / 117, but 512 x 4096 x 4096 41 / 30,
    320 x 8192 x 8192 99 / 76) or, where the fp16 kernels have a long K, one and a half (517 x 3072 x 9472 62.0 / 66.9,
    700 x 2560 x 14336 86.4 / 93.8, 849 x 1832 x 8320 51.3 / 56.5, but 656 x 2560 x 2304 .77 of the time; up to 512 rows it may be
    either, 400 x 5120 x 8192 71.6 / 75.6, 500 x 4096 x 11008 80.3 / 76.0)."""
    if M > Q4_FUSED_MAX_M or not zero_points or M <= 4 * Q4_MAX_M:
        return M > Q4_FUSED_MAX_M
    rounds = 3 if M <= 8 * Q4_MAX_M else (1.5 if K >= 8192 else 2)
    return -(-M // 64) * -(-N // 64) > rounds * _plan_mod.num_cus()


def _run_q4(A, Wq, scales, zeros, C, zero, group, tiled, config, bias, activation):
    if zeros is not None:
        zeros = _zero_points(zeros, scales)  # (row-major like the scales also where the weights are tiled)
    A = _aligned_rows(A)
    _check_matrix(A, "A", torch.float16)
    _check_matrix(Wq, "Wq", torch.uint8)
    _check_matrix(scales, "scales", torch.float16)
    M, K = A.shape
    N = scales.shape[0] if tiled else Wq.shape[0]
    if Wq.shape[1] * 2 != K or not Wq.is_contiguous() or (tiled and Wq.shape[0] != (N + 15) // 16 * 16):
        raise ValueError(f"Wq must be contiguous [N, K/2] (tiled: ceil(N/16)*16 rows); got {tuple(Wq.shape)} for K={K}")
    if tuple(scales.shape) != (N, K // group) or not scales.is_contiguous():
        raise ValueError(f"scales must be contiguous [N, K/group]; got {tuple(scales.shape)}")
    _check_out(C, M, N, torch.float16)
    name = ("q4_zp_tiled" if tiled else "q4_zp") if zeros is not None else ("q4_tiled" if tiled else "q4")
    dequantise = config == "" and not tiled and _dequantises(M, N, K, zeros is not None)
    if M > Q4_MAX_M and not dequantise and not config.startswith("#") and name != "q4" and \
            (tiled and M > 4 * Q4_MAX_M or not _has_plan(config, M, N, K, name, 2 * A.stride(0), K // 2)):
        # Configurations that name kernels for few rows, and tiled weights where the operators' rule takes no kernel for many: up to
        # 256 rows one launch per block of 64.  (Blocks of two rows and more multiply the rounded weights alike; a last block of
        # one row takes the matrix-vector kernels and the unrounded ones.)
        if M <= 4 * Q4_MAX_M:
            for m0 in range(0, M, Q4_MAX_M):
                _run_q4(A[m0:m0 + Q4_MAX_M], Wq, scales, zeros, C[m0:m0 + Q4_MAX_M], zero, group, tiled, config,
                        bias, activation)
            return
        if tiled:
            raise ValueError("more than 256 rows of A need the row-major weights (they are dequantised once)")
        config, dequantise = "", True
    if dequantise:
        # One pass that dequantises the weights (bit-exact device function), then the fp16 tile kernels on them.  The pass costs
        # 26 us for 8192 x 8192 weights, under 7 % of the product from 4096 rows on, where the fused Q4 tile kernels are behind
        # the four-wave fp16 kernel.  The buffer is kept per stream, allocated on first use; with per-group zero points it is
        # the call's own.
        W = (_staging(N * K * 2, A.device).view(torch.float16)[:N * K].view(N, K) if zeros is None
             else torch.empty((N, K), dtype=torch.float16, device=Wq.device))
        _run_dequant_q4(Wq, scales, zeros, W, zero, group)
        _run_16bit(A, W, C, "nt", "", bias, activation, torch.float16, "float16")
        return
    plan = _plan_for(config, M, N, K, name, "nt", 2 * A.stride(0), K // 2)
    if (plan.dtype in (_lib.SK_Q4_TILED, _lib.SK_Q4_ZP_TILED)) != bool(tiled):
        raise ValueError("the plan was made for the other weight layout")
    if (plan.dtype in (_lib.SK_Q4_ZP, _lib.SK_Q4_ZP_TILED)) != (zeros is not None):
        raise ValueError("the plan was made with / without per-group zero points")
    epi = _epilogue(bias, N, torch.float16, A.device, _act(activation))
    tail = _ws_args(plan, A.device)
    L = _lib.lib()
    if epi is not None:
        rc = L.sk_gemm_q4_ex(A.data_ptr(), Wq.data_ptr(), scales.data_ptr(), zeros.data_ptr() if zeros is not None else None,
                             C.data_ptr(), M, N, K, A.stride(0), C.stride(0), group, zero, *tail, ctypes.byref(epi))
    elif zeros is not None:
        rc = L.sk_gemm_q4_zp(A.data_ptr(), Wq.data_ptr(), scales.data_ptr(), zeros.data_ptr(), C.data_ptr(), M, N, K,
                             A.stride(0), C.stride(0), group, *tail)
    else:
        rc = L.sk_gemm_q4(A.data_ptr(), Wq.data_ptr(), scales.data_ptr(), C.data_ptr(), M, N, K, A.stride(0),
                          C.stride(0), group, zero, *tail)
    _lib.check(rc, "sk_gemm_q4")


def _run_dequant_q4(Wq, scales, zeros, W, zero, group):
    _check_matrix(Wq, "Wq", torch.uint8)
    _check_matrix(scales, "scales", torch.float16)
    N, K = Wq.shape[0], Wq.shape[1] * 2
    if not Wq.is_contiguous() or not scales.is_contiguous():
        raise ValueError("Wq and scales must be contiguous")
    _check_out(W, N, K, torch.float16)
    if not W.is_contiguous():
        raise ValueError("the dequantised matrix must be contiguous")
    if zeros is not None:
        zeros = _zero_points(zeros, scales)
        rc = _lib.lib().sk_dequant_q4_zp(Wq.data_ptr(), scales.data_ptr(), zeros.data_ptr(), W.data_ptr(), N, K,
                                         group, _stream_ptr())
        _lib.check(rc, "sk_dequant_q4_zp")
        return
    rc = _lib.lib().sk_dequant_q4(Wq.data_ptr(), scales.data_ptr(), W.data_ptr(), N, K, group, zero, _stream_ptr())
    _lib.check(rc, "sk_dequant_q4")


# ---------------------------------------------------------------------------------------------
# Registration with the dispatcher: `torch.ops.streamk.<name>` (functional, allocates C) and
# `<name>_out` (writes the caller's C).  The functional form's fake implementation is what FakeTensor
# tracing and torch.compile use in place of the kernel.
# ---------------------------------------------------------------------------------------------
_LIBRARY = torch.library.Library("streamk", "DEF")
_EPI = "Tensor? bias=None, str activation=\"none\""


def _register(name, before_out, after_out, run, out_meta):
    """Defines streamk::<name>(before_out, after_out) -> Tensor and streamk::<name>_out(before_out, out,
    after_out) -> ().  run(*args) with C at position len(before_out arguments) performs the launch;
    out_meta(*functional args) -> (shape, dtype) of C."""
    out_pos = before_out.count("Tensor")
    native = name.startswith("gemm_")   # csrc/torch_ops.cpp implements these and calls <name>_general for the rest
    general = "_general" if native else ""
    for suffix in ("", general) if native else ("",):
        _LIBRARY.define(f"{name}{suffix}({before_out}, {after_out}) -> Tensor")
        _LIBRARY.define(f"{name}_out{suffix}({before_out}, Tensor(a!) out, {after_out}) -> ()")

    def functional(*args):
        shape, dtype = out_meta(*args)
        C = torch.empty(shape, dtype=dtype, device=args[0].device)
        if C.numel() > 0:   # an empty batch (no rows of A) has nothing to launch
            run(*args[:out_pos], C, *args[out_pos:])
        return C

    def functional_fake(*args):
        shape, dtype = out_meta(*args)
        return args[0].new_empty(shape, dtype=dtype)

    def out_variant(*args):
        if args[out_pos].numel() > 0 or args[0].shape[0] > 0:
            run(*args)

    # (without the native library the Python implementation stands under both names)
    for suffix in {general} if native and _lib.torch_lib() is not None else {"", general}:
        _LIBRARY.impl(name + suffix, functional, "CUDA")
        _LIBRARY.impl(f"{name}_out{suffix}", out_variant, "CUDA")
    torch.library.register_fake(f"streamk::{name}", functional_fake, lib=_LIBRARY)
    torch.library.register_fake(f"streamk::{name}_out", lambda *args: None, lib=_LIBRARY)


def _mn(A, B, layout):
    return (A.shape[0], _nk_of(B, layout)[0])


_register("gemm_f16", "Tensor A, Tensor B", f"str layout=\"nt\", str config=\"\", {_EPI}",
          lambda A, B, C, layout="nt", config="", bias=None, activation="none":
          _run_16bit(A, B, C, layout, config, bias, activation, torch.float16, "float16"),
          lambda A, B, layout="nt", *rest: (_mn(A, B, layout), torch.float16))
_register("gemm_bf16", "Tensor A, Tensor B", f"str layout=\"nt\", str config=\"\", {_EPI}",
          lambda A, B, C, layout="nt", config="", bias=None, activation="none":
          _run_16bit(A, B, C, layout, config, bias, activation, torch.bfloat16, "bfloat16"),
          lambda A, B, layout="nt", *rest: (_mn(A, B, layout), torch.bfloat16))
_register("gemm_f32", "Tensor A, Tensor B", "str layout=\"nn\", str config=\"\"",
          lambda A, B, C, layout="nn", config="": _run_f32(A, B, C, layout, config),
          lambda A, B, layout="nn", *rest: (_mn(A, B, layout), torch.float32))
_register("gemm_f8", "Tensor A, Tensor B", f"float alpha=1.0, str fmt=\"\", str config=\"\", {_EPI}",
          lambda A, B, C, alpha=1.0, fmt="", config="", bias=None, activation="none":
          _run_f8(A, B, C, alpha, fmt, config, bias, activation),
          lambda A, B, *rest: ((A.shape[0], B.shape[0]), torch.float16))
_register("gemm_i8", "Tensor A, Tensor B", "str config=\"\"",
          lambda A, B, C, config="": _run_i8(A, B, C, config),
          lambda A, B, *rest: ((A.shape[0], B.shape[0]), torch.int32))
_register("gemm_q4", "Tensor A, Tensor Wq, Tensor scales, Tensor? zeros",
          f"int zero=8, int group=128, bool tiled=False, str config=\"\", {_EPI}",
          lambda A, Wq, scales, zeros, C, zero=8, group=128, tiled=False, config="", bias=None, activation="none":
          _run_q4(A, Wq, scales, zeros, C, zero, group, tiled, config, bias, activation),
          lambda A, Wq, scales, *rest: ((A.shape[0], scales.shape[0]), torch.float16))
_register("dequant_q4", "Tensor Wq, Tensor scales, Tensor? zeros", "int zero=8, int group=128",
          lambda Wq, scales, zeros, W, zero=8, group=128: _run_dequant_q4(Wq, scales, zeros, W, zero, group),
          lambda Wq, scales, *rest: ((Wq.shape[0], Wq.shape[1] * 2), torch.float16))

_ops = torch.ops.streamk


# ---------------------------------------------------------------------------------------------
# The reference-shaped entry points
# ---------------------------------------------------------------------------------------------
def streamk_fp16(A, B, *, Wq=None, scales=None, layout="nt", out=None, plan=None, config=None,
                 zero=8, group=128, bias=None, activation=None, **kw):
    """C = A @ B.T (layout 'nt', B is [N,K]) or A @ B (layout 'nn', B is [K,N]) in fp16 with fp32
    accumulation.

    With `Wq` (uint8 [N, K/2], low nibble = even k) and `scales` (fp16 [N, K/group]) the weights
    are dequantised on the fly, w = fp16((q - zero) * scale), and B is ignored (pass None).
    `config`/kwargs: bm, bn, bk, grid, schedule, fixup, raster (see plan.make_config).
    `bias` (fp16 [N]) is added to every row in fp32 before the rounding to fp16; `activation`
    ('relu', 'gelu_tanh', 'silu') is applied after it, also in fp32.
    """
    if Wq is not None:
        return streamk_q4(A, Wq, scales, out=out, plan=plan, config=config, zero=zero, group=group, bias=bias,
                          activation=activation, **kw)
    cfg = _config_string(plan, config, kw)
    if out is None:
        return _ops.gemm_f16(A, B, layout, cfg, bias, activation or "none")
    _ops.gemm_f16_out(A, B, out, layout, cfg, bias, activation or "none")
    return out


def streamk_bf16(A, B, *, layout="nt", out=None, plan=None, config=None, bias=None, activation=None, **kw):
    """streamk_fp16 for bfloat16 operands and output (fp32 accumulation, C rounded to nearest even).
    The reference's scripts are fp16 / fp32 only; this is the bfloat16 instance of the same tile
    kernels."""
    cfg = _config_string(plan, config, kw)
    if out is None:
        return _ops.gemm_bf16(A, B, layout, cfg, bias, activation or "none")
    _ops.gemm_bf16_out(A, B, out, layout, cfg, bias, activation or "none")
    return out


def streamk_fp8(A, B, *, alpha=1.0, fmt=None, out=None, plan=None, config=None, bias=None, activation=None, **kw):
    """C = activation(alpha * (A @ B.T) + bias) for fp8 operands, A [M,K], B [N,K]; fp32 accumulation, alpha applied to the
    fp32 sums, fp16 C.  Both operands are OCP e4m3 (torch.float8_e4m3fn) or both OCP e5m2
    (torch.float8_e5m2); raw uint8 bytes are taken as `fmt` ("e4m3" by default, or "e5m2").  alpha is the
    product of the per-tensor scales of a scaled-fp8 caller; bias (fp16 [N]) and activation as for
    streamk_fp16, applied after alpha.  The reference's scripts stop at fp16; this is
    the same partitioner and fix-ups over the fp8 form of the tile kernel."""
    cfg = _config_string(plan, config, kw)
    if out is None:
        return _ops.gemm_f8(A, B, float(alpha), fmt or "", cfg, bias, activation or "none")
    _ops.gemm_f8_out(A, B, out, float(alpha), fmt or "", cfg, bias, activation or "none")
    return out


def streamk_int8(A, B, *, out=None, plan=None, config=None, **kw):
    """C = A @ B.T for int8 operands, A [M,K], B [N,K]; exact int32 accumulation, int32 C (the accumulator
    type the reference's Triton comparator picks for integer inputs, triton.streamk/first_wave.py:123).
    Every schedule and fix-up returns the same bits."""
    cfg = _config_string(plan, config, kw)
    if out is None:
        return _ops.gemm_i8(A, B, cfg)
    _ops.gemm_i8_out(A, B, out, cfg)
    return out


def tile_q4(Wq):
    """Packed weights Wq[N, K/2] -> the tiled layout (16 rows x 64 bytes per tile, [row block][group]),
    on the device Wq lives on.  Returns a [ceil(N/16)*16, K/2] array (rows past N are zero) to pass to
    streamk_q4(..., tiled=True); the weights then stream faster and the results are the same bit
    for bit.  The counterpart of the reference's offline weight transformation
    (streamk_fp16_ladder_block_reduce_q4.py:568-580)."""
    if Wq.dtype != torch.uint8 or Wq.dim() != 2 or not Wq.is_contiguous():
        raise ValueError("Wq must be a contiguous 2-D uint8 tensor")
    N, K = Wq.shape[0], Wq.shape[1] * 2
    out = torch.empty(((N + 15) // 16 * 16, K // 2), dtype=torch.uint8, device=Wq.device)
    if Wq.is_cuda:
        _lib.check(_lib.lib().sk_q4_tile(Wq.data_ptr(), N, K, out.data_ptr(), _stream_ptr()), "sk_q4_tile")
    else:
        _lib.check(_lib.lib().sk_q4_tile_host(Wq.data_ptr(), N, K, out.data_ptr()), "sk_q4_tile_host")
    return out


def untile_q4(tiled, N):
    """Inverse of tile_q4 for host tensors: the row-major Wq[N, K/2]."""
    if tiled.dtype != torch.uint8 or tiled.dim() != 2 or tiled.is_cuda or not tiled.is_contiguous():
        raise ValueError("tiled must be a contiguous 2-D uint8 tensor in host memory")
    K = tiled.shape[1] * 2
    if tiled.shape[0] != (N + 15) // 16 * 16:
        raise ValueError("tiled has ceil(N/16)*16 rows")
    Wq = torch.empty((N, K // 2), dtype=torch.uint8)
    _lib.check(_lib.lib().sk_q4_untile_host(tiled.data_ptr(), N, K, Wq.data_ptr()), "sk_q4_untile_host")
    return Wq


def streamk_q4(A, Wq, scales, *, out=None, plan=None, config=None, zero=8, group=128, tiled=False, zeros=None,
               bias=None, activation=None, **kw):
    """C[M,N] fp16 = A[M,K] fp16 @ dequant(Wq)[N,K].T, weights in natural nibble order
    (streamk_fp16_ladder_block_reduce_q4.py:552).  tiled=True: Wq is the output of tile_q4 (N is
    then taken from scales).  zeros: one zero point per scale group and row ([N, K/group], integers
    0..15) instead of the scalar `zero`.  bias / activation: as for streamk_fp16."""
    cfg = _config_string(plan, config, kw)
    if out is None:
        return _ops.gemm_q4(A, Wq, scales, zeros, zero, group, bool(tiled), cfg, bias, activation or "none")
    _ops.gemm_q4_out(A, Wq, scales, zeros, out, zero, group, bool(tiled), cfg, bias, activation or "none")
    return out


def dequant_q4(Wq, scales, *, zero=8, group=128, zeros=None):
    """fp16 W[N,K] from packed nibbles, by the same device function the Q4 GEMM uses."""
    return _ops.dequant_q4(Wq, scales, zeros, zero, group)


def pack_q4(q):
    """Wq[N, K/2] from q[N, K] (uint8 values 0..15, host memory): element k of a row goes to nibble
    k & 1 of byte k / 2, the order streamk_fp16_ladder_block_reduce_q4.py:552 expands.  This is the
    array the kernels read: there is no further permutation step (the reference's :568-595)."""
    if q.dtype != torch.uint8 or q.dim() != 2 or q.is_cuda or not q.is_contiguous():
        raise ValueError("q must be a contiguous 2-D uint8 tensor in host memory")
    N, K = q.shape
    Wq = torch.empty((N, K // 2), dtype=torch.uint8)
    _lib.check(_lib.lib().sk_q4_pack_host(q.data_ptr(), N, K, Wq.data_ptr()), "sk_q4_pack_host")
    return Wq


def unpack_q4(Wq):
    """Inverse of pack_q4 (host memory)."""
    if Wq.dtype != torch.uint8 or Wq.dim() != 2 or Wq.is_cuda or not Wq.is_contiguous():
        raise ValueError("Wq must be a contiguous 2-D uint8 tensor in host memory")
    N, K = Wq.shape[0], Wq.shape[1] * 2
    q = torch.empty((N, K), dtype=torch.uint8)
    _lib.check(_lib.lib().sk_q4_unpack_host(Wq.data_ptr(), N, K, q.data_ptr()), "sk_q4_unpack_host")
    return q


def quantize_q4(W, *, group=128, zero=8, asymmetric=False):
    """(Wq[N, K/2] uint8, scales[N, K/group] fp16) from fp16 W[N, K], on the device W lives on.
    scale = fp16(max|w| / levels) per group, q = clamp(rint(w / scale) + zero, 0, 15).
    asymmetric=True: each group's range [min(w, 0), max(w, 0)] is mapped onto 0..15 with its own zero
    point; returns (Wq, scales, zeros[N, K/group] fp16) for streamk_q4(..., zeros=zeros)."""
    if W.dtype != torch.float16 or W.dim() != 2 or W.stride(1) != 1:
        raise ValueError("W must be a 2-D fp16 tensor with unit stride along K")
    N, K = W.shape
    ldw = W.stride(0) if N > 1 else K  # the stride of a single row is arbitrary
    Wq = torch.empty((N, K // 2), dtype=torch.uint8, device=W.device)
    sc = torch.empty((N, K // max(group, 1)), dtype=torch.float16, device=W.device)
    if asymmetric:
        zp = torch.empty_like(sc)
        if W.is_cuda:
            rc = _lib.lib().sk_q4_quantize_zp(W.data_ptr(), N, K, ldw, group, Wq.data_ptr(), sc.data_ptr(),
                                              zp.data_ptr(), _stream_ptr())
        else:
            rc = _lib.lib().sk_q4_quantize_zp_host(W.data_ptr(), N, K, ldw, group, Wq.data_ptr(), sc.data_ptr(),
                                                   zp.data_ptr())
        _lib.check(rc, "sk_q4_quantize_zp")
        return Wq, sc, zp
    if W.is_cuda:
        rc = _lib.lib().sk_q4_quantize(W.data_ptr(), N, K, ldw, group, zero, Wq.data_ptr(), sc.data_ptr(),
                                       _stream_ptr())
        _lib.check(rc, "sk_q4_quantize")
    else:
        rc = _lib.lib().sk_q4_quantize_host(W.data_ptr(), N, K, ldw, group, zero, Wq.data_ptr(),
                                            sc.data_ptr())
        _lib.check(rc, "sk_q4_quantize_host")
    return Wq, sc


def streamk_fp32(A, B, *, layout="nn", out=None, plan=None, config=None, **kw):
    """C = A @ B in fp32 (layout 'nn', B is [K,N]: streamk_fp32.py:65-76)."""
    cfg = _config_string(plan, config, kw)
    if out is None:
        return _ops.gemm_f32(A, B, layout, cfg)
    _ops.gemm_f32_out(A, B, out, layout, cfg)
    return out


class StreamKKernel:
    """A planned GEMM, callable as `kernel(A, B, C)` (C written in place), the role of the
    reference's compiled `tl_mod` (streamk_fp32.py:197-202)."""

    def __init__(self, M, N, K, dtype, layout, plan):
        self.M, self.N, self.K, self.dtype, self.layout, self.plan = M, N, K, dtype, layout, plan

    def __call__(self, A, B, C):
        if self.dtype == "float16":
            return streamk_fp16(A, B, layout=self.layout, out=C, plan=self.plan)
        return streamk_fp32(A, B, layout=self.layout, out=C, plan=self.plan)

    def do_bench(self, fn=None, warmup=25, rep=100):
        """Mean milliseconds per call over `rep` back-to-back launches after `warmup`
        (streamk_fp16.py:394)."""
        if fn is None:
            dt = torch.float16 if self.dtype == "float16" else torch.float32
            A = torch.randn(self.M, self.K, device="cuda", dtype=dt)
            bshape = (self.N, self.K) if self.layout == "nt" else (self.K, self.N)
            B = torch.randn(*bshape, device="cuda", dtype=dt)
            C = torch.empty(self.M, self.N, device="cuda", dtype=dt)
            fn = lambda: self(A, B, C)  # noqa: E731
        return bench_ms(fn, warmup, rep)


def bench_ms(fn, warmup=25, rep=100):
    for _ in range(warmup):
        fn()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    start.record()
    for _ in range(rep):
        fn()
    end.record()
    torch.cuda.synchronize()
    workspace_status()
    return start.elapsed_time(end) / rep


_timing_probes = None  # [(stream, graph of 100 launches of a one-wave kernel)], made on first use


def timing_stream():
    """A side stream for timing microsecond kernels.  The streams of a process are not alike on this part: on some
    of them (which ones changes from process to process and, for the first few streams used, with time) the
    launches of a captured graph start about 0.15 us later each and a launch that streams its operands from HBM
    takes 1.6 us longer, measurement after measurement, while cache-resident launches take the same time.  Eight
    streams are kept, each with a captured probe of 100 one-wave kernels; every call replays the probes and
    returns the stream whose probe is fastest at that moment."""
    global _timing_probes
    if _timing_probes is None:
        x = torch.zeros(64, device="cuda")
        _timing_probes = []
        for _ in range(8):
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                x.add_(1.0)
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=s):
                    for _ in range(100):
                        x.add_(1.0)
                g.replay()
                torch.cuda.synchronize()
            _timing_probes.append((s, g, x))
    st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = None
    for s, g, _ in _timing_probes:
        with torch.cuda.stream(s):
            t = 1e9
            for _ in range(2):
                st.record()
                g.replay()
                en.record()
                torch.cuda.synchronize()
                t = min(t, st.elapsed_time(en))
        if best is None or t < best[0]:
            best = (t, s)
    return best[1]


def graph_ms(fn, launches=20, warmup=3, window_ms=40.0, groups=7, stream=None):
    """Per-launch time in ms of `fn`, for kernels of a few microseconds: `launches` calls are captured into one
    graph (no host cost between them), which is replayed in `groups` separately timed groups that together span
    `window_ms` of GPU time; the median group is returned.  Runs on `stream`, by default on timing_stream()."""
    s = timing_stream() if stream is None else stream
    with torch.cuda.stream(s):
        for _ in range(max(1, warmup)):
            fn()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            for _ in range(launches):
                fn()
        g.replay()
        torch.cuda.synchronize()
        st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        st.record()
        g.replay()
        en.record()
        torch.cuda.synchronize()
        per_group = max(1, int(window_ms / groups / max(st.elapsed_time(en), 1e-3)))
        samples = []
        for _ in range(groups):
            st.record()
            for _ in range(per_group):
                g.replay()
            en.record()
            torch.cuda.synchronize()
            samples.append(st.elapsed_time(en) / (per_group * launches))
    workspace_status()
    return sorted(samples)[len(samples) // 2]


def tl_matmul_streamk(M, N, K, *, dtypeAB="float16", layout=None, block_M=None, block_N=None,
                      block_K=None, streamk_programs=None, schedule="auto", fixup="auto", raster=0):
    """Factory with the reference's name and role (streamk_fp32.py:57-72, streamk_fp16.py:116-124):
    fixes shape, tile and partition, returns the in-place kernel callable."""
    if layout is None:
        layout = "nt" if dtypeAB == "float16" else "nn"
    plan = make_plan(M, N, K, dtypeAB, layout, bm=block_M, bn=block_N, bk=block_K,
                     grid=streamk_programs, schedule=schedule, fixup=fixup, raster=raster)
    return StreamKKernel(M, N, K, dtypeAB, layout, plan)
