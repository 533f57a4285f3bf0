"""ctypes binding of the C-ABI in ``include/cfk_fmha.h``.

Mirrors the reference's host entry ``fmhaForwardDevice`` (src/fmha-pipeline/fmha_forward.cu:86-93): device
pointers for Q/K/V/O in [B,S,H,D], sizes, softmax scale, precision.  torch is used only to own device memory
and streams; all compute happens in ``libcfk_fmha.so``.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import math
import os
import struct
import subprocess
import warnings

_HERE = os.path.dirname(os.path.abspath(__file__))
_LIB_PATH = os.path.join(_HERE, "libcfk_fmha.so")
_lib = None
_launch = None   # (fmha, fmha with workspace, gemm): the launching entry points taking their parameter block as bytes
_BINDING_PATH = os.path.join(_HERE, "cfk_torch.so")
_native = None   # csrc/cfk_torch.cpp, where it can be loaded: plain calls without the interpreter between their steps
_torch = None

CFK_FP16 = 1
CFK_FP8_E4M3 = 2
CFK_FP32 = 3  # GEMM only
CFK_V_BSHD = 0
CFK_V_BDHS = 1
CFK_GEMM_TN = 0
CFK_GEMM_NN = 1
CFK_OPT_PREDICTABLE_LATENCY = 1
CFK_OPT_FAST_E4M3_WEIGHTS = 2


class CfkError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"cfk error {code}: {msg}")
        self.code = code


class FmhaFwdParams(ctypes.Structure):
    """``cfk_fmha_fwd_params`` (include/cfk_fmha.h)."""
    _fields_ = [
        ("dtype", ctypes.c_int32), ("v_dtype", ctypes.c_int32),
        ("batch", ctypes.c_int32), ("heads", ctypes.c_int32),
        ("seqlen_q", ctypes.c_int32), ("seqlen_kv", ctypes.c_int32),
        ("head_dim", ctypes.c_int32), ("v_layout", ctypes.c_int32),
        ("q", ctypes.c_void_p), ("k", ctypes.c_void_p), ("v", ctypes.c_void_p), ("o", ctypes.c_void_p),
        ("softmax_scale", ctypes.c_float),
        ("q_descale", ctypes.c_float), ("k_descale", ctypes.c_float), ("v_descale", ctypes.c_float),
        ("dbg_s", ctypes.c_void_p), ("dbg_row_max", ctypes.c_void_p), ("dbg_row_sum", ctypes.c_void_p),
    ]


class GemmParams(ctypes.Structure):
    """``cfk_gemm_params`` (include/cfk_fmha.h)."""
    _fields_ = [
        ("dtype", ctypes.c_int32), ("layout", ctypes.c_int32),
        ("m", ctypes.c_int32), ("n", ctypes.c_int32), ("k", ctypes.c_int32), ("batch", ctypes.c_int32),
        ("alpha", ctypes.c_float), ("beta", ctypes.c_float),
        ("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("c", ctypes.c_void_p), ("d", ctypes.c_void_p),
    ]


# The same two blocks for the launch path: packing bytes takes a fraction of the time of filling a ctypes structure.
_FMHA_BLOCK = struct.Struct("=8i4Q4f3Q")
_GEMM_BLOCK = struct.Struct("=6i2f4Q")


def _pack(block, *args):
    try:
        return block.pack(*args)
    except (OverflowError, struct.error):   # a factor beyond float32, of whatever type: infinite, as the field of a ctypes structure and native mode make it
        return struct.pack(block.format.replace("=", "@"), *args)


assert _FMHA_BLOCK.size == ctypes.sizeof(FmhaFwdParams) and _GEMM_BLOCK.size == ctypes.sizeof(GemmParams)


def lib_path() -> str:
    return _LIB_PATH


def build(verbose: bool = False) -> str:
    """Compile every HIP source for gfx950 (``make -C csrc``; always recompiles what changed)."""
    cmd = ["make", "-C", os.path.join(_HERE, "csrc"), "-j8"]
    res = subprocess.run(cmd, capture_output=not verbose, text=True)
    if res.returncode != 0:
        raise RuntimeError("building libcfk_fmha.so failed:\n" + (res.stdout or "") + (res.stderr or ""))
    return _LIB_PATH


def lib():
    """The loaded C-ABI library.  Raises if it has not been built -- there is no fallback path."""
    global _lib
    if _lib is None:
        if not os.path.exists(_LIB_PATH):
            raise RuntimeError(
                f"{_LIB_PATH} is missing: build it first (python -c 'import __graft_entry__ as g; g.build()' "
                f"or make -C {os.path.join(_HERE, 'csrc')}). There is no CPU fallback.")
        l = ctypes.CDLL(_LIB_PATH)
        l.cfk_fmha_forward.restype = ctypes.c_int
        l.cfk_fmha_forward.argtypes = [ctypes.POINTER(FmhaFwdParams), ctypes.c_void_p]
        l.cfk_fmha_forward_ws.restype = ctypes.c_int
        l.cfk_fmha_forward_ws.argtypes = [ctypes.POINTER(FmhaFwdParams), ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p]
        l.cfk_fmha_forward_workspace.restype = ctypes.c_int64
        l.cfk_fmha_forward_workspace.argtypes = [ctypes.POINTER(FmhaFwdParams)]
        l.cfk_fmha_forward_or_workspace.restype = ctypes.c_int64
        l.cfk_fmha_forward_or_workspace.argtypes = [ctypes.POINTER(FmhaFwdParams), ctypes.c_void_p]
        l.cfk_fmha_forward_plan.restype = ctypes.c_int
        l.cfk_fmha_forward_plan.argtypes = [ctypes.POINTER(FmhaFwdParams)] + [ctypes.POINTER(ctypes.c_int32)] * 4
        l.cfk_fmha_forward_mfma.restype = ctypes.c_int
        l.cfk_fmha_forward_mfma.argtypes = [ctypes.POINTER(FmhaFwdParams), ctypes.POINTER(ctypes.c_int32)]
        l.cfk_fmha_forward_kernel.restype = ctypes.c_int
        l.cfk_fmha_forward_kernel.argtypes = [ctypes.POINTER(FmhaFwdParams), ctypes.c_char_p, ctypes.c_int32]
        l.cfk_gemm_f16.restype = ctypes.c_int
        l.cfk_gemm_f16.argtypes = [ctypes.c_int32] * 3 + [ctypes.c_void_p] * 3 + [ctypes.c_int32, ctypes.c_void_p]
        l.cfk_gemm.restype = ctypes.c_int
        l.cfk_gemm.argtypes = [ctypes.POINTER(GemmParams), ctypes.c_void_p]
        l.cfk_init.restype = ctypes.c_int
        l.cfk_init.argtypes = []
        l.cfk_set_option.restype = ctypes.c_int
        l.cfk_set_option.argtypes = [ctypes.c_int32, ctypes.c_int32]
        l.cfk_last_error.restype = ctypes.c_char_p
        l.cfk_version.restype = ctypes.c_char_p
        _lib = l
    return _lib


def init() -> None:
    """``cfk_init``: one-time set-up of every kernel on the current device (optional; launches do it on demand)."""
    _check(lib().cfk_init())


def set_option(option: int, value: int) -> None:
    """``cfk_set_option``: process-wide options (``CFK_OPT_PREDICTABLE_LATENCY``, ``CFK_OPT_FAST_E4M3_WEIGHTS``)."""
    _check(lib().cfk_set_option(option, value))


def last_error() -> str:
    return lib().cfk_last_error().decode()


def version() -> str:
    return lib().cfk_version().decode()


def _check(rc):
    if rc != 0:
        raise CfkError(rc, last_error())


def make_params(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, q=0, k=0, v=0, o=0, softmax_scale=None,
                q_descale=1.0, k_descale=1.0, v_descale=1.0, v_layout=CFK_V_BSHD, v_dtype=None,
                dbg_row_max=0, dbg_row_sum=0, dbg_s=0) -> FmhaFwdParams:
    p = FmhaFwdParams()
    p.dtype = dtype
    p.v_dtype = dtype if v_dtype is None else v_dtype
    p.batch, p.heads, p.seqlen_q, p.seqlen_kv, p.head_dim = batch, heads, seqlen_q, seqlen_kv, head_dim
    p.v_layout = v_layout
    p.q, p.k, p.v, p.o = q or None, k or None, v or None, o or None
    p.softmax_scale = (1.0 / math.sqrt(head_dim)) if softmax_scale is None else softmax_scale
    p.q_descale, p.k_descale, p.v_descale = q_descale, k_descale, v_descale
    p.dbg_s = dbg_s or None
    p.dbg_row_max = dbg_row_max or None
    p.dbg_row_sum = dbg_row_sum or None
    return p


def fmha_forward_plan(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, v_layout=CFK_V_BSHD, v_dtype=None):
    """(block_m, block_n, lds_bytes, threads) the library picks; raises CfkError for unsupported shapes.  No GPU needed."""
    p = make_params(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, v_layout=v_layout, v_dtype=v_dtype)
    out = [ctypes.c_int32() for _ in range(4)]
    _check(lib().cfk_fmha_forward_plan(ctypes.byref(p), *[ctypes.byref(x) for x in out]))
    return tuple(x.value for x in out)


def fmha_forward_mfma(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, v_layout=CFK_V_BSHD, v_dtype=None):
    """``cfk_fmha_forward_mfma``: 32 or 16, the MFMA shape of the kernel build the library picks.  No GPU needed."""
    p = make_params(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, v_layout=v_layout, v_dtype=v_dtype)
    out = ctypes.c_int32()
    _check(lib().cfk_fmha_forward_mfma(ctypes.byref(p), ctypes.byref(out)))
    return out.value


def fmha_forward_kernel(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, v_layout=CFK_V_BSHD, v_dtype=None):
    """``cfk_fmha_forward_kernel``: the name of the instantiation the library launches for this call, as a kernel trace
    prints it (``fmha_fwd_kernel16p<128,64,8,2,0,0,0,0,2,0,1,1>``).  No GPU needed."""
    p = make_params(dtype, batch, heads, seqlen_q, seqlen_kv, head_dim, v_layout=v_layout, v_dtype=v_dtype)
    buf = ctypes.create_string_buffer(80)
    _check(lib().cfk_fmha_forward_kernel(ctypes.byref(p), buf, len(buf)))
    return buf.value.decode()


def _load_native(l, torch_version):
    """The extension, or None where it cannot serve -- not built, or built against another torch: every call then goes through ctypes."""
    try:
        loader = importlib.machinery.ExtensionFileLoader("cfk_torch", _BINDING_PATH)
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("cfk_torch", loader))
        loader.exec_module(module)
        if getattr(module, "torch_version", None) != torch_version:
            raise ImportError("it was built against another torch")
    except ImportError as e:
        warnings.warn(f"{_BINDING_PATH} is not used with torch {torch_version}: {e} (make -C {os.path.join(_HERE, 'csrc')} builds it); small "
                      "calls take up to 2 us longer on the host", RuntimeWarning, stacklevel=3)
        return None
    module.setup(*(ctypes.cast(fn, ctypes.c_void_p).value for fn in (l.cfk_fmha_forward_or_workspace, l.cfk_fmha_forward_ws, l.cfk_gemm)))
    return module


def _launchers():
    """torch and the launching entry points, looked up once."""
    global _torch, _launch, _native
    if _launch is None:
        import torch
        l = lib()
        _torch = torch
        _native = _load_native(l, str(torch.__version__))
        _launch = (ctypes.CFUNCTYPE(ctypes.c_int64, ctypes.c_char_p, ctypes.c_void_p)(("cfk_fmha_forward_or_workspace", l)),
                   ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p)(("cfk_fmha_forward_ws", l)),
                   ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p, ctypes.c_void_p)(("cfk_gemm", l)))
    return _launch


def _stream_ptr(stream):
    """The hipStream_t of ``stream`` (a torch stream or a pointer; None: torch's current stream of the current device)."""
    if stream is None:
        # (torch.cuda.current_stream() builds a Stream object: 2.5 us, as much as the launch itself)
        return _torch._C._cuda_getCurrentRawStream(_torch._C._cuda_getDevice())
    return stream if isinstance(stream, int) else stream.cuda_stream


def fmha_forward(q, k, v, o=None, softmax_scale=None, q_descale=1.0, k_descale=1.0, v_descale=1.0,
                 v_layout=CFK_V_BSHD, row_max=None, row_sum=None, scores=None, stream=None, prepare=False):
    """O = softmax(scale * Q K^T) V on device tensors in [B,S,H,D] (D contiguous).
    ``prepare=True`` launches nothing and returns a ``PreparedForward``: a callable that repeats this exact call.

    q,k,v: torch CUDA tensors, float16, or float8_e4m3fn / uint8 holding e4m3 codes (v may be float16 with e4m3
    q,k: hybrid mode).  ``v`` is [B,D,H,S] when
    ``v_layout == CFK_V_BDHS``.  ``row_max`` / ``row_sum`` / ``scores`` are the optional debug taps.  Returns ``o`` (float16 [B,Sq,H,D]); launches asynchronously on ``stream``
    (default: torch's current stream).  A call whose keys are split takes scratch memory from torch's allocator; capture it through
    ``torch.cuda.graph``, which keeps that memory for the replays."""
    if _native is not None and stream is None and row_max is None and row_sum is None and scores is None and not prepare:
        done = _native.fmha(q, k, v, o, softmax_scale, q_descale, k_descale, v_descale, v_layout, _workspace_or_none)
        if done is not None:   # (None: not a plain call)
            return done if type(done) is not int else _check(done)
    launch, launch_ws, _ = _launch or _launchers()
    f16 = _torch.float16
    if not (q.is_cuda and k.is_cuda and v.is_cuda):
        raise ValueError("q, k, v must be device tensors (there is no CPU path)")
    if not (q.is_contiguous() and k.is_contiguous() and v.is_contiguous()):
        raise ValueError("q, k, v must be contiguous [B,S,H,D]")
    qt, vt = q.dtype, v.dtype
    if qt == f16:
        dtype = CFK_FP16
    elif qt in (_torch.float8_e4m3fn, _torch.uint8):
        dtype = CFK_FP8_E4M3
    else:
        raise ValueError(f"unsupported dtype {qt}")
    if k.dtype != qt:
        raise ValueError("q and k must share one dtype")
    if vt == qt:
        v_dtype = dtype
    elif dtype == CFK_FP8_E4M3 and vt == f16:
        v_dtype = CFK_FP16  # hybrid mode: e4m3 Q,K with fp16 P,V (the reference's fp8 build without GEMM2FP8)
    else:
        raise ValueError("v must have the dtype of q, or float16 with fp8 q/k")
    B, Sq, H, D = q_shape = q.shape
    k_shape = k.shape
    Skv = k_shape[1]
    if k_shape != (B, Skv, H, D):
        raise ValueError("k shape mismatch")
    if v.shape != (k_shape if v_layout == CFK_V_BSHD else (B, D, H, Skv)):
        raise ValueError(f"v shape {tuple(v.shape)} does not match layout {v_layout}: expected "
                         f"{(B, Skv, H, D) if v_layout == CFK_V_BSHD else (B, D, H, Skv)}")
    if o is None:
        o = _torch.empty_like(q, dtype=f16)
    elif o.dtype != f16 or o.shape != q_shape or not o.is_contiguous() or not o.is_cuda:
        raise ValueError("o must be a contiguous float16 device tensor [B,Sq,H,D]")
    for t in (row_max, row_sum):
        if t is not None and (t.dtype != _torch.float32 or t.shape != (B, H, Sq) or not t.is_contiguous()):
            raise ValueError("row_max/row_sum must be contiguous float32 [B,H,Sq]")
    if scores is not None and (scores.dtype != _torch.float32 or scores.shape != (B, H, Sq, Skv)
                               or not scores.is_contiguous()):
        raise ValueError("scores must be contiguous float32 [B,H,Sq,Skv]")
    scale = 1.0 / math.sqrt(D) if softmax_scale is None else softmax_scale
    block = _pack(_FMHA_BLOCK, dtype, v_dtype, B, H, Sq, Skv, D, v_layout, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                             scale, q_descale, k_descale, v_descale, *(0 if t is None else t.data_ptr() for t in (scores, row_max, row_sum)))
    if prepare:
        return PreparedForward(FmhaFwdParams.from_buffer_copy(block), (q, k, v, o, row_max, row_sum, scores), stream)
    stream = _stream_ptr(stream)
    rc = launch(block, stream)
    if rc > 0:   # the call is not made yet: it can use this much scratch memory
        ws = _workspace_or_none(rc, stream)
        rc = launch_ws(block, None if ws is None else ws.data_ptr(), rc, stream)
    if rc != 0:
        _check(rc)
    return o


def _workspace(n, stream):
    """n bytes of scratch memory for one call, from torch's allocator for the stream that the call runs on (a hipStream_t of the
    current device): free again when the caller drops it, reused only by later work of that stream (or of the graph being
    captured)."""
    dev = _torch._C._cuda_getDevice()
    device = _torch.device("cuda", dev)
    if stream == _torch._C._cuda_getCurrentRawStream(dev):
        return _torch.empty(n, dtype=_torch.uint8, device=device)
    # (0 is the default stream; to torch.cuda.ExternalStream it is "none given", and its answer a stream of torch's pool)
    with _torch.cuda.stream(_torch.cuda.ExternalStream(stream, device=device) if stream else _torch.cuda.default_stream(device)):
        return _torch.empty(n, dtype=_torch.uint8, device=device)


def _workspace_or_none(n, stream):
    """``_workspace``; None if there is no room: the call runs without it."""
    try:
        return _workspace(n, stream)
    except _torch.OutOfMemoryError:
        return None


def _is_capturing(stream):
    """Whether a graph is being captured from ``stream`` (a c_void_p; the null stream cannot be captured)."""
    status = ctypes.c_int(0)
    return bool(stream.value) and lib().hipStreamIsCapturing(stream, ctypes.byref(status)) == 0 and status.value != 0


class PreparedForward:
    """One ``cfk_fmha_forward`` call with its parameter block filled in once (``fmha_forward(..., prepare=True)``): calling
    the object launches it again on the stream given at preparation (torch's current stream then, if none was given).
    Captured through ``torch.cuda.graph`` the call belongs to the graph, which needs q, k, v, o and not this object.
    What a C++ caller's launch loop does (src/fmha-pipeline/fmha_forward.cu:578-592): the checks and the ctypes
    marshalling of ``fmha_forward`` cost several microseconds per call, as much as a small problem's kernel."""

    def __init__(self, params, tensors, stream):
        self.params, self.tensors = params, tensors   # (the tensors are held so that their memory stays alive)
        self.o = tensors[3]
        self._ref = ctypes.byref(params)
        stream = _stream_ptr(stream)
        self._stream = ctypes.c_void_p(stream)
        self._fn = lib().cfk_fmha_forward_ws
        self._ws_bytes = lib().cfk_fmha_forward_workspace(self._ref)
        # (kept: the calls run one after the other on one stream)
        self._ws = _workspace_or_none(self._ws_bytes, stream) if self._ws_bytes else None
        self._ws_ptr = None if self._ws is None else self._ws.data_ptr()

    def __call__(self):
        ws = self._ws_ptr
        if self._ws_bytes and _is_capturing(self._stream):   # (replays may come when what this object keeps is gone)
            graphs = _workspace_or_none(self._ws_bytes, self._stream.value)
            ws = None if graphs is None else graphs.data_ptr()
        rc = self._fn(self._ref, ws, self._ws_bytes, self._stream)
        if rc != 0:
            _check(rc)
        return self.o


def gemm_f16(a, b, c=None, layout=CFK_GEMM_TN, stream=None):
    """C[M,N] = A[M,K] . B  with B as [N,K] (TN, the reference's form) or [K,N] (NN); fp16 in, fp32 accumulate, fp16 out."""
    _launch or _launchers()
    if a.dtype != _torch.float16 or b.dtype != _torch.float16 or not (a.is_cuda and b.is_cuda):
        raise ValueError("a, b must be float16 device tensors")
    if not (a.is_contiguous() and b.is_contiguous()):
        raise ValueError("a, b must be contiguous")
    M, K = a.shape
    N = b.shape[0] if layout == CFK_GEMM_TN else b.shape[1]
    if tuple(b.shape) != ((N, K) if layout == CFK_GEMM_TN else (K, N)):
        raise ValueError("b shape mismatch")
    if c is None:
        c = a.new_empty((M, N))
    _check(lib().cfk_gemm_f16(M, N, K, a.data_ptr(), b.data_ptr(), c.data_ptr(), layout, _stream_ptr(stream)))
    return c


def gemm(a, b, c=None, alpha=1.0, beta=0.0, out=None, layout=CFK_GEMM_TN, stream=None):
    """D = alpha * A.B + beta * C, fp32 accumulate and epilogue (``cfk_gemm``).

    ``a`` is [M,K] or [L,M,K]; ``b`` is [N,K] (TN, the reference's form, src/cute-gemm-tma-gma/gemm.cu:362-380) or
    [K,N] (NN, fp16 only), with the same leading batch dimension; ``c`` / ``out`` are [M,N] or [L,M,N].  float16 or
    float32 device tensors, all of one dtype (the reference's types 3 and 1, gemm.cu:677-684).
    """
    if _native is not None and stream is None:
        done = _native.gemm(a, b, c, alpha, beta, out, layout)
        if done is not None:   # (None: not a plain call)
            return done if type(done) is not int else _check(done)
    _, _, launch = _launch or _launchers()
    dt = a.dtype
    if dt not in (_torch.float16, _torch.float32) or b.dtype != dt or not (a.is_cuda and b.is_cuda):
        raise ValueError("a, b must be float16 or float32 device tensors of one dtype")
    a_shape, b_shape = a.shape, b.shape
    if len(a_shape) not in (2, 3) or len(b_shape) != len(a_shape):
        raise ValueError("a, b must both be 2-D or both 3-D (leading batch dimension)")
    if not (a.is_contiguous() and b.is_contiguous()):
        raise ValueError("a, b must be contiguous")
    lead = a_shape[:-2]
    M, K = a_shape[-2:]
    N = b_shape[-2] if layout == CFK_GEMM_TN else b_shape[-1]
    if b_shape != (lead + ((N, K) if layout == CFK_GEMM_TN else (K, N))):
        raise ValueError("b shape mismatch")
    shape = lead + (M, N)
    if out is None:
        out = a.new_empty(shape)
    for t in (c, out):
        if t is not None and (t.dtype != dt or t.shape != shape or not t.is_contiguous() or not t.is_cuda):
            raise ValueError("c / out must be contiguous device tensors of a's dtype and shape " + str(tuple(shape)))
    rc = launch(_pack(_GEMM_BLOCK, CFK_FP16 if dt == _torch.float16 else CFK_FP32, layout, M, N, K, lead[0] if lead else 1, alpha, beta,
                                 a.data_ptr(), b.data_ptr(), 0 if c is None else c.data_ptr(), out.data_ptr()), _stream_ptr(stream))
    if rc != 0:
        _check(rc)
    return out
