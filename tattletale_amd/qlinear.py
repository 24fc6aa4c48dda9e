"""``QuantLinear`` -- host-side mirror of the reference's ``Linear`` layer over the C ABI.

Reference interface (workspace/transformers/src/layers/linear.nim:13-57)::

    Linear{weight, bias, in_features, out_features}
    Linear.init(weight, bias = none)      # weight (out_features, in_features)
    forward(self, x)                      # x (..., in_features) -> (..., out_features)

``QuantLinear`` keeps the same shape contract and the same two verbs.  The dense weight is
replaced by a packed buffer (uint8 blocks for Q8_0/Q4_K/Q6_K, u16 trellis words plus the
``suh``/``svh`` vectors for EXL3), so ``init`` takes the dimensions explicitly.  ``forward``
makes one ``ttq_linear_forward`` call; like ``Linear.forward`` it launches asynchronously on
the current stream and returns a tensor.  torch is used for device memory and streams only.
"""
from __future__ import annotations

import ctypes as C
import warnings
from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib
from ._lib import BF16, F16, F32, QLinearStruct, TtqError, check

_DTYPE_CODE = {torch.float32: F32, torch.float16: F16, torch.bfloat16: BF16}


def _code(dt: torch.dtype) -> int:
    try:
        return _DTYPE_CODE[dt]
    except KeyError:
        raise TtqError(_lib.ERR_DTYPE, "dtype %s" % dt) from None


class _PythonHost:
    """In place of the native host half where that is not built: no call is taken, the Python code behind each serves it."""

    @staticmethod
    def linear_forward(*args) -> int:
        return 1

    rmsnorm = silu_and_mul = q4_k_silu_mul = linear_forward


_native_module = None


def _native():
    """The native host half (csrc/ttq_torch.cpp) with the library's entry points bound.  Its functions return the
    output, a negative status, or 1 where the tensors are not what they take: the Python code behind each call then
    finds and raises the error.  Not built, or built for another torch: that Python code makes the calls of the
    library, the same kernels with some 5 us more host time each."""
    global _native_module
    if _native_module is None:
        L = _lib.lib()
        why = ext = None
        try:
            from . import _ttq_torch as ext
        except ImportError as e:
            why = str(e)
        else:
            built_for = getattr(ext, "torch_version", None)
            if built_for != torch.__version__:
                why = "built for torch %s, this is %s" % (built_for, torch.__version__)
        if why is not None:
            warnings.warn("tattletale_amd._ttq_torch is not used (%s): calls cost more host time.  Build it with "
                          "`python -m tattletale_amd.build`" % why, RuntimeWarning, stacklevel=3)
            ext = _PythonHost
        else:
            ext.bind(*(C.cast(fn, C.c_void_p).value for fn in (
                L.ttq_linear_forward, L.ttq_linear_forward_ws, L.ttq_rmsnorm, L.ttq_silu_and_mul,
                L.ttq_gemv_q4_k_silu_mul, L.ttq_gemm_q4_k_silu_mul)))
        _native_module = ext
    return _native_module


def _native_status(r, where: str) -> None:
    """Raises for a status of the library; returns for 1 (the caller goes on in Python)."""
    if r != 1:
        raise TtqError(r, where)


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def _stream(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _require_device(*tensors: Optional[torch.Tensor]) -> torch.device:
    dev = None
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise TtqError(_lib.ERR_UNSUPPORTED, "tensor is not on a GPU (no CPU fallback exists)")
        if dev is not None and t.device != dev:
            raise TtqError(_lib.ERR_UNSUPPORTED, "tensors on different devices")
        dev = t.device
        if not t.is_contiguous():
            raise TtqError(_lib.ERR_SHAPE, "tensor must be contiguous")
    return dev


@dataclass
class QuantLinear:
    """Quantized linear layer; fields follow ``Linear`` (linear.nim:13-27)."""

    qweight: torch.Tensor                 # packed bytes / trellis words, on the GPU
    format: int                           # _lib.Q8_0 | Q4_K | Q6_K | EXL3
    in_features: int
    out_features: int
    bias: Optional[torch.Tensor] = None   # (out_features,)
    suh: Optional[torch.Tensor] = None    # EXL3: (in_features,) float16
    svh: Optional[torch.Tensor] = None    # EXL3: (out_features,) float16
    bits: int = 0
    codebook: int = _lib.CB_MCG
    # PRECISION_F32_SCALES keeps the decode kernels for every batch; PRECISION_BF16_OK lets fp32
    # activations be rounded to bf16 for the matrix-core GEMM
    precision: int = _lib.PRECISION_AUTO

    @classmethod
    def init(cls, qweight: torch.Tensor, format: int, in_features: int, out_features: int,
             bias: Optional[torch.Tensor] = None, suh: Optional[torch.Tensor] = None,
             svh: Optional[torch.Tensor] = None, bits: int = 0,
             codebook: int = _lib.CB_MCG, precision: int = _lib.PRECISION_AUTO) -> "QuantLinear":
        """Creates the layer from existing packed weights (no copy, no repacking), as
        ``Linear.init`` does from a dense weight (linear.nim:29-43)."""
        _require_device(qweight, bias, suh, svh)
        need = _lib.lib().ttq_packed_nbytes(format, out_features, in_features, bits)
        if need < 0:
            raise TtqError(int(need), "QuantLinear.init")
        have = qweight.numel() * qweight.element_size()
        if have != need:
            raise TtqError(_lib.ERR_SHAPE, "QuantLinear.init: packed buffer holds %d bytes, %d expected"
                           % (have, need))
        if bias is not None and bias.numel() != out_features:
            raise TtqError(_lib.ERR_SHAPE, "QuantLinear.init: bias length")
        if format == _lib.EXL3:
            if suh is None or svh is None:
                raise TtqError(_lib.ERR_NULL, "QuantLinear.init: EXL3 needs suh and svh")
            if suh.dtype != torch.float16 or svh.dtype != torch.float16:
                raise TtqError(_lib.ERR_DTYPE, "QuantLinear.init: suh/svh must be float16")
            if suh.numel() != in_features or svh.numel() != out_features:
                raise TtqError(_lib.ERR_SHAPE, "QuantLinear.init: suh/svh length")
        return cls(qweight, format, in_features, out_features, bias, suh, svh, bits, codebook, precision)

    def _struct(self) -> QLinearStruct:
        return QLinearStruct(
            format=self.format, bits=self.bits, codebook=self.codebook,
            bias_dtype=_code(self.bias.dtype) if self.bias is not None else 0,
            precision=self.precision, reserved=0,
            n_out=self.out_features, n_in=self.in_features,
            qweight=_ptr(self.qweight), suh=_ptr(self.suh), svh=_ptr(self.svh), bias=_ptr(self.bias))

    def workspace_bytes(self, m: int, x_dtype: torch.dtype) -> int:
        """Bytes of caller-owned workspace ``forward(..., workspace=...)`` needs for ``m`` rows
        (``ttq_workspace_bytes``); make it with ``torch.zeros`` -- it must be clear before its first use."""
        st = self._struct()
        n = _lib.lib().ttq_workspace_bytes(C.byref(st), m, _code(x_dtype))
        if n < 0:
            raise TtqError(int(n), "ttq_workspace_bytes")
        return int(n)

    def route(self, m: int, x_dtype: torch.dtype, out_dtype: Optional[torch.dtype] = None) -> str:
        """Name of the kernel family ``forward`` launches for ``m`` rows of ``x_dtype`` (``ttq_route``)."""
        st = self._struct()
        r = _lib.lib().ttq_route(C.byref(st), m, _code(x_dtype), _code(out_dtype or x_dtype))
        if r < 0:
            raise TtqError(int(r), "ttq_route")
        return _lib.lib().ttq_route_name(r).decode()

    def route_detail(self, m: int, x_dtype: torch.dtype, out_dtype: Optional[torch.dtype] = None) -> str:
        """What exactly that is: kernel, and for the tiled GEMM its tile, copies along K and way to the activations
        (``ttq_route_detail``)."""
        st, text = self._struct(), C.create_string_buffer(128)
        r = _lib.lib().ttq_route_detail(C.byref(st), m, _code(x_dtype), _code(out_dtype or x_dtype), text, len(text))
        if r < 0:
            raise TtqError(int(r), "ttq_route_detail")
        return text.value.decode()

    def forward(self, x: torch.Tensor, out_dtype: Optional[torch.dtype] = None,
                workspace: Optional[torch.Tensor] = None) -> torch.Tensor:
        """x (..., in_features) -> (..., out_features)  (linear.nim:45-57).

        ``out_dtype`` defaults to ``x.dtype`` (what ``F.linear`` returns); pass
        ``torch.float32`` for fp32 logits from 16-bit activations.  With ``workspace`` (a zero-filled
        uint8 tensor of at least ``workspace_bytes`` bytes) the call allocates nothing inside the
        library (``ttq_linear_forward_ws``)."""
        r = (_native_module or _native()).linear_forward(
            self.qweight, self.suh, self.svh, self.bias, self.format, self.in_features, self.out_features, self.bits,
            self.codebook, self.precision, x, out_dtype, workspace)
        if r.__class__ is not int:
            return r
        _native_status(r, "ttq_linear_forward" if workspace is None else "ttq_linear_forward_ws")
        if x.dim() == 0 or x.shape[-1] != self.in_features:
            raise TtqError(_lib.ERR_SHAPE, "QuantLinear.forward: x has shape %s, in_features is %d"
                           % (tuple(x.shape), self.in_features))
        dev = _require_device(self.qweight, x)
        out_dtype = out_dtype or x.dtype
        m = x.numel() // self.in_features
        y = torch.empty(x.shape[:-1] + (self.out_features,), dtype=out_dtype, device=dev)
        st = self._struct()
        with torch.cuda.device(dev):
            if workspace is not None:
                _require_device(self.qweight, workspace)
                check(_lib.lib().ttq_linear_forward_ws(C.byref(st), x.data_ptr(), _code(x.dtype), m, y.data_ptr(),
                                                       _code(out_dtype), workspace.data_ptr(), _nbytes(workspace),
                                                       _stream(dev)), "ttq_linear_forward_ws")
            else:
                check(_lib.lib().ttq_linear_forward(C.byref(st), x.data_ptr(), _code(x.dtype), m, y.data_ptr(),
                                                    _code(out_dtype), _stream(dev)), "ttq_linear_forward")
        return y

    __call__ = forward


# ------------------------------------------------------------------------- functional API
def _nbytes(t: torch.Tensor) -> int:
    return t.numel() * t.element_size()


def _check_packed(what: str, qweight: torch.Tensor, fmt: int, n_out: int, n_in: int, bits: int = 0) -> None:
    """The packed buffer must hold exactly the (n_out, n_in) matrix the kernels will index."""
    need = _lib.lib().ttq_packed_nbytes(fmt, n_out, n_in, bits)
    if need < 0:
        raise TtqError(int(need), what)
    if need and _nbytes(qweight) != need:     # an empty matrix reads nothing, whatever stands in for it
        raise TtqError(_lib.ERR_SHAPE, "%s: packed buffer holds %d bytes, %d expected for (%d, %d)"
                       % (what, _nbytes(qweight), need, n_out, n_in))


def _rows(what: str, x: torch.Tensor, n_in: int) -> int:
    if x.dim() == 0 or x.shape[-1] != n_in:
        raise TtqError(_lib.ERR_SHAPE, "%s: last dim of x is %s, n_in is %d"
                       % (what, x.shape[-1] if x.dim() else "missing", n_in))
    return x.numel() // n_in


def _check_out(what: str, out: torch.Tensor, m: int, n_out: int, dtype: torch.dtype) -> None:
    if out.dtype != dtype:
        raise TtqError(_lib.ERR_DTYPE, "%s: out is %s, %s expected" % (what, out.dtype, dtype))
    if out.numel() != m * n_out or (out.dim() > 0 and n_out and out.shape[-1] != n_out):
        raise TtqError(_lib.ERR_SHAPE, "%s: out has shape %s, (%d, %d) expected"
                       % (what, tuple(out.shape), m, n_out))


_GEMV = {_lib.Q8_0: "ttq_gemv_q8_0", _lib.Q4_K: "ttq_gemv_q4_k", _lib.Q6_K: "ttq_gemv_q6_k"}
_DEQ = {_lib.Q8_0: "ttq_dequant_q8_0", _lib.Q4_K: "ttq_dequant_q4_k", _lib.Q6_K: "ttq_dequant_q6_k"}


def gemv(fmt: int, qweight: torch.Tensor, x: torch.Tensor, n_out: int, n_in: int,
         out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """fp32 y (m, n_out) = x (m, n_in) * W^T through ``ttq_gemv_<fmt>``."""
    if fmt not in _GEMV:
        raise TtqError(_lib.ERR_FORMAT, f"no block-format GEMV for format {fmt}")
    dev = _require_device(qweight, x, out)
    _check_packed(_GEMV[fmt], qweight, fmt, n_out, n_in)
    m = _rows(_GEMV[fmt], x, n_in)
    if out is None:
        out = torch.empty((m, n_out), dtype=torch.float32, device=dev)
    else:
        _check_out(_GEMV[fmt], out, m, n_out, torch.float32)
    fn = getattr(_lib.lib(), _GEMV[fmt])
    with torch.cuda.device(dev):
        check(fn(qweight.data_ptr(), x.data_ptr(), _code(x.dtype), out.data_ptr(), m, n_out, n_in,
                 _stream(dev)), _GEMV[fmt])
    return out


def gemv_exl3(trellis: torch.Tensor, suh: torch.Tensor, svh: torch.Tensor, x: torch.Tensor,
              n_out: int, n_in: int, bits: int, codebook: int = _lib.CB_MCG,
              out: Optional[torch.Tensor] = None) -> torch.Tensor:
    dev = _require_device(trellis, suh, svh, x, out)
    if x.dtype != torch.float16:
        raise TtqError(_lib.ERR_DTYPE, "ttq_gemv_exl3 takes float16 activations")
    if suh.dtype != torch.float16 or svh.dtype != torch.float16:
        raise TtqError(_lib.ERR_DTYPE, "ttq_gemv_exl3: suh/svh must be float16")
    if suh.numel() != n_in or svh.numel() != n_out:
        raise TtqError(_lib.ERR_SHAPE, "ttq_gemv_exl3: suh/svh length")
    _check_packed("ttq_gemv_exl3", trellis, _lib.EXL3, n_out, n_in, bits)
    m = _rows("ttq_gemv_exl3", x, n_in)
    if out is None:
        out = torch.empty((m, n_out), dtype=torch.float32, device=dev)
    else:
        _check_out("ttq_gemv_exl3", out, m, n_out, torch.float32)
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_gemv_exl3(trellis.data_ptr(), suh.data_ptr(), svh.data_ptr(), x.data_ptr(),
                                       out.data_ptr(), m, n_out, n_in, bits, codebook, _stream(dev)),
              "ttq_gemv_exl3")
    return out


def gemm_exl3(trellis: torch.Tensor, suh: torch.Tensor, svh: torch.Tensor, x: torch.Tensor,
              n_out: int, n_in: int, bits: int, codebook: int = _lib.CB_MCG) -> torch.Tensor:
    """fp32 y (m, n_out) for many activation rows through ``ttq_gemm_exl3`` (activations rotated once,
    rounded to float16; every weight decoded once per 128 rows)."""
    dev = _require_device(trellis, suh, svh, x)
    if suh.dtype != torch.float16 or svh.dtype != torch.float16:
        raise TtqError(_lib.ERR_DTYPE, "ttq_gemm_exl3: suh/svh must be float16")
    if suh.numel() != n_in or svh.numel() != n_out:
        raise TtqError(_lib.ERR_SHAPE, "ttq_gemm_exl3: suh/svh length")
    _check_packed("ttq_gemm_exl3", trellis, _lib.EXL3, n_out, n_in, bits)
    m = _rows("ttq_gemm_exl3", x, n_in)
    out = torch.empty((m, n_out), dtype=torch.float32, device=dev)
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_gemm_exl3(trellis.data_ptr(), suh.data_ptr(), svh.data_ptr(), x.data_ptr(),
                                       _code(x.dtype), out.data_ptr(), m, n_out, n_in, bits, codebook,
                                       _stream(dev)), "ttq_gemm_exl3")
    return out


_GEMM_ENTRY = {_lib.Q4_K: "ttq_gemm_q4_k", _lib.Q6_K: "ttq_gemm_q6_k", _lib.Q8_0: "ttq_gemm_q8_0"}


def gemm(fmt: int, qweight: torch.Tensor, x: torch.Tensor, n_out: int, n_in: int,
         out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """bf16 Y (m, n_out) = bf16 X (m, n_in) * W^T through ``ttq_gemm_<format>``."""
    name = _GEMM_ENTRY.get(fmt)
    if name is None:
        raise TtqError(_lib.ERR_FORMAT, f"no prefill GEMM for format {fmt}")
    dev = _require_device(qweight, x, out)
    if x.dtype != torch.bfloat16:
        raise TtqError(_lib.ERR_DTYPE, f"{name} takes bfloat16 activations")
    _check_packed(name, qweight, fmt, n_out, n_in)
    m = _rows(name, x, n_in)
    if out is None:
        out = torch.empty((m, n_out), dtype=torch.bfloat16, device=dev)
    else:
        _check_out(name, out, m, n_out, torch.bfloat16)
    with torch.cuda.device(dev):
        check(getattr(_lib.lib(), name)(qweight.data_ptr(), x.data_ptr(), out.data_ptr(), m, n_out, n_in,
                                        _stream(dev)), name)
    return out


def gemm_q4_k(qweight: torch.Tensor, x: torch.Tensor, n_out: int, n_in: int,
              out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """bf16 Y (m, n_out) = bf16 X (m, n_in) * W^T through ``ttq_gemm_q4_k``."""
    return gemm(_lib.Q4_K, qweight, x, n_out, n_in, out)


def dequantize(fmt: int, qweight: torch.Tensor, n_out: int, n_in: int,
               dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """Dense (n_out, n_in) weight from packed blocks through ``ttq_dequant_<fmt>``."""
    if fmt not in _DEQ:
        raise TtqError(_lib.ERR_FORMAT, f"no block-format dequantizer for format {fmt}")
    dev = _require_device(qweight)
    _check_packed(_DEQ[fmt], qweight, fmt, n_out, n_in)
    out = torch.empty((n_out, n_in), dtype=dtype, device=dev)
    fn = getattr(_lib.lib(), _DEQ[fmt])
    with torch.cuda.device(dev):
        check(fn(qweight.data_ptr(), out.data_ptr(), _code(dtype), n_out, n_in, _stream(dev)), _DEQ[fmt])
    return out


def dequantize_exl3(trellis: torch.Tensor, n_out: int, n_in: int, bits: int,
                    codebook: int = _lib.CB_MCG) -> torch.Tensor:
    """Decoded (unscaled, unrotated) trellis values, float16 (n_out, n_in)."""
    dev = _require_device(trellis)
    _check_packed("ttq_dequant_exl3", trellis, _lib.EXL3, n_out, n_in, bits)
    out = torch.empty((n_out, n_in), dtype=torch.float16, device=dev)
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_dequant_exl3(trellis.data_ptr(), out.data_ptr(), n_out, n_in, bits, codebook,
                                          _stream(dev)), "ttq_dequant_exl3")
    return out


def hadamard128_(v: torch.Tensor, pre: Optional[torch.Tensor] = None,
                 post: Optional[torch.Tensor] = None) -> torch.Tensor:
    """In-place 128-group Hadamard transform of a float32 tensor (optional fp16 pre/post scale)."""
    dev = _require_device(v, pre, post)
    if v.dtype != torch.float32:
        raise TtqError(_lib.ERR_DTYPE, "hadamard128_ takes float32")
    for t in (pre, post):
        if t is not None and (t.dtype != torch.float16 or t.numel() != v.numel()):
            raise TtqError(_lib.ERR_SHAPE, "hadamard128_: pre/post must be float16 vectors as long as v")
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_hadamard128_f32(v.data_ptr(), _ptr(pre), _ptr(post), v.numel(), _stream(dev)),
              "ttq_hadamard128_f32")
    return v


# ------------------------------------------------------------------------------ gated MLP
def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    """(..., 2h) -> (..., h): silu(x[..., :h]) * x[..., h:]
    (workspace/transformers/src/kernels/activations.nim:14-38), through ``ttq_silu_and_mul``."""
    r = (_native_module or _native()).silu_and_mul(x)
    if r.__class__ is not int:
        return r
    _native_status(r, "ttq_silu_and_mul")
    dev = _require_device(x)
    if x.dim() == 0 or x.shape[-1] == 0 or x.shape[-1] % 2:
        raise TtqError(_lib.ERR_SHAPE, "silu_and_mul: last dim must be even and not empty")
    h = x.shape[-1] // 2
    out = torch.empty(x.shape[:-1] + (h,), dtype=x.dtype, device=dev)
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_silu_and_mul(x.data_ptr(), out.data_ptr(), _code(x.dtype), x.numel() // (2 * h), h,
                                          _stream(dev)), "ttq_silu_and_mul")
    return out


def gemv_q4_k_silu_mul(qweight: torch.Tensor, x: torch.Tensor, n_ff: int, n_in: int,
                       out_dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """y (m, n_ff) = silu(x Wg^T) * (x Wu^T) for the packed (2*n_ff, n_in) Q4_K matrix [Wg; Wu],
    one kernel (``ttq_gemv_q4_k_silu_mul``)."""
    dev = _require_device(qweight, x)
    _check_packed("ttq_gemv_q4_k_silu_mul", qweight, _lib.Q4_K, 2 * n_ff, n_in)
    m = _rows("ttq_gemv_q4_k_silu_mul", x, n_in)
    out = torch.empty((m, n_ff), dtype=out_dtype, device=dev)
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_gemv_q4_k_silu_mul(qweight.data_ptr(), x.data_ptr(), _code(x.dtype), out.data_ptr(),
                                                _code(out_dtype), m, n_ff, n_in, _stream(dev)),
              "ttq_gemv_q4_k_silu_mul")
    return out


def gemm_q4_k_silu_mul(qweight: torch.Tensor, x: torch.Tensor, n_ff: int, n_in: int) -> torch.Tensor:
    """bf16 y (m, n_ff) = silu(x Wg^T) * (x Wu^T) for the packed (2*n_ff, n_in) Q4_K matrix [Wg; Wu] and a
    multi-row bf16 activation: the prefill GEMM with silu_and_mul in its epilogue
    (``ttq_gemm_q4_k_silu_mul``)."""
    dev = _require_device(qweight, x)
    if x.dtype != torch.bfloat16:
        raise TtqError(_lib.ERR_DTYPE, "ttq_gemm_q4_k_silu_mul takes bfloat16 activations")
    _check_packed("ttq_gemm_q4_k_silu_mul", qweight, _lib.Q4_K, 2 * n_ff, n_in)
    m = _rows("ttq_gemm_q4_k_silu_mul", x, n_in)
    out = torch.empty((m, n_ff), dtype=torch.bfloat16, device=dev)
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_gemm_q4_k_silu_mul(qweight.data_ptr(), x.data_ptr(), out.data_ptr(), m, n_ff, n_in,
                                                _stream(dev)), "ttq_gemm_q4_k_silu_mul")
    return out


def rmsnorm(x: torch.Tensor, gamma: torch.Tensor, eps: float, residual: Optional[torch.Tensor] = None):
    """``RmsNorm.forward`` (residual None) / ``forward_with_residual``
    (workspace/transformers/src/layers/norm.nim:23-38) through ``ttq_rmsnorm``.
    Returns (normalized, new_residual or None)."""
    r = (_native_module or _native()).rmsnorm(x, gamma, eps, residual)
    if r.__class__ is not int:
        return r
    _native_status(r, "ttq_rmsnorm")
    dev = _require_device(x, gamma, residual)
    n = x.shape[-1] if x.dim() else 0
    if n == 0 or gamma.numel() != n or gamma.dtype != x.dtype or (residual is not None and
                                                                  (residual.shape != x.shape or residual.dtype != x.dtype)):
        raise TtqError(_lib.ERR_SHAPE, "rmsnorm: x is empty, or gamma / residual do not match it")
    normed = torch.empty_like(x)
    new_res = torch.empty_like(x) if residual is not None else None
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_rmsnorm(x.data_ptr(), _ptr(residual), gamma.data_ptr(), eps, _code(x.dtype),
                                     _ptr(new_res), normed.data_ptr(), x.numel() // n, n, _stream(dev)),
              "ttq_rmsnorm")
    return normed, new_res


def gemv_q4_k_rmsnorm(qweight: torch.Tensor, x: torch.Tensor, gamma: torch.Tensor, eps: float, n_out: int,
                      n_in: int, residual: Optional[torch.Tensor] = None, silu_mul: bool = False,
                      out_dtype: torch.dtype = torch.float32, want_normed: bool = True):
    """y = Linear(RmsNorm(x [, residual])) (optionally followed by silu_and_mul over a gate/up
    weight of 2*n_out rows) in one kernel (``ttq_gemv_q4_k_rmsnorm``).
    Returns (y, normalized or None, new_residual or None)."""
    dev = _require_device(qweight, x, gamma, residual)
    _check_packed("ttq_gemv_q4_k_rmsnorm", qweight, _lib.Q4_K, (2 if silu_mul else 1) * n_out, n_in)
    m = _rows("ttq_gemv_q4_k_rmsnorm", x, n_in)
    if gamma.numel() != n_in or gamma.dtype != x.dtype or (residual is not None and
                                                          (residual.shape != x.shape or residual.dtype != x.dtype)):
        raise TtqError(_lib.ERR_SHAPE, "ttq_gemv_q4_k_rmsnorm: gamma / residual do not match x")
    y = torch.empty((m, n_out), dtype=out_dtype, device=dev)
    normed = torch.empty_like(x) if want_normed else None
    new_res = torch.empty_like(x) if residual is not None else None
    with torch.cuda.device(dev):
        check(_lib.lib().ttq_gemv_q4_k_rmsnorm(qweight.data_ptr(), x.data_ptr(), _ptr(residual), gamma.data_ptr(),
                                               eps, _code(x.dtype), _ptr(new_res), _ptr(normed), y.data_ptr(),
                                               _code(out_dtype), m, n_out, n_in, 1 if silu_mul else 0,
                                               _stream(dev)), "ttq_gemv_q4_k_rmsnorm")
    return y, normed, new_res


@dataclass
class QuantGatedMLP:
    """Quantized counterpart of ``GatedMLP`` (workspace/transformers/src/layers/mlp.nim:25-60):
    one fused gate/up projection, silu_and_mul, down projection."""

    gate_up_proj: QuantLinear            # (2 * intermediate, hidden), gate rows first (mlp.nim:39)
    down_proj: QuantLinear               # (hidden, intermediate)

    @classmethod
    def init(cls, gate_up_proj: QuantLinear, down_proj: QuantLinear) -> "QuantGatedMLP":
        """Takes the already concatenated gate/up weight: rows of the block formats concatenate
        as bytes, so ``torch.cat([gate_packed, up_packed])`` is the ``F.cat`` of mlp.nim:39."""
        if gate_up_proj.out_features != 2 * down_proj.in_features:
            raise TtqError(_lib.ERR_SHAPE, "QuantGatedMLP.init: gate_up rows != 2 * down columns")
        if gate_up_proj.in_features != down_proj.out_features:
            raise TtqError(_lib.ERR_SHAPE, "QuantGatedMLP.init: hidden sizes differ")
        return cls(gate_up_proj, down_proj)

    # From here on silu_and_mul runs in the GEMM's epilogue, for what the result is rather than for speed: the activation
    # gets its sums in fp32 where the separate launches round gate and up to bf16 first (distance from 64-bit
    # arithmetic 2.9e-3 against 3.9e-3), and the (rows, 2 * intermediate) tensor is never made (235 MB at 4096 rows of
    # 28672).  On wide layers that costs time, because the epilogue's exponentials and reciprocals are quarter rate and
    # this GEMM reads its activations through LDS where the plain one reads a packed copy.  Fused / separate, us:
    # 28672 x 4096 466 / 441 at 2048 rows, 910 / 865 at 4096, 1820 / 1748 at 8192; 27648 x 5120 563 / 524 and 1100 / 1030,
    # 37888 x 3584 558 / 523 and 1098 / 1042, 16384 x 2048 168 / 161 and 321 / 310; 6144 x 1024 39.8 / 50.0 and 83.6 / 85.9.
    # Fewer rows take the separate launches (28672 x 4096 131 / 123 at 512 rows, 432 / 404 at 1792): prompts of those lengths
    # keep the faster form.
    FUSED_GEMM_MIN_ROWS = 2048
    # 17 to 64 rows: the same entry point runs the few-row kernel with the activation in its epilogue, one launch and one
    # (rows, 2 * intermediate) round trip less, and the same fp32 sums.  It is faster where the separate GEMM would be the
    # same kernel (fused / separate, us, at 32 rows 6144 x 1024 6.0 / 8.3, 12288 x 2048 10.1 / 12.4, 17920 x 1536 17.1 / 19.4);
    # wide layers (20480 weight rows and more) have a plain GEMM that streams its weights through LDS and no fused form of
    # it, and the fused launch is taken for its sums although it costs time (28672 x 4096 at 32 rows 35.1 / 28.7, at 64
    # 35.1 / 34.2, 27648 x 5120 40.3 / 32.9, 37888 x 3584 46.2 / 30.3).  Below nine rows the decode kernels for several rows
    # plus silu_and_mul are faster on wide layers (28672 x 4096 at 8 rows 27.4 / 24.0, 27648 x 5120 44.4 / 27.8).  From 9 to
    # 16 rows either is (at 16 28672 x 4096 27.0 / 29.4, 37888 x 3584 35.2 / 40.8, 27648 x 5120 40.3 / 29.0); the separate
    # launches are taken.
    FUSED_FEW_ROWS = (17, 64)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        """x (..., hidden) -> (..., hidden)  (mlp.nim:43-60).  On Q4_K weights a 16-bit activation of one to
        four tokens takes the fused GEMV + silu_and_mul kernel and a bf16 activation of 17 to 64 or at least
        ``FUSED_GEMM_MIN_ROWS`` rows the GEMM with silu_and_mul in its epilogue; everything else runs
        the projection, ``silu_and_mul`` and the down projection as three launches."""
        gu = self.gate_up_proj
        n_in, n_ff = gu.in_features, self.down_proj.in_features
        act = None
        if gu.format == _lib.Q4_K and gu.bias is None and x.dtype is not torch.float32 and x.shape[-1] == n_in:
            m = x.numel() // n_in
            # one row, or two to four rows on the shapes whose fused kernel reads the weights once for all of them
            # (rows of 2048 or 4096 values, 2 * n_ff from 4096 to 32768 weight rows)
            few = 2 <= m <= 4 and n_in in (2048, 4096) and n_ff % 8 == 0 and 2048 <= n_ff <= 16384
            decode = m == 1 or few
            if decode or (x.dtype is torch.bfloat16 and n_in % 256 == 0 and
                          (m >= self.FUSED_GEMM_MIN_ROWS or self.FUSED_FEW_ROWS[0] <= m <= self.FUSED_FEW_ROWS[1])):
                act = self._fused_activation(x, m, n_ff, n_in, not decode)
        if act is None:
            act = silu_and_mul(gu.forward(x))
        return self.down_proj.forward(act)

    def _fused_activation(self, x: torch.Tensor, m: int, n_ff: int, n_in: int, gemm: bool) -> Optional[torch.Tensor]:
        """silu(gate) * up in one launch; None where the shape has no fused kernel."""
        qweight = self.gate_up_proj.qweight
        r = (_native_module or _native()).q4_k_silu_mul(qweight, x, n_ff, n_in, gemm)
        if r.__class__ is not int:
            return r
        if r == _lib.ERR_UNSUPPORTED:
            return None
        _native_status(r, "ttq_gemm_q4_k_silu_mul" if gemm else "ttq_gemv_q4_k_silu_mul")
        try:                                     # tensors that the native half does not take
            x2 = x.reshape(m, n_in)
            act = (gemm_q4_k_silu_mul(qweight, x2, n_ff, n_in) if gemm else
                   gemv_q4_k_silu_mul(qweight, x2, n_ff, n_in, out_dtype=x.dtype))
        except TtqError as e:
            if e.status != _lib.ERR_UNSUPPORTED:
                raise
            return None
        return act.reshape(x.shape[:-1] + (n_ff,))

    __call__ = forward
