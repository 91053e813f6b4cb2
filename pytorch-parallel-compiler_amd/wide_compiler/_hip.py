"""
ctypes binding of libwide_hip.so, the gfx950 kernels behind every wide primitive.

The library exposes a plain C ABI (see include/wc_abi.h at the repository root).  This
module loads it once, declares the entry points, and offers thin Python wrappers that

  * check that every tensor lives on a ROCm device, has the dtype / shape / inner
    contiguity the kernel needs, and that no autograd graph is requested (the kernels
    are forward-only);
  * pass raw device pointers, sizes and strides plus torch's current HIP stream;
  * turn a non-zero status into an exception carrying ``wc_last_error()``.

There is no CPU path and no fallback: when the library is missing, or a tensor is on
the CPU, the call raises.
"""

from __future__ import annotations

import ctypes
import os
import struct
from typing import Dict, List, Optional, Sequence

import torch
from torch import Tensor

ABI_VERSION = 7

F32, BF16, F16 = 0, 1, 2
ACT_NONE, ACT_RELU = 0, 1
CELL_GRU, CELL_LSTM = 0, 1
ERR_LIMIT = -5                  # WC_ERR_LIMIT: a size or layout the kernel does not take

_DTYPES = {torch.float32: F32, torch.bfloat16: BF16, torch.float16: F16}

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libwide_hip.so")

_lib = None


class WideKernelError(RuntimeError):
    """A libwide_hip.so entry point returned a non-zero status."""


class _RnnArgs(ctypes.Structure):
    _fields_ = [
        ("cell", ctypes.c_int32), ("dtype", ctypes.c_int32),
        ("n", ctypes.c_int64), ("batch", ctypes.c_int64), ("steps", ctypes.c_int64),
        ("input_size", ctypes.c_int64), ("hidden", ctypes.c_int64),
        ("x", ctypes.c_void_p),
        ("x_stride_n", ctypes.c_int64), ("x_stride_b", ctypes.c_int64), ("x_stride_t", ctypes.c_int64),
        ("w_ih", ctypes.c_void_p), ("w_hh", ctypes.c_void_p),
        ("b_ih", ctypes.c_void_p), ("b_hh", ctypes.c_void_p),
        ("h0", ctypes.c_void_p), ("c0", ctypes.c_void_p),
        ("out", ctypes.c_void_p), ("h_n", ctypes.c_void_p), ("c_n", ctypes.c_void_p),
        ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_int64),
        ("status", ctypes.c_void_p),
    ]


class _GemmArgs(ctypes.Structure):
    _fields_ = [
        ("dtype", ctypes.c_int32), ("out_dtype", ctypes.c_int32),
        ("bias_dtype", ctypes.c_int32), ("act", ctypes.c_int32),
        ("n", ctypes.c_int64), ("m", ctypes.c_int64), ("o", ctypes.c_int64), ("k", ctypes.c_int64),
        ("a", ctypes.c_void_p),
        ("a_stride_n", ctypes.c_int64), ("a_stride_outer", ctypes.c_int64),
        ("a_stride_inner", ctypes.c_int64), ("a_rows_inner", ctypes.c_int64),
        ("w", ctypes.c_void_p), ("w_stride_n", ctypes.c_int64),
        ("bias", ctypes.c_void_p), ("bias_stride_n", ctypes.c_int64),
        ("residual", ctypes.c_void_p),
        ("r_stride_n", ctypes.c_int64), ("r_stride_outer", ctypes.c_int64), ("r_stride_inner", ctypes.c_int64),
        ("c", ctypes.c_void_p),
        ("c_stride_n", ctypes.c_int64), ("c_stride_outer", ctypes.c_int64),
        ("c_stride_inner", ctypes.c_int64), ("c_rows_inner", ctypes.c_int64),
    ]


class _GemmPairArgs(ctypes.Structure):
    _fields_ = [
        *_GemmArgs._fields_,                     # the embedded wc_gemm_args
        ("w2", ctypes.c_void_p), ("w2_stride_n", ctypes.c_int64),
        ("bias2", ctypes.c_void_p), ("bias2_stride_n", ctypes.c_int64), ("o1", ctypes.c_int64),
    ]


class _Mlp2Args(ctypes.Structure):
    entry = "wc_mlp2"                  # the entry point the block is for
    _fields_ = [
        ("dtype", ctypes.c_int32), ("act1", ctypes.c_int32), ("act2", ctypes.c_int32),
        ("n", ctypes.c_int64), ("m", ctypes.c_int64), ("in_features", ctypes.c_int64),
        ("hidden", ctypes.c_int64), ("out_features", ctypes.c_int64),
        ("x", ctypes.c_void_p), ("x_stride_n", ctypes.c_int64), ("x_stride_outer", ctypes.c_int64),
        ("x_stride_inner", ctypes.c_int64), ("x_rows_inner", ctypes.c_int64),
        ("w1", ctypes.c_void_p), ("b1", ctypes.c_void_p), ("w2", ctypes.c_void_p), ("b2", ctypes.c_void_p),
        ("y", ctypes.c_void_p), ("y_stride_n", ctypes.c_int64), ("y_stride_outer", ctypes.c_int64),
        ("y_stride_inner", ctypes.c_int64), ("y_rows_inner", ctypes.c_int64),
    ]


class _ConvArgs(ctypes.Structure):
    _fields_ = [
        ("dtype", ctypes.c_int32), ("param_dtype", ctypes.c_int32), ("act", ctypes.c_int32),
        ("n", ctypes.c_int64), ("batch", ctypes.c_int64), ("c_in", ctypes.c_int64), ("c_out", ctypes.c_int64),
        ("h", ctypes.c_int64), ("w", ctypes.c_int64), ("kh", ctypes.c_int64), ("kw", ctypes.c_int64),
        ("stride_h", ctypes.c_int64), ("stride_w", ctypes.c_int64), ("pad_h", ctypes.c_int64),
        ("pad_w", ctypes.c_int64), ("dil_h", ctypes.c_int64), ("dil_w", ctypes.c_int64),
        ("h_out", ctypes.c_int64), ("w_out", ctypes.c_int64),
        ("x", ctypes.c_void_p), ("x_stride_n", ctypes.c_int64), ("x_stride_b", ctypes.c_int64),
        ("packed_weight", ctypes.c_void_p), ("bias", ctypes.c_void_p),
        ("bn_weight", ctypes.c_void_p), ("bn_bias", ctypes.c_void_p), ("bn_mean", ctypes.c_void_p),
        ("bn_var", ctypes.c_void_p), ("bn_eps", ctypes.c_float),
        ("residual", ctypes.c_void_p), ("r_stride_n", ctypes.c_int64), ("r_stride_b", ctypes.c_int64),
        ("y", ctypes.c_void_p), ("y_stride_n", ctypes.c_int64), ("y_stride_b", ctypes.c_int64),
        ("weight", ctypes.c_void_p),
    ]


class _Conv3dArgs(ctypes.Structure):
    _fields_ = [
        ("dtype", ctypes.c_int32), ("param_dtype", ctypes.c_int32), ("act", ctypes.c_int32),
        ("n", ctypes.c_int64), ("batch", ctypes.c_int64), ("c_in", ctypes.c_int64), ("c_out", ctypes.c_int64),
        ("d", ctypes.c_int64), ("h", ctypes.c_int64), ("w", ctypes.c_int64),
        ("kd", ctypes.c_int64), ("kh", ctypes.c_int64), ("kw", ctypes.c_int64),
        ("stride_d", ctypes.c_int64), ("stride_h", ctypes.c_int64), ("stride_w", ctypes.c_int64),
        ("pad_d", ctypes.c_int64), ("pad_h", ctypes.c_int64), ("pad_w", ctypes.c_int64),
        ("dil_d", ctypes.c_int64), ("dil_h", ctypes.c_int64), ("dil_w", ctypes.c_int64),
        ("d_out", ctypes.c_int64), ("h_out", ctypes.c_int64), ("w_out", ctypes.c_int64),
        ("x", ctypes.c_void_p), ("x_stride_n", ctypes.c_int64), ("x_stride_b", ctypes.c_int64),
        ("packed_weight", ctypes.c_void_p), ("bias", ctypes.c_void_p),
        ("y", ctypes.c_void_p), ("y_stride_n", ctypes.c_int64), ("y_stride_b", ctypes.c_int64),
    ]


class _AttnArgs(ctypes.Structure):
    _fields_ = [
        ("dtype", ctypes.c_int32), ("causal", ctypes.c_int32),
        ("nb", ctypes.c_int64), ("heads", ctypes.c_int64), ("sq", ctypes.c_int64), ("skv", ctypes.c_int64),
        ("head_dim", ctypes.c_int64), ("scale", ctypes.c_float),
        ("q", ctypes.c_void_p), ("q_stride_nb", ctypes.c_int64), ("q_stride_s", ctypes.c_int64),
        ("k", ctypes.c_void_p), ("k_stride_nb", ctypes.c_int64), ("k_stride_s", ctypes.c_int64),
        ("v", ctypes.c_void_p), ("v_stride_nb", ctypes.c_int64), ("v_stride_s", ctypes.c_int64),
        ("o", ctypes.c_void_p), ("o_stride_nb", ctypes.c_int64), ("o_stride_s", ctypes.c_int64),
        ("mask", ctypes.c_void_p), ("mask_stride_nb", ctypes.c_int64), ("mask_stride_head", ctypes.c_int64),
        ("mask_stride_q", ctypes.c_int64),
    ]


class _SelfAttnArgs(ctypes.Structure):
    _fields_ = [
        ("dtype", ctypes.c_int32), ("causal", ctypes.c_int32),
        ("n", ctypes.c_int64), ("b", ctypes.c_int64), ("s", ctypes.c_int64), ("d_model", ctypes.c_int64),
        ("heads", ctypes.c_int64), ("scale", ctypes.c_float),
        ("x", ctypes.c_void_p), ("x_stride_n", ctypes.c_int64), ("x_stride_b", ctypes.c_int64),
        ("x_stride_s", ctypes.c_int64),
        ("q_weight", ctypes.c_void_p), ("q_weight_stride_n", ctypes.c_int64),
        ("kv_weight", ctypes.c_void_p), ("kv_weight_stride_n", ctypes.c_int64),
        ("q_bias", ctypes.c_void_p), ("q_bias_stride_n", ctypes.c_int64),
        ("kv_bias", ctypes.c_void_p), ("kv_bias_stride_n", ctypes.c_int64),
        ("o", ctypes.c_void_p), ("o_stride_nb", ctypes.c_int64), ("o_stride_s", ctypes.c_int64),
    ]


def _packer(cls):
    """struct.pack for the fields of an argument struct in order (pointers as integers, 0 for NULL):
    the bytes of the C struct.  Packing a call's ~25 fields at once costs a third of setting them
    one by one on a ctypes structure."""
    codes = {ctypes.c_int32: "i", ctypes.c_int64: "q", ctypes.c_void_p: "P", ctypes.c_float: "f"}
    s = struct.Struct("@" + "".join(codes[t] for _, t in cls._fields_) + "0q")
    if s.size != ctypes.sizeof(cls):
        raise ImportError(f"wide_compiler: {cls.__name__} packs to {s.size} bytes, not {ctypes.sizeof(cls)}")
    return s.pack


_pack_gemm, _pack_gemm_pair, _pack_conv = _packer(_GemmArgs), _packer(_GemmPairArgs), _packer(_ConvArgs)
_pack_attn, _pack_self_attn = _packer(_AttnArgs), _packer(_SelfAttnArgs)

_P = ctypes.c_void_p
_I32 = ctypes.c_int32
_I64 = ctypes.c_int64
_F = ctypes.c_float

# name -> (restype, argtypes); the single source of truth for the exported ABI
SIGNATURES = {
    "wc_abi_version": (_I32, []),
    "wc_last_error": (ctypes.c_char_p, []),
    "wc_device_count": (_I32, []),
    "wc_pack_rows": (_I32, [ctypes.POINTER(_P), ctypes.POINTER(_I64), _I64, _I64, _I64, _P, _P]),
    "wc_swap01": (_I32, [_P, _I64, _I64, _I64, _I64, _I64, _P, _P]),
    "wc_embedding_gather": (_I32, [_P, _I64, _I64, _I64, _I32, _P, _I64, _I32, _P, _P, _P]),
    "wc_layernorm": (_I32, [_P, _I64, _I64, _P, _P, _P, _I64, _I64, _I64, _I64, _I64, _F, _I32, _I32, _P]),
    "wc_embedding_layernorm": (_I32, [_P, _I64, _I64, _I64, _P, _I64, _I32, _P, _P, _F, _I32, _I32, _P, _P, _P]),
    "wc_bn_eval": (_I32, [_P, _I64, _I64, _P, _P, _P, _P, _F, _P, _I64, _I64, _I64, _I64, _I32, _I32, _I32, _P]),
    "wc_group_norm": (_I32, [_P, _P, _I64, _I64, _I64, _I64, _I64, _P, _P, _F, _I32, _I32, _I32, _P]),
    "wc_rnn_workspace_bytes": (_I64, [ctypes.POINTER(_RnnArgs)]),
    "wc_rnn_status_offset": (_I64, [ctypes.POINTER(_RnnArgs)]),
    "wc_rnn_noalloc_scratch_bytes": (_I64, []),
    "wc_rnn_forward_noalloc": (_I32, [ctypes.POINTER(_RnnArgs), _P]),
    "wc_rnn_forward": (_I32, [ctypes.POINTER(_RnnArgs), _P]),
    "wc_rnn_set_spin_limit": (_I32, [_I32]),
    "wc_rnn_input_projection": (_I32, [ctypes.POINTER(_RnnArgs), _P]),
    "wc_rnn_recurrence": (_I32, [ctypes.POINTER(_RnnArgs), _P]),
    "wc_grouped_gemm": (_I32, [ctypes.POINTER(_GemmArgs), _P]),
    "wc_grouped_gemm_pair": (_I32, [ctypes.POINTER(_GemmPairArgs), _P]),
    "wc_mlp2_supported": (_I32, [_I32, _I64, _I64, _I64]),
    "wc_mlp2": (_I32, [ctypes.POINTER(_Mlp2Args), _P]),
    "wc_mlp2_any_supported": (_I32, [_I32, _I64, _I64, _I64, _I64, _I64]),
    "wc_mlp2_any": (_I32, [ctypes.POINTER(_Mlp2Args), _P]),
    "wc_conv_pack_weights": (_I32, [_P, _I64, _I64, _I64, _I64, _I64, _I32, _P, _P]),
    "wc_conv_packed_weight_elems": (_I64, [_I64, _I64, _I64, _I64, _I64]),
    "wc_conv2d": (_I32, [ctypes.POINTER(_ConvArgs), _P]),
    "wc_conv2d_direct_weights": (_I32, [ctypes.POINTER(_ConvArgs)]),
    "wc_conv3d": (_I32, [ctypes.POINTER(_Conv3dArgs), _P]),
    "wc_attention": (_I32, [ctypes.POINTER(_AttnArgs), _P]),
    "wc_self_attention": (_I32, [ctypes.POINTER(_SelfAttnArgs), _P]),
}


def lib():
    """Load libwide_hip.so (once) after torch's HIP runtime; raise if it is not built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            f"wide_compiler: {LIB_PATH} is not built. Build it with "
            f"`make -C {os.path.dirname(os.path.dirname(LIB_PATH))}` or __graft_entry__.build(); "
            "this build has no fallback path."
        )
    # torch is imported first so its libamdhip64.so.7 is the runtime the library binds to
    handle = ctypes.CDLL(LIB_PATH)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(handle, name)
        fn.restype = res
        fn.argtypes = args
    got = handle.wc_abi_version()
    if got != ABI_VERSION:
        raise ImportError(f"wide_compiler: libwide_hip.so ABI {got} != expected {ABI_VERSION}")
    _lib = handle
    return _lib


def last_error() -> str:
    return lib().wc_last_error().decode(errors="replace")


def _check(rc: int, what: str) -> None:
    if rc != 0:
        raise WideKernelError(f"{what} failed (status {rc}): {last_error()}")


def dtype_code(t: torch.dtype, what: str) -> int:
    try:
        return _DTYPES[t]
    except KeyError:
        raise TypeError(f"{what}: dtype {t} is not supported (float32, bfloat16, float16)") from None


def require_device(what: str, *tensors: Optional[Tensor]) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError(
                f"{what}: wide_compiler's MI355X build executes on ROCm device tensors only "
                f"(got a tensor on {t.device}); move the model and inputs to 'cuda'"
            )


def require_forward_only(what: str, *tensors: Optional[Tensor]) -> None:
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors):
        raise RuntimeError(
            f"{what}: the HIP wide kernels are forward-only; run under torch.no_grad() or "
            "torch.inference_mode()"
        )


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_of(t: Tensor) -> int:
    """The current HIP stream of t's device as an address (what the ABI's void* stream takes).
    torch's raw accessor costs a tenth of building a torch.cuda.Stream object per launch."""
    if _raw_stream is not None:
        return _raw_stream(t.get_device())
    return torch.cuda.current_stream(t.device).cuda_stream


def ptr(t: Optional[Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


try:
    # CPython launcher of the entry points (built beside libwide_hip.so): a call through it
    # costs a fraction of a ctypes call, which dominates a small forward's host time
    from . import _wc_launch
except ImportError:     # not built: the ctypes binding of the same entry points
    _wc_launch = None
_entries: Dict[str, int] = {}


def entry_address(name: str) -> int:
    """Address of libwide_hip.so's entry point `name` (looked up once)."""
    a = _entries.get(name)
    if a is None:
        a = _entries[name] = ctypes.cast(getattr(lib(), name), ctypes.c_void_p).value
    return a


def _launch(name: str, cls, block: bytes, stream: int) -> None:
    """Call the entry point `name` with the packed argument struct `block` (of type cls)."""
    if _wc_launch is not None:
        rc = _wc_launch.callb(_entries.get(name) or entry_address(name), block, stream)
    else:
        rc = getattr(lib(), name)(ctypes.byref(cls.from_buffer_copy(block)), stream)
    if rc:
        _check(rc, name)


# ---------------------------------------------------------------------------------------
# wrappers
# ---------------------------------------------------------------------------------------

def pack_rows(srcs: Sequence[Tensor], dst: Tensor, rows: int, row_bytes: int,
              row_strides_bytes: Sequence[int]) -> None:
    n = len(srcs)
    arr_p = (_P * n)(*[s.data_ptr() for s in srcs])
    arr_s = (_I64 * n)(*row_strides_bytes)
    _check(lib().wc_pack_rows(arr_p, arr_s, n, rows, row_bytes, dst.data_ptr(), stream_of(dst)),
           "wc_pack_rows")


def swap01(src: Tensor, d0: int, d1: int, s0_bytes: int, s1_bytes: int, inner_bytes: int,
           dst: Tensor) -> None:
    _check(lib().wc_swap01(src.data_ptr(), d0, d1, s0_bytes, s1_bytes, inner_bytes, dst.data_ptr(),
                           stream_of(src)), "wc_swap01")


def embedding_gather(weight: Tensor, ids: Tensor, out: Tensor, shared: bool,
                     err_flag: Optional[Tensor] = None) -> None:
    n, vocab, dim = weight.shape
    rows = ids.numel() if shared else ids.numel() // max(n, 1)
    _check(lib().wc_embedding_gather(weight.data_ptr(), n, vocab, dim, dtype_code(weight.dtype, "embedding"),
                                     ids.data_ptr(), rows, 1 if shared else 0, out.data_ptr(),
                                     ptr(err_flag), stream_of(weight)), "wc_embedding_gather")


def embedding_layernorm(weight: Tensor, ids: Tensor, gamma: Tensor, beta: Optional[Tensor], eps: float,
                        out: Tensor, shared: bool, err_flag: Optional[Tensor] = None) -> bool:
    """Gather + LayerNorm in one launch (wc_embedding_layernorm); False (nothing launched) where
    the fused kernel does not take the row size or alignment."""
    n, vocab, dim = weight.shape
    rows = ids.numel() if shared else ids.numel() // max(n, 1)
    rc = lib().wc_embedding_layernorm(weight.data_ptr(), n, vocab, dim, ids.data_ptr(), rows, 1 if shared else 0,
                                      gamma.data_ptr(), ptr(beta), float(eps), dtype_code(weight.dtype, "embedding"),
                                      dtype_code(gamma.dtype, "layernorm"), out.data_ptr(), ptr(err_flag),
                                      stream_of(weight))
    if rc == ERR_LIMIT:
        return False
    _check(rc, "wc_embedding_layernorm")
    return True


def layernorm(x: Tensor, x_ms: int, x_rs: int, gamma: Tensor, beta: Optional[Tensor], y: Tensor,
              y_ms: int, y_rs: int, n: int, rows_per_model: int, dim: int, eps: float) -> None:
    args = (x.data_ptr(), x_ms, x_rs, gamma.data_ptr(), 0 if beta is None else beta.data_ptr(), y.data_ptr(), y_ms,
            y_rs, n, rows_per_model, dim, float(eps), dtype_code(x.dtype, "layernorm"),
            dtype_code(gamma.dtype, "layernorm"), stream_of(x))
    if _wc_launch is not None:
        rc = _wc_launch.layernorm(_entries.get("wc_layernorm") or entry_address("wc_layernorm"), *args)
    else:
        rc = lib().wc_layernorm(*args)
    if rc:
        _check(rc, "wc_layernorm")


def bn_eval(x: Tensor, xsn: int, xsb: int, weight: Optional[Tensor], bias: Optional[Tensor],
            rmean: Tensor, rvar: Tensor, eps: float, y: Tensor, n: int, b: int, c: int, hw: int,
            relu: bool = False) -> None:
    _check(lib().wc_bn_eval(x.data_ptr(), xsn, xsb, ptr(weight), ptr(bias), rmean.data_ptr(), rvar.data_ptr(),
                            float(eps), y.data_ptr(), n, b, c, hw, dtype_code(x.dtype, "batchnorm"),
                            dtype_code(rmean.dtype, "batchnorm"), ACT_RELU if relu else ACT_NONE,
                            stream_of(x)), "wc_bn_eval")


def group_norm(x: Tensor, y: Tensor, n: int, b: int, c: int, s: int, groups: int,
               weight: Optional[Tensor], bias: Optional[Tensor], eps: float, relu: bool = False) -> None:
    """x, y contiguous [n, b, c, s]; statistics per (model, batch row, group of c // groups channels)."""
    pdt = weight.dtype if weight is not None else x.dtype
    _check(lib().wc_group_norm(x.data_ptr(), y.data_ptr(), n, b, c, s, groups, ptr(weight), ptr(bias), float(eps),
                               dtype_code(x.dtype, "group_norm"), dtype_code(pdt, "group_norm"),
                               ACT_RELU if relu else ACT_NONE, stream_of(x)), "wc_group_norm")


def grouped_gemm(*, n: int, m: int, o: int, k: int,
                 a: Tensor, a_sn: int, a_so: int, a_si: int, a_rows_inner: int,
                 w: Tensor, w_sn: int,
                 c: Tensor, c_sn: int, c_so: int, c_si: int, c_rows_inner: int,
                 bias: Optional[Tensor] = None, bias_sn: int = 0,
                 residual: Optional[Tensor] = None, r_sn: int = 0, r_so: int = 0, r_si: int = 0,
                 relu: bool = False) -> None:
    dt = dtype_code(a.dtype, "grouped_gemm")
    _launch("wc_grouped_gemm", _GemmArgs, _pack_gemm(
        dt, dtype_code(c.dtype, "grouped_gemm"), dt if bias is None else dtype_code(bias.dtype, "grouped_gemm"),
        ACT_RELU if relu else ACT_NONE, n, m, o, k, a.data_ptr(), a_sn, a_so, a_si, a_rows_inner,
        w.data_ptr(), w_sn, 0 if bias is None else bias.data_ptr(), bias_sn,
        0 if residual is None else residual.data_ptr(), r_sn, r_so, r_si,
        c.data_ptr(), c_sn, c_so, c_si, c_rows_inner), stream_of(a))


def grouped_gemm_pair(*, n: int, m: int, k: int, o1: int, o2: int, a: Tensor, a_sn: int, a_so: int, a_si: int,
                      a_rows_inner: int, w1: Tensor, bias1: Optional[Tensor], w2: Tensor, bias2: Optional[Tensor],
                      c: Tensor) -> None:
    """Columns [0, o1) of c [n, m, o1 + o2] (contiguous) from w1 [n, o1, k] / bias1 [n, o1], the rest from
    w2 [n, o2, k] / bias2 (wc_grouped_gemm_pair); weights contiguous and of a's dtype, biases
    contiguous and of one dtype."""
    dt = dtype_code(a.dtype, "grouped_gemm")
    o = o1 + o2
    bias = bias1 if bias1 is not None else bias2
    _launch("wc_grouped_gemm_pair", _GemmPairArgs, _pack_gemm_pair(
        dt, dt, dt if bias is None else dtype_code(bias.dtype, "grouped_gemm"), ACT_NONE, n, m, o, k, a.data_ptr(), a_sn, a_so, a_si, a_rows_inner,
        w1.data_ptr(), o1 * k, 0 if bias1 is None else bias1.data_ptr(), o1, 0, 0, 0, 0,
        c.data_ptr(), m * o, 0, o, max(m, 1), w2.data_ptr(), o2 * k, 0 if bias2 is None else bias2.data_ptr(), o2, o1),
        stream_of(a))


def mlp2_supported(dtype: torch.dtype, in_features: int, hidden: int, out_features: int) -> bool:
    """True when two chained layers of these widths run as one launch, at least for few rows."""
    return mlp2_entry(dtype, 1, 1, in_features, hidden, out_features) is not None


def mlp2_entry(dtype: torch.dtype, n: int, m: int, in_features: int, hidden: int, out_features: int) -> Optional[str]:
    """The entry point that runs n models of m rows as one launch: wc_mlp2 for the widths it takes,
    else wc_mlp2_any where one launch is faster than two GEMMs; None: two GEMMs."""
    if dtype not in _DTYPES:
        return None
    code = dtype_code(dtype, "mlp2")
    if lib().wc_mlp2_supported(code, in_features, hidden, out_features):
        return "wc_mlp2"
    return "wc_mlp2_any" if lib().wc_mlp2_any_supported(code, n, m, in_features, hidden, out_features) else None


def mlp2_args(*, n: int, m: int, in_features: int, hidden: int, out_features: int,
              x: Tensor, x_sn: int, x_so: int, x_si: int, x_rows_inner: int,
              w1: Tensor, b1: Optional[Tensor], w2: Tensor, b2: Optional[Tensor],
              y: Tensor, y_sn: int, y_so: int, y_si: int, y_rows_inner: int,
              relu1: bool, relu2: bool, entry: str = "wc_mlp2") -> "_Mlp2Args":
    """The filled argument block of wc_mlp2 or wc_mlp2_any (launch with mlp2_launch; a caller may
    keep it and change only the x / y addresses between launches)."""
    a = _Mlp2Args()
    if entry != a.entry:
        a.entry = entry
    a.dtype = dtype_code(x.dtype, "mlp2")
    a.act1 = ACT_RELU if relu1 else ACT_NONE
    a.act2 = ACT_RELU if relu2 else ACT_NONE
    a.n, a.m, a.in_features, a.hidden, a.out_features = n, m, in_features, hidden, out_features
    a.x, a.x_stride_n, a.x_stride_outer, a.x_stride_inner, a.x_rows_inner = x.data_ptr(), x_sn, x_so, x_si, x_rows_inner
    a.w1, a.b1, a.w2, a.b2 = w1.data_ptr(), ptr(b1), w2.data_ptr(), ptr(b2)
    a.y, a.y_stride_n, a.y_stride_outer, a.y_stride_inner, a.y_rows_inner = y.data_ptr(), y_sn, y_so, y_si, y_rows_inner
    return a


def mlp2_launch(a: "_Mlp2Args", stream: int) -> None:
    name = a.entry
    if _wc_launch is not None:
        rc = _wc_launch.call2(_entries.get(name) or entry_address(name), ctypes.addressof(a), stream)
    else:
        rc = getattr(lib(), name)(ctypes.byref(a), stream)
    if rc:
        _check(rc, name)


def mlp2(**kw) -> None:
    """wc_mlp2 with the arguments of mlp2_args, on x's current stream."""
    mlp2_launch(mlp2_args(**kw), stream_of(kw["x"]))


def rnn_args(*, cell: int, x: Tensor, w_ih: Tensor, w_hh: Tensor, b_ih: Optional[Tensor],
             b_hh: Optional[Tensor], h0: Optional[Tensor], c0: Optional[Tensor], out: Tensor,
             h_n: Optional[Tensor], c_n: Optional[Tensor], workspace: Optional[Tensor] = None,
             allocate: bool = True, status: Optional[Tensor] = None):
    """Fill the wc_rnn_args struct; allocates the workspace unless one is given or
    allocate is False (then the struct carries no workspace).  ``status`` is an optional
    int32 device word that a give-up of the partitioned recurrence's bounded waits sets (never
    cleared by the library).  Returns (args, workspace)."""
    n, batch, steps, in_size = x.shape
    hidden = w_hh.shape[-1]
    a = _RnnArgs()
    a.cell = cell
    a.dtype = dtype_code(x.dtype, "rnn")
    a.n, a.batch, a.steps, a.input_size, a.hidden = n, batch, steps, in_size, hidden
    a.x = x.data_ptr()
    a.x_stride_n, a.x_stride_b, a.x_stride_t = x.stride(0), x.stride(1), x.stride(2)
    a.w_ih, a.w_hh, a.b_ih, a.b_hh = w_ih.data_ptr(), w_hh.data_ptr(), ptr(b_ih), ptr(b_hh)
    a.h0, a.c0 = ptr(h0), ptr(c0)
    a.out, a.h_n, a.c_n = out.data_ptr(), ptr(h_n), ptr(c_n)
    if status is not None:
        if status.dtype != torch.int32 or status.device != x.device:
            raise ValueError("rnn status word must be an int32 tensor on the input's device")
        a.status = status.data_ptr()
    if not allocate and workspace is None:
        a.workspace, a.workspace_bytes = None, 0
        return a, None
    need = int(lib().wc_rnn_workspace_bytes(ctypes.byref(a)))
    ws = workspace
    if ws is None or ws.numel() * ws.element_size() < need:
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device=x.device)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel() * ws.element_size()
    return a, ws


# The partitioned recurrence's bounded cross-workgroup waits report a give-up (its outputs are
# then invalid) in a status word.  Every launch made through rnn_forward /
# rnn_forward_noalloc is given this device's own word, which the library never clears:
# it collects the verdict of every eager launch and of every replay of a captured graph
# until rnn_sync_check reads it, raises, and clears it.  After an eager launch a copy of
# the word is queued to pinned host memory behind an event, so a later check raises
# without blocking the stream; replays of captured launches queue no copy of their own,
# so the next check queues one for every device whose word a capture used.
_status_words: Dict[int, Tensor] = {}
_status_captured: set = set()
_rnn_pending: List = []


def rnn_status_word(device: torch.device) -> Tensor:
    """This device's status word (created, zeroed, at the first recurrent call outside
    graph capture)."""
    idx = torch.device(device).index
    idx = torch.cuda.current_device() if idx is None else idx
    w = _status_words.get(idx)
    if w is None:
        if torch.cuda.is_current_stream_capturing():
            raise WideKernelError("wide_compiler: run a recurrent layer once outside graph capture before "
                                  "capturing it (its status word is created then)")
        w = _status_words[idx] = torch.zeros(1, dtype=torch.int32, device=torch.device("cuda", idx))
    return w


def _queue_status_copy(word: Tensor) -> None:
    host = torch.empty(1, dtype=torch.int32, pin_memory=True)
    host.copy_(word, non_blocking=True)
    ev = torch.cuda.Event()
    ev.record(torch.cuda.current_stream(word.device))
    _rnn_pending.append((ev, host, word))


def _rnn_watch(word: Tensor) -> None:
    if torch.cuda.is_current_stream_capturing():
        _status_captured.add(word.device.index)
    else:
        _queue_status_copy(word)


def rnn_sync_check(block: bool = False) -> None:
    """Raise WideKernelError if a finished partitioned-recurrence launch or graph replay reported
    a bounded wait that gave up (its outputs are then invalid), and clear the word.
    block=True waits for every launch still in flight; otherwise launches whose status
    has not landed yet are checked by a later call."""
    global _rnn_pending
    if torch.cuda.is_current_stream_capturing():
        return                       # events cannot be queried while a graph is captured
    for idx in _status_captured:
        _queue_status_copy(_status_words[idx])
    if not _rnn_pending:
        return
    keep, failed = [], []
    for ev, host, word in _rnn_pending:
        if block:
            ev.synchronize()
        if ev.query():
            if int(host[0]) != 0 and all(word is not f for f in failed):
                failed.append(word)
        else:
            keep.append((ev, host, word))
    _rnn_pending = keep
    if failed:
        for word in failed:
            word.zero_()
        # copies still in flight may hold the verdict just reported
        _rnn_pending = [e for e in _rnn_pending if all(e[2] is not f for f in failed)]
        raise WideKernelError("wc_rnn_recurrence: a cross-workgroup wait of the partitioned recurrence gave up; "
                              "the outputs of that launch (or graph replay) are invalid")


def rnn_set_spin_limit(polls: int) -> int:
    """Poll rounds after which a partitioned-recurrence wait gives up for launches made from now
    on (0: at the first wait; < 0: the default); returns the previous value."""
    return int(lib().wc_rnn_set_spin_limit(int(polls)))


def _part_status(a: _RnnArgs, x: Tensor) -> Optional[Tensor]:
    """This device's status word, set in ``a``, when these sizes run the partitioned recurrence
    (the one recurrent kernel with cross-workgroup waits); None otherwise, and for a captured fp32
    launch, which takes the kernel without such waits."""
    if x.dtype == torch.float32 and torch.cuda.is_current_stream_capturing():
        return None
    if int(lib().wc_rnn_status_offset(ctypes.byref(a))) < 0:
        return None
    word = rnn_status_word(x.device)
    a.status = word.data_ptr()
    return word


def rnn_forward(**kw) -> None:
    """wc_rnn_forward with a fresh workspace (and, on the partitioned plan, this device's
    status word); a give-up of an earlier launch is raised here (non-blocking), or by
    rnn_sync_check."""
    rnn_sync_check()
    a, ws = rnn_args(**kw)
    word = _part_status(a, kw["x"])
    _launch("wc_rnn_forward", _RnnArgs, bytes(a), stream_of(kw["x"]))
    if word is not None:
        _rnn_watch(word)


def rnn_forward_noalloc(**kw) -> None:
    """wc_rnn_forward_noalloc: the same forward with the workspace in the library's static
    per-device scratch; nothing is allocated for the call (the status word is this
    device's persistent one)."""
    rnn_sync_check()
    a, _ = rnn_args(allocate=False, **kw)
    word = _part_status(a, kw["x"])
    _check(lib().wc_rnn_forward_noalloc(ctypes.byref(a), stream_of(kw["x"])), "wc_rnn_forward_noalloc")
    if word is not None:
        _rnn_watch(word)


def rnn_phase(a: _RnnArgs, phase: str, like: Tensor) -> None:
    """Run one phase ('input_projection' or 'recurrence') of a prepared rnn_args struct."""
    fn = getattr(lib(), f"wc_rnn_{phase}")
    _check(fn(ctypes.byref(a), stream_of(like)), f"wc_rnn_{phase}")


def conv_pack_weights(w: Tensor, n: int, c_out: int, c_in: int, kh: int, kw: int) -> Tensor:
    elems = int(lib().wc_conv_packed_weight_elems(n, c_out, c_in, kh, kw))
    out = torch.empty(max(elems, 8), dtype=w.dtype, device=w.device)
    args = (w.data_ptr(), n, c_out, c_in, kh, kw, dtype_code(w.dtype, "conv"), out.data_ptr(), stream_of(w))
    if _wc_launch is not None:
        rc = _wc_launch.conv_pack(_entries.get("wc_conv_pack_weights") or entry_address("wc_conv_pack_weights"), *args)
    else:
        rc = lib().wc_conv_pack_weights(*args)
    if rc:
        _check(rc, "wc_conv_pack_weights")
    return out


def conv2d(*, x: Tensor, weight: Tensor, n: int, c_in: int, c_out: int, kernel, stride, padding, dilation,
           y: Tensor, bias: Optional[Tensor] = None, bn=None, residual: Optional[Tensor] = None,
           relu: bool = False, packed: bool = False) -> None:
    """x / y / residual are [n, b, C, H, W] with dense [C, H, W] blocks; ``weight`` is the
    contiguous grouped filter bank [n*C_out, C_in, kh, kw]; bn = (weight, bias, running_mean,
    running_var, eps) or None.  The filters go to the kernel as they are where the library
    reads that layout (wc_conv2d_direct_weights), else (or with ``packed``) through one
    packing pass."""
    params = [t for t in (bias, *(bn[:4] if bn else ())) if t is not None]
    dt = dtype_code(x.dtype, "conv")
    bn_ptrs = (0, 0, 0, 0, 0.0) if bn is None else (ptr(bn[0]) or 0, ptr(bn[1]) or 0, ptr(bn[2]) or 0,
                                                    ptr(bn[3]) or 0, float(bn[4]))
    kh, kw = kernel
    xs, ys = x.shape, y.shape
    head = (dt, dtype_code(params[0].dtype, "conv") if params else dt, ACT_RELU if relu else ACT_NONE,
            n, xs[1], c_in, c_out, xs[3], xs[4], kh, kw, *stride, *padding, *dilation, ys[3], ys[4],
            x.data_ptr(), x.stride(0), x.stride(1))
    tail = (0 if bias is None else bias.data_ptr(), *bn_ptrs,
            *((0, 0, 0) if residual is None else (residual.data_ptr(), residual.stride(0), residual.stride(1))),
            y.data_ptr(), y.stride(0), y.stride(1), weight.data_ptr())
    a = None
    # sizes that one of the two kernels reading the filter bank may take (the tile kernel: short
    # filters, at least this many workgroups in one round); the library decides
    if not packed and (c_in * kh * kw <= 160 and kh * kw <= 9 and
                       n * xs[1] * ((ys[3] * ys[4] + 127) // 128) * ((c_out + 63) // 64) <= 256
                       or dt == BF16 and kw == 3 and c_in in (32, 64)):
        a = _pack_conv(*head, 0, *tail)
        if not lib().wc_conv2d_direct_weights(ctypes.byref(_ConvArgs.from_buffer_copy(a))):
            a = None
    if a is None:
        packed_w = conv_pack_weights(weight, n, c_out, c_in, kh, kw)
        a = _pack_conv(*head, packed_w.data_ptr(), *tail)
    _launch("wc_conv2d", _ConvArgs, a, stream_of(x))


def conv3d(*, x: Tensor, packed_w: Tensor, n: int, c_in: int, c_out: int, kernel, stride, padding, dilation,
           y: Tensor, bias: Optional[Tensor] = None, relu: bool = False) -> None:
    """x / y are [n, b, C, D, H, W] with dense [C, D, H, W] blocks."""
    a = _Conv3dArgs()
    a.dtype = dtype_code(x.dtype, "conv3d")
    a.param_dtype = dtype_code(bias.dtype, "conv3d") if bias is not None else a.dtype
    a.act = ACT_RELU if relu else ACT_NONE
    a.n, a.batch, a.c_in, a.c_out = n, x.shape[1], c_in, c_out
    a.d, a.h, a.w = x.shape[3], x.shape[4], x.shape[5]
    a.kd, a.kh, a.kw = kernel
    a.stride_d, a.stride_h, a.stride_w = stride
    a.pad_d, a.pad_h, a.pad_w = padding
    a.dil_d, a.dil_h, a.dil_w = dilation
    a.d_out, a.h_out, a.w_out = y.shape[3], y.shape[4], y.shape[5]
    a.x, a.x_stride_n, a.x_stride_b = x.data_ptr(), x.stride(0), x.stride(1)
    a.packed_weight = packed_w.data_ptr()
    a.bias = ptr(bias)
    a.y, a.y_stride_n, a.y_stride_b = y.data_ptr(), y.stride(0), y.stride(1)
    _check(lib().wc_conv3d(ctypes.byref(a), stream_of(x)), "wc_conv3d")


def attention(*, q: Tensor, k: Tensor, v: Tensor, o: Tensor, nb: int, heads: int, sq: int, skv: int,
              head_dim: int, q_strides, k_strides, v_strides, o_strides, scale: float, causal: bool,
              mask: Optional[Tensor] = None) -> None:
    """q/k/v/o are base pointers (views) of [nb, S, heads*head_dim]-shaped data with the given
    (stride_nb, stride_s) element strides; ``mask`` is an additive fp32 [nb, heads, sq, skv]
    view with a unit key stride (other strides may be 0)."""
    mask_fields = (0, 0, 0, 0)
    if mask is not None:
        if mask.dtype != torch.float32 or tuple(mask.shape) != (nb, heads, sq, skv) or \
                (skv > 1 and mask.stride(3) != 1) or mask.device != q.device:
            raise ValueError("attention mask must be an fp32 [nb, heads, sq, skv] view with unit key stride "
                             "on the query's device")
        mask_fields = (mask.data_ptr(), mask.stride(0), mask.stride(1), mask.stride(2))
    _launch("wc_attention", _AttnArgs, _pack_attn(
        dtype_code(q.dtype, "attention"), 1 if causal else 0, nb, heads, sq, skv, head_dim, float(scale),
        q.data_ptr(), *q_strides, k.data_ptr(), *k_strides, v.data_ptr(), *v_strides, o.data_ptr(), *o_strides,
        *mask_fields), stream_of(q))


def self_attention(*, x: Tensor, q_weight: Tensor, kv_weight: Tensor, q_bias: Optional[Tensor],
                   kv_bias: Optional[Tensor], o: Tensor, heads: int, scale: float, causal: bool) -> None:
    """Fused self-attention core with the Q and K|V projections inside (wc_self_attention):
    x [N, B, S, D] (unit last stride), q_weight [N, D, D] and kv_weight [N, 2D, D] with
    contiguous rows, biases [N, D] / [N, 2D] or None, o [N, B, S, D] contiguous (the attention
    output before the output projection)."""
    n, b, s, d = x.shape
    _launch("wc_self_attention", _SelfAttnArgs, _pack_self_attn(
        dtype_code(x.dtype, "self_attention"), 1 if causal else 0, n, b, s, d, heads, float(scale),
        x.data_ptr(), x.stride(0), x.stride(1), x.stride(2), q_weight.data_ptr(), q_weight.stride(0),
        kv_weight.data_ptr(), kv_weight.stride(0),
        *((0, 0) if q_bias is None else (q_bias.data_ptr(), q_bias.stride(0))),
        *((0, 0) if kv_bias is None else (kv_bias.data_ptr(), kv_bias.stride(0))),
        o.data_ptr(), o.stride(1), o.stride(2)), stream_of(x))


def exported_symbols() -> List[str]:
    return list(SIGNATURES)


# Every entry point that launches kernels is a compile boundary: under torch.compile
# (compile_model=True) dynamo does not trace into the ctypes call and its stream handle,
# but ends the compiled region there and runs the call as is, so inductor never generates
# code for the hot path.
for _name in ("pack_rows", "swap01", "embedding_gather", "layernorm", "bn_eval", "group_norm", "grouped_gemm", "grouped_gemm_pair",
              "mlp2", "mlp2_entry", "mlp2_args", "mlp2_launch", "embedding_layernorm", "rnn_forward", "rnn_forward_noalloc", "rnn_phase", "conv_pack_weights", "conv2d", "conv3d",
              "attention", "self_attention", "rnn_sync_check", "rnn_status_word", "rnn_set_spin_limit"):
    globals()[_name] = torch.compiler.disable(globals()[_name])
del _name
