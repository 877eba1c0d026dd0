"""Python mirror of ``ops::Mul`` over the C-ABI, for torch tensors that live on the GPU.

Validation follows the reference's ``ops::Mul`` (src/ops.cpp:540-556), extended as the HIP backend
is: a rank-3 A may multiply a rank-2 B, which is then broadcast over the batch (batch stride 0).
The result dtype follows the GPU backends' ``compute_type(a, b)`` (include/core/type_traits.h:270-287,
src/backend/cuda/mul.cu:63); ``out_dtype=FLOAT32`` for half inputs gives the CPU backend's widened
result type instead (src/backend/cpu/mul.cpp:110-112).
"""
from __future__ import annotations

import ctypes
import struct

import torch

from . import (BFLOAT16, FLOAT16, FLOAT32, FLOAT64, INT8, INT16, INT32, INT64, TvGemmArgs, check,
               lib)

_T2TV = {torch.int8: INT8, torch.int16: INT16, torch.int32: INT32, torch.int64: INT64,
         torch.bfloat16: BFLOAT16, torch.float16: FLOAT16, torch.float32: FLOAT32, torch.float64: FLOAT64}
_TV2T = {v: k for k, v in _T2TV.items()}


def torch_to_tv(dt: torch.dtype) -> int:
    try:
        return _T2TV[dt]
    except KeyError:
        raise RuntimeError(f"unsupported dtype {dt}") from None


def tv_to_torch(dt: int) -> torch.dtype:
    return _TV2T[dt]


def storage_to_torch(arr, dt: int, device="cuda") -> torch.Tensor:
    """Host storage array (uint16 bit patterns for bf16/fp16) -> torch tensor of tv dtype ``dt``."""
    import numpy as np
    arr = np.ascontiguousarray(arr)
    if dt in (BFLOAT16, FLOAT16):
        return torch.from_numpy(arr.view(np.int16)).view(tv_to_torch(dt)).to(device)
    return torch.from_numpy(arr).to(device)


def torch_to_storage(t: torch.Tensor):
    """torch tensor -> host numpy storage array (uint16 bit patterns for bf16/fp16)."""
    import numpy as np
    t = t.detach().cpu().contiguous()
    if t.dtype in (torch.bfloat16, torch.float16):
        return t.view(torch.int16).numpy().view(np.uint16)
    return t.numpy()


def compute_type(a: int, b: int) -> int:
    """Result dtype of a binary op (reference include/core/type_traits.h:270-287)."""
    if a == b:
        return a
    if a <= INT64 and b <= INT64:
        return max(a, b)
    if a > INT64 and b > INT64:
        return max(max(a, FLOAT32), max(b, FLOAT32))
    if a == INT64 or b == INT64:
        return FLOAT64
    return max(max(a, FLOAT32), max(b, FLOAT32))


def _check_shapes(a: torch.Tensor, b: torch.Tensor) -> None:
    """The reference's checks in its order (src/ops.cpp:542-556), with the broadcast extension."""
    if a.device != b.device:
        raise RuntimeError("Tensors a and b device mismatch!")
    if b.dim() != a.dim() and not (a.dim() == 3 and b.dim() == 2):
        raise RuntimeError(f"Tensors a and b must have the same rank,but got {a.dim()} and {b.dim()}")
    if a.dim() not in (2, 3):
        raise RuntimeError(f"Tensors a and b dims must be 2 or 3,but got {a.dim()}")
    if a.dim() == 3:
        if b.dim() == 3 and a.shape[0] != b.shape[0]:
            raise RuntimeError("Tensors a and b must have the same batch size")
        if a.shape[2] != b.shape[-2]:
            raise RuntimeError(f"Tensors common dim must match,but {a.shape[2]} and {b.shape[-2]}")
    elif a.shape[1] != b.shape[0]:
        # the reference's 2-d message names dimension 0 of both operands (src/ops.cpp:555)
        raise RuntimeError(f"Tensors common dim must match,but {a.shape[0]} and {b.shape[0]}")


def make_args(a: torch.Tensor, b: torch.Tensor, c: torch.Tensor) -> TvGemmArgs:
    """Pack the strided descriptor: element strides, data pointers that include the view offset."""
    args = TvGemmArgs()
    args.dtype_a, args.dtype_b, args.dtype_c = torch_to_tv(a.dtype), torch_to_tv(b.dtype), torch_to_tv(c.dtype)
    args.flags = 0
    if a.dim() == 3:
        args.batch, args.M, args.K = a.shape
        args.sa_b, args.sa_m, args.sa_k = a.stride()
    else:
        args.batch = 1
        args.M, args.K = a.shape
        args.sa_b = 0
        args.sa_m, args.sa_k = a.stride()
    if b.dim() == 3:
        args.N = b.shape[2]
        args.sb_b, args.sb_k, args.sb_n = b.stride()
    else:
        args.N = b.shape[1]
        args.sb_b = 0
        args.sb_k, args.sb_n = b.stride()
    if c.dim() == 3:
        args.sc_b, args.sc_m, args.sc_n = c.stride()
    else:
        args.sc_b = 0
        args.sc_m, args.sc_n = c.stride()
    args.A, args.B, args.C = a.data_ptr(), b.data_ptr(), c.data_ptr()
    return args


# tv_gemm_args as bytes, in native layout (the fields of make_args in order).
_pack_args = struct.Struct("4i 4q P3q P3q P3q").pack
assert struct.calcsize("4i 4q P3q P3q P3q") == ctypes.sizeof(TvGemmArgs)
_entries: dict[str, object] = {}  # entry point -> ctypes function that takes the packed bytes


def _entry(name: str):
    fn = _entries.get(name)
    if fn is None:
        fn = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p, ctypes.c_void_p)((name, lib()))
        _entries[name] = fn
    return fn


def _public_current_stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _stream_getter():
    """The handle of torch.cuda.current_stream(), without building the Stream object (2.8 us of a 10.5 us call) where
    this torch has the functions for it, which are not part of its public interface."""
    raw, device = getattr(torch._C, "_cuda_getCurrentRawStream", None), getattr(torch._C, "_cuda_getDevice", None)
    if raw is None or device is None:
        return _public_current_stream
    return lambda: raw(device())


_current_stream = _stream_getter()


def _stream(stream) -> int:
    if stream is None:
        return _current_stream()
    return stream if isinstance(stream, int) else stream.cuda_stream


def _run(name: str, a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None, out_dtype: int | None, stream) -> torch.Tensor:
    """Checks, output and descriptor of one call.  A small product is bound by this host code, so it reads
    each tensor attribute once and packs the descriptor in one step: 10.5 -> 7.0 us a call."""
    sa, sb = a.shape, b.shape
    if a.device != b.device or not (len(sa) == len(sb) or (len(sa) == 3 and len(sb) == 2)) or \
            not (len(sa) == 2 or (len(sa) == 3 and (len(sb) == 2 or sa[0] == sb[0]))) or sa[-1] != sb[-2]:
        _check_shapes(a, b)  # raises the message that applies
    da, db = torch_to_tv(a.dtype), torch_to_tv(b.dtype)
    dc = out_dtype if out_dtype is not None else compute_type(da, db)
    batched = len(sa) == 3
    m, k, n = sa[-2], sa[-1], sb[-1]
    shape = (sa[0], m, n) if batched else (m, n)
    if out is None:
        out = a.new_empty(shape, dtype=_TV2T[dc])
    elif tuple(out.shape) != shape or torch_to_tv(out.dtype) != dc:
        raise RuntimeError(f"out has shape {tuple(out.shape)}/{out.dtype}, expected {shape}/{tv_to_torch(dc)}")
    if batched:
        args = _pack_args(da, db, dc, 0, sa[0], m, n, k, a.data_ptr(), *a.stride(), b.data_ptr(),
                          *(b.stride() if len(sb) == 3 else (0, *b.stride())), out.data_ptr(), *out.stride())
    else:
        args = _pack_args(da, db, dc, 0, 1, m, n, k, a.data_ptr(), 0, *a.stride(), b.data_ptr(), 0, *b.stride(),
                          out.data_ptr(), 0, *out.stride())
    check(_entry(name)(args, _current_stream() if stream is None else _stream(stream)))
    return out


def gemm(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None, out_dtype: int | None = None,
         stream=None) -> torch.Tensor:
    """C = A @ B on the HIP kernels (asynchronous on ``stream``, default torch's current stream)."""
    return _run("tv_hip_gemm", a, b, out, out_dtype, stream)


def gemv(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None, out_dtype: int | None = None,
         stream=None) -> torch.Tensor:
    """Skinny-M (M <= 8) path; raises TensorviaHipError(TV_E_UNSUPPORTED) if it does not serve the call."""
    return _run("tv_hip_gemv", a, b, out, out_dtype, stream)


def matmul(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """``ops::Mul`` / ``ops::matmul``: synchronous, like the reference (src/backend/cuda/mul.cu:122)."""
    c = gemm(a, b)
    torch.cuda.current_stream().synchronize()
    return c
