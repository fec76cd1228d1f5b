"""`gpu_step::matmul` on MI355X: MatRef, Epilogue, matmul / matmul_f32 / matmul_with.

Mirrors gpu_step/matmul.rs:26-112: same type and argument meaning, buffers are
torch device tensors (float32, contiguous) standing in for cubecl Handles, and
offsets/strides are in elements of the whole buffer.  A failed call raises
ScratchtapeError with the message the reference would panic with.
"""
from __future__ import annotations

import ctypes
import struct
from dataclasses import dataclass
from typing import Optional, Tuple

import torch

from . import _lib


def _ptr(t: torch.Tensor) -> int:
    if not isinstance(t, torch.Tensor):
        raise TypeError("buffers are torch tensors")
    if t.dtype != torch.float32 or not t.is_contiguous():
        raise ValueError("buffers are contiguous float32 tensors")
    if not t.is_cuda:
        raise ValueError("buffers live on the GPU")
    return t.data_ptr()


# The handle of a device's current stream without a Stream object around it (a third of the call's host time).
_current_raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)

# st_matref, st_epilogue and st_gemm (scratchtape_hip.h) as the C compiler lays them out.
_REF = struct.Struct("=Qqqiiqqq")
_EPI = struct.Struct("=QqqQqQqiiiiqq")
_GEMM = struct.Struct("=" + 3 * "Qqqiiqqq" + "QqqQqQqiiiiqq" + "qqqqii")
_NO_EPI = 13 * (0,)


def _stream(stream) -> int:
    if stream is None:
        if _current_raw is not None:
            return _current_raw(torch.cuda.current_device())
        return torch.cuda.current_stream().cuda_stream
    return stream.cuda_stream if hasattr(stream, "cuda_stream") else int(stream)


@dataclass(frozen=True)
class MatRef:
    """A matrix inside a device buffer (matmul.rs:26-40).

    Matrix z starts at off + (z // group)*stride + (z % group)*inner; its stored
    rows are `ld` apart (0: packed); `trans`: a logical [r, c] stored as [c, r].
    """
    h: torch.Tensor
    off: int = 0
    stride: int = 0
    trans: bool = False
    ld: int = 0
    group: int = 1
    inner: int = 0

    @staticmethod
    def new(h: torch.Tensor) -> "MatRef":
        """The whole buffer from 0, one batch, not transposed (matmul.rs:44-46)."""
        return MatRef(h)

    @staticmethod
    def heads(h: torch.Tensor, col0: int, cols: int, t: int, heads: int, width: int) -> "MatRef":
        """Attention heads in place (matmul.rs:48-54): matrix z = b*heads + h is rows
        b*t .. b*t + t, columns col0 + h*width .. + width of a row-major [B*t, cols] buffer."""
        return MatRef(h, off=col0, stride=t * cols, ld=cols, group=heads, inner=width)

    def with_(self, **kw) -> "MatRef":
        for name in kw:
            if name not in _MATREF_FIELDS:
                raise TypeError(f"MatRef has no field {name!r}")
        new = object.__new__(type(self))  # dataclasses.replace, without its walk over the fields
        new.__dict__.update(self.__dict__)
        new.__dict__.update(kw)
        return new

    def _fields(self) -> tuple:
        """st_matref's fields in order."""
        return (_ptr(self.h), self.off, self.stride, 1 if self.trans else 0, 0, self.ld, self.group, self.inner)


_MATREF_FIELDS = frozenset(MatRef.__dataclass_fields__)


@dataclass
class Epilogue:
    """matmul.rs:62-79.  bias/mask/residual are (buffer, offset) pairs; col_sum is
    (offset, stride) into out's buffer (always +=)."""
    bias: Optional[Tuple[torch.Tensor, int]] = None
    bias_stride: int = 0
    relu: bool = False
    mask: Optional[Tuple[torch.Tensor, int]] = None
    residual: Optional[Tuple[torch.Tensor, int]] = None
    accumulate: bool = False
    col_sum: Optional[Tuple[int, int]] = None

    def _fields(self) -> tuple:
        """st_epilogue's fields in order."""
        bias, mask, residual, col_sum = self.bias, self.mask, self.residual, self.col_sum
        return (_ptr(bias[0]) if bias is not None else 0, bias[1] if bias is not None else 0, self.bias_stride,
                _ptr(mask[0]) if mask is not None else 0, mask[1] if mask is not None else 0,
                _ptr(residual[0]) if residual is not None else 0, residual[1] if residual is not None else 0,
                int(self.relu), int(self.accumulate), 0 if col_sum is None else 1, 0,
                *(col_sum if col_sum is not None else (0, 0)))


def _pack(layout: struct.Struct, *fields) -> bytes:
    try:
        return layout.pack(*fields)
    except struct.error as e:
        raise TypeError(str(e)) from None


def _call(name, a: MatRef, b: MatRef, out: MatRef, batch, m, k, n, epi, *extra, stream=None):
    _lib.check(_lib.packed(name)(_pack(_REF, *a._fields()), _pack(_REF, *b._fields()), _pack(_REF, *out._fields()),
                                 batch, m, k, n, _pack(_EPI, *(epi._fields() if epi else _NO_EPI)), *extra,
                                 _stream(stream)))


def matmul(a: MatRef, b: MatRef, out: MatRef, batch: int, m: int, k: int, n: int,
           epi: Optional[Epilogue] = None, stream=None) -> None:
    """out[z] (+)= epi(a[z] @ b[z]) (matmul.rs:86); f16-in/f32-acc when enabled and the shape tiles."""
    _call("st_matmul", a, b, out, batch, m, k, n, epi, stream=stream)


def matmul_f32(a: MatRef, b: MatRef, out: MatRef, batch: int, m: int, k: int, n: int,
               epi: Optional[Epilogue] = None, stream=None) -> None:
    """`matmul` always in f32 (matmul.rs:93), the reference's attention route."""
    _call("st_matmul_f32", a, b, out, batch, m, k, n, epi, stream=stream)


def matmul_with(a: MatRef, b: MatRef, out: MatRef, batch: int, m: int, k: int, n: int,
                epi: Optional[Epilogue], use_f16: bool, stream=None) -> None:
    """`matmul` with the f16 route chosen by the caller (matmul.rs:106)."""
    _call("st_matmul_with", a, b, out, batch, m, k, n, epi, int(bool(use_f16)), stream=stream)


def matmul_plan(a: MatRef, b: MatRef, out: MatRef, batch: int, m: int, k: int, n: int, epi: Optional[Epilogue],
                use_f16: bool) -> Tuple[int, int, int, int, int]:
    """What matmul_with launches for these arguments (st_matmul_plan; no reference counterpart): the kernel (0 any
    shape, 1 LDS-DMA tiles, 2 grouped 256 x 128 tiles), kernel 0's tile rows and columns and slices of k, and the bytes
    of split-k scratch."""
    plan = (ctypes.c_int64 * 5)()
    _lib.check(_lib.packed("st_matmul_plan")(_pack(_REF, *a._fields()), _pack(_REF, *b._fields()),
                                             _pack(_REF, *out._fields()), batch, m, k, n,
                                             _pack(_EPI, *(epi._fields() if epi else _NO_EPI)), int(bool(use_f16)),
                                             ctypes.addressof(plan)))
    return tuple(plan)


def matmul_grouped(calls, stream=None, noalloc: bool = False) -> None:
    """Several independent `matmul_with` calls in one submission (st_matmul_grouped).

    `calls` holds (a, b, out, batch, m, k, n, epi, use_f16) tuples, the arguments
    of matmul_with, e.g. a Linear backward's dW and dx (gpu_step/tape.rs:324-347).
    No call may read or write memory that another one writes.  noalloc: the
    same through st_matmul_grouped_noalloc (split-k partials in the library's
    fixed per-device scratch; no device allocation)."""
    gemms = [_pack(_GEMM, *a._fields(), *b._fields(), *out._fields(), *(epi._fields() if epi else _NO_EPI), batch, m, k,
                   n, 1 if use_f16 else 0, 0) for a, b, out, batch, m, k, n, epi, use_f16 in calls]
    # (One empty struct for an empty group: the library takes no NULL array.)
    _lib.check(_lib.packed("st_matmul_grouped_noalloc" if noalloc else "st_matmul_grouped")(
        b"".join(gemms) or bytes(_GEMM.size), len(gemms), _stream(stream)))


def f16_enabled() -> bool:
    """matmul.rs:97-102: on unless TRAIN_F16=0."""
    return bool(_lib.lib().st_f16_enabled())


def f16_route(m: int, k: int, n: int, col_sum: bool = False, b_trans: bool = False) -> bool:
    """Whether a shape takes the f16 route (matmul.rs:108-112, 524-534)."""
    return not (col_sum and b_trans) and k > 0 and k % 32 == 0 and m % 64 == 0 and n % 32 == 0


def sync(stream=None) -> None:
    """st_sync: waits for `stream`, then raises ScratchtapeError if a bounded slot wait of the grouped f16 kernel gave
    up since the last check: the outputs of matmul_grouped's f16 GEMMs, and of single f16 calls that matmul_plan puts on
    that kernel (2), are then not valid."""
    _lib.call("st_sync", _stream(stream))


def set_wait_limit(polls: int) -> None:
    """st_set_wait_limit: polls before a slot wait of the grouped f16 kernel gives up (negative: the default)."""
    _lib.call("st_set_wait_limit", int(polls))
