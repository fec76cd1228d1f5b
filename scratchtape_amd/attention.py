"""Batched causal attention forward and backward as the device tape runs it.

The call sequence of DeviceTape::batched_matmul / backward and the softmax
between them (gpu_step/tape.rs:196-212, 349-372, 475-491; rows.rs:101-123):
Q, K, V are head views of a fused [B*T, 3D] buffer, the scores S and
probabilities P are stacked [B*H*T, T], the context is written into the merged
[B*T, D] layout.  Every product goes through the GEMM of this package and the
softmax through its row kernels, or, where all six products run in f32 and that
is faster (_f32_step_pays), through three launches that keep a block of score
rows on chip and write the same buffers; `use_f16` picks the f16-in/f32-acc
route for the six products (the reference keeps them f32: matmul.rs:90-95).

`fused_forward` / `fused_backward` compute the same attention in two launches
that never write S or P (the reference's next step, docs/tiers_design.md:891-893):
the forward keeps each row's log-sum-exp, from which the backward recomputes P.
They run the f16-in/f32-acc route for head_dim 64 and sequence lengths that are
multiples of 32 up to 256.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib, rows
from .matmul import MatRef, _ptr, _stream, f16_route, matmul_with


@dataclass
class AttnBuffers:
    s: torch.Tensor     # [B*H*T, T] scores
    p: torch.Tensor     # [B*H*T, T] probabilities
    ctx: torch.Tensor   # [B*T, D] context
    dp: torch.Tensor    # [B*H*T, T]
    ds: torch.Tensor    # [B*H*T, T]
    dqkv: torch.Tensor  # [B*T, 3D] gradient of the fused QKV buffer

    @staticmethod
    def empty(b: int, h: int, t: int, hd: int, device) -> "AttnBuffers":
        d = h * hd
        z = lambda n: torch.zeros(n, dtype=torch.float32, device=device)
        return AttnBuffers(z(b * h * t * t), z(b * h * t * t), z(b * t * d), z(b * h * t * t), z(b * h * t * t),
                           z(b * t * 3 * d))


def _share(a: torch.Tensor, b: torch.Tensor) -> bool:
    """Whether the two contiguous float32 tensors have memory in common."""
    p, q = a.data_ptr(), b.data_ptr()
    return p < q + 4 * b.numel() and q < p + 4 * a.numel()


def _f32_step(qkv, dctx, buf: AttnBuffers, b: int, h: int, t: int, hd: int, use_f16: bool) -> bool:
    """Whether st_attention_fwd / _bwd take the step: its products all run in f32 (the six have one f16 rule: t % 64 ==
    0 and hd % 32 == 0), the sizes fit, the buffers hold the whole problems, and none shares memory in a way that only
    the separate launches' order allows: ctx written over the scores, or dS over P or dctx (st_attention_bwd reads both
    for dV after it has written dS; the separate launches make dV first)."""
    if (use_f16 and f16_route(t, hd, t)) or b < 1 or h < 1 or not _lib.lib().st_attention_fits(t, hd):
        return False
    n, tokens = b * h * t * t, b * t * h * hd
    sizes = [(qkv, 3 * tokens), (buf.s, n), (buf.p, n), (buf.ctx, tokens)] if dctx is None else \
        [(qkv, 3 * tokens), (dctx, tokens), (buf.p, n), (buf.dp, n), (buf.ds, n), (buf.dqkv, 3 * tokens)]
    if not all(x.numel() >= least for x, least in sizes):
        return False
    return not (_share(buf.s, buf.ctx) if dctx is None else _share(buf.ds, buf.p) or _share(buf.ds, dctx))


def _f32_step_pays(b: int, h: int, t: int, hd: int) -> bool:
    """Whether st_attention_fwd / _bwd are faster than the separate launches, forward and backward timed in HIP graphs
    for 1 to 384 problems x T = 8 to 512 x head widths of 16 to 128 (us, separate / one-launch, forward + backward):

    - Head widths above 80 (compiled as 128), and above 64 off 4, run separately: 96 x 128 x 96 77 / 94, 96 x 448 x 96
      410 / 1108, 96 x 256 x 128 198 / 204, 96 x 512 x 128 594 / 778; 96 x 100 x 128 is the exception (91 / 75).
    - A workgroup holds 32 x T scores and a 64-row tile in LDS; with one workgroup per CU (over 80 KB) nothing hides its
      chain of steps: 96 x 512 x 64 423 / 500, against 320 / 312 at T = 448.
    - Widths off 4 are loaded element by element, and widths off 16 pad the 80-wide form: separate from T = 257 on (48 x
      350 x 30 139 / 171, 64 x 288 x 72 178 / 194), as the 64-wide form with its T from 128 on.
    - Narrow heads pay for any T up to 128 (4 x 128 x 32 32 / 28) and from 16 problems on (8 x 256 x 32 38 / 41, 16 x 256
      x 32 47 / 42); widths up to 16 always (8 x 192 x 16 51 / 37), except where k_gemm_dma's 16 x 16 tiles take T x T x
      T products (4 x 256 x 16 34 / 45).
    - Otherwise a launch needs its workgroups: 128 of them (16 x 224 x 80 60 / 61, 24 x 224 x 80 67 / 62, 32 x 128 x 80 51 /
      44, 8 x 256 x 80 49 / 63), or 192 where the products tile and run on the LDS-DMA kernel (16 x 256 x 64 47 / 55, 24 x
      256 x 64 62 / 56, 96 x 128 x 64 67 / 51) or the width is padded.  Short sequences off 32 pay from one problem on
      (1 x 50 x 64 33 / 27)."""
    if hd > 80 or (hd > 64 and hd % 4):
        return False
    width = 32 if hd <= 32 and hd % 4 == 0 else 64 if hd <= 64 else 80
    if 128 * ((t + 15) // 16 * 16 + 4) + 256 * (width + 4) > 80 << 10:  # bytes of LDS per workgroup
        return False
    padded = hd > 64 and hd % 16 != 0
    if (hd % 4 or padded) and t > 256:
        return False
    if hd <= 32:
        return t <= 128 or b * h >= 16 or (hd <= 16 and hd % 4 == 0 and t % 256 != 0)
    if hd <= 64 and hd % 4 == 0 and t <= 112 and t % 32:
        return True
    tiled = t % 32 == 0 and hd % 32 == 0
    return b * h * ((t + 31) // 32) >= (192 if tiled or padded else 128)


def forward(qkv: torch.Tensor, buf: AttnBuffers, b: int, h: int, t: int, hd: int, use_f16: bool,
            stream=None) -> None:
    d = h * hd
    batch, scale = b * h, hd ** -0.5
    if _f32_step_pays(b, h, t, hd) and _f32_step(qkv, None, buf, b, h, t, hd, use_f16):
        _lib.call("st_attention_fwd", _ptr(qkv), _ptr(buf.s), _ptr(buf.p), _ptr(buf.ctx), b, h, t, hd, scale,
                  _stream(stream))
        return
    stacked = MatRef(buf.s, stride=t * t)
    matmul_with(MatRef.heads(qkv, 0, 3 * d, t, h, hd), MatRef.heads(qkv, d, 3 * d, t, h, hd).with_(trans=True),
                stacked, batch, t, hd, t, None, use_f16, stream=stream)
    rows.softmax(buf.s, batch * t, t, t, scale, True, False, out=buf.p, stream=stream)
    matmul_with(MatRef(buf.p, stride=t * t), MatRef.heads(qkv, 2 * d, 3 * d, t, h, hd),
                MatRef.heads(buf.ctx, 0, d, t, h, hd), batch, t, t, hd, None, use_f16, stream=stream)


def backward(qkv: torch.Tensor, dctx: torch.Tensor, buf: AttnBuffers, b: int, h: int, t: int, hd: int,
             use_f16: bool, stream=None) -> None:
    """dV = Pᵀ dO, dP = dO Vᵀ, dS = softmax backward, dQ = dS K, dK = dSᵀ Q, written into buf.dqkv."""
    d = h * hd
    batch, scale = b * h, hd ** -0.5
    if _f32_step_pays(b, h, t, hd) and _f32_step(qkv, dctx, buf, b, h, t, hd, use_f16):
        _lib.call("st_attention_bwd", _ptr(qkv), _ptr(dctx), _ptr(buf.p), _ptr(buf.dp), _ptr(buf.ds), _ptr(buf.dqkv), b,
                  h, t, hd, scale, _stream(stream))
        return
    p = MatRef(buf.p, stride=t * t)
    do = MatRef.heads(dctx, 0, d, t, h, hd)
    v = MatRef.heads(qkv, 2 * d, 3 * d, t, h, hd)
    # c = p v: dp = dc vᵀ, dv = pᵀ dc
    matmul_with(do, v.with_(trans=True), MatRef(buf.dp, stride=t * t), batch, t, hd, t, None, use_f16,
                stream=stream)
    matmul_with(p.with_(trans=True), do, MatRef.heads(buf.dqkv, 2 * d, 3 * d, t, h, hd), batch, t, t, hd, None,
                use_f16, stream=stream)
    rows.softmax_backward(buf.dp, buf.p, batch * t, t, scale, out=buf.ds, stream=stream)
    # s = q kᵀ: dq = ds k, dk = dsᵀ q
    ds = MatRef(buf.ds, stride=t * t)
    matmul_with(ds, MatRef.heads(qkv, d, 3 * d, t, h, hd), MatRef.heads(buf.dqkv, 0, 3 * d, t, h, hd), batch, t, t,
                hd, None, use_f16, stream=stream)
    matmul_with(ds.with_(trans=True), MatRef.heads(qkv, 0, 3 * d, t, h, hd),
                MatRef.heads(buf.dqkv, d, 3 * d, t, h, hd), batch, t, t, hd, None, use_f16, stream=stream)


def step(qkv: torch.Tensor, dctx: torch.Tensor, buf: AttnBuffers, b: int, h: int, t: int, hd: int,
         use_f16: bool, stream: Optional[object] = None) -> None:
    forward(qkv, buf, b, h, t, hd, use_f16, stream)
    backward(qkv, dctx, buf, b, h, t, hd, use_f16, stream)


@dataclass
class FusedBuffers:
    ctx: torch.Tensor   # [B*T, D] context
    lse: torch.Tensor   # [B*H*T] log-sum-exp of each score row (kept for the backward)
    dqkv: torch.Tensor  # [B*T, 3D] gradient of the fused QKV buffer

    @staticmethod
    def empty(b: int, h: int, t: int, hd: int, device) -> "FusedBuffers":
        d = h * hd
        z = lambda n: torch.zeros(n, dtype=torch.float32, device=device)
        return FusedBuffers(z(b * t * d), z(b * h * t), z(b * t * 3 * d))


def _f32(t: torch.Tensor, what: str) -> int:
    if not isinstance(t, torch.Tensor) or not t.is_cuda or t.dtype != torch.float32 or not t.is_contiguous():
        raise ValueError(f"{what} must be a contiguous float32 GPU tensor")
    return t.data_ptr()


def fused_forward(qkv: torch.Tensor, buf: FusedBuffers, b: int, h: int, t: int, hd: int, one: bool = False,
                  stream=None) -> None:
    """O = softmax(hd^-1/2 Q K^T, causal) V into buf.ctx, row log-sum-exp into buf.lse."""
    _lib.call("st_attention_fused_fwd", _f32(qkv, "qkv"), _f32(buf.ctx, "ctx"), _f32(buf.lse, "lse"), b, h, t, hd,
              hd ** -0.5, int(one), _stream(stream))


def fused_backward(qkv: torch.Tensor, dctx: torch.Tensor, buf: FusedBuffers, b: int, h: int, t: int, hd: int,
                   stream=None) -> None:
    """dQ, dK, dV of the fused forward for the upstream gradient dctx, into buf.dqkv."""
    _lib.call("st_attention_fused_bwd", _f32(qkv, "qkv"), _f32(buf.ctx, "ctx"), _f32(dctx, "dctx"),
              _f32(buf.lse, "lse"), _f32(buf.dqkv, "dqkv"), b, h, t, hd, hd ** -0.5, _stream(stream))


def fused_step(qkv: torch.Tensor, dctx: torch.Tensor, buf: FusedBuffers, b: int, h: int, t: int, hd: int,
               one: bool = False, stream: Optional[object] = None) -> None:
    fused_forward(qkv, buf, b, h, t, hd, one, stream)
    fused_backward(qkv, dctx, buf, b, h, t, hd, stream)
