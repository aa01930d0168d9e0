"""Tensor-level wrappers over the C ABI: shape/dtype/device checks in Python, raw pointers and
the current torch stream handed to libflashsvd_hip.  PyTorch only provides device memory and
streams here; every arithmetic step runs in the HIP library."""
from __future__ import annotations

import math
import os
from typing import Optional

import torch

from . import _lib
from .torch_ops import ops as _OPS

_BF16 = torch.bfloat16


def _stream() -> int:
    """The handle of the current stream of the current device, without the Stream object around it (0.3 us instead of 4)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def _need(t: torch.Tensor, name: str, *, dtype=_BF16) -> None:
    if not t.is_cuda:
        raise ValueError(f"{name} must be a GPU tensor, got device {t.device}")
    if t.dtype != dtype:
        raise ValueError(f"{name} must be {dtype}, got {t.dtype}")


_ELEM_CODES = {torch.bfloat16: 0, torch.float16: 1}     # FSVD_BF16, FSVD_FP16


def _elem(t: torch.Tensor, name: str):
    """Element type of a call on the fused product path, named by its first operand: (torch dtype, C-ABI code).  Every
    other 16-bit tensor of the call must be of the same type."""
    if not t.is_cuda:
        raise ValueError(f"{name} must be a GPU tensor, got device {t.device}")
    code = _ELEM_CODES.get(t.dtype)
    if code is None:
        raise ValueError(f"{name} must be torch.bfloat16 or torch.float16, got {t.dtype}")
    return t.dtype, code


def _rows(t: torch.Tensor, name: str) -> torch.Tensor:
    """View as [rows, last] with unit stride on the last axis (copies only if it must)."""
    if t.stride(-1) != 1:
        t = t.contiguous()
    if t.dim() == 1:
        return t.unsqueeze(0)
    if t.dim() == 2:
        return t
    try:
        return t.view(-1, t.shape[-1])
    except RuntimeError:
        return t.reshape(-1, t.shape[-1])


def _row_operand(t: torch.Tensor, name: str):
    """``_rows(t)`` as (tensor to keep alive, address, row stride, rows, row length); no view is made of contiguous tensors."""
    n = t.shape[-1]
    if n and t.dim() > 1 and t.is_contiguous():
        return t, t.data_ptr(), t.stride(0) if t.dim() == 2 else n, t.numel() // n, n
    t = _rows(t, name)
    return t, t.data_ptr(), t.stride(0), t.shape[0], n


_SPLIT_WS: dict = {}                      # device index -> scratch tensor registered with the library (kept alive here)
_SPLIT_WS_BYTES = (64 << 20) + (64 << 10)
_SPLIT_WS_OLD: dict = {}                  # device index -> replaced buffers: graphs captured earlier may hold their addresses
_SPLIT_WS_MAX = 1 << 30


def _splitk_enabled() -> bool:
    """``FLASHSVD_AMD_SPLITK=0``: no call gets scratch to split K in, neither the device's nor one of its own."""
    return os.environ.get("FLASHSVD_AMD_SPLITK", "1") != "0"


def ensure_split_workspace(device: torch.device, min_bytes: int = 0) -> bool:
    """Register, once per device, the scratch the library's K-split projections (three rows and more, K a multiple of 64 and
    rows on the 16-byte grid; others run without it) work in.  The library allocates nothing itself; this hands it 64 MiB of torch memory, or ``min_bytes`` rounded up to a power of two (up to
    1 GiB) when a caller needs more: a larger buffer then replaces the registered one (a doubling each time at least, so
    a growing demand costs a logarithmic number of replacements), and the old one is kept alive until
    ``release_split_workspace`` because graphs captured earlier hold its address.  ``FLASHSVD_AMD_SPLITK=0`` keeps the
    library without scratch (and the calls of 128 rows and more without scratch of their own); so does a first call made under stream capture (an allocation there would belong to the
    graph's pool), and a registered buffer is never replaced under capture.  Launches that use the scratch must be
    ordered on one stream per device.  Returns whether a buffer of at least ``min_bytes`` is registered."""
    idx = device.index if device.index is not None else torch.cuda.current_device()
    need = max(int(min_bytes), _SPLIT_WS_BYTES)
    have = _SPLIT_WS.get(idx)
    if have is not None and have.numel() >= need:
        return True
    if not _splitk_enabled() or torch.cuda.is_current_stream_capturing() or need > _SPLIT_WS_MAX:
        return have is not None and min_bytes <= 0
    if need > _SPLIT_WS_BYTES:
        need = min(_SPLIT_WS_MAX, 1 << (need - 1).bit_length())
    with torch.cuda.device(idx):
        ws = torch.empty(need, dtype=torch.uint8, device=f"cuda:{idx}")
        rc = _lib.load().fsvd_set_workspace(ws.data_ptr(), ws.numel(), _stream())
        _lib.check("fsvd_set_workspace", rc)
        torch.cuda.current_stream().synchronize()      # cleared before any other stream can use it
    if have is not None:
        _SPLIT_WS_OLD.setdefault(idx, []).append(have)
    _SPLIT_WS[idx] = ws
    return True


def release_split_workspace(device: Optional[torch.device] = None) -> None:
    """Unregister (and free) the scratch of ``device`` and the buffers it replaced; the library runs without scratch
    until it is registered again.  Graphs captured while a buffer was registered must not be replayed afterwards."""
    idx = torch.cuda.current_device() if device is None or device.index is None else device.index
    _SPLIT_WS_OLD.pop(idx, None)
    if _SPLIT_WS.pop(idx, None) is not None:
        with torch.cuda.device(idx):
            torch.cuda.synchronize()
            _lib.check("fsvd_set_workspace", _lib.load().fsvd_set_workspace(None, 0, None))


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None, *,
           norm_weight: Optional[torch.Tensor] = None, eps: float = 1e-6,
           residual: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None, cfg: int = 0) -> torch.Tensor:
    """out = (residual +) linear(rmsnorm?(x), weight, bias); weight is nn.Linear layout [N, K].
    Dispatches to the custom operator flashsvd_hip::linear (``.out`` when ``out`` is given).  From three rows on, with K a
    multiple of 64 and rows on the 16-byte grid, the call may split K through the device's one scratch buffer
    (``ensure_split_workspace``): such calls are to be ordered on one stream."""
    if out is None:
        return _OPS.linear.default(x, weight, bias, norm_weight, float(eps), residual, int(cfg))
    return _OPS.linear.out(x, weight, bias, norm_weight, float(eps), residual, int(cfg), out=out)


def _linear_impl(x, weight, bias, norm_weight, eps, residual, out, cfg):
    dt, code = _elem(x, "x")
    _need(weight, "weight", dtype=dt)
    if weight.dim() != 2 or weight.stride(1) != 1:
        raise ValueError(f"weight must be [N, K] with unit inner stride, got {tuple(weight.shape)} strides {weight.stride()}")
    N, K = weight.shape
    if x.shape[-1] != K:
        raise ValueError(f"x last dim {x.shape[-1]} != weight in_features {K}")
    x2, xp, ldx, B, _ = _row_operand(x, "x")
    if out is None:
        out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=dt)
    _need(out, "out", dtype=dt)
    _, op, ldo, rows, cols = _row_operand(out, "out")
    if rows != B or cols != N or op != out.data_ptr():
        raise ValueError("out must be a dense [..., N] tensor matching x")
    r2, rp, ldr = None, None, 0
    if residual is not None:
        _need(residual, "residual", dtype=dt)
        r2, rp, ldr, rows, cols = _row_operand(residual, "residual")
        if rows != B or cols != N:
            raise ValueError(f"residual shape {tuple(residual.shape)} does not match output [{B}, {N}]")
    for t, nm, n in ((bias, "bias", N), (norm_weight, "norm_weight", K)):
        if t is not None:
            _need(t, nm, dtype=dt)
            if t.shape != (n,) or not t.is_contiguous():
                raise ValueError(f"{nm} must be a contiguous [{n}] tensor")
    lib = _lib.load()
    if B >= 3:
        ensure_split_workspace(x.device)
    if norm_weight is not None and B >= 3 and cfg == 0:
        # three rows and more run on the matrix cores, which take the activations as they are: normalise once
        # up front (same rounding points as the fused prologue)
        x2, xp, ldx, _, _ = _row_operand(_rmsnorm_impl(x2, norm_weight, eps, None), "x")
        norm_weight = None
    wp, ldw = weight.data_ptr(), weight.stride(0)
    scratch, nbytes = None, 0
    if B >= 128 and K >= 4096 and cfg == 0 and _splitk_enabled():
        nbytes = lib.fsvd_linear_scratch_bytes(xp, ldx, wp, ldw, rp, ldr, op, ldo, B, N, K)
        if nbytes:
            scratch = torch.empty(nbytes, dtype=torch.uint8, device=x.device)      # of this call and stream
    rc = lib.fsvd_linear_scratch(xp, ldx, wp, ldw, _ptr(bias), _ptr(norm_weight), float(eps), rp, ldr, op, ldo, B, N, K, int(cfg), code,
                                 _ptr(scratch), nbytes, _stream())
    _lib.check("fsvd_linear", rc)
    return out


def linear_rankkv_append(x: torch.Tensor, weight: torch.Tensor, pk_cache: torch.Tensor, pv_cache: torch.Tensor, positions: torch.Tensor, *,
                         ranks, norm_weight: Optional[torch.Tensor] = None, eps: float = 1e-6) -> torch.Tensor:
    """The packed rank projection of one or two decoded tokens, ``p = norm(x) @ weight.T`` with ``weight = [q_v; k_v; v_v]``
    and ``ranks = (rq, rk, rv)``, which also stores the Pk | Pv parts of every row at ``pk_cache[b, positions[b]]`` /
    ``pv_cache[b, positions[b]]`` (caches [>=B, S, R]): ``linear`` followed by ``rankkv_append`` in one launch, same bits.
    Custom operator flashsvd_hip::linear_rankkv_append (the caches are mutated arguments)."""
    rq, rk, rv = (int(r) for r in ranks)
    return _OPS.linear_rankkv_append.default(x, weight, pk_cache, pv_cache, positions, rq, rk, rv, norm_weight, float(eps))


def _linear_rankkv_append_impl(x, weight, pk_cache, pv_cache, positions, rq, rk, rv, norm_weight, eps):
    dt, code = _elem(x, "x")
    _need(weight, "weight", dtype=dt); _need(pk_cache, "pk_cache", dtype=dt); _need(pv_cache, "pv_cache", dtype=dt)
    _need(positions, "positions", dtype=torch.int32)
    if weight.dim() != 2 or weight.stride(1) != 1 or weight.shape[0] != rq + rk + rv:
        raise ValueError(f"weight must be [rq + rk + rv, K] = [{rq + rk + rv}, K] with unit inner stride, got {tuple(weight.shape)}")
    K = weight.shape[1]
    x2 = _rows(x, "x")
    B = x2.shape[0]
    if x2.shape[1] != K or B > 2:
        raise ValueError(f"x must be one or two rows of {K} values, got {tuple(x.shape)}")
    for c, r, nm in ((pk_cache, rk, "pk_cache"), (pv_cache, rv, "pv_cache")):
        if c.dim() != 3 or c.shape[0] < B or c.shape[2] != r or c.stride(2) != 1 or c.shape[1] != pk_cache.shape[1]:
            raise ValueError(f"{nm} must be [>={B}, S, {r}] with unit inner stride, got {tuple(c.shape)}")
    if positions.numel() != B or not positions.is_contiguous():
        raise ValueError(f"positions must be a contiguous int32 [{B}] tensor")
    if norm_weight is not None:
        _need(norm_weight, "norm_weight", dtype=dt)
        if norm_weight.shape != (K,) or not norm_weight.is_contiguous():
            raise ValueError(f"norm_weight must be a contiguous [{K}] tensor")
    out = torch.empty(*x.shape[:-1], rq + rk + rv, device=x.device, dtype=dt)
    o2 = _rows(out, "out")
    rc = _lib.load().fsvd_linear_rankkv_append(x2.data_ptr(), x2.stride(0), weight.data_ptr(), weight.stride(0), _ptr(norm_weight), float(eps),
                                               o2.data_ptr(), o2.stride(0), B, rq, rk, rv, K, pk_cache.data_ptr(), pk_cache.stride(0),
                                               pk_cache.stride(1), pv_cache.data_ptr(), pv_cache.stride(0), pv_cache.stride(1),
                                               positions.data_ptr(), int(pk_cache.shape[1]), code, _stream())
    _lib.check("fsvd_linear_rankkv_append", rc)
    return out


def swiglu_linear(p: torch.Tensor, gate_u: torch.Tensor, up_u: torch.Tensor, *, up_off: int, mode: int = 0,
                  out: Optional[torch.Tensor] = None, cfg: int = 0) -> torch.Tensor:
    """h = silu(p[..., :R] @ gate_u.T) * (p[..., up_off:up_off+R] @ up_u.T); gate_u/up_u are [D, R].
    Custom operator flashsvd_hip::swiglu_linear.  3 to 127 rows with R a multiple of 64 on the 16-byte grid may split R
    through the device's one scratch buffer, as :func:`linear` does."""
    if out is None:
        return _OPS.swiglu_linear.default(p, gate_u, up_u, int(up_off), int(mode), int(cfg))
    return _OPS.swiglu_linear.out(p, gate_u, up_u, int(up_off), int(mode), int(cfg), out=out)


def _swiglu_linear_impl(p, gate_u, up_u, up_off, mode, out, cfg):
    dt, code = _elem(p, "p")
    _need(gate_u, "gate_u", dtype=dt); _need(up_u, "up_u", dtype=dt)
    if gate_u.dim() != 2 or gate_u.shape != up_u.shape or gate_u.stride() != up_u.stride() or gate_u.stride(1) != 1:
        raise ValueError(f"gate_u/up_u must be matching [D, R] weights, got {tuple(gate_u.shape)} / {tuple(up_u.shape)}")
    D, R = gate_u.shape
    p2, pp, ldp, B, width = _row_operand(p, "p")
    if width < up_off + R:
        raise ValueError(f"p last dim {width} too small for up_off {up_off} + R {R}")
    if out is None:
        out = torch.empty(*p.shape[:-1], D, device=p.device, dtype=dt)
    _need(out, "out", dtype=dt)
    o2, op, ldo, _, _ = _row_operand(out, "out")
    lib = _lib.load()
    if 3 <= B < 128:
        ensure_split_workspace(p.device)
    rc = lib.fsvd_swiglu_linear(pp, ldp, int(up_off), gate_u.data_ptr(), up_u.data_ptr(),
                                gate_u.stride(0), op, ldo, B, D, R, int(mode), int(cfg), code, _stream())
    _lib.check("fsvd_swiglu_linear", rc)
    return out


def _q4_check(qweight, scales, zeros, N: int, K: int, group_size: int, name: str) -> int:
    """Validate one int4 matrix; returns the group width the kernel is given (0 = one group per row)."""
    if qweight.dtype != torch.uint8 or scales.dtype != torch.float16 or zeros.dtype != torch.int16:
        raise TypeError(f"{name}: expected uint8 weights, float16 scales and int16 zeros, got {qweight.dtype}, {scales.dtype}, "
                        f"{zeros.dtype}")
    if not (qweight.is_cuda and scales.is_cuda and zeros.is_cuda):
        raise ValueError(f"{name}: quantised buffers must be on the GPU")
    if qweight.dim() != 2 or qweight.shape != (N, (K + 1) // 2) or qweight.stride(1) != 1:
        raise ValueError(f"{name}: packed weight must be [{N}, {(K + 1) // 2}] bytes, got {tuple(qweight.shape)}")
    group = 0 if group_size <= 0 or group_size >= K else int(group_size)
    G = 1 if group == 0 else -(-K // group)
    if scales.shape != (N, G) or zeros.shape != (N, G) or scales.stride() != zeros.stride() or scales.stride(1) != 1:
        raise ValueError(f"{name}: scales / zeros must be matching [{N}, {G}] tensors, got {tuple(scales.shape)} / {tuple(zeros.shape)}")
    return group


def linear_q4(x: torch.Tensor, qweight: torch.Tensor, scales: torch.Tensor, zeros: torch.Tensor, *, group_size: int,
              bias: Optional[torch.Tensor] = None, norm_weight: Optional[torch.Tensor] = None, eps: float = 1e-6,
              residual: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = (residual +) linear(rmsnorm?(x), s * (q - z), bias) on group-wise int4 weights [N, K/2] bytes."""
    dt, code = _elem(x, "x")
    N, K = qweight.shape[0], x.shape[-1]
    group = _q4_check(qweight, scales, zeros, N, K, group_size, "linear_q4")
    x2 = _rows(x, "x")
    B = x2.shape[0]
    if out is None:
        out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=dt)
    _need(out, "out", dtype=dt)
    o2 = out if out.dim() == 2 else _rows(out, "out")
    if o2.shape != (B, N) or o2.stride(1) != 1:
        raise ValueError("out must be a [rows, N] tensor with unit inner stride matching x")
    r2 = None
    if residual is not None:
        _need(residual, "residual", dtype=dt)
        r2 = _rows(residual, "residual")
        if r2.shape != (B, N):
            raise ValueError(f"residual shape {tuple(residual.shape)} does not match output [{B}, {N}]")
    for t, nm, n in ((bias, "bias", N), (norm_weight, "norm_weight", K)):
        if t is not None:
            _need(t, nm, dtype=dt)
            if t.shape != (n,) or not t.is_contiguous():
                raise ValueError(f"{nm} must be a contiguous [{n}] tensor")
    lib = _lib.load()
    rc = lib.fsvd_linear_q4(x2.data_ptr(), x2.stride(0), qweight.data_ptr(), qweight.stride(0), scales.data_ptr(), zeros.data_ptr(),
                            scales.stride(0), group, _ptr(bias), _ptr(norm_weight), float(eps), _ptr(r2),
                            0 if r2 is None else r2.stride(0), o2.data_ptr(), o2.stride(0), B, N, K, code, _stream())
    _lib.check("fsvd_linear_q4", rc)
    return out


def swiglu_linear_q4(p: torch.Tensor, gate: tuple, up: tuple, *, up_off: int, group_size: int, mode: int = 0,
                     out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """h = silu(p[..., :R] @ Wg.T) * (p[..., up_off:up_off+R] @ Wu.T); gate / up are (qweight, scales, zeros) of [D, R]."""
    dt, code = _elem(p, "p")
    (gq, gs, gz), (uq, us, uz) = gate, up
    D = gq.shape[0]
    R = 2 * gq.shape[1]
    p2 = _rows(p, "p")
    if p2.shape[1] < up_off + R:
        raise ValueError(f"p last dim {p2.shape[1]} too small for up_off {up_off} + R {R}")
    group = _q4_check(gq, gs, gz, D, R, group_size, "swiglu_linear_q4 gate")
    _q4_check(uq, us, uz, D, R, group_size, "swiglu_linear_q4 up")
    if gq.stride() != uq.stride() or gs.stride() != us.stride():
        raise ValueError("gate and up must share one layout")
    B = p2.shape[0]
    if out is None:
        out = torch.empty(*p.shape[:-1], D, device=p.device, dtype=dt)
    _need(out, "out", dtype=dt)
    o2 = _rows(out, "out")
    lib = _lib.load()
    rc = lib.fsvd_swiglu_linear_q4(p2.data_ptr(), p2.stride(0), int(up_off), gq.data_ptr(), gs.data_ptr(), gz.data_ptr(),
                                   uq.data_ptr(), us.data_ptr(), uz.data_ptr(), gq.stride(0), gs.stride(0), group,
                                   o2.data_ptr(), o2.stride(0), B, D, R, int(mode), code, _stream())
    _lib.check("fsvd_swiglu_linear_q4", rc)
    return out


def dequant_q4(qweight: torch.Tensor, scales: torch.Tensor, zeros: torch.Tensor, *, in_features: int, group_size: int,
               out: Optional[torch.Tensor] = None, dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """[N, K] = s * (q - z), rounded once to ``dtype`` (bf16 or fp16; the type of ``out`` when that is given, else bf16)."""
    N, K = qweight.shape[0], int(in_features)
    group = _q4_check(qweight, scales, zeros, N, K, group_size, "dequant_q4")
    if out is None:
        out = torch.empty(N, K, device=qweight.device, dtype=dtype or _BF16)
    dt, code = _elem(out, "out")
    if out.shape != (N, K) or (dtype is not None and dt != dtype) or out.stride(1) != 1:
        raise ValueError(f"out must be a {dtype or 'bf16 / fp16'} [{N}, {K}] tensor with unit inner stride")
    lib = _lib.load()
    rc = lib.fsvd_dequant_q4(qweight.data_ptr(), qweight.stride(0), scales.data_ptr(), zeros.data_ptr(), scales.stride(0), group,
                             out.data_ptr(), out.stride(0), N, K, code, _stream())
    _lib.check("fsvd_dequant_q4", rc)
    return out


def qkv_rope_append(p: torch.Tensor, q_u: torch.Tensor, k_u: torch.Tensor, v_u: torch.Tensor,
                    cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], positions: torch.Tensor,
                    k_cache: torch.Tensor, v_cache: torch.Tensor, *, num_heads: int, num_kv_heads: int, head_dim: int,
                    q_out: Optional[torch.Tensor] = None, cfg: int = 0) -> torch.Tensor:
    """q (rotated) -> q_out [B,H,Dh]; rotated k and v written into the caches [B,S,Hk,Dh] at positions[b].
    Custom operator flashsvd_hip::qkv_rope_append (the caches are mutated arguments)."""
    a = (p, q_u, k_u, v_u, cos, sin, positions, k_cache, v_cache, int(num_heads), int(num_kv_heads), int(head_dim), int(cfg))
    return _OPS.qkv_rope_append.default(*a) if q_out is None else _OPS.qkv_rope_append.out(*a, q_out=q_out)


def _qkv_rope_append_impl(p, q_u, k_u, v_u, cos, sin, positions, k_cache, v_cache, num_heads, num_kv_heads, head_dim, q_out, cfg):
    dt, code = _elem(p, "p")
    for t, nm in ((q_u, "q_u"), (k_u, "k_u"), (v_u, "v_u"), (k_cache, "k_cache"), (v_cache, "v_cache")):
        _need(t, nm, dtype=dt)
    _need(positions, "positions", dtype=torch.int32)
    H, Hk, Dh = int(num_heads), int(num_kv_heads), int(head_dim)
    Rq, Rk, Rv = q_u.shape[1], k_u.shape[1], v_u.shape[1]
    if q_u.shape[0] != H * Dh or k_u.shape[0] != Hk * Dh or v_u.shape[0] != Hk * Dh:
        raise ValueError(f"u_proj rows do not match heads: {tuple(q_u.shape)}/{tuple(k_u.shape)}/{tuple(v_u.shape)} "
                         f"for H={H} Hk={Hk} Dh={Dh}")
    p2 = _rows(p, "p")
    B = p2.shape[0]
    if p2.shape[1] != Rq + Rk + Rv:
        raise ValueError(f"p last dim {p2.shape[1]} != Rq+Rk+Rv = {Rq + Rk + Rv}")
    if k_cache.dim() != 4 or k_cache.shape != v_cache.shape or k_cache.stride() != v_cache.stride() \
            or k_cache.shape[2:] != (Hk, Dh) or k_cache.shape[0] < B or k_cache.stride(3) != 1:
        raise ValueError(f"caches must be matching [B>={B}, S, {Hk}, {Dh}] tensors, got {tuple(k_cache.shape)}")
    if positions.numel() != B or not positions.is_contiguous():
        raise ValueError(f"positions must be a contiguous int32 [{B}] tensor")
    rope_len = 0
    if cos is not None:
        _need(cos, "cos", dtype=dt); _need(sin, "sin", dtype=dt)
        if cos.shape != sin.shape or cos.dim() != 2 or cos.shape[1] != Dh // 2 or not cos.is_contiguous() or not sin.is_contiguous():
            raise ValueError(f"cos/sin must be contiguous [len, {Dh // 2}] tables")
        rope_len = cos.shape[0]
    if q_out is None:
        q_out = torch.empty(B, H, Dh, device=p.device, dtype=dt)
    elif q_out.shape != (B, H, Dh) or not q_out.is_contiguous() or q_out.dtype != dt:
        raise ValueError("q_out must be contiguous [B,H,Dh]")
    lib = _lib.load()
    rc = lib.fsvd_qkv_rope_append(p2.data_ptr(), p2.stride(0), q_u.data_ptr(), q_u.stride(0), k_u.data_ptr(), k_u.stride(0),
                                  v_u.data_ptr(), v_u.stride(0), _ptr(cos), _ptr(sin), rope_len, positions.data_ptr(),
                                  q_out.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                                  k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
                                  B, H, Hk, Dh, Rq, Rk, Rv, k_cache.shape[1], int(cfg), code, _stream())
    _lib.check("fsvd_qkv_rope_append", rc)
    return q_out


def pick_nsplit(max_len: int, batch: int, heads: int, head_dim: int = 128, own_row: bool = False) -> int:
    """Key-axis split: about 128 keys per workgroup (one pass of loads in flight), bounded so that
    batch*heads*nsplit stays within ~2048 workgroups.  Up to 256 rows in one range, which saves the merge, with head_dim 64 (8 heads,
    137 keys 5.6 -> 4.4 us) and for 256 pairs and more (16 x 32 heads over 8 of 128 9.4 -> 8.0; fewer lose: 32 heads, 250 keys 6.4 -> 6.7).
    ``own_row``: every head has a kv head of its own and the call appends its row.  The rows are then read behind the write's way to
    memory, and a second round of workgroups that is less than five eighths full waits for that once more: two ranges there (17 / 20 / 24 x 16 heads of up to 248 keys 10.1,
    10.9, 11.4 in two, 11.2, 11.7, 12.1 in one; 26 x 16 12.0 and 10.9).  It goes by the room in the cache: how many keys there are is not known here."""
    pairs = batch * heads
    if max_len <= 256 and (head_dim < 128 or (pairs >= 256 and not (own_row and 256 < pairs < 416))):
        return 1
    n = max(1, math.ceil(max_len / 128))
    cap = max(1, 2048 // max(1, pairs))
    return int(max(1, min(n, cap)))


def attn_workspace(batch: int, heads: int, head_dim: int, nsplit: int, device) -> torch.Tensor:
    lib = _lib.load()
    nbytes = lib.fsvd_attn_decode_workspace_bytes(batch, heads, head_dim, nsplit)
    return torch.zeros(max(1, (nbytes + 3) // 4), dtype=torch.int32, device=device)


def attn_decode_densekv(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, cache_seqlens: torch.Tensor, *,
                        k_new: Optional[torch.Tensor] = None, v_new: Optional[torch.Tensor] = None,
                        cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None, seqlen_add: int = 0,
                        nsplit: Optional[int] = None, workspace: Optional[torch.Tensor] = None,
                        out: Optional[torch.Tensor] = None, softmax_scale: Optional[float] = None,
                        static_scratch: bool = False) -> torch.Tensor:
    """q [B,H,Dh] over caches [B,S,Hk,Dh]; see fsvd_attn_decode_densekv in include/flashsvd_hip.h.
    static_scratch=True takes fsvd_attn_decode_densekv_static (the library's own fixed scratch array).
    Custom operator flashsvd_hip::attn_decode_densekv."""
    a = (q, k_cache, v_cache, cache_seqlens, k_new, v_new, cos, sin, int(seqlen_add), None if nsplit is None else int(nsplit),
         workspace, None if not softmax_scale else float(softmax_scale), bool(static_scratch))
    return _OPS.attn_decode_densekv.default(*a) if out is None else _OPS.attn_decode_densekv.out(*a, out=out)


def _attn_decode_densekv_impl(q, k_cache, v_cache, cache_seqlens, k_new, v_new, cos, sin, seqlen_add, nsplit, workspace, out,
                              softmax_scale, static_scratch):
    dt, code = _elem(q, "q")
    _need(k_cache, "k_cache", dtype=dt); _need(v_cache, "v_cache", dtype=dt)
    _need(cache_seqlens, "cache_seqlens", dtype=torch.int32)
    if q.dim() != 3 or q.stride(2) != 1:
        raise ValueError(f"q must be [B,H,Dh] with unit inner stride, got {tuple(q.shape)}")
    B, H, Dh = q.shape
    if k_cache.dim() != 4 or k_cache.shape != v_cache.shape or k_cache.stride() != v_cache.stride() \
            or k_cache.shape[3] != Dh or k_cache.shape[0] < B or k_cache.stride(3) != 1:
        raise ValueError(f"caches must be matching [B>={B}, S, Hk, {Dh}] tensors, got {tuple(k_cache.shape)} / {tuple(v_cache.shape)}")
    S, Hk = k_cache.shape[1], k_cache.shape[2]
    if H % Hk != 0:
        raise ValueError(f"H={H} is not a multiple of Hk={Hk}")
    if cache_seqlens.numel() != B or not cache_seqlens.is_contiguous():
        raise ValueError(f"cache_seqlens must be a contiguous int32 [{B}] tensor")
    sk_b = sk_h = sv_b = sv_h = 0
    if k_new is not None:
        _need(k_new, "k_new", dtype=dt); _need(v_new, "v_new", dtype=dt)
        if k_new.shape != (B, Hk, Dh) or v_new.shape != (B, Hk, Dh) or k_new.stride(2) != 1 or v_new.stride(2) != 1:
            raise ValueError(f"k_new/v_new must be [B,Hk,Dh] tensors with unit inner stride, got {tuple(k_new.shape)} / {tuple(v_new.shape)}")
        sk_b, sk_h, sv_b, sv_h = k_new.stride(0), k_new.stride(1), v_new.stride(0), v_new.stride(1)
    rope_len = 0
    if cos is not None:
        _need(cos, "cos", dtype=dt); _need(sin, "sin", dtype=dt)
        if cos.shape != sin.shape or cos.dim() != 2 or cos.shape[1] != Dh // 2 or not cos.is_contiguous() or not sin.is_contiguous():
            raise ValueError(f"cos/sin must be contiguous [len, {Dh // 2}] tables")
        rope_len = cos.shape[0]
    if nsplit is None:
        nsplit = pick_nsplit(S, B, H, Dh, own_row=k_new is not None and Hk == H)
    if out is None:
        out = torch.empty(B, H, Dh, device=q.device, dtype=dt)
    elif out.shape != (B, H, Dh) or out.stride(2) != 1 or out.dtype != dt:
        raise ValueError("out must be [B,H,Dh] with unit inner stride")
    lib = _lib.load()
    if static_scratch:
        # library-owned scratch: no workspace tensor, nothing allocated inside the call (out must then be given too
        # by a caller that may not allocate)
        rc = lib.fsvd_attn_decode_densekv_static(q.data_ptr(), q.stride(0), q.stride(1), k_cache.data_ptr(), v_cache.data_ptr(),
                                                 k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
                                                 _ptr(k_new), sk_b, sk_h, _ptr(v_new), sv_b, sv_h, cache_seqlens.data_ptr(),
                                                 int(seqlen_add), _ptr(cos), _ptr(sin), rope_len, out.data_ptr(), out.stride(0),
                                                 out.stride(1), B, H, Hk, Dh, S, int(nsplit),
                                                 float(softmax_scale) if softmax_scale else 0.0, code, _stream())
        _lib.check("fsvd_attn_decode_densekv_static", rc)
        return out
    ws_ptr, ws_bytes = None, 0
    if nsplit > 1:
        if workspace is None:
            workspace = attn_workspace(B, H, Dh, nsplit, q.device)
        ws_ptr, ws_bytes = workspace.data_ptr(), workspace.numel() * workspace.element_size()
    rc = lib.fsvd_attn_decode_densekv(q.data_ptr(), q.stride(0), q.stride(1), k_cache.data_ptr(), v_cache.data_ptr(),
                                      k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
                                      _ptr(k_new), sk_b, sk_h, _ptr(v_new), sv_b, sv_h, cache_seqlens.data_ptr(), int(seqlen_add),
                                      _ptr(cos), _ptr(sin), rope_len, out.data_ptr(), out.stride(0), out.stride(1),
                                      ws_ptr, ws_bytes, B, H, Hk, Dh, S, int(nsplit),
                                      float(softmax_scale) if softmax_scale else 0.0, code, _stream())
    _lib.check("fsvd_attn_decode_densekv", rc)
    return out


def greedy_token_(logits: torch.Tensor, tokens: torch.Tensor, positions: Optional[torch.Tensor] = None) -> None:
    """``tokens[b] = logits[b].argmax()`` (ties to the lowest index, NaN above everything) and ``positions[b] += 1`` in one
    launch; logits [B, V] with unit inner stride, tokens int64 [B, 1] or [B], positions int32 [B].  Custom operator
    flashsvd_hip::greedy_token_ (tokens and positions are mutated arguments)."""
    _OPS.greedy_token_.default(logits, tokens, positions)


def _greedy_token_impl(logits, tokens, positions):
    _, code = _elem(logits, "logits")
    if logits.dim() != 2 or logits.stride(1) != 1:
        raise ValueError(f"logits must be [B, V] with unit inner stride, got {tuple(logits.shape)} strides {logits.stride()}")
    B, V = logits.shape
    _need(tokens, "tokens", dtype=torch.long)
    if tokens.numel() != B or tokens.shape[0] != B:
        raise ValueError(f"tokens must hold {B} rows of one id, got {tuple(tokens.shape)}")
    if positions is not None:
        _need(positions, "positions", dtype=torch.int32)
        if positions.shape != (B,) or not positions.is_contiguous():
            raise ValueError(f"positions must be a contiguous [{B}] tensor")
    if logits.device != tokens.device or (positions is not None and positions.device != tokens.device):
        raise ValueError("logits, tokens and positions must be on one device")
    rc = _lib.load().fsvd_greedy_token(logits.data_ptr(), logits.stride(0), tokens.data_ptr(), tokens.stride(0), _ptr(positions), B, V, code,
                                       _stream())
    _lib.check("fsvd_greedy_token", rc)


def set_token_rows_(tokens: torch.Tensor, src: torch.Tensor, positions: torch.Tensor, position: int) -> None:
    """``tokens.copy_(src)`` and ``positions.fill_(position)`` in one launch (contiguous int64 / int64 / int32 of the same
    number of rows on one device).  Custom operator flashsvd_hip::set_token_rows_ (tokens and positions are mutated arguments)."""
    _OPS.set_token_rows_.default(tokens, src, positions, int(position))


def _set_token_rows_impl(tokens, src, positions, position):
    _need(tokens, "tokens", dtype=torch.long)
    _need(src, "src", dtype=torch.long)
    _need(positions, "positions", dtype=torch.int32)
    if not tokens.device == src.device == positions.device:
        raise ValueError(f"tokens, src and positions must be on one device, got {tokens.device}, {src.device} and {positions.device}")
    if not (tokens.is_contiguous() and src.is_contiguous() and positions.is_contiguous() and tokens.numel() == src.numel() == positions.numel()):
        raise ValueError("tokens, src and positions must be contiguous and of one length")
    with torch.cuda.device(tokens.device):
        rc = _lib.load().fsvd_set_token_rows(tokens.data_ptr(), src.data_ptr(), positions.data_ptr(), int(position), tokens.numel(), _stream())
    _lib.check("fsvd_set_token_rows", rc)


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """w * bf16(x * rsqrt(mean(x^2) + eps)); custom operator flashsvd_hip::rmsnorm."""
    return _OPS.rmsnorm.default(x, weight, float(eps)) if out is None else _OPS.rmsnorm.out(x, weight, float(eps), out=out)


def _rmsnorm_impl(x, weight, eps, out):
    dt, code = _elem(x, "x")
    _need(weight, "weight", dtype=dt)
    K = x.shape[-1]
    if weight.shape != (K,) or not weight.is_contiguous():
        raise ValueError(f"weight must be contiguous [{K}]")
    x2, xp, ldx, rows, _ = _row_operand(x, "x")
    if out is None:
        out = torch.empty_like(x, memory_format=torch.contiguous_format)
    _need(out, "out", dtype=dt)
    o2, op, ldo, _, _ = _row_operand(out, "out")
    lib = _lib.load()
    rc = lib.fsvd_rmsnorm(xp, ldx, weight.data_ptr(), float(eps), op, ldo, rows, K, code, _stream())
    _lib.check("fsvd_rmsnorm", rc)
    return out


def _expand_operands(p, u, heads, Dh, out, bias, head_stride):
    """Checks of one head expansion; returns (B, M, R, coefficient strides, element code)."""
    dt, code = _elem(p, "p")
    _need(u, "u", dtype=dt); _need(out, "out", dtype=dt)
    if p.dim() == 3:
        B, M, R = p.shape
        sp = (p.stride(0), p.stride(1), 0 if head_stride is None else int(head_stride))
    elif p.dim() == 4:
        B, M, hp, R = p.shape
        if hp != heads:
            raise ValueError(f"p has {hp} heads, expected {heads}")
        sp = (p.stride(0), p.stride(1), p.stride(2))
    else:
        raise ValueError(f"p must be [B,M,R] or [B,M,heads,R], got {tuple(p.shape)}")
    if p.stride(-1) != 1 or u.stride(1) != 1 or out.stride(-1) != 1:
        raise ValueError("p, u and out need unit stride on the last axis")
    if u.shape != (heads * Dh, R):
        raise ValueError(f"u must be [{heads * Dh}, {R}], got {tuple(u.shape)}")
    if out.dim() != 4 or out.shape[0] < B or out.shape[2] != heads or out.shape[3] != Dh:
        raise ValueError(f"out must be [B>={B}, rows, {heads}, {Dh}], got {tuple(out.shape)}")
    if bias is not None:
        _need(bias, "bias", dtype=dt)
        if bias.numel() != heads * Dh or not bias.is_contiguous():
            raise ValueError(f"bias must be contiguous [{heads * Dh}]")
    return B, M, R, sp, code


def _rope_tables(cos, sin, Dh, dt):
    if cos is None:
        return 0
    _need(cos, "cos", dtype=dt); _need(sin, "sin", dtype=dt)
    if cos.shape != sin.shape or cos.dim() != 2 or cos.shape[1] != Dh // 2 or not cos.is_contiguous() or not sin.is_contiguous():
        raise ValueError(f"cos/sin must be contiguous [len, {Dh // 2}] tables")
    return cos.shape[0]


def lowrank_expand_heads(p: torch.Tensor, u: torch.Tensor, *, num_heads: int, head_dim: int, out: torch.Tensor,
                         cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None,
                         positions: Optional[torch.Tensor] = None, bias: Optional[torch.Tensor] = None,
                         dst_by_position: bool = False, head_stride: Optional[int] = None) -> torch.Tensor:
    """out[b, row, h, :] = rope(p[b, m, (h), :] @ u[h*Dh:(h+1)*Dh].T + bias); see fsvd_lowrank_expand_heads.
    p is [B, M, R] (shared by all heads) or [B, M, heads, R]; out is [B, rows, heads, Dh].
    Custom operator flashsvd_hip::lowrank_expand_heads (``out`` is the mutated argument)."""
    _OPS.lowrank_expand_heads.default(p, u, int(num_heads), int(head_dim), out, cos, sin, positions, bias, bool(dst_by_position),
                                      None if head_stride is None else int(head_stride))
    return out


def _lowrank_expand_heads_impl(p, u, num_heads, head_dim, out, cos, sin, positions, bias, dst_by_position, head_stride):
    heads, Dh = int(num_heads), int(head_dim)
    B, M, R, sp, code = _expand_operands(p, u, heads, Dh, out, bias, head_stride)
    rope_len = _rope_tables(cos, sin, Dh, p.dtype)
    if positions is not None:
        _need(positions, "positions", dtype=torch.int32)
        if positions.numel() != B:
            raise ValueError(f"positions must be int32 [{B}]")
    lib = _lib.load()
    rc = lib.fsvd_lowrank_expand_heads(p.data_ptr(), sp[0], sp[1], sp[2], u.data_ptr(), u.stride(0), _ptr(bias), _ptr(cos), _ptr(sin),
                                       rope_len, _ptr(positions), out.data_ptr(), out.stride(0), out.stride(1), out.stride(2),
                                       int(bool(dst_by_position)), out.shape[1], B, M, heads, Dh, R, code, _stream())
    _lib.check("fsvd_lowrank_expand_heads", rc)
    return out


def _weights2d(dt, **ts) -> None:
    for nm, t in ts.items():
        _need(t, nm, dtype=dt)
        if t.dim() != 2 or t.stride(1) != 1:
            raise ValueError(f"{nm} must be a 2-d weight with unit inner stride, got {tuple(t.shape)} strides {t.stride()}")


def _row_vector(dt, t, n: int, nm: str) -> Optional[int]:
    if t is None:
        return None
    _need(t, nm, dtype=dt)
    if t.shape != (n,) or not t.is_contiguous():
        raise ValueError(f"{nm} must be a contiguous [{n}] tensor")
    return t.data_ptr()


def _residual_rows(dt, t, B: int, N: int):
    """(tensor to keep alive, address, row stride) of a residual of B rows of N."""
    if t is None:
        return None, None, 0
    _need(t, "residual", dtype=dt)
    t, p, ld, rows, cols = _row_operand(t, "residual")
    if rows != B or cols != N:
        raise ValueError(f"residual shape {tuple(t.shape)} does not match output [{B}, {N}]")
    return t, p, ld


def _buffers(dt, device, *counts):
    """One allocation for the intermediates of a block: (tensor, addresses), each 512-byte aligned as an allocation of its own."""
    ends, n = [], 0
    for c in counts:
        ends.append(n)
        n += (c + 255) // 256 * 256
    buf = torch.empty(max(n, 1), dtype=dt, device=device)
    base = buf.data_ptr()
    return buf, [base + 2 * e for e in ends]


def _block_scratch(b, device, nbytes_of):
    """Scratch of this call and stream for the K shares of a block's projections; the tensor to keep alive."""
    n = nbytes_of(b) if _splitk_enabled() else 0
    if not n:
        return None
    t = torch.empty(n, dtype=torch.uint8, device=device)
    b.scratch, b.scratch_bytes = t.data_ptr(), n
    return t


def lowrank_mlp(x: torch.Tensor, gu_v: torch.Tensor, gate_u: torch.Tensor, up_u: torch.Tensor, down_v: torch.Tensor, down_u: torch.Tensor, *,
                norm_weight: Optional[torch.Tensor] = None, eps: float = 1e-6, residual: Optional[torch.Tensor] = None, mode: int = 0) -> torch.Tensor:
    """(residual +) down_u(down_v(silu(gate_u g) * up_u u)) with [g | u] = gu_v norm(x): the launches of :func:`linear`,
    :func:`swiglu_linear` and twice :func:`linear` issued by one native call.  Custom operator flashsvd_hip::lowrank_mlp."""
    return _OPS.lowrank_mlp.default(x, gu_v, gate_u, up_u, down_v, down_u, norm_weight, float(eps), residual, int(mode))


def _lowrank_mlp_impl(x, gu_v, gate_u, up_u, down_v, down_u, norm_weight, eps, residual, mode):
    dt, code = _elem(x, "x")
    _weights2d(dt, gu_v=gu_v, gate_u=gate_u, up_u=up_u, down_v=down_v, down_u=down_u)
    (two_r, K), (D, R), (Rd, Dv), (N, Ru) = gu_v.shape, gate_u.shape, down_v.shape, down_u.shape
    if two_r != 2 * R or up_u.shape != gate_u.shape or up_u.stride() != gate_u.stride() or Dv != D or Ru != Rd or x.shape[-1] != K:
        raise ValueError(f"factors do not match: x [.., {x.shape[-1]}], gu_v {tuple(gu_v.shape)}, gate_u {tuple(gate_u.shape)}, up_u {tuple(up_u.shape)}, "
                         f"down_v {tuple(down_v.shape)}, down_u {tuple(down_u.shape)}")
    nw = _row_vector(dt, norm_weight, K, "norm_weight")
    x2, xp, ldx, B, _ = _row_operand(x, "x")
    out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=dt)
    keep, rp, ldr = _residual_rows(dt, residual, B, N)
    if B >= 3:
        ensure_split_workspace(x.device)
    # the normalised rows are read by the rank projection only: the down projection's coefficients take their place
    buf, (xs, p, h) = _buffers(dt, x.device, max(B * K if nw and B >= 3 else 0, B * Rd), B * two_r, B * D)
    b = _lib.MlpBlock(xp, ldx, nw, xs, gu_v.data_ptr(), gu_v.stride(0), p, two_r, None, gate_u.data_ptr(), up_u.data_ptr(), gate_u.stride(0),
                      h, down_v.data_ptr(), down_v.stride(0), xs, down_u.data_ptr(), down_u.stride(0), None, rp, ldr, out.data_ptr(), N,
                      float(eps), B, K, R, D, Rd, N, int(mode), code)
    scratch = _block_scratch(b, x.device, _lib.load().fsvd_mlp_block_scratch_bytes) if B >= 128 and max(K, D, Rd) >= 4096 else None
    _lib.check("fsvd_mlp_block_run", _lib.load().fsvd_mlp_block_run(b, _stream()))
    return out


def _mlp_from_coefficients(pg, pu, gate_u, up_u, down_v, down_u, bias, mode):
    """The same from gate and up coefficients [B, R] of one row stride, which may be tensors of their own."""
    dt, code = _elem(pg, "pg")
    _weights2d(dt, gate_u=gate_u, up_u=up_u, down_v=down_v, down_u=down_u, pg=pg, pu=pu)
    (D, R), (Rd, Dv), (N, Ru) = gate_u.shape, down_v.shape, down_u.shape
    if pg.shape != pu.shape or pg.stride() != pu.stride() or pg.shape[1] != R or up_u.shape != gate_u.shape or up_u.stride() != gate_u.stride() \
            or Dv != D or Ru != Rd:
        raise ValueError("coefficients and factors do not match")
    if pg.device != pu.device:
        raise ValueError(f"gate and up coefficients must be on one device, got {pg.device} and {pu.device}")
    B = pg.shape[0]
    bp = _row_vector(dt, bias, N, "bias")
    out = torch.empty(B, N, device=pg.device, dtype=dt)
    if B >= 3:
        ensure_split_workspace(pg.device)
    buf, (h, s) = _buffers(dt, pg.device, B * D, B * Rd)
    b = _lib.MlpBlock(None, 0, None, None, None, 0, pg.data_ptr(), pg.stride(0), pu.data_ptr(), gate_u.data_ptr(), up_u.data_ptr(), gate_u.stride(0),
                      h, down_v.data_ptr(), down_v.stride(0), s, down_u.data_ptr(), down_u.stride(0), bp, None, 0, out.data_ptr(), N,
                      0.0, B, 0, R, D, Rd, N, int(mode), code)
    scratch = _block_scratch(b, pg.device, _lib.load().fsvd_mlp_block_scratch_bytes) if B >= 128 and max(D, Rd) >= 4096 else None
    _lib.check("fsvd_mlp_block_run", _lib.load().fsvd_mlp_block_run(b, _stream()))
    return out


def lowrank_attn_prefill(x: torch.Tensor, qkv_v: torch.Tensor, q_u: torch.Tensor, k_u: torch.Tensor, v_u: torch.Tensor, o_v: torch.Tensor,
                         o_u: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, *, start: int,
                         num_heads: int, num_kv_heads: int, norm_weight: Optional[torch.Tensor] = None, eps: float = 1e-6,
                         residual: Optional[torch.Tensor] = None, o_v_bias: Optional[torch.Tensor] = None,
                         o_u_bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The attention half of a prompt pass over the dense cache: x [B, T, K] at positions start .. start + T - 1, keys and values
    into the cache rows of those positions, (residual +) o_u(o_v(attention)).  The launches of :func:`linear`,
    :func:`lowrank_expand_heads_multi`, :func:`attn_prefill` and twice :func:`linear` issued by one native call.  Custom
    operator flashsvd_hip::lowrank_attn_prefill (the caches are mutated arguments)."""
    return _OPS.lowrank_attn_prefill.default(x, qkv_v, q_u, k_u, v_u, o_v, o_u, k_cache, v_cache, cos, sin, int(start), int(num_heads),
                                             int(num_kv_heads), norm_weight, float(eps), residual, o_v_bias, o_u_bias)


def _lowrank_attn_prefill_impl(x, qkv_v, q_u, k_u, v_u, o_v, o_u, k_cache, v_cache, cos, sin, start, num_heads, num_kv_heads, norm_weight, eps,
                               residual, o_v_bias, o_u_bias):
    dt, code = _elem(x, "x")
    _weights2d(dt, qkv_v=qkv_v, q_u=q_u, k_u=k_u, v_u=v_u, o_v=o_v, o_u=o_u)
    _need(k_cache, "k_cache", dtype=dt); _need(v_cache, "v_cache", dtype=dt)
    if x.dim() != 3 or k_cache.dim() != 4 or k_cache.shape != v_cache.shape or k_cache.stride() != v_cache.stride() or k_cache.stride(3) != 1:
        raise ValueError("x must be [B, T, K] and the caches matching [B, S, Hk, Dh] with unit inner stride")
    H, Hk = int(num_heads), int(num_kv_heads)
    (B, T, K), (_, S, hk, Dh) = x.shape, k_cache.shape
    (Rt, Kw), (qn, rq), (kn, rk), (vn, rv), (Ro, w), (N, Ru) = (t.shape for t in (qkv_v, q_u, k_u, v_u, o_v, o_u))
    if k_cache.shape[0] < B or hk != Hk or qn != H * Dh or kn != Hk * Dh or vn != Hk * Dh or Rt != rq + rk + rv or Kw != K or w != H * Dh or Ru != Ro:
        raise ValueError("factors and caches do not match")
    rope_len = _rope_tables(cos, sin, Dh, dt)
    nw, bv, bu = _row_vector(dt, norm_weight, K, "norm_weight"), _row_vector(dt, o_v_bias, Ro, "o_v_bias"), _row_vector(dt, o_u_bias, N, "o_u_bias")
    x2, xp, ldx, rows, _ = _row_operand(x, "x")
    out = torch.empty(B, T, N, device=x.device, dtype=dt)
    keep, rp, ldr = _residual_rows(dt, residual, rows, N)
    if rows >= 3:
        ensure_split_workspace(x.device)
    buf, (xs, p, q, a) = _buffers(dt, x.device, max(rows * K if nw and rows >= 3 else 0, rows * Ro), rows * Rt, rows * w, rows * w)
    b = _lib.AttnBlock(xp, ldx, nw, xs, qkv_v.data_ptr(), qkv_v.stride(0), p, q_u.data_ptr(), k_u.data_ptr(), v_u.data_ptr(), q_u.stride(0),
                       k_u.stride(0), v_u.stride(0), cos.data_ptr(), sin.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), k_cache.stride(0),
                       k_cache.stride(1), k_cache.stride(2), q, a, o_v.data_ptr(), o_v.stride(0), bv, xs, o_u.data_ptr(), o_u.stride(0), bu,
                       rp, ldr, out.data_ptr(), N, float(eps), B, T, K, rq, rk, rv, H, Hk, Dh, S, int(start), rope_len, Ro, N, code)
    scratch = _block_scratch(b, x.device, _lib.load().fsvd_attn_block_scratch_bytes) if rows >= 128 and max(K, w, Ro) >= 4096 else None
    _lib.check("fsvd_attn_block_prefill", _lib.load().fsvd_attn_block_prefill(b, _stream()))
    return out


def prefill_head_groups(B: int, M: int, n_ctx: int, H: int, Hk: int, Dh: int, itemsize: int = 2) -> int:
    """How many kv heads (with their query heads) the expand-then-attend prompt pass takes at a time.

    The pass rebuilds q [B,M,H,Dh] and K, V [B,n_ctx,Hk,Dh] from rank coefficients into temporaries and runs the prompt
    attention over them; nothing forces all heads to exist at once.  The largest group of kv heads whose temporaries
    fit FLASHSVD_AMD_PREFILL_TEMP_BYTES (default 1 GiB) is taken, at least one; 0 or a negative budget means all heads in
    one pass.  Groups cost a few per cent of the pass (8 x 2048 tokens at rank 1664: +4 % at 64 MiB, five kv heads per
    group), so the default only bounds the temporaries of very long batches."""
    import os
    budget = int(float(os.getenv("FLASHSVD_AMD_PREFILL_TEMP_BYTES", str(1 << 30))))
    if budget <= 0:
        return Hk
    per_kv_head = (B * M * (H // Hk) + 2 * B * n_ctx) * Dh * itemsize
    return max(1, min(Hk, budget // max(per_kv_head, 1)))


def lowrank_expand_heads_multi(items, *, head_dim: int, cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None,
                               positions: Optional[torch.Tensor] = None) -> None:
    """The q / k / v expansions of one prompt pass in one call (fsvd_lowrank_expand_heads_multi): ``items`` is a list of one
    to three dicts with the keyword arguments of :func:`lowrank_expand_heads` for one expansion (``p``, ``u``,
    ``num_heads``, ``out``, optional ``bias``, ``dst_by_position``, ``head_stride``) plus ``rotate`` (apply cos / sin).
    The same results as separate calls; a single launch when every expansion takes the tiled kernel."""
    Dh = int(head_dim)
    if not 1 <= len(items) <= 3:
        raise ValueError(f"{len(items)} expansions (1..3)")
    rope_len = _rope_tables(cos, sin, Dh, items[0]["p"].dtype)
    descs = (_lib.ExpandDesc * len(items))()
    shape = code = None
    for d, it in zip(descs, items):
        heads, out, bias = int(it["num_heads"]), it["out"], it.get("bias")
        B, M, R, sp, c = _expand_operands(it["p"], it["u"], heads, Dh, out, bias, it.get("head_stride"))
        if shape is None:
            shape, code = (B, M), c
        elif shape != (B, M):
            raise ValueError(f"expansions of one call cover the same token rows: {shape} vs {(B, M)}")
        elif c != code:
            raise ValueError("expansions of one call are of one element type")
        if it.get("rotate") and cos is None:
            raise ValueError("rotate asked for without cos / sin")
        d.p, d.sp_b, d.sp_m, d.sp_h = it["p"].data_ptr(), sp[0], sp[1], sp[2]
        d.u, d.ldu, d.bias = it["u"].data_ptr(), it["u"].stride(0), _ptr(bias)
        d.y, d.sy_b, d.sy_m, d.sy_h = out.data_ptr(), out.stride(0), out.stride(1), out.stride(2)
        d.heads, d.R, d.rotate = heads, R, int(bool(it.get("rotate")))
        d.dst_by_position, d.dst_rows, d.rsv0 = int(bool(it.get("dst_by_position"))), out.shape[1], 0
    B, M = shape
    if positions is not None:
        _need(positions, "positions", dtype=torch.int32)
        if positions.numel() != B:
            raise ValueError(f"positions must be int32 [{B}]")
    lib = _lib.load()
    rc = lib.fsvd_lowrank_expand_heads_multi(descs, len(items), _ptr(cos), _ptr(sin), rope_len, _ptr(positions), B, M, Dh, code, _stream())
    _lib.check("fsvd_lowrank_expand_heads_multi", rc)


def rope_tables(position_ids: torch.Tensor, inv_freq: torch.Tensor, dtype: torch.dtype):
    """cos, sin [rows, half] of ``position_ids.float() * inv_freq`` (contiguous int64 and fp32 tensors), rounded to ``dtype``,
    in one launch.  Custom operator flashsvd_hip::rope_tables."""
    return _OPS.rope_tables.default(position_ids, inv_freq, dtype)


def rope_tables_mask(position_ids: torch.Tensor, inv_freq: torch.Tensor, dtype: torch.dtype, mask: torch.Tensor):
    """:func:`rope_tables` and ``(mask != 0)`` as the uint8 padding mask of :func:`attn_prefill` (mask: contiguous int64), in one
    launch.  Custom operator flashsvd_hip::rope_tables_mask."""
    return _OPS.rope_tables_mask.default(position_ids, inv_freq, dtype, mask)


def _rope_tables_impl(position_ids, inv_freq, dtype, mask=None):
    code = _ELEM_CODES.get(dtype)
    if code is None:
        raise ValueError(f"rotation tables are torch.bfloat16 or torch.float16, got {dtype}")
    _need(position_ids, "position_ids", dtype=torch.long); _need(inv_freq, "inv_freq", dtype=torch.float32)
    if not position_ids.is_contiguous() or inv_freq.dim() != 1 or not inv_freq.is_contiguous():
        raise ValueError("position_ids and inv_freq must be contiguous, inv_freq one-dimensional")
    if position_ids.device != inv_freq.device:
        raise ValueError(f"position_ids and inv_freq must be on one device, got {position_ids.device} and {inv_freq.device}")
    rows, half = position_ids.numel(), inv_freq.numel()
    cos = torch.empty(rows, half, dtype=dtype, device=position_ids.device)
    sin = torch.empty_like(cos)
    if mask is None:
        _lib.check("fsvd_rope_tables", _lib.load().fsvd_rope_tables(position_ids.data_ptr(), inv_freq.data_ptr(), cos.data_ptr(), sin.data_ptr(), rows,
                                                                    half, code, _stream()))
        return cos, sin
    _need(mask, "mask", dtype=torch.long)
    if not mask.is_contiguous() or mask.device != position_ids.device:
        raise ValueError(f"mask must be contiguous and on {position_ids.device}, got strides {mask.stride()} on {mask.device}")
    pad = torch.empty(mask.shape, dtype=torch.uint8, device=mask.device)
    _lib.check("fsvd_rope_tables_mask", _lib.load().fsvd_rope_tables_mask(position_ids.data_ptr(), inv_freq.data_ptr(), cos.data_ptr(), sin.data_ptr(), rows,
                                                                          half, mask.data_ptr(), pad.data_ptr(), mask.numel(), code, _stream()))
    return cos, sin, pad


def attn_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, *, q_pos0: Optional[torch.Tensor] = None, causal: bool = True,
                 pad_mask: Optional[torch.Tensor] = None, add_mask: Optional[torch.Tensor] = None,
                 out: Optional[torch.Tensor] = None, softmax_scale: Optional[float] = None) -> torch.Tensor:
    """q [B,M,H,Dh] (rotated), k/v [B,S,Hk,Dh] -> out [B,M,H,Dh]; keys n < q_pos0[b]+M, causal n <= q_pos0[b]+m.
    Custom operator flashsvd_hip::rope_attn_prefill."""
    a = (q, k, v, q_pos0, bool(causal), pad_mask, add_mask, None if not softmax_scale else float(softmax_scale))
    return _OPS.rope_attn_prefill.default(*a) if out is None else _OPS.rope_attn_prefill.out(*a, out=out)


def _attn_prefill_impl(q, k, v, q_pos0, causal, pad_mask, add_mask, out, softmax_scale):
    dt, code = _elem(q, "q")
    _need(k, "k", dtype=dt); _need(v, "v", dtype=dt)
    if q.dim() != 4 or k.dim() != 4 or k.shape != v.shape or k.stride() != v.stride():
        raise ValueError(f"q must be [B,M,H,Dh] and k/v matching [B,S,Hk,Dh], got {tuple(q.shape)} {tuple(k.shape)} {tuple(v.shape)}")
    B, M, H, Dh = q.shape
    S, Hk = k.shape[1], k.shape[2]
    if k.shape[0] < B or k.shape[3] != Dh or H % Hk:
        raise ValueError("k/v do not match q")
    if q.stride(3) != 1 or k.stride(3) != 1:
        raise ValueError("q, k, v need unit stride on the last axis")
    if out is None:
        out = torch.empty(B, M, H, Dh, device=q.device, dtype=dt)
    _need(out, "out", dtype=dt)
    spm = sam_b = sam_q = 0
    for t, nm in ((pad_mask, "pad_mask"), (add_mask, "add_mask")):
        if t is not None and t.device != q.device:
            raise ValueError(f"{nm} must be on the device of q, {q.device}, got {t.device}")
    if pad_mask is not None:
        if pad_mask.dtype != torch.uint8 or pad_mask.dim() != 2 or pad_mask.shape[0] != B or pad_mask.stride(1) != 1:
            raise ValueError("pad_mask must be uint8 [B, keys]")
        spm = pad_mask.stride(0)
    if add_mask is not None:
        if add_mask.dtype != torch.float32 or add_mask.dim() != 3 or add_mask.shape[0] != B or add_mask.shape[1] != M or add_mask.stride(2) != 1:
            raise ValueError("add_mask must be float32 [B, M, keys]")
        sam_b, sam_q = add_mask.stride(0), add_mask.stride(1)
    if q_pos0 is not None:
        _need(q_pos0, "q_pos0", dtype=torch.int32)
    lib = _lib.load()
    rc = lib.fsvd_attn_prefill(q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), k.data_ptr(), v.data_ptr(), k.stride(0),
                               k.stride(1), k.stride(2), _ptr(q_pos0), _ptr(pad_mask), spm, _ptr(add_mask), sam_b, sam_q,
                               out.data_ptr(), out.stride(0), out.stride(1), out.stride(2), B, M, H, Hk, Dh, S, int(bool(causal)),
                               float(softmax_scale) if softmax_scale else 0.0, code, _stream())
    _lib.check("fsvd_attn_prefill", rc)
    return out
