"""Torch-tensor wrappers over the C ABI (device memory and streams only).

Every function requires CUDA (ROCm) tensors and launches the gfx950 kernels on
the current stream of the tensor's device; there is no CPU path.
"""
from __future__ import annotations

import ctypes
import functools
import os
from typing import Tuple

import torch

from . import _lib
from ._lib import PratchyaError, PratchyaUnsupported, PratchyaWaitTimeout  # noqa: F401  (re-exported)

E4M3 = torch.float8_e4m3fn
E8M0 = torch.float8_e8m0fnu


# The wrappers' own time is what a small call costs (a Linear of 4 tokens: 69
# us for 12 us of kernels), so they take addresses and the current stream as
# plain integers, allocate outputs in their own dtypes and keep the layouts of
# shapes they have seen.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _ptr(t: torch.Tensor) -> int:
    return t.data_ptr()


def _stream(t: torch.Tensor) -> int:
    if _raw_stream is not None:
        return _raw_stream(t.device.index)
    return torch.cuda.current_stream(t.device).cuda_stream


def _require_gpu(*ts: torch.Tensor) -> None:
    for t in ts:
        if not t.is_cuda:
            raise RuntimeError("pratchya_amd runs on the GPU only; got a tensor on "
                               f"{t.device} (there is no CPU fallback)")


def _dtype_code(dt: torch.dtype) -> int:
    if dt == torch.float32:
        return _lib.DT_F32
    if dt == torch.bfloat16:
        return _lib.DT_BF16
    raise TypeError(f"unsupported dtype {dt}; expected float32 or bfloat16")


def slices_hw(shape) -> Tuple[int, int, int]:
    """(slices, H, W) of a tensor shape: 0-d -> (1,1,1), 1-d -> (1,1,n)
    (pratchya/_qualia/_qarr.py:461-464); leading dims are independent slices."""
    shape = tuple(int(s) for s in shape)
    if len(shape) == 0:
        return 1, 1, 1
    if len(shape) == 1:
        return 1, 1, shape[0]
    s = 1
    for d in shape[:-2]:
        s *= d
    return s, shape[-2], shape[-1]


@functools.lru_cache(maxsize=4096)
def _group_layout(H: int, W: int, a: int, b: int) -> Tuple[int, int, int]:
    lib = _lib.load()
    n_blk, K, M = ctypes.c_int64(), ctypes.c_int64(), ctypes.c_int64()
    _lib.check(lib.pratchya_quant_layout(H, W, a, b, ctypes.byref(n_blk), ctypes.byref(K), ctypes.byref(M)),
               "quantize layout")
    return n_blk.value, K.value, M.value


def group_layout(H: int, W: int, tgrid) -> Tuple[int, int, int]:
    """(n_blk, K, M) of one [H, W] slice (pratchya/_qualia/_qarr.py:474-480)."""
    return _group_layout(int(H), int(W), int(tgrid[0]), int(tgrid[1]))


@functools.lru_cache(maxsize=4096)
def _ws_bytes_of(query: str, device: int, *sizes: int) -> int:
    return int(getattr(_lib.load(), query)(*sizes))


def _ws_bytes(query: str, *sizes: int) -> int:
    """A workspace query of the library (they depend on the sizes and on the
    device's compute units only)."""
    return _ws_bytes_of(query, torch.cuda.current_device(), *sizes)


def _aligned(t: torch.Tensor, n: int) -> bool:
    return t.data_ptr() % n == 0


def _check_out(out, shapes, what):
    """Caller-provided output buffers: contiguous, on the device, of the right
    byte sizes (dtype views of uint8 / e4m3fn / e8m0 and f32 are accepted)."""
    if len(out) != len(shapes):
        raise ValueError(f"{what}: expected {len(shapes)} output buffers")
    for t, (shape, esz) in zip(out, shapes):
        n = 1
        for d in shape:
            n *= int(d)
        if not t.is_cuda or not t.is_contiguous() or t.numel() * t.element_size() != n * esz:
            raise ValueError(f"{what}: output buffer of {tuple(t.shape)} {t.dtype} does not fit {shape}")


def quantize(x: torch.Tensor, tgrid, out=None) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Quantize ``x`` (bf16 or f32) with block grid ``tgrid``.

    Returns ``(x_fp8 [x.shape] e4m3fn, sc_fp8 [..., M, K] e8m0, sc_fp32
    [..., M, 1, 1] f32)`` exactly as pratchya/_qualia/_qarr.py:506.  ``out``
    may hold preallocated (payload, e8m0, f32) buffers to write instead.
    """
    _require_gpu(x)
    if x.dtype not in (torch.float32, torch.bfloat16):
        x = x.float()
    a, b = int(tgrid[0]), int(tgrid[1])
    S, H, W = slices_hw(x.shape)
    n_blk, K, M = group_layout(H, W, (a, b))
    lead = tuple(x.shape[:-2]) if x.dim() >= 2 else ()
    if not x.is_contiguous() or not _aligned(x, 16):
        x = x.contiguous() if not x.is_contiguous() else x.clone()
    if out is None:
        x8 = torch.empty(x.shape, dtype=E4M3, device=x.device)
        sc8 = torch.empty(lead + (M, K), dtype=E8M0, device=x.device)
        sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=x.device)
    else:
        _check_out(out, [(x.shape, 1), (lead + (M, K), 1), (lead + (M, 1, 1), 4)], "quantize")
        x8, sc8, sc32 = out[0].view(E4M3), out[1].view(E8M0), out[2]
    lib = _lib.load()
    code = _dtype_code(x.dtype)
    ws_bytes = _ws_bytes("pratchya_quantize_workspace_bytes", code, S, H, W, a, b)
    if ws_bytes == 0 and not _aligned(x8, 8 if x.dtype == torch.bfloat16 else 4):
        ws_bytes = S * n_blk * 4      # a misaligned caller payload buffer: the general path runs
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=x.device) if ws_bytes else None
    _lib.check(lib.pratchya_quantize(_ptr(x), code, S, H, W, a, b, _ptr(x8), _ptr(sc8), _ptr(sc32),
                                     _ptr(ws) if ws is not None else None, ws_bytes, _stream(x)), "quantize")
    return x8, sc8, sc32


def quantize_dequantize(x: torch.Tensor, tgrid, dtype: torch.dtype, fix_nan: bool = False, out=None):
    """Fake quantization in one pass: ``dequantize_impl(*quantize_impl(x, tgrid),
    dtype, tgrid)``, i.e. ``QArrayImpl(x, tgrid).astype(dtype)``
    (pratchya/_qualia/_qarr.py:339-342, 458-506, 541-569), without writing
    the payload.  ``fix_nan`` dequantizes NaN e8m0 scales as 1.0, as
    quantize_impl's backward does for a requantized cotangent (Q:512-526).

    Returns ``(y [x.shape] dtype, sc_fp8 [..., M, K] e8m0, sc_fp32 [..., M, 1, 1])``;
    the scales are quantize_impl's, unrepaired.  ``out`` may hold preallocated
    (y, e8m0, f32) buffers.
    """
    _require_gpu(x)
    if x.dtype not in (torch.float32, torch.bfloat16):
        x = x.float()
    if dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"quantize_dequantize: output dtype {dtype} is not float32 or bfloat16")
    a, b = int(tgrid[0]), int(tgrid[1])
    S, H, W = slices_hw(x.shape)
    n_blk, K, M = group_layout(H, W, (a, b))
    lead = tuple(x.shape[:-2]) if x.dim() >= 2 else ()
    if not x.is_contiguous() or not _aligned(x, 16):
        x = x.contiguous() if not x.is_contiguous() else x.clone()
    if out is None:
        y = torch.empty(x.shape, dtype=dtype, device=x.device)
        sc8 = torch.empty(lead + (M, K), dtype=E8M0, device=x.device)
        sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=x.device)
    else:
        esz = 2 if dtype == torch.bfloat16 else 4
        _check_out(out, [(x.shape, esz), (lead + (M, K), 1), (lead + (M, 1, 1), 4)], "quantize_dequantize")
        y, sc8, sc32 = out[0], out[1].view(E8M0), out[2]
    lib = _lib.load()
    code = _dtype_code(x.dtype)
    ws_bytes = _ws_bytes("pratchya_quantize_dequantize_workspace_bytes", code, S, H, W, a, b)
    if ws_bytes == 0 and not (_aligned(y, 16) and _aligned(sc8, 8)):
        ws_bytes = S * n_blk * 4      # misaligned caller buffers: the general path runs
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=x.device) if ws_bytes else None
    _lib.check(lib.pratchya_quantize_dequantize(
        _ptr(x), code, S, H, W, a, b, _ptr(y), _dtype_code(dtype), 1 if fix_nan else 0, _ptr(sc8),
        _ptr(sc32), _ptr(ws) if ws is not None else None, ws_bytes, _stream(x)), "quantize_dequantize")
    return y, sc8, sc32


def requantize_cotangent(g: torch.Tensor, g_sc8: torch.Tensor, g_sc32: torch.Tensor, out=None):
    """``quantize_impl(dequantize_impl_bwd(g, g_sc8, g_sc32, (1, 128)), (1, 128))``
    in one pass (pratchya/_qualia/_qarr.py:575-601 then 458-506): the cotangent
    of a Linear output requantized for the FP8 dgrad.  ``g`` bf16 / f32 with the
    (1, 128) scales of the tensor it is the cotangent of.  Returns
    ``(g_fp8, sc_fp8, sc_fp32)`` as ``quantize(g1, (1, 128))``; raises
    ``PratchyaUnsupported`` unless the layout has 8 blocks per group."""
    _require_gpu(g, g_sc8, g_sc32)
    if g.dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"requantize_cotangent: dtype {g.dtype} is not float32 or bfloat16")
    S, H, W = slices_hw(g.shape)
    n_blk, K, M = group_layout(H, W, (1, 128))
    lead = tuple(g.shape[:-2]) if g.dim() >= 2 else ()
    if not g.is_contiguous() or not _aligned(g, 16):
        g = g.contiguous() if not g.is_contiguous() else g.clone()
    gs8, gs32 = _u8(g_sc8).contiguous(), g_sc32.contiguous().float()
    if gs8.numel() != S * n_blk or gs32.numel() != S * M:
        raise ValueError("requantize_cotangent: scales do not match a (1, 128) quantization of g's shape")
    if out is None:
        x8 = torch.empty(g.shape, dtype=torch.uint8, device=g.device)
        sc8 = torch.empty(lead + (M, K), dtype=torch.uint8, device=g.device)
        sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=g.device)
    else:
        _check_out(out, [(g.shape, 1), (lead + (M, K), 1), (lead + (M, 1, 1), 4)], "requantize_cotangent")
        x8, sc8, sc32 = _u8(out[0]), _u8(out[1]), out[2]
    lib = _lib.load()
    _lib.check(lib.pratchya_requantize_cotangent(_ptr(g), _dtype_code(g.dtype), _ptr(gs8), _ptr(gs32), S, H, W,
                                                 _ptr(x8), _ptr(sc8), _ptr(sc32), _stream(g)),
               "requantize_cotangent")
    return x8.view(E4M3), sc8.view(E8M0), sc32


def _u8(t: torch.Tensor) -> torch.Tensor:
    return t.view(torch.uint8) if t.dtype != torch.uint8 else t


def quantize_t1x128(x: torch.Tensor, x_sc8: torch.Tensor = None, x_sc32: torch.Tensor = None):
    """``quantize_impl(x^T, (1, 128))`` (pratchya/_qualia/_qarr.py:458-506)
    of a [T, C] tensor, without materialising x^T: fp8_matmul's quantization
    of its transposed raw inputs (Q:786-788).  Blocks are 128 tokens of one
    channel, groups 8 consecutive blocks of one channel.  ``x`` and the input
    scales as for ``quantize_t128``.  Returns ``(xt_fp8 [C, T] e4m3fn,
    sc_fp8 [C*T/1024, 8] e8m0, sc_fp32 [C*T/1024, 1, 1] f32)``, the
    K-contiguous (1, 128) row operand of a GEMM that contracts over tokens.
    The kernel takes T a multiple of 1024; other token counts go through the
    general quantizer on the explicitly transposed (dequantized) tensor."""
    _require_gpu(x)
    if x.dim() != 2:
        raise ValueError("quantize_t1x128 needs a [T, C] tensor")
    T, C = int(x.shape[0]), int(x.shape[1])
    if x.dtype in (E4M3, torch.uint8):
        if x_sc8 is None or x_sc32 is None:
            raise ValueError("an fp8 input needs its (1, 128) scales")
        code, xin = _lib.DT_E4M3, _u8(x)
        xs8, xs32 = _u8(x_sc8).contiguous(), x_sc32.contiguous().float()
    elif x.dtype == torch.bfloat16 and x_sc8 is not None and x_sc32 is not None:
        code, xin = _lib.DT_BF16, x
        xs8, xs32 = _u8(x_sc8).contiguous(), x_sc32.contiguous().float()
    else:
        if x_sc8 is not None or x_sc32 is not None:
            raise ValueError("input scales apply to an fp8 payload or a bf16 cotangent only")
        xin = x if x.dtype in (torch.float32, torch.bfloat16) else x.float()
        code = _dtype_code(xin.dtype)
        xs8 = xs32 = None
    if T % 1024 or C % 8:
        # the reference's composition: the values (dequantized / taken through
        # dequantize_impl_bwd as the kernel does), transposed, quantized
        if code == _lib.DT_E4M3:
            v = dequantize(xin.view(E4M3), xs8.view(E8M0), xs32, torch.float32, (1, 128))
        elif xs8 is not None:
            v = dequantize_bwd(xin, xs8.view(E8M0), xs32, (1, 128))
        else:
            v = xin
        return quantize(v.t().contiguous(), (1, 128))
    if not xin.is_contiguous() or not _aligned(xin, 16):
        xin = xin.contiguous() if not xin.is_contiguous() else xin.clone()
    M = C * T // 1024
    xt8 = torch.empty((C, T), dtype=torch.uint8, device=x.device)
    sc8 = torch.empty((M, 8), dtype=torch.uint8, device=x.device)
    sc32 = torch.empty((M, 1, 1), dtype=torch.float32, device=x.device)
    _lib.check(_lib.load().pratchya_quantize_t1x128(_ptr(xin), code,
                                                    _ptr(xs8) if xs8 is not None else None,
                                                    _ptr(xs32) if xs32 is not None else None,
                                                    1, T, C, _ptr(xt8), _ptr(sc8), _ptr(sc32), _stream(xin)),
               "quantize_t1x128")
    return xt8.view(E4M3), sc8.view(E8M0), sc32


def quantize_128x1(x: torch.Tensor, x_sc8: torch.Tensor = None, x_sc32: torch.Tensor = None, out=None):
    """``quantize_impl(x, (128, 1))`` (pratchya/_qualia/_qarr.py:458-506) with
    the payload in ``x``'s own [..., T, C] layout, from the same inputs as
    ``quantize_t128`` (bf16 / f32, an fp8 payload with its (1, 128) scales, or
    a bf16 cotangent with them).  Returns ``(q_fp8 [..., T, C] e4m3fn, sc_fp8
    [..., M, 8] e8m0, sc_fp32 [..., M, 1, 1] f32)``, exactly quantize_impl's.
    """
    return _quantize_128x1(x, x_sc8, x_sc32, out, rows=True)


def quantize_dual(x: torch.Tensor):
    """``quantize_impl(x, (1, 128))`` and, from the same pass,
    ``quantize_impl(dequantize_impl(that), (128, 1))`` with the second payload
    in ``x``'s own [..., T, C] layout (pratchya/_qualia/_qarr.py:458-506,
    :541-569): a quantized Linear's input and the FP8 weight gradient's
    token-axis requantization of it (Q:784-789).  ``x``: bf16 or f32
    [..., T, C] with T a multiple of 128 and C of 1024
    (``PratchyaUnsupported`` for other C).  Returns ``((q, sc8, sc32), (q2,
    sc8b, sc32b))``, bit-identical to ``quantize(x, (1, 128))`` and
    ``quantize_128x1`` of its payload."""
    _require_gpu(x)
    if x.dim() < 2:
        raise ValueError("quantize_dual needs a [..., T, C] tensor")
    if x.dtype not in (torch.float32, torch.bfloat16):
        x = x.float()
    if not x.is_contiguous() or not _aligned(x, 16):
        x = x.contiguous() if not x.is_contiguous() else x.clone()
    lead = tuple(x.shape[:-2])
    T, C = int(x.shape[-2]), int(x.shape[-1])
    S = 1
    for d in lead:
        S *= int(d)
    _, K1, M1 = group_layout(T, C, (1, 128))
    _, K2, M2 = group_layout(T, C, (128, 1))
    dev = x.device
    q = torch.empty(x.shape, dtype=torch.uint8, device=dev)
    sc8 = torch.empty(lead + (M1, K1), dtype=torch.uint8, device=dev)
    sc32 = torch.empty(lead + (M1, 1, 1), dtype=torch.float32, device=dev)
    q2 = torch.empty(x.shape, dtype=torch.uint8, device=dev)
    sc8b = torch.empty(lead + (M2, K2), dtype=torch.uint8, device=dev)
    sc32b = torch.empty(lead + (M2, 1, 1), dtype=torch.float32, device=dev)
    _lib.check(_lib.load().pratchya_quantize_dual(_ptr(x), _dtype_code(x.dtype), S, T, C, _ptr(q), _ptr(sc8),
                                                  _ptr(sc32), _ptr(q2), _ptr(sc8b), _ptr(sc32b), _stream(x)),
               "quantize_dual")
    return (q.view(E4M3), sc8.view(E8M0), sc32), (q2.view(E4M3), sc8b.view(E8M0), sc32b)


def quantize_t128(x: torch.Tensor, x_sc8: torch.Tensor = None, x_sc32: torch.Tensor = None, out=None):
    """``quantize_impl(x, (128, 1))`` (pratchya/_qualia/_qarr.py:458-506) with
    the payload transposed per slice.

    ``x``: [..., T, C] bf16 or f32, or an e4m3fn payload quantized with tgrid
    (1, 128) whose scales are ``x_sc8`` / ``x_sc32`` (dequantized to f32 first,
    as ``dequantize_impl`` does).  A bf16 ``x`` given with scales is the
    cotangent of a tensor quantized (1, 128) with them: it goes through
    ``dequantize_impl_bwd`` (Q:575-601) first, in registers.  Returns ``(xt_fp8 [..., C, T] e4m3fn,
    sc_fp8 [..., M, 8] e8m0, sc_fp32 [..., M, 1, 1] f32)``: the scales are
    exactly ``quantize_impl(x, (128, 1))``'s, the payload is its payload with
    the last two axes swapped.  ``out`` may hold preallocated buffers.
    """
    return _quantize_128x1(x, x_sc8, x_sc32, out, rows=False)


def _quantize_128x1(x, x_sc8, x_sc32, out, rows):
    name = "quantize_128x1" if rows else "quantize_t128"
    _require_gpu(x)
    if x.dim() < 2:
        raise ValueError(f"{name} needs a [..., T, C] tensor")
    lead = tuple(x.shape[:-2])
    T, C = int(x.shape[-2]), int(x.shape[-1])
    S = 1
    for d in lead:
        S *= int(d)
    if x.dtype in (E4M3, torch.uint8):
        if x_sc8 is None or x_sc32 is None:
            raise ValueError("an fp8 input needs its (1, 128) scales")
        code = _lib.DT_E4M3
        xs8, xs32 = _u8(x_sc8).contiguous(), x_sc32.contiguous().float()
        xin = _u8(x)
    elif x.dtype == torch.bfloat16 and x_sc8 is not None and x_sc32 is not None:
        code = _lib.DT_BF16
        xs8, xs32 = _u8(x_sc8).contiguous(), x_sc32.contiguous().float()
        xin = x
    else:
        if x_sc8 is not None or x_sc32 is not None:
            raise ValueError("input scales apply to an fp8 payload or a bf16 cotangent only")
        code = _dtype_code(x.dtype if x.dtype in (torch.float32, torch.bfloat16) else torch.float32)
        xin = x if x.dtype in (torch.float32, torch.bfloat16) else x.float()
        xs8 = xs32 = None
    if not xin.is_contiguous() or not _aligned(xin, 16):
        xin = xin.contiguous() if not xin.is_contiguous() else xin.clone()
    _, K, M = group_layout(T, C, (128, 1))
    qshape = lead + ((T, C) if rows else (C, T))
    if out is None:
        xt = torch.empty(qshape, dtype=torch.uint8, device=x.device)
        sc8 = torch.empty(lead + (M, K), dtype=torch.uint8, device=x.device)
        sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=x.device)
    else:
        _check_out(out, [(qshape, 1), (lead + (M, K), 1), (lead + (M, 1, 1), 4)], name)
        xt, sc8, sc32 = _u8(out[0]), _u8(out[1]), out[2]
    lib = _lib.load()
    fn = lib.pratchya_quantize_128x1 if rows else lib.pratchya_quantize_t128
    _lib.check(fn(_ptr(xin), code, _ptr(xs8) if xs8 is not None else None,
                  _ptr(xs32) if xs32 is not None else None,
                  S, T, C, _ptr(xt), _ptr(sc8), _ptr(sc32), _stream(xin)), name)
    return xt.view(E4M3), sc8.view(E8M0), sc32


def dequantize(x_fp8: torch.Tensor, sc_fp8: torch.Tensor, sc_fp32: torch.Tensor,
               dtype: torch.dtype, tgrid) -> torch.Tensor:
    """``(f32(x8) * (f32(e<<23) * G)) / 128`` cast to ``dtype``
    (pratchya/_qualia/_qarr.py:541-569)."""
    _require_gpu(x_fp8, sc_fp8, sc_fp32)
    a, b = int(tgrid[0]), int(tgrid[1])
    S, H, W = slices_hw(x_fp8.shape)
    out_dtype = dtype if dtype in (torch.float32, torch.bfloat16) else torch.float32
    x8 = x_fp8.contiguous()
    sc8 = sc_fp8.contiguous()
    sc32 = sc_fp32.contiguous().float()
    out = torch.empty(x_fp8.shape, dtype=out_dtype, device=x_fp8.device)
    lib = _lib.load()
    _lib.check(lib.pratchya_dequantize(_ptr(x8), _ptr(sc8), _ptr(sc32), S, H, W, a, b, _ptr(out),
                                       _dtype_code(out_dtype), _stream(x8)), "dequantize")
    return out if out_dtype == dtype else out.to(dtype)


def gather_dequantize(x_fp8: torch.Tensor, sc_fp8: torch.Tensor, sc_fp32: torch.Tensor, tgrid,
                      idx: torch.Tensor, dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """``dequantize_impl(x)[idx]`` for a 2-D quantized table and an integer index
    array of any shape (pratchya/_qualia/_qarr.py:263-284 without the full
    dequantization): returns ``idx.shape + (W,)`` in ``dtype``.  Negative
    indices count from the end; indices are clamped to the table."""
    _require_gpu(x_fp8, sc_fp8, sc_fp32, idx)
    if x_fp8.dim() != 2:
        raise ValueError("gather_dequantize needs a 2-D table")
    if dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"gather_dequantize: output dtype {dtype} is not float32 or bfloat16")
    H, W = int(x_fp8.shape[0]), int(x_fp8.shape[1])
    a, b = int(tgrid[0]), int(tgrid[1])
    ids = idx.reshape(-1).to(torch.int64).contiguous()
    out = torch.empty(tuple(idx.shape) + (W,), dtype=dtype, device=x_fp8.device)
    x8 = x_fp8.contiguous()
    sc8 = sc_fp8.contiguous()
    sc32 = sc_fp32.contiguous().float()
    lib = _lib.load()
    _lib.check(lib.pratchya_gather_dequantize(_ptr(x8), _ptr(sc8), _ptr(sc32), H, W, a, b, _ptr(ids),
                                              ids.numel(), _ptr(out), _dtype_code(dtype), _stream(x8)),
               "gather_dequantize")
    return out


ELEMENTWISE_OPS = ("add", "sub", "mul", "div", "floordiv", "mod")


def elementwise(op: str, x, grid_x, y, grid_y, tgrid, out=None):
    """``QArrayImpl(op(dequantize_impl(x, f32), dequantize_impl(y, f32)), tgrid)``
    in one fused pass (pratchya/_qualia/_qarr.py:121-261, 715-720): ``x`` and
    ``y`` are quantized (payload, e8m0, f32) triples of one shape with block
    grids ``grid_x`` / ``grid_y``; ``op`` one of ELEMENTWISE_OPS (jnp's add,
    subtract, multiply, divide, floor_divide, remainder).  Returns the result's
    ``(payload, sc_fp8, sc_fp32)`` as ``quantize`` lays them out; ``out`` may
    hold preallocated buffers."""
    if op not in ELEMENTWISE_OPS:
        raise ValueError(f"elementwise: operator {op!r} is not one of {ELEMENTWISE_OPS}")
    x8, xs8, xs32 = x
    y8, ys8, ys32 = y
    _require_gpu(x8, xs8, xs32, y8, ys8, ys32)
    if tuple(x8.shape) != tuple(y8.shape):
        raise ValueError(f"elementwise: operand shapes {tuple(x8.shape)} and {tuple(y8.shape)} differ")
    a, b = int(tgrid[0]), int(tgrid[1])
    S, H, W = slices_hw(x8.shape)
    n_blk, K, M = group_layout(H, W, (a, b))
    lead = tuple(x8.shape[:-2]) if x8.dim() >= 2 else ()
    xq, yq = _u8(x8).contiguous(), _u8(y8).contiguous()
    xs8c, ys8c = _u8(xs8).contiguous(), _u8(ys8).contiguous()
    xs32c, ys32c = xs32.contiguous().float(), ys32.contiguous().float()
    if out is None:
        q = torch.empty(x8.shape, dtype=torch.uint8, device=x8.device)
        sc8 = torch.empty(lead + (M, K), dtype=torch.uint8, device=x8.device)
        sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=x8.device)
    else:
        _check_out(out, [(x8.shape, 1), (lead + (M, K), 1), (lead + (M, 1, 1), 4)], "elementwise")
        q, sc8, sc32 = _u8(out[0]), _u8(out[1]), out[2]
    (xa, xb), (ya, yb) = (int(v) for v in grid_x), (int(v) for v in grid_y)
    lib = _lib.load()
    ws_bytes = _ws_bytes("pratchya_elementwise_workspace_bytes", S, H, W, xa, xb, ya, yb, a, b)
    if ws_bytes == 0 and not (_aligned(xq, 16) and _aligned(yq, 16) and _aligned(q, 16)):
        ws_bytes = S * n_blk * 4          # unaligned payloads take the general path
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=x8.device) if ws_bytes else None
    _lib.check(lib.pratchya_elementwise(ELEMENTWISE_OPS.index(op), _ptr(xq), _ptr(xs8c), _ptr(xs32c), xa, xb,
                                        _ptr(yq), _ptr(ys8c), _ptr(ys32c), ya, yb, S, H, W, a, b, _ptr(q),
                                        _ptr(sc8), _ptr(sc32), _ptr(ws) if ws is not None else None, ws_bytes,
                                        _stream(xq)), "elementwise")
    return q.view(E4M3), sc8.view(E8M0), sc32


def gather_quantize(x_fp8: torch.Tensor, sc_fp8: torch.Tensor, sc_fp32: torch.Tensor, tgrid, idx: torch.Tensor,
                    out_grid):
    """``quantize_impl(dequantize_impl(x)[idx], out_grid)`` for a 2-D quantized
    table and an integer index array of any shape, in one fused pass
    (pratchya/_qualia/_qarr.py:263-284 then 458-506): returns the
    ``(payload, sc_fp8, sc_fp32)`` of ``idx.shape + (W,)`` as ``quantize``
    lays them out."""
    _require_gpu(x_fp8, sc_fp8, sc_fp32, idx)
    if x_fp8.dim() != 2:
        raise ValueError("gather_quantize needs a 2-D table")
    H, W = int(x_fp8.shape[0]), int(x_fp8.shape[1])
    shape = tuple(idx.shape) + (W,)
    S, T, Wd = slices_hw(shape)
    a, b = int(out_grid[0]), int(out_grid[1])
    n_blk, K, M = group_layout(T, Wd, (a, b))
    lead = shape[:-2] if len(shape) >= 2 else ()
    ids = idx.reshape(-1).to(torch.int64).contiguous()
    q = torch.empty(shape, dtype=torch.uint8, device=x_fp8.device)
    sc8 = torch.empty(lead + (M, K), dtype=torch.uint8, device=x_fp8.device)
    sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=x_fp8.device)
    ws_bytes = S * n_blk * 4
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=x_fp8.device)
    x8 = _u8(x_fp8).contiguous()
    lib = _lib.load()
    _lib.check(lib.pratchya_gather_quantize(_ptr(x8), _ptr(_u8(sc_fp8).contiguous()), _ptr(sc_fp32.contiguous().float()),
                                            H, W, int(tgrid[0]), int(tgrid[1]), _ptr(ids), S, T, a, b, _ptr(q),
                                            _ptr(sc8), _ptr(sc32), _ptr(ws), ws_bytes, _stream(x8)),
               "gather_quantize")
    return q.view(E4M3), sc8.view(E8M0), sc32


def dequantize_bwd(g: torch.Tensor, sc_fp8: torch.Tensor, sc_fp32: torch.Tensor, tgrid) -> torch.Tensor:
    """Cotangent of the payload: ``(g * (f32(e<<23) * G) / 128).astype(g.dtype)``
    (pratchya/_qualia/_qarr.py:575-601)."""
    _require_gpu(g, sc_fp8, sc_fp32)
    a, b = int(tgrid[0]), int(tgrid[1])
    S, H, W = slices_hw(g.shape)
    orig = g.dtype
    gg = g if g.dtype in (torch.float32, torch.bfloat16) else g.float()
    gg = gg.contiguous()
    sc8 = sc_fp8.contiguous()
    sc32 = sc_fp32.contiguous().float()
    out = torch.empty(gg.shape, dtype=gg.dtype, device=g.device)
    lib = _lib.load()
    _lib.check(lib.pratchya_dequantize_bwd(_ptr(gg), _dtype_code(gg.dtype), _ptr(sc8), _ptr(sc32),
                                           S, H, W, a, b, _ptr(out), _stream(gg)), "dequantize_bwd")
    return out if out.dtype == orig else out.to(orig)


def debug_bf16_to_e4m3(bits: torch.Tensor, mode: int) -> torch.Tensor:
    """Run the kernels' bf16 -> e4m3fn conversion (mode 0 software, 1 gfx950
    instructions) over uint16/int16 bf16 bit patterns."""
    _require_gpu(bits)
    bits = bits.contiguous()
    out = torch.empty(bits.shape, dtype=torch.uint8, device=bits.device)
    _lib.check(_lib.load().pratchya_debug_bf16_to_e4m3(_ptr(bits), _ptr(out), bits.numel(), mode,
                                                       _stream(bits)), "debug_bf16_to_e4m3")
    return out


def debug_f32_to_bf16(x: torch.Tensor, mode: int) -> torch.Tensor:
    """Run the kernels' f32 -> bf16 rounding (mode 0 software, 1 gfx950)."""
    _require_gpu(x)
    x = x.contiguous().float()
    out = torch.empty(x.shape, dtype=torch.int16, device=x.device)
    _lib.check(_lib.load().pratchya_debug_f32_to_bf16(_ptr(x), _ptr(out), x.numel(), mode,
                                                      _stream(x)), "debug_f32_to_bf16")
    return out


# --------------------------------------------------------------------------
# Block-scaled FP8 GEMM operands
# --------------------------------------------------------------------------
class Operand:
    """An FP8 GEMM operand in the K-contiguous layout the GEMM reads.

    ``payload``: e4m3fn/uint8 [rows, K]; ``sc8``/``sc32``: the quantizer's
    scale arrays; ``desc``: (rdiv, sr, sk, kg) addressing the block of
    (row, 128-wide K block kb) as (row // rdiv) * sr + kb * sk, its group as
    block // kg.
    """

    __slots__ = ("payload", "sc8", "sc32", "desc", "k_major")

    def __init__(self, payload, sc8, sc32, desc, k_major=False):
        self.payload = payload
        self.sc8 = sc8
        self.sc32 = sc32
        self.desc = tuple(int(v) for v in desc)
        self.k_major = bool(k_major)      # payload [K, rows] instead of [rows, K]

    @property
    def rows(self) -> int:
        return int(self.payload.shape[1 if self.k_major else 0])

    @property
    def k(self) -> int:
        return int(self.payload.shape[0 if self.k_major else 1])


def operand_rows(x8: torch.Tensor, sc8: torch.Tensor, sc32: torch.Tensor, tgrid) -> Operand:
    """Operand from a 2-D tensor quantized as [rows, K] with tgrid (a, 128)
    (activations (1,128), dY, weights used as W[k_out, n] in dgrad)."""
    a, b = int(tgrid[0]), int(tgrid[1])
    if b != 128 or x8.dim() != 2:
        raise ValueError(f"operand_rows needs a 2-D payload quantized with tgrid (a, 128), got {tgrid}")
    R, K = x8.shape
    _, kg, _ = group_layout(R, K, (a, b))
    return Operand(x8, sc8, sc32, (a, K // 128, 1, kg))


def operand_transposed(x8: torch.Tensor, sc8: torch.Tensor, sc32: torch.Tensor, tgrid,
                       payload_t: torch.Tensor = None) -> Operand:
    """Operand from a 2-D tensor quantized as [K, rows] with tgrid (128, b) and
    contracted over its first axis (weights W[K, N] in the forward; (128,1)
    token-axis quantized A and dY in wgrad).  The payload is transposed to
    [rows, K] (or ``payload_t`` is used if the caller already holds it)."""
    a, b = int(tgrid[0]), int(tgrid[1])
    if a != 128 or x8.dim() != 2:
        raise ValueError(f"operand_transposed needs a 2-D payload quantized with tgrid (128, b), got {tgrid}")
    K, R = x8.shape
    _, kg, _ = group_layout(K, R, (a, b))
    pt = transpose_u8(x8) if payload_t is None else payload_t
    return Operand(pt, sc8, sc32, (b, 1, R // b, kg))


def operand_t128(xt8: torch.Tensor, sc8: torch.Tensor, sc32: torch.Tensor) -> Operand:
    """Operand from ``quantize_t128`` of a 2-D [T, C] tensor: rows are the C
    channels, the contraction runs over the T tokens (wgrad)."""
    if xt8.dim() != 2:
        raise ValueError("operand_t128 needs the payload of a 2-D tensor")
    C, T = xt8.shape
    return Operand(xt8, sc8, sc32, (1, 1, C, 8))


def operand_k128(x8: torch.Tensor, sc8: torch.Tensor, sc32: torch.Tensor) -> Operand:
    """Operand from a 2-D [T, C] tensor quantized with tgrid (128, 1) in its own
    layout (``quantize(x, (128, 1))``): rows are the C channels, the
    contraction runs over the T tokens, and the payload is read K-major."""
    if x8.dim() != 2:
        raise ValueError("operand_k128 needs the payload of a 2-D tensor")
    T, C = x8.shape
    return Operand(x8, sc8, sc32, (1, 1, C, 8), k_major=True)


def transpose_u8(x8: torch.Tensor) -> torch.Tensor:
    """[rows, cols] fp8 payload -> [cols, rows] (same dtype)."""
    _require_gpu(x8)
    src = _u8(x8).contiguous()
    R, C = src.shape
    out = torch.empty((C, R), dtype=torch.uint8, device=src.device)
    _lib.check(_lib.load().pratchya_transpose_u8(_ptr(src), R, C, _ptr(out), _stream(src)), "transpose")
    return out.view(x8.dtype) if x8.dtype != torch.uint8 else out


GEMM_TILE_ROWS = 256


def _tile_readable(p: torch.Tensor) -> torch.Tensor:
    """A [rows, K] payload whose buffer is readable for at least
    GEMM_TILE_ROWS rows: the kernel reads an operand of fewer rows as one full
    tile (rows beyond ``rows`` feed only outputs that are not stored).  A
    payload whose storage already extends that far is used in place; a
    shorter one is copied into a zero-padded buffer."""
    rows, K = int(p.shape[0]), int(p.shape[1])
    if rows >= GEMM_TILE_ROWS:
        return p
    avail = p.untyped_storage().nbytes() - p.storage_offset() * p.element_size()
    if avail >= GEMM_TILE_ROWS * K * p.element_size():
        return p
    padded = torch.zeros((GEMM_TILE_ROWS, K), dtype=p.dtype, device=p.device)
    padded[:rows].copy_(p)
    return padded[:rows]


def _aligned_payload(p: torch.Tensor) -> torch.Tensor:
    """A contiguous [rows, K] payload for the 128-row-tile kernels, which read no
    row past the last but whole 16-byte chunks: a misaligned one that
    _tile_readable copies for the 256x256 kernel is copied alike."""
    p = p.contiguous()
    return p if _aligned(p, 16) else _tile_readable(_u8(p))


def _word_readable(e8: torch.Tensor) -> torch.Tensor:
    """An e8m0 array readable up to the next multiple of 4 bytes (the GEMM
    reads each byte as the aligned word that holds it): used in place when its
    storage extends that far, else copied into a padded buffer."""
    n = e8.numel()
    need = (n + 3) & ~3
    avail = e8.untyped_storage().nbytes() - e8.storage_offset()
    if avail >= need:
        return e8
    padded = torch.zeros(need, dtype=torch.uint8, device=e8.device)
    padded[:n].copy_(e8.reshape(-1))
    return padded[:n]


def gemm_nt(a: Operand, b: Operand, out_dtype: torch.dtype = torch.bfloat16,
            out: torch.Tensor = None, few: bool = False) -> torch.Tensor:
    """C[M, N] = dequant(a) @ dequant(b)^T on the FP8 MFMA kernel (any M, N;
    K a multiple of 128).  ``few``: a product of few tiles may run as gemm_t128,
    whose sums are in another order."""
    _require_gpu(a.payload, b.payload)
    if a.k != b.k:
        raise ValueError(f"contraction mismatch: {a.k} vs {b.k}")
    M, N, K = a.rows, b.rows, a.k
    if few and out is None and not a.k_major and prefers_t128(M, a.desc[3], b):
        return gemm_t128(a, b, out_dtype)
    if a.k_major or b.k_major:
        if not (a.k_major and b.k_major):
            raise PratchyaUnsupported("gemm_nt: K-major FP8 operands are supported as a pair")
        ap, bp = _u8(a.payload).contiguous(), _u8(b.payload).contiguous()
    else:
        ap, bp = _tile_readable(_u8(a.payload).contiguous()), _tile_readable(_u8(b.payload).contiguous())
    as8, bs8 = _word_readable(_u8(a.sc8).contiguous()), _word_readable(_u8(b.sc8).contiguous())
    as32, bs32 = a.sc32.contiguous().float(), b.sc32.contiguous().float()
    if out is None:
        out = torch.empty((M, N), dtype=out_dtype, device=ap.device)
    lib = _lib.load()
    if a.k_major:
        _lib.check(lib.pratchya_gemm_bs_kmajor(_ptr(ap), M, _ptr(as8), _ptr(as32), *a.desc,
                                               _ptr(bp), N, _ptr(bs8), _ptr(bs32), *b.desc,
                                               M, N, K, _ptr(out), out.stride(0), _dtype_code(out.dtype),
                                               _stream(ap)), "gemm_kmajor")
        return out
    _lib.check(lib.pratchya_gemm_bs_nt(_ptr(ap), K, _ptr(as8), _ptr(as32), *a.desc,
                                       _ptr(bp), K, _ptr(bs8), _ptr(bs32), *b.desc,
                                       M, N, K, _ptr(out), out.stride(0), _dtype_code(out.dtype),
                                       _stream(ap)), "gemm")
    return out


def gemm_nt_blockmax(a: Operand, b: Operand) -> Tuple[torch.Tensor, torch.Tensor]:
    """``gemm_nt(a, b, float32)`` plus the 128 x 128 block maxima of the
    product (max |c| as f32 bits, [M / 128, N / 128] int32) from the GEMM's
    epilogue: the first pass of the product's (128, 128) requantization.
    Operands K-contiguous or both K-major; M and N multiples of 128
    (``PratchyaUnsupported`` otherwise)."""
    _require_gpu(a.payload, b.payload)
    if a.k != b.k:
        raise ValueError(f"contraction mismatch: {a.k} vs {b.k}")
    M, N, K = a.rows, b.rows, a.k
    if a.k_major != b.k_major:
        raise PratchyaUnsupported("gemm_blockmax: K-major FP8 operands are supported as a pair")
    if a.k_major:
        ap, bp = _u8(a.payload).contiguous(), _u8(b.payload).contiguous()
    else:
        ap, bp = _tile_readable(_u8(a.payload).contiguous()), _tile_readable(_u8(b.payload).contiguous())
    as8, bs8 = _word_readable(_u8(a.sc8).contiguous()), _word_readable(_u8(b.sc8).contiguous())
    as32, bs32 = a.sc32.contiguous().float(), b.sc32.contiguous().float()
    out = torch.empty((M, N), dtype=torch.float32, device=ap.device)
    bmax = torch.empty((max(M // 128, 1), max(N // 128, 1)), dtype=torch.int32, device=ap.device)
    lda, ldb = (M, N) if a.k_major else (K, K)
    _lib.check(_lib.load().pratchya_gemm_bs_blockmax(_ptr(ap), lda, _ptr(as8), _ptr(as32), *a.desc,
                                                     _ptr(bp), ldb, _ptr(bs8), _ptr(bs32), *b.desc,
                                                     M, N, K, 1 if a.k_major else 0, _ptr(out), N, _ptr(bmax),
                                                     _stream(ap)), "gemm_blockmax")
    return out, bmax


def quantize_dequantize_premax(x: torch.Tensor, block_max: torch.Tensor, tgrid, dtype: torch.dtype,
                               fix_nan: bool = False):
    """``quantize_dequantize(x, tgrid, dtype, fix_nan)`` of an f32 ``x`` whose
    block maxima ``block_max`` (f32 bits of max |x| per block, as
    ``gemm_nt_blockmax`` returns them) are already known: only the group
    scales and the cast run.  Returns ``(y, sc_fp8, sc_fp32)``."""
    _require_gpu(x, block_max)
    if x.dtype != torch.float32:
        raise ValueError("quantize_dequantize_premax: x must be float32")
    if dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"quantize_dequantize_premax: output dtype {dtype} is not float32 or bfloat16")
    a, b = int(tgrid[0]), int(tgrid[1])
    S, H, W = slices_hw(x.shape)
    n_blk, K, M = group_layout(H, W, (a, b))
    if block_max.numel() != S * n_blk or block_max.dtype not in (torch.int32, torch.uint32):
        raise ValueError(f"quantize_dequantize_premax: block_max must hold {S * n_blk} 32-bit maxima")
    lead = tuple(x.shape[:-2]) if x.dim() >= 2 else ()
    x = x.contiguous()
    bm = block_max.contiguous()
    y = torch.empty(x.shape, dtype=dtype, device=x.device)
    sc8 = torch.empty(lead + (M, K), dtype=torch.uint8, device=x.device)
    sc32 = torch.empty(lead + (M, 1, 1), dtype=torch.float32, device=x.device)
    _lib.check(_lib.load().pratchya_quantize_dequantize_premax(
        _ptr(x), S, H, W, a, b, _ptr(bm), _ptr(y), _dtype_code(dtype), 1 if fix_nan else 0, _ptr(sc8), _ptr(sc32),
        _stream(x)), "quantize_dequantize_premax")
    return y, sc8.view(E8M0), sc32


def few_tiles(M: int, N: int) -> bool:
    """Whether a bf16 product leaves half of the chip idle on 256x256 tiles: it
    then runs on 128x128 ones with its K steps split (gemm_planes).  Measured
    (us, 256x256 / 128x128): [1024, 6144] . [6144, 1024] 124 / 27, [2048, 12288]
    . [12288, 2048] (64 tiles) 254 / 104, [4096, 2048] . [2048, 2048] (128) 50 /
    37, [3000, 3072] . [3072, 3000] (144) 75 / 78, [4096, 2048] . [2048, 4096]
    (256) 64 / 70."""
    return 0 < -(-M // GEMM_TILE_ROWS) * -(-N // GEMM_TILE_ROWS) <= 128


def gemm_bf16_nt(a: torch.Tensor, b: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """C[M, N] = a @ b^T for bf16 ``a`` [M, K] and ``b`` [N, K] with f32
    accumulation, rounded once to ``out_dtype``: the bf16 dots of
    newton_schulz (pratchya/_nnx_impl/_optimizer.py:20-22) on the MFMA kernel.
    K must be a multiple of 64 (``PratchyaUnsupported`` otherwise)."""
    _require_gpu(a, b)
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16 or a.dim() != 2 or b.dim() != 2:
        raise ValueError("gemm_bf16_nt: a and b must be 2-D bfloat16")
    if a.shape[1] != b.shape[1]:
        raise ValueError(f"contraction mismatch: {a.shape[1]} vs {b.shape[1]}")
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"gemm_bf16_nt: output dtype {out_dtype} is not float32 or bfloat16")
    M, N, Kd = int(a.shape[0]), int(b.shape[0]), int(a.shape[1])
    ap, bp = _tile_readable(a.contiguous()), _tile_readable(b.contiguous())
    out = torch.empty((M, N), dtype=out_dtype, device=ap.device)
    _lib.check(_lib.load().pratchya_gemm_bf16_nt(_ptr(ap), Kd, _ptr(bp), Kd, M, N, Kd, _ptr(out), N,
                                                 _dtype_code(out_dtype), _stream(ap)), "gemm_bf16")
    return out


def prefers_t128(M: int, a_kg: int, b: Operand) -> bool:
    """Whether an FP8 product of M rows (a_kg blocks per group) with ``b`` is one
    that gemm_t128 takes and runs faster than on the persistent
    256x256 kernel, which takes about 10 us and 10 us per 1024 of K however few
    tiles there are.  Measured (us, with the output's requantization, 256x256 /
    t128): 4 x [4096, 4096] 62.6 / 11.8; 512 x [4096, 4096] 60 / 33; 1000 x
    [2176, 2944] 50 / 34; 2048 x [2048, 2048] (64 tiles) 41 / 37; 4096 x [1024,
    1024] (64 tiles) 31 / 32; 2048 x [4096, 4096] (128 tiles) 60 / 63."""
    N, Kd = b.rows, b.k
    tiles = -(-M // GEMM_TILE_ROWS) * -(-N // GEMM_TILE_ROWS)
    if 0 in (M, N, Kd) or not (M <= 32 or (tiles <= 64 and Kd >= 32 * tiles)) or b.k_major or N % 8:
        return False
    brd, bsr, bsk, bkg = b.desc
    rows4 = brd % 4 == 0 or (brd == 1 and bsr > 0 and bkg % (4 * bsr) == 0 and bsk % (4 * bsr) == 0)
    return rows4 and a_kg & (a_kg - 1) == 0 and bkg & (bkg - 1) == 0


def gemm_t128(a: Operand, b: Operand, out_dtype: torch.dtype = torch.float32) -> torch.Tensor:
    """``gemm_nt(a, b, out_dtype)`` on 128-row tiles with the K steps split over
    workgroups (pratchya_gemm_bs_t128): for products of few 256 x 256 tiles.
    ``PratchyaUnsupported`` for K-major operands and scale layouts it does not
    take."""
    _require_gpu(a.payload, b.payload)
    if a.k != b.k:
        raise ValueError(f"contraction mismatch: {a.k} vs {b.k}")
    if a.k_major or b.k_major:
        raise PratchyaUnsupported("gemm_t128: K-contiguous operands only")
    M, N, Kd = a.rows, b.rows, a.k
    ap, bp = _aligned_payload(a.payload), _aligned_payload(b.payload)
    as8, bs8 = a.sc8.contiguous(), b.sc8.contiguous()
    as32, bs32 = a.sc32.contiguous().float(), b.sc32.contiguous().float()
    lib = _lib.load()
    c = torch.empty((M, N), dtype=out_dtype, device=ap.device)
    ws_bytes = _ws_bytes("pratchya_gemm_t128_workspace_bytes", M, N, Kd // 128, 1)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=ap.device) if ws_bytes else None
    _lib.check(lib.pratchya_gemm_bs_t128(_ptr(ap), Kd, _ptr(as8), _ptr(as32), *a.desc, _ptr(bp), Kd, _ptr(bs8),
                                         _ptr(bs32), *b.desc, M, N, Kd, _ptr(c), N, _dtype_code(out_dtype),
                                         _ptr(ws) if ws is not None else None, ws_bytes, _stream(ap)), "gemm_t128")
    return c


# bf16 piece pairs of an f32 product (see pratchya_split_pack_bf16): the six
# pairs whose weight is at least 2^-24 of the leading product
_F32_PAIRS = ((0, 0), (0, 1), (1, 0), (0, 2), (1, 1), (2, 0))


def _split_pack(src: torch.Tensor, transpose: bool, planes, kp: int, out_rows_min: int = 0) -> torch.Tensor:
    """bf16 [max(out_rows, out_rows_min), len(planes) * kp] operand of the
    bf16 GEMM: segment s holds piece planes[s] of each source row (or column,
    ``transpose``); rows beyond the source's are zero."""
    src = src.contiguous()
    R, C = int(src.shape[0]), int(src.shape[1])
    out_rows = C if transpose else R
    rows = max(out_rows, out_rows_min)
    dst = (torch.zeros if rows > out_rows else torch.empty)((rows, len(planes) * kp), dtype=torch.bfloat16,
                                                             device=src.device)
    pl = (ctypes.c_int * len(planes))(*planes)
    _lib.check(_lib.load().pratchya_split_pack_bf16(_ptr(src), _dtype_code(src.dtype), R, C, C, 1 if transpose else 0,
                                                    len(planes), pl, _ptr(dst), len(planes) * kp, kp, _stream(src)),
               "split_pack")
    return dst


# The pairs of planes (PLANE_SPLIT4) of a product of two f32 operands: the six
# whose weight is at least 2^-24 of the leading product (_F32_PAIRS), a
# non-finite value in the first only
F32_PLANE_PAIRS = ((0, 0), (3, 1), (1, 3), (3, 2), (1, 1), (2, 3))


def _matmul_f32_planes(a, b, a_t, b_t, M, N, Kd):
    """matmul_f32 on 128x128 tiles, the operands' planes in their own layouts
    (each written once, no transposed copies)."""
    # what planes() and gemm_planes() take: whole chunks of 8 of every plane's
    # rows (4 of the output's), K a multiple of 64 unless both are padded along it
    if a.dtype == torch.bfloat16 or ((not a_t or b_t) and Kd % 64) or (a_t and M % 8) or N % (4 if b_t else 8):
        raise PratchyaUnsupported("matmul_f32: packed pieces")
    if b.dtype == torch.bfloat16:
        flags = torch.zeros(2, dtype=torch.int32, device=a.device)
        pb = planes(PLANE_BF16, b, None, None, None, flags, pad=1 if b_t else 64)
        pa = planes(PLANE_SPLIT4, a, None, None, None, pad=64 if a_t else 1)
        return gemm_planes(pa, pb, ((0, 0), (1, 0), (2, 0)), a_t, b_alt=(0, 1, 1), flags=flags, b_k_major=not b_t,
                           short=3)
    pa = planes(PLANE_SPLIT4, a, None, None, None, pad=64 if a_t else 1)
    same = b is a and a_t == (not b_t)
    pb = pa if same else planes(PLANE_SPLIT4, b, None, None, None, pad=1 if b_t else 64)
    return gemm_planes(pa, pb, F32_PLANE_PAIRS, a_t, b_k_major=not b_t)


def _packed_on_few_tiles(M: int, N: int, Kd: int) -> bool:
    """Whether a product of packed pieces (Kd columns in all) takes 128x128 tiles:
    few_tiles, where those are the faster ones also for a short K.  Measured (us,
    whole products of bf16 operands, 256x256 / 128x128 tiles): [2048, 512] . [512,
    2048] 31 / 41, K 768 39 / 42, K 1024 47 / 44 (from 512 on K is split in two
    there, which pays from 1024); [4096, 256] . [256, 2048] 26 / 30, K 512 36 /
    35 (128 tiles: K is not split).  Fewer than 256 rows or columns would have
    to be padded for the 256x256 kernel."""
    if not few_tiles(M, N) or min(M, N) < GEMM_TILE_ROWS:
        return few_tiles(M, N)
    if -(-M // GEMM_TILE_ROWS) * -(-N // GEMM_TILE_ROWS) > 64:
        return Kd >= 512
    return Kd < 512 or Kd >= 1024


def matmul_f32(a: torch.Tensor, b: torch.Tensor, a_t: bool = False, b_t: bool = False) -> torch.Tensor:
    """f32 ``op(a) @ op(b)`` for 2-D f32 / bf16 tensors on the bf16 MFMA
    kernel: ``op(a)`` is ``a`` [M, K] (``a_t``: ``a`` is [K, M] and is used
    transposed), ``op(b)`` is ``b`` [K, N] (``b_t``: ``b`` is [N, K]).  Each
    f32 operand is split into three exact bf16 pieces and the piece products
    of weight >= 2^-24 run as one bf16 GEMM along a K six times as long (three
    times for a bf16 operand, once for two): f32 products to f32 accuracy, up
    to summation order (the f32 dots of pratchya/_qualia/_qarr.py:645-712,
    :618-622)."""
    _require_gpu(a, b)
    if a.dim() != 2 or b.dim() != 2:
        raise ValueError("matmul_f32: 2-D operands expected")
    for t in (a, b):
        if t.dtype not in (torch.float32, torch.bfloat16):
            raise TypeError(f"matmul_f32: unsupported dtype {t.dtype}")
    M, Kd = (int(a.shape[1]), int(a.shape[0])) if a_t else (int(a.shape[0]), int(a.shape[1]))
    Kb, N = (int(b.shape[1]), int(b.shape[0])) if b_t else (int(b.shape[0]), int(b.shape[1]))
    if Kd != Kb:
        raise ValueError(f"contraction mismatch: {Kd} vs {Kb}")
    if M == 0 or N == 0:
        return torch.empty((M, N), dtype=torch.float32, device=a.device)
    if Kd == 0:
        return torch.zeros((M, N), dtype=torch.float32, device=a.device)
    # (a bf16 b of a short K: two packs of it cost the host and the chip no more
    # than a flag word, two passes of planes and a pass that repairs them:
    # [256, 256] . [256, 256] 34 us packed, 38 as planes; K 512 48 / 42)
    if few_tiles(M, N) and M > 32 and (b.dtype == torch.float32 or Kd >= 384):
        try:
            return _matmul_f32_planes(a, b, a_t, b_t, M, N, Kd)
        except PratchyaUnsupported:
            pass
    na = 1 if a.dtype == torch.bfloat16 else 3
    nb = 1 if b.dtype == torch.bfloat16 else 3
    pairs = [(i, j) for i, j in _F32_PAIRS if i < na and j < nb]
    # a non-finite value takes part only in the (0, 0) pair (plane 3: piece 0
    # with non-finite values as 0)
    a_planes = [3 if (i == 0 and j > 0) else i for i, j in pairs]
    b_planes = [3 if (j == 0 and i > 0) else j for i, j in pairs]
    kp = (Kd + 63) // 64 * 64
    # the GEMM's operand rows: A = op(a) rows, B = op(b) columns (N-major);
    # an N below one tile is padded to a multiple of 4 with zero rows
    n_rows = N if N >= GEMM_TILE_ROWS else (N + 3) // 4 * 4
    A = _split_pack(a, a_t, a_planes, kp)
    B = _split_pack(b, not b_t, b_planes, kp, n_rows)
    c = None
    if _packed_on_few_tiles(M, n_rows, len(pairs) * kp):
        try:
            c = gemm_planes(A[None], B[None], [(0, 0)], False)
        except PratchyaUnsupported:      # few rows of more than 2^24 columns
            pass
    if c is None:
        c = gemm_bf16_nt(A, B, torch.float32)
    return c if n_rows == N else c[:, :N]


# Planes of an operand of ``gemm_planes`` (pratchya_planes)
PLANE_POW2, PLANE_SPLIT3, PLANE_SPLIT4, PLANE_BF16, PLANE_SPLIT4Q = 0, 1, 2, 3, 4
_PLANE_COUNT = {PLANE_POW2: 1, PLANE_SPLIT3: 3, PLANE_SPLIT4: 4, PLANE_BF16: 2, PLANE_SPLIT4Q: 4}


def planes(mode: int, src: torch.Tensor, sc8, sc32, tgrid, flags=None, pad: int = 1) -> torch.Tensor:
    """The bf16 planes [planes, rows padded to ``pad``, W] of a 2-D payload with
    its scales (PLANE_POW2, PLANE_SPLIT3, PLANE_SPLIT4Q), an f32 matrix (PLANE_SPLIT4) or a bf16
    one (PLANE_BF16), the last two taken through dequantize_impl_bwd with the
    scales if given.  ``flags``: two zeroed uint32 words that say which planes
    the product needs (PLANE_POW2: if given, a second plane as PLANE_BF16's).  ``PratchyaUnsupported`` for layouts it does not take."""
    _require_gpu(src)
    T, W = int(src.shape[0]), int(src.shape[1])
    Tp = -(-T // pad) * pad
    x = src.contiguous()
    if not _aligned(x, 16):
        x = x.clone()
    a, b = (int(tgrid[0]), int(tgrid[1])) if sc8 is not None else (1, 8)
    e8 = sc8.contiguous() if sc8 is not None else None
    g32 = sc32.contiguous().float() if sc8 is not None else None
    count = 2 if mode == PLANE_POW2 and flags is not None else _PLANE_COUNT[mode]
    out = torch.empty((count, Tp, W), dtype=torch.bfloat16, device=src.device)
    _lib.check(_lib.load().pratchya_planes(mode, _ptr(x), _ptr(e8) if e8 is not None else None,
                                           _ptr(g32) if g32 is not None else None, T, W, a, b, Tp, _ptr(out),
                                           _ptr(flags) if flags is not None else None, _stream(x)), "planes")
    return out


@functools.lru_cache(maxsize=64)
def _nibbles(seq) -> int:
    return sum(int(v) << (4 * i) for i, v in enumerate(seq))


def gemm_planes(a: torch.Tensor, b: torch.Tensor, pairs, k_major: bool, out_dtype=torch.float32, short: int = 0,
                b_alt=None, flags=None, units=None, x=None, b_k_major=None) -> torch.Tensor:
    """``sum over (i, j) in pairs of op(a[i]) @ op(b[j])^T`` for bf16 planes
    ``a`` [planes, M, K] and ``b`` [planes, N, K] (``k_major``: [planes, K, M] and
    [planes, K, N]; ``b_k_major``: b's layout where it differs) with f32
    accumulation.  ``short`` pairs are enough where flags[0] is 0; ``b_alt`` are
    b's planes where flags[1] is not.  ``units``: ``(sc32, tgrid, blocks per
    group)`` of the payload that b is the power-of-two plane of.  ``x`` [M, N]
    bf16: the result is ``1.5 x - 0.5 product`` in bf16."""
    _require_gpu(a, b)
    return _gemm_planes(a[None], b[None], pairs, k_major, out_dtype, short, b_alt, flags, units,
                        None if x is None else x[None], b_k_major)[0]


def gemm_planes_batch(a: torch.Tensor, b: torch.Tensor, k_major: bool, out_dtype=torch.float32, x=None,
                      b_k_major=None) -> torch.Tensor:
    """``gemm_planes`` of each slice's single planes: a [batch, M, K], b [batch,
    N, K], x [batch, M, N]."""
    _require_gpu(a, b)
    return _gemm_planes(a[:, None], b[:, None], ((0, 0),), k_major, out_dtype, x=x, b_k_major=b_k_major)


def _gemm_planes(a, b, pairs, k_major, out_dtype, short=0, b_alt=None, flags=None, units=None, x=None, b_k_major=None):
    b_km = k_major if b_k_major is None else b_k_major
    L, ha, a0, a1 = a.shape
    b0, b1 = b.shape[2:]
    (M, Kd), N = ((a1, a0) if k_major else (a0, a1)), (b1 if b_km else b0)
    short = short or len(pairs)
    c = torch.empty((L, M, N), dtype=out_dtype, device=a.device)
    ws_bytes = _ws_bytes("pratchya_gemm_t128_workspace_bytes", M, N, short * (Kd // 64), L)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=a.device) if ws_bytes else None
    pa, pb = _nibbles(tuple(i for i, _ in pairs)), _nibbles(tuple(j for _, j in pairs))
    g32, brow, bcol, kg = (units[0].contiguous().float(), int(units[1][0]), int(units[1][1]), int(units[2])) \
        if units is not None else (None, 1, 1, 1)
    (sa, ta, lda, _), (sb, tb, ldb, _) = a.stride(), b.stride()
    _lib.check(_lib.load().pratchya_gemm_bf16_planes(
        _ptr(a), lda, ta, 1 if k_major else 0, ha, pa, _ptr(b), ldb, tb, 1 if b_km else 0, b.shape[1], pb,
        pb if b_alt is None else _nibbles(tuple(b_alt)), M, N, Kd, len(pairs), short,
        _ptr(flags) if flags is not None else None, _ptr(g32) if g32 is not None else None, brow, bcol, kg,
        _ptr(c), N, _dtype_code(out_dtype), _ptr(x) if x is not None else None, x.stride(1) if x is not None else 0,
        L, sa, sb, M * N, x.stride(0) if x is not None else 0, _ptr(ws) if ws is not None else None, ws_bytes,
        _stream(a)), "gemm_planes")
    return c


def gemm_fine(a: torch.Tensor, a_sc32: torch.Tensor, b: torch.Tensor, b_sc32: torch.Tensor, b_kg: int,
              blk: int) -> torch.Tensor:
    """f32 ``dequant(x) @ dequant(W)`` to f32 accuracy for x [M, K] quantized
    (1, blk) and W [K, N] quantized (blk, blk), blk 16 or 32, given as their
    power-of-two planes ``a`` and ``b`` and group maxima (W with ``b_kg`` blocks
    per group)."""
    _require_gpu(a, b)
    M, Kd, N = int(a.shape[0]), int(a.shape[1]), int(b.shape[1])
    lib = _lib.load()
    ag, bg = a_sc32.contiguous().float(), b_sc32.contiguous().float()
    if ag.numel() != M * Kd // (16 if blk == 16 else 64):
        raise PratchyaUnsupported("gemm_fine: x's groups are not one block of 16 or two of 32")
    if not _aligned(ag, 16):      # a view into a larger array: four maxima are one load
        ag = ag.clone()
    c = torch.empty((M, N), dtype=torch.float32, device=a.device)
    ws_bytes = _ws_bytes("pratchya_gemm_t128_workspace_bytes", M, N, Kd // 64, 1)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=a.device) if ws_bytes else None
    _lib.check(lib.pratchya_gemm_fine(_ptr(a), int(a.stride(0)), _ptr(ag), _ptr(b), int(b.stride(0)), _ptr(bg), b_kg, blk,
                                      M, N, Kd, _ptr(c), N, _ptr(ws) if ws is not None else None, ws_bytes, _stream(a)),
               "gemm_fine")
    return c


def transpose_b16(x: torch.Tensor) -> torch.Tensor:
    """[rows, cols] 16-bit matrix -> its transpose [cols, rows], contiguous."""
    _require_gpu(x)
    if x.dim() != 2 or x.element_size() != 2:
        raise ValueError("transpose_b16: a 2-D 16-bit tensor is required")
    src = x.contiguous()
    R, C = int(src.shape[0]), int(src.shape[1])
    out = torch.empty((C, R), dtype=x.dtype, device=src.device)
    _lib.check(_lib.load().pratchya_transpose_b16(_ptr(src), R, C, _ptr(out), _stream(src)), "transpose_b16")
    return out


def ns_normalize(g: torch.Tensor) -> torch.Tensor:
    """``g / (||g||_F + 1e-7)`` (pratchya/_nnx_impl/_optimizer.py:17) in g's
    dtype.  bf16: the roundings of the bf16 jnp expression -- the squares,
    their sum, the square root, the sum with 1e-7 and every quotient rounded
    to bf16; f32: f32 squares, sum, square root and quotients.  The sum is
    accumulated in f32 in a fixed order.  Returns a new contiguous tensor of
    g's shape."""
    _require_gpu(g)
    if g.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("ns_normalize: g must be bfloat16 or float32")
    gc = g.contiguous()
    if not _aligned(gc, 16):      # a slice of a larger array
        gc = gc.clone()
    out = torch.empty_like(gc)
    lib = _lib.load()
    ws = torch.empty(_ws_bytes("pratchya_ns_normalize_workspace_bytes"), dtype=torch.uint8, device=gc.device)
    fn = lib.pratchya_ns_normalize if g.dtype == torch.bfloat16 else lib.pratchya_ns_normalize_f32
    _lib.check(fn(_ptr(gc), _ptr(out), gc.numel(), _ptr(ws), ws.numel(), _stream(gc)), "ns_normalize")
    return out


def ns_normalize_batch(g: torch.Tensor) -> torch.Tensor:
    """``ns_normalize`` of each slice of a bf16 [batch, m, n] array (m * n a
    multiple of 8)."""
    _require_gpu(g)
    if g.dtype != torch.bfloat16 or g.dim() != 3:
        raise ValueError("ns_normalize_batch: g must be a 3-D bfloat16 array")
    gc = g.contiguous()
    if not _aligned(gc, 16):
        gc = gc.clone()
    out = torch.empty_like(gc)
    L = int(g.shape[0])
    ws = torch.empty(L * _ws_bytes("pratchya_ns_normalize_workspace_bytes"), dtype=torch.uint8, device=gc.device)
    _lib.check(_lib.load().pratchya_ns_normalize_batch(_ptr(gc), _ptr(out), gc.numel() // max(L, 1), L, _ptr(ws),
                                                       ws.numel(), _stream(gc)), "ns_normalize_batch")
    return out


# The Gram product and the requantizing GEMM exchange data between
# workgroups with bounded waits; a wait that runs out sets a status word in
# the call's workspace (and NaN in the outputs concerned) instead of hanging.
# With checks on (check_waits(True), or PRATCHYA_CHECK_WAITS=1 in the
# environment) each such call synchronizes its stream and raises
# PratchyaWaitTimeout when the word is set (not while the stream is being
# captured into a graph); either call also copies the word into a caller's
# ``status`` tensor (int32, on the device, no sync).
_CHECK_WAITS = os.environ.get("PRATCHYA_CHECK_WAITS", "0") not in ("", "0")


def check_waits(enable: bool = True) -> bool:
    """Turn the synchronous status check of the bounded waits on or off;
    returns the previous setting."""
    global _CHECK_WAITS
    prev, _CHECK_WAITS = _CHECK_WAITS, bool(enable)
    return prev


def _wait_status(ws: torch.Tensor, offset: int, status, what: str) -> None:
    word = ws[offset:offset + 4].view(torch.int32)
    if status is not None:
        if status.dtype != torch.int32 or status.device != ws.device or status.numel() < 1:
            raise ValueError(f"{what}: status must be an int32 tensor on {ws.device}")
        status.view(-1)[:1].copy_(word)
    if _CHECK_WAITS and not torch.cuda.is_current_stream_capturing() and int(word.item()) != 0:
        raise PratchyaWaitTimeout(f"{what}: a bounded wait between workgroups ran out (outputs hold NaN)")


_GRAM_WS = {}


def _gram_workspace(device: torch.device, stream) -> torch.Tensor:
    """The Gram product's workspace for ``stream``: sized once for the largest
    grid (one range per CU) and never replaced, so that a graph that captured
    a Gram call keeps a valid workspace whatever later calls need."""
    key = (device.index, stream.cuda_stream)
    ws = _GRAM_WS.get(key)
    if ws is None:
        # a shape whose grid is one range per CU: the largest workspace
        big = int(_lib.load().pratchya_gemm_bf16_gram_workspace_bytes(256 * 64, 64 * 4096))
        ws = torch.empty(big, dtype=torch.uint8, device=device)
        _GRAM_WS[key] = ws
    return ws


def gemm_bf16_gram(a: torch.Tensor, k_major: bool = False, status: torch.Tensor = None) -> torch.Tensor:
    """The symmetric bf16 product ``a @ a^T`` (f32 accumulation, rounded once
    to bf16) of a bf16 ``a`` [M, K], the Gram product of newton_schulz
    (pratchya/_nnx_impl/_optimizer.py:20-22): only the tiles on and above the
    diagonal are computed and the lower triangle is their transpose, so the
    result is exactly symmetric.  With ``k_major``, ``a`` is given as its
    [K, M] transpose and the result is ``a^T @ a`` [M, M] (the Gram product of
    a tall iterate, read without a transposed copy).  M must be a multiple of
    256 and K of 64 (``PratchyaUnsupported`` otherwise).  The partial-tile
    workspace is kept per device and stream; calls on one stream run in
    order.  ``status``: an int32 device tensor that receives the bounded
    wait's status word (0: every partial tile arrived)."""
    _require_gpu(a)
    if a.dtype != torch.bfloat16 or a.dim() != 2:
        raise ValueError("gemm_bf16_gram: a must be 2-D bfloat16")
    M, Kd = (int(a.shape[1]), int(a.shape[0])) if k_major else (int(a.shape[0]), int(a.shape[1]))
    lib = _lib.load()
    ws_bytes = _ws_bytes("pratchya_gemm_bf16_gram_workspace_bytes", M, Kd)
    if ws_bytes <= 0:
        raise PratchyaUnsupported(f"gemm_bf16_gram: M must be a multiple of 256 and K of 64 (got {M}, {Kd})")
    ap = a.contiguous()
    ws = _gram_workspace(ap.device, torch.cuda.current_stream(ap.device))
    if ws.numel() < ws_bytes:
        raise PratchyaError(f"gemm_bf16_gram: workspace of {ws.numel()} bytes, {ws_bytes} needed")
    out = torch.empty((M, M), dtype=torch.bfloat16, device=ap.device)
    _lib.check(lib.pratchya_gemm_bf16_gram(_ptr(ap), int(ap.stride(0)), M, Kd, 1 if k_major else 0, _ptr(out), M,
                                           _ptr(ws), int(ws.numel()), _stream(ap)), "gemm_bf16_gram")
    _wait_status(ws, int(lib.pratchya_gemm_bf16_gram_status_offset(M, Kd)), status, "gemm_bf16_gram")
    return out


def gemm_bf16_nt_ns(a: torch.Tensor, b: torch.Tensor, x: torch.Tensor, out: torch.Tensor = None,
                    b_k_major: bool = False) -> torch.Tensor:
    """One Newton-Schulz step ``1.5 x - 0.5 (a @ b^T)`` (pratchya/_nnx_impl/
    _optimizer.py:20-27) with the combination in the bf16 GEMM's epilogue: the
    same bits as ``ns_combine(x, gemm_bf16_nt(a, b))``.  ``a`` [M, K], ``b``
    [N, K] (with ``b_k_major``: ``b`` given as its [K, N] transpose, read
    without a transposed copy), ``x`` [M, N], all bf16; ``out`` must not
    overlap ``x``."""
    _require_gpu(a, b, x)
    if any(t.dtype != torch.bfloat16 or t.dim() != 2 for t in (a, b, x)):
        raise ValueError("gemm_bf16_nt_ns: a, b and x must be 2-D bfloat16")
    bk = int(b.shape[0]) if b_k_major else int(b.shape[1])
    if a.shape[1] != bk:
        raise ValueError(f"contraction mismatch: {a.shape[1]} vs {bk}")
    M, N, Kd = int(a.shape[0]), int(b.shape[1] if b_k_major else b.shape[0]), int(a.shape[1])
    if tuple(x.shape) != (M, N):
        raise ValueError(f"gemm_bf16_nt_ns: x is {tuple(x.shape)}, the product is {(M, N)}")
    ap = _tile_readable(a.contiguous())
    bp = b.contiguous() if b_k_major else _tile_readable(b.contiguous())
    xc = x.contiguous()
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=ap.device)
    _lib.check(_lib.load().pratchya_gemm_bf16_nt_ns(_ptr(ap), Kd, _ptr(bp), int(bp.stride(0)), 1 if b_k_major else 0,
                                                    M, N, Kd, _ptr(xc), N, _ptr(out), out.stride(0), _stream(ap)),
               "gemm_bf16_ns")
    return out


def mfma_ceiling(a: torch.Tensor, b: torch.Tensor, bf16: bool, iters: int) -> int:
    """Launch the MFMA-rate probe (``pratchya_mfma_ceiling``, a measurement aid
    with no reference counterpart) on the bytes of ``a`` and ``b`` (2-D,
    contiguous, at least 256 rows of 128 bytes); returns the launch's FLOP count
    for the caller's timing."""
    _require_gpu(a, b)
    if a.dim() != 2 or b.dim() != 2 or a.shape[0] < 256 or b.shape[0] < 256:
        raise ValueError("mfma_ceiling: operands of at least 256 rows")
    ld = int(a.stride(0)) * a.element_size()
    if int(b.stride(0)) * b.element_size() != ld:
        raise ValueError("mfma_ceiling: a and b need the same row stride")
    sink = torch.empty(1, dtype=torch.float32, device=a.device)
    flop = ctypes.c_int64(0)
    _lib.check(_lib.load().pratchya_mfma_ceiling(_ptr(a), _ptr(b), ld, 1 if bf16 else 0, int(iters), _ptr(sink),
                                                 ctypes.byref(flop), _stream(a)), "mfma_ceiling")
    return int(flop.value)


def _few_then_requantize(a: Operand, b: Operand, out_dtype, lead, scales: bool):
    """gemm_nt_q11 of a product of few tiles, as its two steps, the second of
    which stores the scales of every element (dropped without ``scales``).
    Measured (us, without scales, the epilogue's one launch / the two steps): 4 x
    [2048, 4096] 48 / 30, x [2048, 32768] 48 / 31, x [2048, 131072] 89 / 46; 1000 x
    [2048, 4096] 44 / 39; 4096 x [2048, 1024] 44 / 39."""
    lead = tuple(lead) if lead else (a.rows,)
    c = gemm_t128(a, b, torch.float32)
    y, s8, s32 = quantize_dequantize(c.view(lead + (b.rows,)), (1, 1), out_dtype)
    return (y.view(a.rows, b.rows),) + ((s8, s32) if scales else (None, None))


def gemm_t128_fq(a: Operand, b: Operand, out_dtype: torch.dtype, fix_nan: bool = False, lead=None,
                 scales: bool = True):
    """``gemm_t128(a, b, float32)`` and its requantization as gemm_nt_fq
    returns them, in two launches: the slices of K are summed as the
    requantization reads them.  N a multiple of 128 and every slice of ``lead``
    whole groups of 8 blocks (``PratchyaUnsupported`` otherwise).  ``scales``
    False: the scale arrays are not stored (None)."""
    _require_gpu(a.payload, b.payload)
    if a.k != b.k:
        raise ValueError(f"contraction mismatch: {a.k} vs {b.k}")
    M, N, Kd = a.rows, b.rows, a.k
    lead = tuple(lead) if lead else (M,)
    H = int(lead[-1])
    if a.k_major or b.k_major or N % 128 or H * N % 1024 or M < 1:
        raise PratchyaUnsupported("gemm_t128_fq: K-contiguous operands, outputs in whole groups of 8 blocks")
    ap, bp = _aligned_payload(a.payload), _aligned_payload(b.payload)
    as8, bs8 = a.sc8.contiguous(), b.sc8.contiguous()
    as32, bs32 = a.sc32.contiguous().float(), b.sc32.contiguous().float()
    lib, dev = _lib.load(), ap.device
    y = torch.empty((M, N), dtype=out_dtype, device=dev)
    sc8 = sc32 = None
    if scales:
        sc8 = torch.empty(lead[:-1] + (H * N // 1024, 8), dtype=E8M0, device=dev)
        sc32 = torch.empty(lead[:-1] + (H * N // 1024, 1, 1), dtype=torch.float32, device=dev)
    ws_bytes = _ws_bytes("pratchya_gemm_t128_fq_workspace_bytes", M, N, Kd // 128)
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=dev)
    _lib.check(lib.pratchya_gemm_bs_t128_fq(
        _ptr(ap), Kd, _ptr(as8), _ptr(as32), *a.desc, _ptr(bp), Kd, _ptr(bs8), _ptr(bs32), *b.desc, M, N, Kd, _ptr(y),
        _dtype_code(out_dtype), 1 if fix_nan else 0, _ptr(sc8) if scales else None, _ptr(sc32) if scales else None,
        _ptr(ws), ws_bytes, _stream(ap)), "gemm_t128_fq")
    return y, sc8, sc32


def gemm_nt_fq(a: Operand, b: Operand, out_dtype: torch.dtype, fix_nan: bool = False, lead=None,
               status: torch.Tensor = None, few: bool = False, scales: bool = True):
    """``QArrayImpl(dequant(a) @ dequant(b)^T, (1, 128)).astype(out_dtype)``
    with the requantization in the GEMM's epilogue: returns ``(y [M, N],
    sc_fp8, sc_fp32)`` bit-identical to ``quantize_dequantize(gemm_nt(a, b,
    float32), (1, 128), out_dtype, fix_nan)``.  ``lead``: leading dimensions
    of the product (its rows are ``prod(lead) * H`` flattened; the scales are
    shaped per slice as quantize_impl returns them).  Raises
    ``PratchyaUnsupported`` unless N is a multiple of 1024 and B's scale
    groups span at least 32 rows.  ``status``: an int32 device tensor that
    receives the strip exchange's status word (0: every wait completed).
    ``few``: a product of few tiles may run as gemm_t128_fq, whose sums are in
    another order; N then a multiple of 128, of 1024 where K is not split.
    ``scales`` False: the caller keeps only y, the scales may be None."""
    _require_gpu(a.payload, b.payload)
    if a.k != b.k:
        raise ValueError(f"contraction mismatch: {a.k} vs {b.k}")
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"gemm_nt_fq: output dtype {out_dtype} is not float32 or bfloat16")
    M, N, K = a.rows, b.rows, a.k
    # (N not of whole groups of a row: worth it where there are slices to sum)
    if few and status is None and b.desc[0] % 32 == 0 and not a.k_major and prefers_t128(M, a.desc[3], b) \
            and (N % 1024 == 0 or _ws_bytes("pratchya_gemm_t128_workspace_bytes", M, N, K // 128, 1)):
        return gemm_t128_fq(a, b, out_dtype, fix_nan, lead, scales)
    lib = _lib.load()
    ws_bytes = _ws_bytes("pratchya_gemm_bs_nt_fq_workspace_bytes", M, N)
    if ws_bytes <= 0:
        raise PratchyaUnsupported(f"gemm_fq: N must be a multiple of 1024 (got {N})")
    ap, bp = _tile_readable(_u8(a.payload).contiguous()), _tile_readable(_u8(b.payload).contiguous())
    as8, bs8 = _word_readable(_u8(a.sc8).contiguous()), _word_readable(_u8(b.sc8).contiguous())
    as32, bs32 = a.sc32.contiguous().float(), b.sc32.contiguous().float()
    lead = tuple(lead) if lead else (1,)
    S = 1
    for d in lead[:-1]:
        S *= int(d)
    H = M // S
    y = torch.empty((M, N), dtype=out_dtype, device=ap.device)
    sc8 = torch.empty(tuple(lead[:-1]) + (H * N // 1024, 8), dtype=torch.uint8, device=ap.device)
    sc32 = torch.empty(tuple(lead[:-1]) + (H * N // 1024, 1, 1), dtype=torch.float32, device=ap.device)
    ws = torch.empty(int(ws_bytes), dtype=torch.uint8, device=ap.device)
    _lib.check(lib.pratchya_gemm_bs_nt_fq(_ptr(ap), K, _ptr(as8), _ptr(as32), *a.desc,
                                          _ptr(bp), K, _ptr(bs8), _ptr(bs32), *b.desc,
                                          M, N, K, _ptr(y), N, _dtype_code(out_dtype), 1 if fix_nan else 0,
                                          _ptr(sc8), _ptr(sc32), _ptr(ws), int(ws_bytes), _stream(ap)), "gemm_fq")
    _wait_status(ws, int(lib.pratchya_gemm_bs_nt_fq_status_offset(M, N)), status, "gemm_fq")
    return y, sc8.view(E8M0), sc32


def gemm_nt_q11(a: Operand, b: Operand, out_dtype: torch.dtype, lead=None, few: bool = False,
                scales: bool = True):
    """``QArrayImpl(dequant(a) @ dequant(b)^T, (1, 1)).astype(out_dtype)``
    with the requantization in the GEMM's epilogue (the output grid of a
    weight quantized (a, 1): lm_head, LoRA): returns ``(y [M, N], sc_fp8,
    sc_fp32)`` bit-identical to ``quantize_dequantize(gemm_nt(a, b, float32),
    (1, 1), out_dtype)``, the scales shaped per slice of ``lead`` as there.
    Raises ``PratchyaUnsupported`` unless N is a multiple of 16.  ``few``: as
    for gemm_nt_fq.  Without ``scales`` the scale arrays, five of the seven
    bytes written per bf16 element, are not returned (None), and unless the
    product ran as one of few tiles neither allocated nor stored."""
    _require_gpu(a.payload, b.payload)
    if a.k != b.k:
        raise ValueError(f"contraction mismatch: {a.k} vs {b.k}")
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"gemm_nt_q11: output dtype {out_dtype} is not float32 or bfloat16")
    M, N, K = a.rows, b.rows, a.k
    if N % 16:
        raise PratchyaUnsupported(f"gemm_q11: N must be a multiple of 16 (got {N})")
    if few and not a.k_major and prefers_t128(M, a.desc[3], b):
        return _few_then_requantize(a, b, out_dtype, lead, scales)
    lib = _lib.load()
    ap, bp = _tile_readable(_u8(a.payload).contiguous()), _tile_readable(_u8(b.payload).contiguous())
    as8, bs8 = _word_readable(_u8(a.sc8).contiguous()), _word_readable(_u8(b.sc8).contiguous())
    as32, bs32 = a.sc32.contiguous().float(), b.sc32.contiguous().float()
    lead = tuple(lead) if lead else (1,)
    S = 1
    for d in lead[:-1]:
        S *= int(d)
    H = M // S
    y = torch.empty((M, N), dtype=out_dtype, device=ap.device)
    sc8 = sc32 = None
    if scales:
        sc8 = torch.empty(tuple(lead[:-1]) + (H * N, 1), dtype=torch.uint8, device=ap.device)
        sc32 = torch.empty(tuple(lead[:-1]) + (H * N, 1, 1), dtype=torch.float32, device=ap.device)
    _lib.check(lib.pratchya_gemm_bs_nt_q11(_ptr(ap), K, _ptr(as8), _ptr(as32), *a.desc,
                                           _ptr(bp), K, _ptr(bs8), _ptr(bs32), *b.desc,
                                           M, N, K, _ptr(y), N, _dtype_code(out_dtype),
                                           _ptr(sc8) if scales else None, _ptr(sc32) if scales else None,
                                           _stream(ap)), "gemm_q11")
    return y, None if sc8 is None else sc8.view(E8M0), sc32


def gemm_nt_qa(x: torch.Tensor, b: Operand, out_dtype: torch.dtype, fq: bool = False, lead=None,
               status: torch.Tensor = None):
    """``quantize_impl(x, (1, 128))`` of a bf16 activation ``x`` [..., K] and
    the GEMM ``dequant(x_q) @ dequant(b)^T`` in one launch (the quantize
    prologue, pratchya_gemm_bs_nt_qa): each row of ``x`` is quantized once,
    by the GEMM's workgroups before their first tiles.  Returns ``(y [M, N], (x8, sc8,
    sc32), out_scales)``: ``(x8, sc8, sc32)`` bit-identical to
    ``quantize(x, (1, 128))`` (what the backward keeps), ``y`` bit-identical to
    ``gemm_nt(operand_rows(*that), b, out_dtype)``, or with ``fq`` to
    ``gemm_nt_fq(..., out_dtype)``, whose output scales are ``out_scales``
    (else None).  ``lead`` shapes the output scales as in gemm_nt_fq.  Raises ``PratchyaUnsupported`` where the fused path does not
    apply (x not bf16, fewer than 256 rows, K not a multiple of 1024, B's scale
    groups narrower than 32 rows, N not a multiple of 1024 with ``fq``)."""
    _require_gpu(x, b.payload)
    if x.dtype != torch.bfloat16:
        raise PratchyaUnsupported(f"gemm_qa: the quantize prologue takes bf16 activations (got {x.dtype})")
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise ValueError(f"gemm_qa: output dtype {out_dtype} is not float32 or bfloat16")
    K = int(x.shape[-1])
    if b.k != K:
        raise ValueError(f"contraction mismatch: {K} vs {b.k}")
    if b.k_major:
        raise PratchyaUnsupported("gemm_qa: B must be K-contiguous")
    M, N = x.numel() // K, b.rows
    if not x.is_contiguous() or not _aligned(x, 16):
        x = x.contiguous() if not x.is_contiguous() else x.clone()
    S, H, W = slices_hw(x.shape)
    _, Kg, Mg = group_layout(H, W, (1, 128))
    xlead = tuple(x.shape[:-2]) if x.dim() >= 2 else ()
    x8 = torch.empty(x.shape, dtype=torch.uint8, device=x.device)
    xs8 = torch.empty(xlead + (Mg, Kg), dtype=torch.uint8, device=x.device)
    xs32 = torch.empty(xlead + (Mg, 1, 1), dtype=torch.float32, device=x.device)
    lib = _lib.load()
    ws_bytes = lib.pratchya_gemm_bs_nt_qa_workspace_bytes(M, N, 1 if fq else 0)
    if ws_bytes <= 0:
        raise PratchyaUnsupported(f"gemm_qa: unsupported shape M={M} N={N} fq={fq}")
    bp = _tile_readable(_u8(b.payload).contiguous())
    bs8, bs32 = _word_readable(_u8(b.sc8).contiguous()), b.sc32.contiguous().float()
    y = torch.empty((M, N), dtype=out_dtype, device=x.device)
    if fq:
        lead = tuple(lead) if lead else (1,)
        Sl = 1
        for d in lead[:-1]:
            Sl *= int(d)
        Hl = M // Sl
        osc8 = torch.empty(tuple(lead[:-1]) + (Hl * N // 1024, 8), dtype=torch.uint8, device=x.device)
        osc32 = torch.empty(tuple(lead[:-1]) + (Hl * N // 1024, 1, 1), dtype=torch.float32, device=x.device)
    else:
        osc8 = osc32 = None
    ws = torch.empty(int(ws_bytes), dtype=torch.uint8, device=x.device)
    _lib.check(lib.pratchya_gemm_bs_nt_qa(_ptr(x), K, _ptr(x8), _ptr(xs8), _ptr(xs32),
                                          _ptr(bp), K, _ptr(bs8), _ptr(bs32), *b.desc,
                                          M, N, K, _ptr(y), N, _dtype_code(out_dtype), 1 if fq else 0,
                                          _ptr(osc8) if fq else None, _ptr(osc32) if fq else None,
                                          _ptr(ws), int(ws_bytes), _stream(x)), "gemm_qa")
    _wait_status(ws, int(lib.pratchya_gemm_bs_nt_qa_status_offset(M, N, 1 if fq else 0)), status, "gemm_qa")
    xq = (x8.view(E4M3), xs8.view(E8M0), xs32)
    return y, xq, ((osc8.view(E8M0), osc32) if fq else None)


def _as_operand(x, what):
    """(tensor, dtype code, sc8, sc32) of an optimizer operand: an fp8 payload
    given as a (payload, sc8, sc32) triple, or a bf16 / f32 tensor."""
    if isinstance(x, (tuple, list)):
        x8, s8, s32 = x
        _require_gpu(x8, s8, s32)
        return _u8(x8).contiguous(), _lib.DT_E4M3, _u8(s8).contiguous(), s32.contiguous().float()
    _require_gpu(x)
    if x.dtype not in (torch.float32, torch.bfloat16):
        raise TypeError(f"{what}: unsupported dtype {x.dtype}")
    return x.contiguous(), _dtype_code(x.dtype), None, None


def momentum(m, g, tgrid, arith: torch.dtype, beta1: float, beta1c: float, beta2: float, beta2c: float):
    """``c = beta1*m + beta1c*g`` and ``m_new = beta2*m + beta2c*g`` of the
    Miulion step (pratchya/_nnx_impl/_optimizer.py:124-135, :157-176), one
    rounding per operation in ``arith`` (float32 or bfloat16), in one pass.
    ``m``: the quantized momentum as a (payload, sc8, sc32) triple with tgrid
    ``tgrid``; ``g``: a triple in the same layout or a bf16 / f32 tensor.  The
    constants must be values of ``arith``.  Returns ``(c, m_new)`` in ``arith``."""
    m8, _, ms8, ms32 = _as_operand(m, "momentum")
    gt, gcode, gs8, gs32 = _as_operand(g, "momentum gradient")
    if tuple(gt.shape) != tuple(m8.shape):
        raise ValueError(f"momentum: gradient shape {tuple(gt.shape)} != momentum shape {tuple(m8.shape)}")
    S, H, W = slices_hw(m8.shape)
    c = torch.empty(m8.shape, dtype=arith, device=m8.device)
    nm = torch.empty(m8.shape, dtype=arith, device=m8.device)
    lib = _lib.load()
    _lib.check(lib.pratchya_momentum(_ptr(m8), _ptr(ms8), _ptr(ms32), _ptr(gt), gcode,
                                     _ptr(gs8) if gs8 is not None else None,
                                     _ptr(gs32) if gs32 is not None else None,
                                     S, H, W, int(tgrid[0]), int(tgrid[1]), _dtype_code(arith),
                                     beta1, beta1c, beta2, beta2c, _ptr(c), _ptr(nm), _stream(m8)), "momentum")
    return c, nm


def ns_combine(x: torch.Tensor, b: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """``1.5 * x - 0.5 * b`` with each operation rounded to ``x.dtype`` (bf16 or
    f32), one Newton-Schulz step's combination (pratchya/_nnx_impl/_optimizer.py:
    26-27), in one pass.  ``out`` may be ``x``."""
    _require_gpu(x, b)
    if x.dtype != b.dtype or tuple(x.shape) != tuple(b.shape):
        raise ValueError("ns_combine: x and b must share dtype and shape")
    xx, bb = x.contiguous(), b.contiguous()
    if out is None:
        out = torch.empty_like(xx)
    elif not out.is_contiguous() or tuple(out.shape) != tuple(xx.shape) or out.dtype != xx.dtype:
        raise ValueError("ns_combine: out must be a contiguous tensor like x")
    lib = _lib.load()
    _lib.check(lib.pratchya_ns_combine(_ptr(xx), _ptr(bb), _ptr(out), xx.numel(), _dtype_code(xx.dtype),
                                       _stream(xx)), "ns_combine")
    return out


def apply_update(u: torch.Tensor, use_sign: bool, scale: float, p, tgrid, arith: torch.dtype,
                 lr: float, lr_wd: float, out_dtype: torch.dtype) -> torch.Tensor:
    """``-(lr * u' + lr_wd * p)`` with ``u' = sign(u)`` (Lion) or ``u * scale``
    (Muon) (pratchya/_nnx_impl/_optimizer.py:147-153, :189-197): ``p`` and
    ``u * scale`` rounded to the leaf dtype ``arith``, the products and the sum
    in f32 (``lr``, ``lr_wd`` f32 values), one rounding to ``out_dtype``.
    ``p``: a (payload, sc8, sc32) triple with tgrid ``tgrid`` or a bf16 / f32
    tensor of ``u``'s shape."""
    _require_gpu(u)
    uu = u.contiguous()
    pt, pcode, ps8, ps32 = _as_operand(p, "update parameter")
    if tuple(pt.shape) != tuple(uu.shape):
        raise ValueError(f"apply_update: parameter shape {tuple(pt.shape)} != direction shape {tuple(uu.shape)}")
    S, H, W = slices_hw(uu.shape)
    a, b = (int(tgrid[0]), int(tgrid[1])) if pcode == _lib.DT_E4M3 else (1, 1)
    out = torch.empty(uu.shape, dtype=out_dtype, device=uu.device)
    lib = _lib.load()
    _lib.check(lib.pratchya_apply_update(_ptr(uu), _dtype_code(uu.dtype), 1 if use_sign else 0, scale,
                                         _ptr(pt), pcode, _ptr(ps8) if ps8 is not None else None,
                                         _ptr(ps32) if ps32 is not None else None, S, H, W, a, b,
                                         _dtype_code(arith), lr, lr_wd, _ptr(out), _dtype_code(out_dtype),
                                         _stream(uu)), "apply_update")
    return out
