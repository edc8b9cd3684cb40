"""Quantization primitives with the reference's names and signatures
(core/quantization.py:4-45), computed by the gfx950 kernels of libdscq.

``weight_codes`` / ``activation_codes`` return the same float-valued codes,
scales and zero-points as the reference (round half to even, IEEE fp32
division, the 1e-8 scale floor), bit for bit, for finite inputs on a CUDA
(HIP) device.  These are inference primitives: the codes carry no gradient
(the reference's straight-through estimator serves calibration, which stays
outside this path).  A CPU tensor raises -- there is no CPU fallback.
"""
from __future__ import annotations

import torch

from .. import _lib

__all__ = ["ste_round", "weight_codes", "activation_codes", "quantize_weight",
           "quantize_activation", "pack_int4", "unpack_int4"]

_CODE = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16, torch.float32: _lib.F32}


def ste_round(x):
    """core/quantization.py:4-5: round in the forward pass, identity gradient."""
    return x + (x.round() - x).detach()


def _as_kernel_input(t: torch.Tensor, what: str) -> torch.Tensor:
    if not t.is_cuda:
        raise RuntimeError(f"{what}: dscquant_amd runs on the GPU (HIP); got a "
                           f"{t.device.type} tensor")
    if t.dtype not in _CODE:
        t = t.float()  # fp64, integers -> fp32; the reference widens with .float() too
    return t.contiguous()


def _clip_value(clip) -> float:
    return float(clip.detach().float().item()) if torch.is_tensor(clip) else float(clip)


def _fake_quant(rows, bits: int, clip: float, weight: int):
    """``rows`` [M, K] quantized and put back on their scales, in their own dtype."""
    out = torch.empty_like(rows)
    _lib.require_gfx950(rows.device)
    if rows.shape[0] or weight:
        with _lib.on(rows.device):
            _lib.call("dscq_fake_quant", rows.data_ptr(), _CODE[rows.dtype], rows.shape[0],
                      rows.shape[1], clip, bits, weight, out.data_ptr(),
                      _lib.stream(rows.device))
    return out


def _float_codes(rows, bits: int, clip: float, weight: int):
    """(code f32 [M, K], scale f32 [M], zero f32 [M]) of ``rows`` [M, K]."""
    M, K = rows.shape
    dev = rows.device
    code = torch.empty((M, K), dtype=torch.float32, device=dev)
    scale = torch.empty((M,), dtype=torch.float32, device=dev)
    zero = None if weight else torch.empty((M,), dtype=torch.float32, device=dev)
    _lib.require_gfx950(dev)
    if M or weight:
        with _lib.on(dev):
            _lib.call("dscq_float_codes", rows.data_ptr(), _CODE[rows.dtype], M, K, clip, bits,
                      weight, code.data_ptr(), scale.data_ptr(), _lib.ptr(zero),
                      _lib.stream(dev))
    return code, scale, zero


def weight_codes(weight, bits, clip=1.0):
    """core/quantization.py:7-11 -> (code f32 [N, K], scale f32 [N, 1])."""
    w = _as_kernel_input(weight, "weight_codes")
    if w.dim() != 2:
        raise ValueError("weight_codes expects a [out_features, in_features] matrix")
    code, scale, _ = _float_codes(w, int(bits), _clip_value(clip), 1)
    return code, scale[:, None]


def activation_codes(x, bits, clip=1.0):
    """core/quantization.py:13-21 -> (code, scale, zero), codes in [0, 2^bits-1].

    Shapes follow the reference: code like x, scale / zero ``x.shape[:-1] + (1,)``,
    all float32.
    """
    xk = _as_kernel_input(x, "activation_codes")
    bits, clip = int(bits), _clip_value(clip)
    K = xk.shape[-1]
    code, scale, zero = _float_codes(xk.reshape(-1, K), bits, clip, 0)
    lead = x.shape[:-1]
    return code.reshape(*lead, K), scale.reshape(*lead, 1), zero.reshape(*lead, 1)


def quantize_weight(weight, bits, clip=1.0):
    """core/quantization.py:23-25: fake-quantized weight in its own dtype."""
    w = _as_kernel_input(weight, "weight_codes")
    if w.dim() != 2:
        raise ValueError("weight_codes expects a [out_features, in_features] matrix")
    return _fake_quant(w, int(bits), _clip_value(clip), 1).to(weight.dtype)


def quantize_activation(x, bits, clip=1.0):
    """core/quantization.py:27-29: fake-quantized activation in its own dtype."""
    xk = _as_kernel_input(x, "activation_codes")
    bits, clip = int(bits), _clip_value(clip)
    rows = xk.reshape(-1, xk.shape[-1])
    return _fake_quant(rows, bits, clip, 0).reshape(x.shape).to(x.dtype)


def pack_int4(codes):
    """core/quantization.py:31-40: signed [-8, 7] codes -> u8 [R, ceil(C/2)]."""
    if codes.ndim != 2:
        raise ValueError('Packed weights must be a matrix.')
    if not codes.is_cuda:
        c = codes.to(torch.int8)
        if bool(((c < -8) | (c > 7)).any()):
            raise ValueError('Signed INT4 code out of range.')
        raise RuntimeError("pack_int4: dscquant_amd runs on the GPU (HIP); got a "
                           f"{c.device.type} tensor")
    # Codes as weight_codes gives them (fp32) are converted in the kernel; the
    # range check is the kernel's too, one flag read back.
    c = (codes if codes.dtype in (torch.float32, torch.int8) else codes.to(torch.int8)).contiguous()
    R, C = c.shape
    out = torch.empty((R, (C + 1) // 2), dtype=torch.uint8, device=c.device)
    bad = torch.zeros((1,), dtype=torch.int32, device=c.device)
    with _lib.on(c.device):
        _lib.call("dscq_pack_int4_checked", _lib.ptr(c), 1 if c.dtype == torch.float32 else 0,
                  R, C, _lib.ptr(out), bad.data_ptr(), _lib.stream(c.device))
    if bool(bad):
        raise ValueError('Signed INT4 code out of range.')
    return out


def unpack_int4(packed, width):
    """core/quantization.py:42-45: u8 [R, CB] -> signed int8 [R, width]."""
    if not packed.is_cuda:
        raise RuntimeError("unpack_int4: dscquant_amd runs on the GPU (HIP); got a "
                           f"{packed.device.type} tensor")
    p = packed.to(torch.uint8).contiguous()
    R, CB = p.shape
    width = int(width)
    width = min(width, 2 * CB)  # slicing semantics of the reference's [:, :width]
    out = torch.empty((R, width), dtype=torch.int8, device=p.device)
    with _lib.on(p.device):
        _lib.call("dscq_unpack_int4", _lib.ptr(p), R, CB, width, _lib.ptr(out),
                  _lib.stream(p.device))
    return out
