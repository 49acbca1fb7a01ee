"""FP8 KV cache rows for :func:`dsa_amd.forward` (no reference counterpart: the
reference takes a contiguous bf16 cache only, dsa/api.py:30-33).

One row per token, 656 bytes -- the layout of DeepSeek-V3.2's FP8 MLA cache:

* bytes   0..511: the 512 latent values as OCP float8 e4m3 (bias 7, max 448),
* bytes 512..527: 4 fp32 scales, scale i for dims 128 i .. 128 i + 127,
* bytes 528..655: the 64 rope values as bf16 (not quantized).

The attention kernels compute with ``bf16(fp32(e4m3) * scale)`` for the latent
values, for any positive scale; with power-of-two scales (2^-100 .. 2^100)
that value is exact and they expand the rows with one conversion
instruction per two values.  :func:`quantize_kv_fp8` writes such rows from a
bf16 cache: per 128-dim block the scale is the smallest power of two with
``amax / scale <= 448`` (e4m3 is floating point, so a power-of-two scale
costs no relative precision), or ``amax / 448`` with ``pow2_scales=False``.

Tensors on a ROCm GPU are written by one kernel (``csrc/kv_rows.hip``), any
other call (CPU tensors, traced or transformed ones, a package whose library is
not built) by the same arithmetic as tensor code.  The kernel's bytes are those
of the tensor code on the same GPU.  On the CPU the two differ in the last place
of some scales: ``amax / 448`` is a product with the rounded reciprocal on the
GPU, and powers of two beyond 2^15 or below 2^-15 (block maxima above about 10^7
or below 0.01) are what the GPU's ``powf`` gives.
"""
from __future__ import annotations

import torch
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import _lib
from .api import _on_device

FP8_ROW = 656
E4M3_MAX = 448.0


def quantize_kv_fp8(kv, k_rope, pow2_scales: bool = True):
    """``kv [..., 512]`` bf16 and ``k_rope [..., 64]`` bf16 (same leading dims)
    -> uint8 rows ``[..., 656]`` on the same device."""
    if kv.shape[-1] != 512 or k_rope.shape[-1] != 64 or kv.shape[:-1] != k_rope.shape[:-1]:
        raise ValueError("expected kv[..., 512] and k_rope[..., 64] with the same leading dims")
    if kv.dtype != torch.bfloat16 or k_rope.dtype != torch.bfloat16:
        raise ValueError("kv and k_rope must be bfloat16")
    lead = kv.shape[:-1]
    if _plain_gpu_pair(kv, k_rope):
        return _quantize_gpu(kv.contiguous(), k_rope.contiguous(), lead, pow2_scales)
    x = kv.float().reshape(*lead, 4, 128)
    amax = x.abs().amax(-1, keepdim=True)
    scale = torch.where(amax > 0, amax / E4M3_MAX, torch.ones_like(amax))
    if pow2_scales:  # the smallest power of two >= amax / 448: frexp gives s = m 2^e, m in [0.5, 1)
        m, e = torch.frexp(scale)
        scale = torch.ldexp(torch.ones_like(scale), e - (m == 0.5).to(e.dtype))
    codes = (x / scale).clamp(-E4M3_MAX, E4M3_MAX).to(torch.float8_e4m3fn).reshape(*lead, 512)
    rows = torch.cat([codes.view(torch.uint8),
                      scale.reshape(*lead, 4).contiguous().view(torch.uint8),
                      k_rope.contiguous().view(torch.uint8)], dim=-1)
    return rows.contiguous()


def _plain_gpu_pair(kv, k_rope):
    """Whether the kernel may read these two tensors: ordinary eager tensors
    of one ROCm GPU (no subclass, tracing, function or dispatch mode or
    functorch level between the caller and the storage) with at least one row,
    and the library built (the rows can be written without it, unlike the
    attention's results)."""
    return ((_lib._lib is not None or _lib.built()) and type(kv) is torch.Tensor and type(k_rope) is torch.Tensor
            and kv.is_cuda and kv.device == k_rope.device and torch.version.hip is not None and kv.numel() > 0
            and not torch.compiler.is_compiling() and not torch.jit.is_tracing()
            and not torch._C._are_functorch_transforms_active() and torch._C._len_torch_dispatch_stack() == 0
            and (torch._C._len_torch_function_stack() == 0 or _only_default_devices())
            and not (kv.is_neg() or k_rope.is_neg()))


def _only_default_devices() -> bool:
    """Whether the torch_function modes are default devices
    (``torch.set_default_device``), which only place tensors that name no
    device: any other mode watches the operations."""
    return all(type(m) is DeviceContext for m in _get_current_function_mode_stack())


def _quantize_gpu(kv, k_rope, lead, pow2_scales):
    device = kv.device
    # a view may start anywhere in its storage: the kernel's loads are 16 and 4 bytes wide
    kv = kv.clone() if kv.data_ptr() % 16 else kv
    k_rope = k_rope.clone() if k_rope.data_ptr() % 4 else k_rope
    rows = torch.empty((*lead, FP8_ROW), device=device, dtype=torch.uint8)
    with _on_device(device):
        rc = _lib.load().dsa_kv_quantize_rows(kv.data_ptr(), k_rope.data_ptr(), rows.data_ptr(), kv.numel() // 512,
                                              1 if pow2_scales else 0,
                                              torch._C._cuda_getCurrentRawStream(device.index))
    _lib.check(rc, "dsa_kv_quantize_rows")
    return rows
