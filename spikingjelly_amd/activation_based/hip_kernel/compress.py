"""Spike bit-packing on the device: 8 binary spikes per byte, LSB first over the flattened tensor.

Counterpart of the device kernels of the reference's ``triton_kernel/compress.py:114-221``
(``bit_spike_compress`` / ``bit_spike_decompress``).  These functions run ``libsjhip.so`` on ROCm tensors only
and raise for anything else; the torch path the reference keeps for non-CUDA tensors (compress.py:19-44,
150-151) lives with the compressor classes in ``memopt/compress.py``.
"""

from __future__ import annotations

import torch

from . import library as L
from . import native

__all__ = ["bit_spike_compress", "bit_spike_decompress"]


def bit_spike_compress(s_seq: torch.Tensor) -> torch.Tensor:
    """Pack a strictly binary tensor into ``(numel + 7) // 8`` bytes (uint8, 1-D)."""
    L.require_device_tensor("s_seq", s_seq)
    if s_seq.numel() > 0:
        L.dtype_id(s_seq.dtype, allow_u8=True)
    return native.load().bit_pack(s_seq)


def bit_spike_decompress(s_seq_compressed: torch.Tensor, shape, dtype: torch.dtype = torch.uint8) -> torch.Tensor:
    """Unpack to a 0/1 tensor of ``shape``.  ``dtype`` defaults to ``uint8`` like the reference's
    device kernel; passing the final dtype saves the separate cast pass."""
    shape = torch.Size(shape)
    L.require_device_tensor("s_seq_compressed", s_seq_compressed)
    n = shape.numel()
    if s_seq_compressed.dtype != torch.uint8 or s_seq_compressed.numel() < (n + 7) // 8:
        raise ValueError(f"compressed tensor must be uint8 with at least {(n + 7) // 8} bytes")
    if n > 0:
        L.dtype_id(dtype, allow_u8=True)
    return native.load().bit_unpack(s_seq_compressed, shape, dtype)
