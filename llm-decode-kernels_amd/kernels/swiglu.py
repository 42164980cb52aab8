"""Fused SwiGLU activation on gfx950: out = silu(gate) * up, in one pass.

Drop-in for the reference's `kernels/swiglu.py`: accepts two tensors or one fused [.., 2*I]
tensor (gate first, then up) whose halves are read in place. silu is computed in fp32 and
rounded to fp16 like F.silu, then multiplied by `up` in fp16 (kernels/reference.py:22-24).
"""

from __future__ import annotations

import torch

from kernels import _lib


def _launch(gate: int, ldg: int, up: int, ldu: int, M: int, I: int, dev) -> torch.Tensor:
    """gate, up: device addresses of fp16 rows of I values, strides ldg and ldu, that the caller's
    locals keep alive."""
    out = torch.empty((M, I), dtype=torch.float16, device=dev)
    with _lib.device_guard(dev):
        st = _lib.load().ldk_swiglu(gate, ldg, up, ldu, out.data_ptr(), I, M, I, _lib.stream(dev))
    _lib.check(st, "swiglu")
    return out


def swiglu(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up for two same-shape tensors (swiglu.py:49-53)."""
    I = gate.shape[-1]
    gate2, up2 = gate.reshape(-1, I), up.reshape(-1, I)
    assert gate2.stride(-1) == 1 and up2.stride(-1) == 1
    dev = _lib.require_gpu(gate2, up2, what="swiglu")
    if gate2.dtype != torch.float16 or up2.dtype != torch.float16:
        raise ValueError("swiglu: gate and up must be float16")
    out = _launch(gate2.data_ptr(), gate2.stride(0), up2.data_ptr(), up2.stride(0), gate2.shape[0], I, dev)
    return out.view(gate.shape)


def swiglu_fused(gate_up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up where gate_up = cat([gate, up], dim=-1); reads the halves in place
    (swiglu.py:56-61)."""
    I = gate_up.shape[-1] // 2
    flat = gate_up.dim() == 2 and gate_up.shape[1] == 2 * I
    gu = gate_up if flat else gate_up.reshape(-1, 2 * I)
    assert gu.stride(-1) == 1
    dev = _lib.require_gpu(gu, what="swiglu")
    if gu.dtype != torch.float16:
        raise ValueError("swiglu: gate and up must be float16")
    ld = gu.stride(0)
    out = _launch(gu.data_ptr(), ld, gu.data_ptr() + 2 * I, ld, gu.shape[0], I, dev)  # fp16: 2 bytes
    return out if flat else out.view(*gate_up.shape[:-1], I)


def swiglu_bytes(M: int, I: int, elem: int = 2) -> int:
    """Read gate and up, write out (swiglu.py:64-65)."""
    return 3 * M * I * elem
