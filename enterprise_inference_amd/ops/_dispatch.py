"""Device dispatch helpers shared by the op wrappers."""

from __future__ import annotations

import os

import torch

from .. import _native

# Debug switch: run the PyTorch reference ops even on the GPU (never the default).
FORCE_TORCH = os.environ.get("EIA_FORCE_TORCH_OPS", "0") == "1"
# Debug switch (SURVEY §5.2 "HIP_LAUNCH_BLOCKING test mode"): synchronise after every native
# kernel launch and surface asynchronous faults at the op that caused them.
SYNC_KERNELS = (os.environ.get("EIA_SYNC_KERNELS", "0") == "1"
                or os.environ.get("HIP_LAUNCH_BLOCKING", "0") == "1"
                or os.environ.get("AMD_SERIALIZE_KERNEL", "0") == "3")


def use_hip(*tensors: torch.Tensor) -> bool:
    """True when the HIP kernels must be used for these tensors."""
    if FORCE_TORCH:
        return False
    hip = False
    for t in tensors:
        if t is not None:
            if not t.is_cuda:
                return False
            hip = True
    return hip


def ptr(t):
    return None if t is None else t.data_ptr()


def workspace(device, *sizes: int):
    """One allocation of so many bytes each, at multiples of 512 bytes from its start, large ones of 2 MiB (8 experts of
    1024 x 512, 2000 rows 41.4 -> 40.4 us, other ops and sizes the same) -> (the tensor that owns it, addresses).  An
    allocation costs the host 1.3 us, and small steps are bound by their launches."""
    at, total = [], 0
    for n in sizes:
        step = 512 if n < 1 << 21 else 1 << 21
        total = -(-total // step) * step
        at.append(total)
        total += n
    ws = torch.empty(total, dtype=torch.uint8, device=device)
    base = ws.data_ptr()
    return ws, [base + a for a in at]


def stream(t: torch.Tensor) -> int:
    # (the raw handle: torch.cuda.current_stream builds a Stream object around it, 1.5 us a call)
    return torch._C._cuda_getCurrentRawStream(t.device.index)


def lib():
    return _native.kernels()


def check(status: int, name: str) -> None:
    _native.check(status, name)
    if SYNC_KERNELS and torch.cuda.is_available() and not torch.cuda.is_current_stream_capturing():
        try:
            torch.cuda.synchronize()
        except RuntimeError as e:   # asynchronous fault: name the op that launched it
            raise RuntimeError(f"{name}: device fault after launch: {e}") from e


def require(cond: bool, msg: str) -> None:
    if not cond:
        raise ValueError(msg)
