"""Device-memory plumbing: torch tensors carry the buffers and the stream.

Arrays may be given as numpy arrays or torch tensors; they are moved to the
current HIP device as contiguous float32/float64 tensors.  Results are
returned as the same kind of array as the primary input.
"""
import ctypes as C
import threading

import numpy as np
import torch

from . import _lib


def require_device():
    if not torch.cuda.is_available():
        raise RuntimeError(
            "jubik_amd computes on an AMD GPU through libjubik_hip.so; no HIP "
            "device is visible")
    _lib.load()


def float_dtype(*arrays):
    """float32 if every floating input is float32, else float64 (jubik
    enforces float64, jubik/enforce_float64.py:1-2)."""
    seen = []
    for a in arrays:
        if a is None:
            continue
        dt = a.dtype
        if isinstance(a, torch.Tensor):
            seen.append(dt == torch.float32)
        else:
            seen.append(np.dtype(dt) == np.float32)
    return torch.float32 if seen and all(seen) else torch.float64


def code(dtype):
    return _lib.FLOAT32 if dtype == torch.float32 else _lib.FLOAT64


def to_device(a, dtype):
    """Contiguous device tensor of ``dtype`` holding ``a``."""
    if isinstance(a, torch.Tensor):
        if (a.is_cuda and a.dtype == dtype and a.get_device() == torch.cuda.current_device()
                and a.is_contiguous()):
            return a
        t = a.to(device="cuda", dtype=dtype)
    else:
        t = torch.as_tensor(np.asarray(a), dtype=dtype, device="cuda")
    return t.contiguous()


# Pinned (page-locked) staging buffers for device-to-host results, one per
# (device, dtype, element count), reused across calls: a download from
# device memory into pinned host memory runs at the DMA rate, several times
# the rate of a download into pageable memory (measured on MI355X: 2 x 4 MB
# in 0.18 ms pinned against 1.6 ms pageable).  The caller receives a fresh
# numpy copy, never a view of the staging buffer.
_STAGING = {}
_STAGING_MAX_BYTES = 256 << 20
_STAGING_LOCK = threading.Lock()


def _download(t):
    t = t.detach()
    if t.device.type != "cuda" or t.numel() * t.element_size() > _STAGING_MAX_BYTES:
        return t.cpu().numpy()
    key = (t.device.index, t.dtype, t.numel())
    with _STAGING_LOCK:
        pin = _STAGING.get(key)
        if pin is None:
            pin = torch.empty(t.numel(), dtype=t.dtype, pin_memory=True)
            _STAGING[key] = pin
        pin.copy_(t.reshape(-1), non_blocking=True)
        torch.cuda.current_stream(t.device).synchronize()
        return pin.numpy().reshape(tuple(t.shape)).copy()


def like_input(t, ref):
    """Return ``t`` as the kind of array ``ref`` is (torch stays on device)."""
    if isinstance(ref, torch.Tensor):
        return t
    return _download(t)


def ptr(t):
    return C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p(0)


def ptrs(tensors):
    """Host array of the tensors' device pointers."""
    return (C.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)
