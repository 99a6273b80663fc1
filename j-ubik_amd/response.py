"""Exposure and read-out: drop-in for jubik/response.py on the GPU.

The builders keep the reference's host-side behaviour exactly (argument
checks, in-place cut of the caller's array, key handling); the closures
they return run as HIP kernels (broadcast multiply, gather of the kept pixels
in C order).
"""
import math

import numpy as np
import torch

from . import _device as dev
from . import _lib
from .data import Vector


def build_exposure_function(exposures, exposure_cut=None):
    """jubik/response.py:12-45: returns ``x -> exposures * x``.

    Entries below ``exposure_cut`` are zeroed in place in ``exposures`` (the
    reference mutates the caller's array, which Chandra relies on).  Like
    the reference's closure, each call multiplies by the array as it is at
    that call: later in-place edits of ``exposures`` are seen (a device
    tensor of the working dtype is used without a copy; a host array is
    copied to the device per call).
    """
    if exposure_cut is not None:
        if exposure_cut < 0:
            raise ValueError("exposure_cut should be non-negative or None!")
        exposures[exposures < exposure_cut] = 0

    def exposure(x):
        dtype = dev.float_dtype(exposures, x)
        dev.require_device()
        e = dev.to_device(exposures, dtype)
        xt = dev.to_device(x, dtype)
        try:
            oshape = tuple(torch.broadcast_shapes(tuple(e.shape), tuple(xt.shape)))
        except RuntimeError as err:
            raise ValueError(str(err)) from None
        ev, xv = e, xt
        # The kernel broadcasts operands whose shape is a suffix of the
        # output shape; any other broadcast is materialised first.
        if tuple(ev.shape) != oshape[len(oshape) - ev.dim():]:
            ev = ev.expand(oshape).contiguous()
        if tuple(xv.shape) != oshape[len(oshape) - xv.dim():]:
            xv = xv.expand(oshape).contiguous()
        out = torch.empty(oshape, dtype=dtype, device="cuda")
        _lib.call("jubik_exposure_apply", dev.code(dtype), dev.ptr(ev), max(ev.numel(), 1),
                  dev.ptr(xv), max(xv.numel(), 1), dev.ptr(out), out.numel(), dev.stream())
        return dev.like_input(out, x)

    return exposure


# Set bits of every byte (numpy counts bits by itself from version 2.0 on only).
_BITS = np.unpackbits(np.arange(256, dtype=np.uint8)[:, None], axis=1).sum(axis=1)


def kept_words(kept):
    """Bit words of the kept pixels (``kept``: one boolean map per module):
    an int64 array (2, modules, words) that holds the words, bit b of word k
    for pixel 64 k + b, and the kept pixels before each word; and the number
    of kept pixels of every module."""
    modules = kept.shape[0]
    per = int(np.prod(kept.shape[1:]))
    words = np.zeros((2, modules, (per + 63) // 64), dtype=np.int64)
    bits = words[0].view(np.uint8).reshape(modules, -1)
    for i in range(modules):
        packed = np.packbits(kept[i].reshape(-1), bitorder="little")
        bits[i, :packed.size] = packed
    upto = np.cumsum(_BITS[bits].reshape(words[0].shape + (8,)).sum(axis=-1), axis=1,
                     dtype=np.int64)
    words[1, :, 1:] = upto[:, :-1]
    return words, (upto[:, -1].tolist() if words.shape[2] else [0] * modules)


def build_readout_function(flags, threshold=None, keys=None):
    """jubik/response.py:48-112: returns ``x -> Vector({key_i: x[i][~mask[i]]})``.

    ``mask = (flags == 0)`` after zeroing the flags below ``threshold`` in
    place.  The kept pixels are held as a bit each (``kept_words``) and read out
    in C order, all modules in one launch.
    """
    if threshold is not None and threshold < 0:
        raise ValueError("threshold should be positive!")
    if threshold is not None:
        flags[flags < threshold] = 0
    mask = np.asarray(flags) == 0

    if keys is None:
        keys = ['masked input']
    elif len(keys) != flags.shape[0]:
        raise ValueError("length of keys should match the number of flag maps.")
    word_cache = {}
    pixels = math.prod(mask.shape[1:])

    def _words():
        """Kept pixels of the modules that are read out, on the current
        device: pointers to the bit words and to the kept pixels before each
        word, and the number of kept pixels per module (and the tensor that
        the pointers lie in)."""
        dkey = torch.cuda.current_device()
        if dkey not in word_cache:
            host, counts = kept_words(~mask[:len(keys)])
            words = torch.as_tensor(host, device="cuda")
            word_cache[dkey] = (dev.ptr(words[0]), dev.ptr(words[1]), counts, words)
        return word_cache[dkey][:3]

    def _apply_readout(x):
        if len(mask.shape) != 4:
            raise ValueError("flags should have shape (n, m, q, l)!")
        if len(x.shape) != 4:
            raise ValueError("input should have shape (n, m, q, l)!")
        dev.require_device()
        dtype = dev.float_dtype(x)
        xt = dev.to_device(x, dtype)
        per = math.prod(xt.shape[1:])
        if xt.shape[0] < len(keys):
            raise IndexError("input has fewer modules than there are keys")
        if per < pixels:
            raise ValueError("input module shape does not match the flags")
        words, before, counts = _words()
        out = [torch.empty(c, dtype=dtype, device="cuda") for c in counts]
        _lib.call("jubik_readout_gather_words", dev.code(dtype), len(keys), words, before, pixels,
                  dev.ptr(xt), per, dev.ptrs(out), dev.stream())
        return Vector({key: dev.like_input(v, x) for key, v in zip(keys, out)})

    def _transpose(vec, like_shape=None):
        """Scatter read-out vectors back into a zero (M, E, H, W) array."""
        dev.require_device()
        shape = mask.shape
        first = vec[keys[0]]
        dtype = dev.float_dtype(first)
        words, before, counts = _words()
        vs = [dev.to_device(vec[key], dtype) for key in keys]
        if any(v.numel() < c for v, c in zip(vs, counts)):
            raise ValueError("read-out vectors are shorter than the kept pixels")
        # modules that are not read out stay zero
        new = torch.empty if len(keys) == shape[0] else torch.zeros
        out = new(shape, dtype=dtype, device="cuda")
        _lib.call("jubik_readout_scatter_words", dev.code(dtype), len(keys), words, before, pixels,
                  dev.ptrs(vs), dev.ptr(out), dev.stream())
        return dev.like_input(out, first)

    _apply_readout.transpose = _transpose
    _apply_readout.mask = mask
    _apply_readout.keys = tuple(keys)
    return _apply_readout
