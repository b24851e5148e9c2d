"""Autocast handling for the autograd functions.

Same behaviour as stk/backend/autocast.py:19-37: under torch.autocast the
forward casts every floating-point GPU tensor argument (float64 excepted) to
the autocast GPU dtype and then runs with autocast switched off; the backward
always runs with autocast switched off.
"""
import functools

import torch


def _castable(x):
    return isinstance(x, torch.Tensor) and x.is_cuda and x.is_floating_point() and x.dtype != torch.float64


def _cast_tree(x, dtype):
    if _castable(x):
        return x.to(dtype)
    if isinstance(x, (list, tuple)):
        return type(x)(_cast_tree(y, dtype) for y in x)
    if isinstance(x, dict):
        return {k: _cast_tree(v, dtype) for k, v in x.items()}
    return x


def casts(*tensors):
    """Whether a function wrapped by custom_fwd would be called on other tensors than these."""
    return torch.is_autocast_enabled() and any(_castable(t) and t.dtype != torch.get_autocast_gpu_dtype() for t in tensors)


def custom_fwd(fwd):
    @functools.wraps(fwd)
    def wrapper(*args, **kwargs):
        if not torch.is_autocast_enabled():
            return fwd(*args, **kwargs)
        dtype = torch.get_autocast_gpu_dtype()
        with torch.autocast(device_type="cuda", enabled=False):
            return fwd(*_cast_tree(args, dtype), **_cast_tree(kwargs, dtype))
    return wrapper


def custom_bwd(bwd):
    @functools.wraps(bwd)
    def wrapper(*args, **kwargs):
        with torch.autocast(device_type="cuda", enabled=False):
            return bwd(*args, **kwargs)
    return wrapper
