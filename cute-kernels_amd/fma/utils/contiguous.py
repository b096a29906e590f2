"""`ensure_contiguous` decorator (the reference's fma/utils/contiguous.py:15-21): every tensor argument, also inside
containers, is made contiguous before the wrapped function sees it."""

from enum import Enum
from functools import wraps
from typing import Any, Callable

import torch
from torch.utils._pytree import tree_map


def _leaf(x: Any) -> Any:
    return x.contiguous() if isinstance(x, torch.Tensor) else x


# arguments of this package's functions that no tensor can be inside of (the first argument of an autograd function is a context)
_PLAIN = (int, float, str, type(None), torch.dtype, Enum, torch.autograd.function.FunctionCtx)


def _contiguous(x: Any) -> Any:
    # a tensor or a plain value is handled without building a tree (which took 11 us of host time per call); anything else may be
    # a container, of a type that torch's pytree knows by itself or that a program has registered with it
    if isinstance(x, torch.Tensor):
        return x.contiguous()
    return x if isinstance(x, _PLAIN) else tree_map(_leaf, x)


def ensure_contiguous(func: Callable) -> Callable:
    @wraps(func)
    def inner(*args, **kwargs):
        return func(*[_contiguous(x) for x in args], **{name: _contiguous(x) for name, x in kwargs.items()})

    return inner
