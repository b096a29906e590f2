"""`ensure_contiguous` decorator (the reference's fma/utils/contiguous.py:15-21): every tensor argument, also inside
containers, is made contiguous before the wrapped function sees it."""

from functools import wraps
from typing import Any, Callable

import torch
from torch.utils._pytree import tree_map


def _leaf(x: Any) -> Any:
    return x.contiguous() if isinstance(x, torch.Tensor) else x


def _contiguous(x: Any) -> Any:
    # an argument that is no container is handled without building a tree (which took 11 us of host time per call)
    if isinstance(x, torch.Tensor):
        return x.contiguous()
    return tree_map(_leaf, x) if isinstance(x, (tuple, list, dict)) else x


def ensure_contiguous(func: Callable) -> Callable:
    @wraps(func)
    def inner(*args, **kwargs):
        return func(*[_contiguous(x) for x in args], **{name: _contiguous(x) for name, x in kwargs.items()})

    return inner
