"""Registration of this package's operators.

`hip_op` stands where torch.library.custom_op would: same operator namespace and name, schema inferred from the function's
annotations, mutated arguments declared, a body that tracing does not look into. The difference is the price of a call: the
wrappers that custom_op puts around every call take 14 us of host time here against 2.7 us for an operator defined on the
dispatcher directly, and a step of this package is a dozen calls.

What the wrappers do beside dispatching is kept:
 * a call advances the version counters of the arguments it declares as mutated (0.5 us; as a kernel of its own in front of
   the body, where custom_op does it, 7 to 10 us), so that autograd still refuses a backward pass through a buffer that an
   operator has overwritten since it was saved;
 * the body runs without recording gradients, whatever the grad mode around the call;
 * under a functorch transform (torch.func.grad, vmap, ...) the call goes to an operator that custom_op has made.
"""

import inspect
from operator import itemgetter
from typing import Callable, Iterable

import torch
from torch._C import _increment_version

from .constants import LIBRARY_NAME

_library = torch.library.Library(LIBRARY_NAME, "FRAGMENT")


def hip_op(name: str, mutates_args: Iterable[str]) -> Callable:
    def register(fn: Callable) -> torch._ops.OpOverload:
        parameters = inspect.signature(fn).parameters.values()
        mutated = [i for i, p in enumerate(parameters) if p.name in mutates_args]
        optional = any(p.annotation is not torch.Tensor for p in parameters if p.name in mutates_args)
        written = itemgetter(*mutated) if len(mutated) > 1 else itemgetter(slice(mutated[0], mutated[0] + 1))

        def body(*args) -> None:
            # (what torch.autograd.graph.increment_version calls; inference tensors have no version and are passed over)
            if optional:
                _increment_version([args[i] for i in mutated if i < len(args) and args[i] is not None])
            else:
                _increment_version(written(args))
            if not torch.is_grad_enabled():
                return fn(*args)
            torch._C._set_grad_enabled(False)  # (torch.no_grad() would take 1.9 us)
            try:
                return fn(*args)
            finally:
                torch._C._set_grad_enabled(True)

        _library.define(name + torch.library.infer_schema(fn, mutates_args=mutates_args))
        # every backend key: a tensor that is not on the GPU reaches the body, which says so
        _library.impl(name, body, "CompositeExplicitAutograd")
        torch.library.register_fake(f"{LIBRARY_NAME}::{name}", lambda *args, **kwargs: None, lib=_library)
        transformed = torch.library.custom_op(f"{LIBRARY_NAME}::{name}_in_transform", fn, mutates_args=mutates_args)
        _library.impl(name, transformed, "FuncTorchDynamicLayerFrontMode")
        op = getattr(getattr(torch.ops, LIBRARY_NAME), name).default
        op.__doc__ = fn.__doc__
        return op

    return register
