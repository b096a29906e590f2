"""What torch.library.custom_op promises of an operator with mutated arguments holds for the operators registered by hip_op
(fma/_ops.py). Runs on CPU tensors: a body that refuses them has had its arguments marked before it was entered, as with custom_op."""

import pytest
import torch
from torch.library import custom_op

import fma  # noqa: F401  (registers the operators)
import fma.modules.moe.cuda_implementation  # noqa: F401
from fma._ops import hip_op
from fma.constants import LIBRARY_NAME


def _fill(x: torch.Tensor, y: torch.Tensor) -> None:
    assert not (x * 1).requires_grad
    y.zero_()
    y.numpy()[...] = 5.0


hip_fill = hip_op("test_fill", mutates_args={"y"})(_fill)
custom_fill = custom_op("fma_test::fill", mutates_args={"y"})(_fill)
_OPERATORS = sorted(n.split("::")[1].split(".")[0] for n in torch._C._dispatch_get_all_op_names()
                    if n.startswith(LIBRARY_NAME + "::") and not n.endswith("_in_transform") and "test_" not in n)  # fmt: skip


def test_every_operator_is_here():
    assert len(_OPERATORS) >= 20 and "grouped_gemm_cuda" in _OPERATORS and "moe_decode_cuda" in _OPERATORS


@pytest.mark.parametrize("name", _OPERATORS)
def test_mutated_arguments_advance_their_version(name):
    op = getattr(getattr(torch.ops, LIBRARY_NAME), name).default
    args = []
    for a in op._schema.arguments:
        kind = str(a.type)
        args.append(torch.ones(2) if "Tensor" in kind else False if kind == "bool" else 1.0 if kind == "float" else 1)
    before = [a._version if isinstance(a, torch.Tensor) else 0 for a in args]
    with pytest.raises((RuntimeError, AssertionError)):  # CPU tensors
        op(*args)
    mutated = [bool(a.alias_info and a.alias_info.is_write) for a in op._schema.arguments]
    assert any(mutated)
    for a, was, writes in zip(args, before, mutated):
        if isinstance(a, torch.Tensor):
            assert a._version == was + (1 if writes else 0)


@pytest.mark.parametrize("fill", [custom_fill, hip_fill], ids=["custom_op", "hip_op"])
def test_backward_through_an_overwritten_buffer_is_refused(fill):
    w, saved = torch.ones(3, requires_grad=True), torch.ones(6)
    loss = (w * saved[:3]).sum()
    fill(torch.ones(6), saved)  # through the base of the saved view
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


@pytest.mark.parametrize("fill", [custom_fill, hip_fill], ids=["custom_op", "hip_op"])
def test_modes(fill):
    one = torch.ones(3)
    for x in (one, torch.ones(3, requires_grad=True)):
        for y in (torch.ones(3), torch.ones(3, requires_grad=True).detach()):
            fill(x, y)
            assert y._version >= 1 and not y.requires_grad and torch.equal(y, torch.full((3,), 5.0))
            assert torch.is_grad_enabled()
    leaf = torch.ones(3, requires_grad=True)
    with torch.no_grad():
        fill(one, leaf)
        assert not torch.is_grad_enabled()
    assert leaf._version >= 1
    with torch.inference_mode():
        inside, version = torch.ones(3), leaf._version
        fill(one, inside)
        fill(inside, leaf)
    assert leaf._version > version


@pytest.mark.parametrize("fill", [custom_fill, hip_fill], ids=["custom_op", "hip_op"])
def test_functorch_transforms(fill):
    def f(v, use):
        y = torch.ones(3)
        fill(use(v), y)
        return (v * y).sum()

    one = torch.ones(3)
    assert torch.equal(torch.func.grad(f)(one, lambda v: one), torch.full((3,), 5.0))
    with pytest.raises(RuntimeError):  # there is no derivative: not a gradient that leaves it out
        torch.func.grad(f)(one, lambda v: v)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda v: (fill(v, torch.ones(3)), v)[1])(torch.ones(2, 3))
