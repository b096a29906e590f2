"""What the host decides and records about the fp32 SwiGLU layer, on the CPU: the operators are replaced by the same values from torch."""

import pytest
import torch
import torch.nn.functional as F
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from fma import KernelBackend, MoE, swiglu_packed
from fma.modules.moe import cuda_implementation as ci

TOL = 1e-5  # fp32 sums of 24 terms of size one


def _router_in_torch(x, gate_weight, top_k, logits, weights, selected, token_block_hist, kept):
    with torch.no_grad():
        logits.copy_(x @ gate_weight.t())
        top, chosen = logits.topk(top_k, dim=-1)
        weights.copy_(top.softmax(-1))
        selected.copy_(chosen)
        kept.copy_(top)


def _router_backward_in_torch(kept, selected, weights_grad, logits_output_grad, logits_grad):
    with torch.no_grad():
        columns = selected.long()
        s = kept.softmax(-1)
        logits_grad.copy_(torch.zeros_like(logits_grad) if logits_output_grad is None else logits_output_grad)
        if weights_grad is not None:
            logits_grad.scatter_add_(1, columns, s * (weights_grad - (s * weights_grad).sum(-1, keepdim=True)))


class _GatedSum:
    """stands for the experts' node: depends on tokens and gates as they do, and is differentiated by autograd"""

    @staticmethod
    def apply(x, gates, *_):
        return x * gates.pow(2).sum(-1, keepdim=True)


@pytest.mark.parametrize("strided", ["tokens", "gate", "neither"])
def test_second_derivative_with_strided_arguments(strided, monkeypatch):
    T, H, E, k = 12, 24, 6, 2
    torch.manual_seed(0)
    wide = torch.randn(T, H + 8)
    x = wide[:, :H] if strided == "tokens" else wide[:, :H].contiguous()
    w = torch.randn(H, E).t() if strided == "gate" else torch.randn(E, H)
    assert (x.is_contiguous(), w.is_contiguous()) == (strided != "tokens", strided != "gate")
    monkeypatch.setattr(ci, "router_topk_f32_cuda", _router_in_torch)
    monkeypatch.setattr(ci, "router_topk_backward_f32_cuda", _router_backward_in_torch)
    monkeypatch.setattr(ci, "build_routing_index", lambda *_: (None,) * 5)
    monkeypatch.setattr(ci, "_Fp32SwigluExperts", _GatedSum)

    def layer(x, w):
        y, logits = ci.fp32_swiglu_layer(x, w, *[None] * 6, k)
        return y, logits

    def library(x, w):
        logits = F.linear(x, w)
        gates = logits.topk(k, dim=-1).values.softmax(-1)
        return _GatedSum.apply(x, gates), logits

    results = []
    for fn in (layer, library):
        xi, wi = x.detach().requires_grad_(), w.detach().requires_grad_()
        assert xi.stride() == x.stride() and wi.stride() == w.stride()
        y, logits = fn(xi, wi)
        first = torch.autograd.grad(y.sin().sum() + logits.logsumexp(-1).pow(2).sum(), (xi, wi), create_graph=True)
        results.append([*first, *torch.autograd.grad(sum(g.pow(2).sum() for g in first), (xi, wi))])
    for got, expect in zip(*results):
        assert float((got - expect).norm() / expect.norm()) < TOL


@pytest.mark.parametrize("how", ["logits changed in place", "is_grads_batched", "vmap"])
def test_what_the_library_calls_allow(how, monkeypatch):
    T, H, E, k = 12, 24, 6, 2
    torch.manual_seed(0)
    x, w, v = torch.randn(T, H, requires_grad=True), torch.randn(E, H), torch.randn(3, T, E)
    monkeypatch.setattr(ci, "router_topk_f32_cuda", _router_in_torch)
    monkeypatch.setattr(ci, "router_topk_backward_f32_cuda", _router_backward_in_torch)
    results = []
    for node in (True, False):
        if node:
            logits, gates = ci._Fp32Router.apply(x, w, k)[:2]
        else:
            logits = F.linear(x, w)
            gates = logits.topk(k, dim=-1).values.softmax(-1)
        if how == "logits changed in place":
            logits.mul_(2.0)
            results.append(torch.autograd.grad(gates.sin().sum() + logits.pow(2).sum(), x)[0])
        elif how == "is_grads_batched":
            results.append(torch.autograd.grad(logits, x, v, is_grads_batched=True)[0])
        else:
            results.append(torch.vmap(lambda g: torch.autograd.grad(logits, x, g)[0])(v))
    assert float((results[0] - results[1]).norm() / results[1].norm()) < TOL


class _Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func.name())
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("how", ["fake mode", "make_fx"])
@pytest.mark.filterwarnings("error")
def test_tracing_takes_the_general_path(how):
    """a traced layer is made of the library's router and the operators of the general path, and no address is asked for"""
    fake = FakeTensorMode(allow_non_fake_inputs=True)
    with fake, torch.device("cuda"):
        moe = MoE(8, 2, 64, 32, swiglu_packed, True, False, 0.02)
        x = torch.randn(20, 64)

    def layer(x):
        return moe(x, kernel_backend=KernelBackend.cuda)

    if how == "make_fx":
        with fake:
            names = [str(n.target) for n in make_fx(layer)(x).graph.nodes]
        linear, of_layer = "aten.mm.default", "f32_cuda.default"
    else:
        with fake, _Names() as seen:
            layer(x)
        names, linear, of_layer = seen.names, "aten::mm", "f32_cuda"
    assert linear in names and not any(n.endswith(of_layer) for n in names), names
    # outside the mode its tensors are still no tensors with an address
    assert moe._fp32_operands(x, KernelBackend.cuda) is None
