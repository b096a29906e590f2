"""The fp32 SwiGLU layer as three operators (router, routing index, experts) against the general path (the switch
fuse_swiglu_backward off), which runs the library's router and an autograd node per product, and against the same layer in float64:
both paths round fp32 sums of up to a few hundred terms of size one, so each stays within 1e-5 of float64 (2-norms) and of the other."""

import pytest
import torch
import torch.nn.functional as F

from fma import KernelBackend, MoE, swiglu_packed
from fma.modules.moe import cuda_implementation as ci

from gpu_util import DEV

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _layer(E, k, H, I, seed=0):
    torch.manual_seed(seed)
    moe = MoE(E, k, H, I, swiglu_packed, True, False, 0.2).to(DEV)
    with torch.no_grad():
        moe.gate.weight.normal_(0, 0.3)
    return moe


def _step(moe, x, dy, dlogits):
    moe.zero_grad()
    x = x.clone().requires_grad_()
    y, logits = moe(x, kernel_backend=KernelBackend.cuda)
    torch.autograd.backward((y, logits), (dy, dlogits))
    return dict(y=y.detach(), logits=logits.detach(), x=x.grad, **{n: p.grad.clone() for n, p in moe.named_parameters()})


def _reference(moe, x, dy, dlogits):
    x = x.double().requires_grad_()
    gate, w1, w2 = (p.detach().double().requires_grad_() for p in (moe.gate.weight, moe.c_fc.weight, moe.c_proj.weight))
    logits = x @ gate.T
    top, chosen = logits.topk(moe.top_k, dim=-1)
    weights = top.softmax(-1)
    y = torch.zeros_like(x)
    for e in range(moe.num_experts):
        t, j = (chosen == e).nonzero(as_tuple=True)
        up, g = (x[t] @ w1[e].T).chunk(2, -1)
        y = y.index_add(0, t, weights[t, j, None] * ((up * F.silu(g)) @ w2[e].T))
    torch.autograd.backward((y, logits), (dy.double(), dlogits.double()))
    return {"y": y.detach(), "logits": logits.detach(), "x": x.grad, "gate.weight": gate.grad, "c_fc.weight": w1.grad,
            "c_proj.weight": w2.grad}  # fmt: skip


def _close(a, b):
    for n in b:
        scale = b[n].double().norm() + 1e-30
        assert float((a[n].double() - b[n].double()).norm() / scale) <= TOL, n


@pytest.mark.parametrize(
    "E,k,H,I,T",
    [(8, 2, 256, 512, 512), (8, 2, 256, 512, 1), (5, 5, 24, 8, 17), (64, 8, 72, 40, 33), (65, 1, 40, 16, 16), (130, 64, 64, 24, 50)],
)
def test_against_the_general_path_and_float64(E, k, H, I, T, monkeypatch):
    moe = _layer(E, k, H, I)
    x, dy = torch.randn(T, H, device=DEV), torch.randn(T, H, device=DEV)
    dlogits = torch.randn(T, E, device=DEV)
    calls = []
    real = ci.swiglu_experts_f32_cuda
    monkeypatch.setattr(ci, "swiglu_experts_f32_cuda", lambda *a: (calls.append(1), real(*a))[1])
    got = _step(moe, x, dy, dlogits)
    assert calls == [1]
    moe.fuse_swiglu_backward = False
    general = _step(moe, x, dy, dlogits)
    assert calls == [1]
    _close(got, general)
    _close(got, _reference(moe, x, dy, dlogits))
    moe.fuse_swiglu_backward = True
    with torch.no_grad():
        y, logits = moe(x, kernel_backend=KernelBackend.cuda)
    assert torch.equal(y, got["y"]) and torch.equal(logits, got["logits"])


def test_some_gradients_only():
    moe = _layer(8, 2, 64, 32)
    x, dy = torch.randn(40, 64, device=DEV), torch.randn(40, 64, device=DEV)
    every = _step(moe, x, dy, torch.zeros(40, 8, device=DEV))
    for name in ("gate.weight", "c_fc.weight", "c_proj.weight"):
        for n, p in moe.named_parameters():
            p.requires_grad_(n == name)
        moe.zero_grad()
        moe(x, kernel_backend=KernelBackend.cuda)[0].backward(dy)
        for n, p in moe.named_parameters():
            assert torch.equal(p.grad, every[n]) if n == name else p.grad is None


def test_choice_of_equal_values_infinities_and_nan():
    """largest first, NaN above every number, equal values (and zeros of either sign) in ascending column order"""
    inf, nan = float("inf"), float("nan")
    rows = torch.tensor([[1, 3, 3, 2, 3, 0], [0, -0.0, 0, -1, -0.0, 0], [inf, 1, inf, -inf, 2, 2], [nan, 5, inf, nan, 1, 0],
                         [-inf] * 6, [-1, -2, -3, -1, -2, -3]], device=DEV)  # fmt: skip
    T, E, k = 6, 6, 4
    eye = torch.zeros(E, 8, device=DEV)
    eye[:, :6] = torch.eye(6, device=DEV)
    finite = rows.nan_to_num(nan=0.0, posinf=0.0, neginf=0.0)
    logits, weights = torch.empty(T, E, device=DEV), torch.empty(T, k, device=DEV)
    selected = torch.empty(T, k, dtype=torch.int32, device=DEV)
    hist = torch.empty(1, E, dtype=torch.uint32, device=DEV)
    x = torch.zeros(T, 8, device=DEV)
    x[:, :6] = finite
    ci.router_topk_f32_cuda(x, eye, k, logits, weights, selected, hist)
    for t in (0, 1, 5):
        expect = sorted(range(E), key=lambda n: (-float(finite[t, n]), n))[:k]
        assert selected[t].tolist() == expect
        assert torch.allclose(weights[t], finite[t][expect].softmax(-1), rtol=1e-6)
    assert hist.to(torch.int64).sum() == T * k
    # a single reduction element per logit: the values arrive as they are
    one = torch.zeros(T, 8, device=DEV)
    one[:, 0] = 1.0
    for t in (2, 3, 4):
        gate = torch.zeros(E, 8, device=DEV)
        gate[:, 0] = rows[t]
        ci.router_topk_f32_cuda(one, gate, k, logits, weights, selected, hist)
        ref = rows[t].nan_to_num(nan=float("inf")) if t == 3 else rows[t]
        key = lambda n: (not bool(torch.isnan(rows[t, n])), -float(ref[n]), n)  # noqa: E731
        assert selected[0].tolist() == sorted(range(E), key=key)[:k]


def test_second_derivative_of_the_logits():
    moe = _layer(8, 2, 64, 32)
    x = torch.randn(20, 64, device=DEV)
    results = []
    for fused in (True, False):
        moe.fuse_swiglu_backward = fused
        xi = x.clone().requires_grad_()
        _, logits = moe(xi, kernel_backend=KernelBackend.cuda)
        (g,) = torch.autograd.grad(logits.logsumexp(-1).pow(2).sum(), xi, create_graph=True)
        results.append(torch.autograd.grad(g.pow(2).sum(), (xi, moe.gate.weight)))
    for a, b in zip(*results):
        assert float((a - b).norm() / b.norm()) < TOL


@pytest.mark.parametrize("case", ["hook", "subclass", "instance", "autocast", "misaligned", "gate"])
def test_what_takes_the_general_path(case, monkeypatch):
    moe = _layer(8, 2, 64, 32)
    x = torch.randn(20, 64, device=DEV)
    expect = moe(x, kernel_backend=KernelBackend.cuda)
    calls, seen = [], []
    real = ci.swiglu_experts_f32_cuda
    monkeypatch.setattr(ci, "swiglu_experts_f32_cuda", lambda *a: (calls.append(1), real(*a))[1])
    context = torch.no_grad()
    if case == "hook":
        moe.gate.register_forward_hook(lambda m, i, o: seen.append(1))
    elif case == "subclass":
        moe.__class__ = type("Sub", (MoE,), {"_get_topk": lambda self, l: (seen.append(1), MoE._get_topk(self, l))[1]})
    elif case == "instance":
        own = moe.c_fc.cuda_forward
        moe.c_fc.cuda_forward = lambda **kw: (seen.append(1), own(**kw))[1]
    elif case == "autocast":
        context = torch.autocast("cuda", dtype=torch.bfloat16)
        seen.append(1)
        moe.fuse_swiglu_backward = False
        with context:
            expect = moe(x, kernel_backend=KernelBackend.cuda)
        moe.fuse_swiglu_backward = True
    elif case == "misaligned":
        x = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(20, 64)
        seen.append(1)
    elif case == "gate":
        moe.gate = type("Gate", (torch.nn.Linear,), {"forward": lambda self, v: (seen.append(1), F.linear(v, self.weight))[1]})(
            64, 8, bias=False, device=DEV
        )
        moe.gate.weight = torch.nn.Parameter(_layer(8, 2, 64, 32).gate.weight.detach().clone())
    with context:
        got = moe(x, kernel_backend=KernelBackend.cuda)
    assert seen and calls == []
    for a, b in zip(got, expect):
        assert a.dtype == b.dtype and float((a.float() - b.float()).norm() / b.float().norm()) < TOL


@pytest.mark.parametrize("H,inter", [(64, 36), (60, 64), (64, 33), (12, 16)])
def test_sizes_that_are_no_multiples_of_eight_are_refused(H, inter):
    moe = _layer(4, 2, H, inter)
    with pytest.raises(AssertionError):
        moe(torch.randn(20, H, device=DEV), kernel_backend=KernelBackend.cuda)


@pytest.mark.parametrize("strided", ["tokens", "gate"])
def test_second_derivative_of_strided_tokens_and_gate(strided):
    moe = _layer(8, 2, 64, 32)
    wide = torch.randn(20, 72, device=DEV)
    x = wide[:, :64] if strided == "tokens" else wide[:, :64].contiguous()
    if strided == "gate":
        moe.gate.weight = torch.nn.Parameter(moe.gate.weight.detach().t().contiguous().t())
    results = []
    for fused in (True, False):
        moe.fuse_swiglu_backward = fused
        xi = x.detach().requires_grad_()
        assert xi.is_contiguous() == (strided != "tokens")
        _, logits = moe(xi, kernel_backend=KernelBackend.cuda)
        first = torch.autograd.grad(logits.logsumexp(-1).pow(2).sum(), (xi, moe.gate.weight), create_graph=True)
        results.append([*first, *torch.autograd.grad(sum(g.pow(2).sum() for g in first), (xi, moe.gate.weight))])
    for a, b in zip(*results):
        assert float((a - b).norm() / b.norm()) < TOL


@pytest.mark.parametrize(
    "E,H,k,fused",
    [(64, 1152, 8, True), (128, 576, 8, True), (1000, 24, 4, True), (64, 256, 32, True), (64, 256, 1, True), (64, 1664, 2, False), (129, 576, 2, False),
     (64, 1024, 64, False), (64, 264, 1, False), (8, 2048, 2, False)],
)  # fmt: skip
def test_large_routers_are_the_library_s(E, H, k, fused, monkeypatch):
    moe = _layer(E, k, H, 16)
    x, dy, dlogits = torch.randn(30, H, device=DEV), torch.randn(30, H, device=DEV), torch.randn(30, E, device=DEV)
    calls = []
    for name in ("router_topk_f32_cuda", "swiglu_experts_f32_cuda"):
        real = getattr(ci, name)
        monkeypatch.setattr(ci, name, lambda *a, real=real, name=name: (calls.append(name), real(*a))[1])
    got = _step(moe, x, dy, dlogits)
    assert calls == ["router_topk_f32_cuda"] * fused + ["swiglu_experts_f32_cuda"]
    moe.fuse_swiglu_backward = False
    _close(got, _step(moe, x, dy, dlogits))


def _peak(step):
    step()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    step()
    return torch.cuda.max_memory_allocated() - before


@pytest.mark.parametrize("T,fused", [(9000, True), (9600, False)])  # 28096 bytes a token
def test_memory_of_large_passes(T, fused):
    """past the size where host time matters a pass takes no more memory than the general path; up to it, without a backward, no more
    than the rows of the tokens, the pre-activation and the activation (and the output) at once"""
    moe = _layer(8, 2, 512, 1000)
    x, dy = torch.randn(T, 512, device=DEV), torch.randn(T, 512, device=DEV)

    def infer():
        with torch.no_grad():
            moe(x, kernel_backend=KernelBackend.cuda)

    def train():
        moe.zero_grad(set_to_none=True)
        moe(x, kernel_backend=KernelBackend.cuda)[0].backward(dy)

    peaks = []
    for switch in (True, False):
        moe.fuse_swiglu_backward = switch
        peaks.append([_peak(infer), _peak(train)])
    few = 1 << 22  # logits, weights, choices and index
    assert peaks[0][0] <= T * 4 * (2 * (512 + 3000) + 512) + few
    if not fused:
        assert peaks[0] == peaks[1]


def test_scratch_of_a_backward_for_the_second_projection_alone(monkeypatch):
    moe = _layer(8, 2, 64, 32)
    moe.c_fc.weight.requires_grad_(False)
    moe.gate.weight.requires_grad_(False)
    seen = []
    real = ci.swiglu_experts_backward_f32_cuda
    monkeypatch.setattr(ci, "swiglu_experts_backward_f32_cuda", lambda *a: (seen.append(a), real(*a))[1])
    moe(torch.randn(40, 64, device=DEV), kernel_backend=KernelBackend.cuda)[0].sum().backward()
    ((*_, o_grad, act_grad, h_grad, x_grad, gates_grad, weight1_grad, weight2_grad),) = seen
    assert act_grad is h_grad is x_grad is weight1_grad is None and o_grad is not None and weight2_grad is not None
