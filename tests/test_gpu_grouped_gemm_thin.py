"""The grouped product for a few rows per group (fma_grouped_gemm_thin) against the tile kernel's entry points, bit for bit:
both walk the reduction in the same order with the same instruction. Sizes around the edges of its units: 16 / 32 / 64 rows
of a pass, 32 / 64 weight rows of a wavefront, 64 reduction elements of a step, more than 64 groups."""

import pytest
import torch
from torch.autograd import forward_ad

from fma.modules.moe import cuda_implementation as ci

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize(
    "sizes,N,K",
    [
        ([1], 16, 8),
        ([0, 1, 0, 2, 15, 16, 17, 0], 48, 72),  # 32 weight rows per wavefront
        ([33, 1, 0, 32], 96, 64),  # 64 weight rows per wavefront from here on
        ([64, 65, 0, 130, 16, 17], 144, 2056),
        ([7, 31, 64], 4096, 1408),
        ([1] * 70 + [0] * 20 + [3] * 7, 64, 192),
        # several passes of an expert, side by side and more of them than that (16): 32 rows each, then 64
        ([1] * 70 + [600, 0, 33, 2, 64], 336, 136),
        ([1100, 0, 65, 3], 336, 136),
    ],
)
def test_thin_product_equals_the_tile_kernel(sizes, N, K, swiglu, bias, dtype):
    E, R, k = len(sizes), sum(sizes), 2
    g = torch.Generator().manual_seed(N + K)
    counts = torch.tensor(sizes, dtype=torch.int32, device=DEV).view(torch.uint32)
    offsets = torch.tensor(sizes).cumsum(0).to(torch.int32).to(DEV).view(torch.uint32)
    W = (torch.randn(E, N, K, generator=g) * 0.1).to(dtype).to(DEV)
    b = torch.randn(E, N, generator=g).to(dtype).to(DEV) if bias else None
    T = R // k + 1
    x = torch.randn(T, K, generator=g).to(dtype).to(DEV)
    slots = torch.randperm(T * k, generator=g)[:R].to(torch.int32).to(DEV)
    packed = x[(slots // k).long()].contiguous()
    cols = N // 2 if swiglu else N

    expect = torch.empty(R, cols, device=DEV, dtype=dtype)
    if swiglu:
        ci.grouped_gemm_swiglu_cuda(packed, W, counts, None, expect, b)
    else:
        ci.grouped_gemm_ragged_cuda(packed, W, expect, counts, False, 0, N, K, False, True, b)
    for rows, index, divisor in ((packed, None, 1), (x, slots, k)):
        got = torch.full_like(expect, float("nan"))
        ci.grouped_gemm_thin_cuda(rows, index, divisor, W, b, counts, offsets, got, swiglu)
        assert torch.equal(got, expect), f"gathered={index is not None}"


@pytest.mark.parametrize("T,k,E", [(1, 8, 64), (5, 2, 8), (129, 2, 8), (33, 4, 130)])
@pytest.mark.parametrize("bias", [False, True])
def test_layer_without_backward_equals_the_training_forward(T, k, E, bias):
    from fma import KernelBackend, MoE, swiglu_packed

    torch.manual_seed(T)
    moe = MoE(E, k, 328, 200, swiglu_packed, True, bias, 0.05).to(torch.bfloat16).to(DEV)
    x = torch.randn(T, 328, device=DEV).bfloat16()
    expect, expect_logits = moe(x, kernel_backend=KernelBackend.cuda)
    with torch.no_grad():
        y, logits = moe(x, kernel_backend=KernelBackend.cuda)
    assert torch.equal(logits, expect_logits) and torch.equal(y, expect)


# Routing on which the streaming kernel keeps the products, and on which it leaves them to the tile kernel (the choice is made on
# the device where an expert can take more than four passes): passes of 32 rows, of 64 rows, the one-call forward pass.
@pytest.mark.parametrize("hot", [0, 1, 4, 8])
@pytest.mark.parametrize("T,k,E", [(129, 8, 128), (192, 8, 128), (333, 8, 128), (300, 2, 128), (1030, 8, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_layer_without_backward_under_uneven_routing(T, k, E, hot, bias):
    from fma import KernelBackend, MoE, swiglu_packed

    torch.manual_seed(T + hot)
    moe = MoE(E, k, 136, 72, swiglu_packed, True, bias, 0.05).to(torch.bfloat16).to(DEV)
    x = torch.randn(T, 136, device=DEV).bfloat16()
    x[:, 0] = 8.0
    with torch.no_grad():  # these experts are in every token's choice
        moe.gate.weight[torch.randperm(E)[: min(hot, k)], 0] = 4.0
    expect, expect_logits = moe(x, kernel_backend=KernelBackend.cuda)
    with torch.no_grad():
        for _ in range(2):  # (the second finds what the first left in the workspace)
            y, logits = moe(x, kernel_backend=KernelBackend.cuda)
            assert torch.equal(logits, expect_logits) and torch.equal(y, expect)


def test_replays_take_either_kernel():
    """a captured pass in which the device chooses between the two kernels: even and collapsed routing in turn"""
    from fma import KernelBackend, MoE, swiglu_packed

    T, k, E, H = 200, 8, 128, 136
    torch.manual_seed(3)
    moe = MoE(E, k, H, 72, swiglu_packed, True, True, 0.05).to(torch.bfloat16).to(DEV)
    with torch.no_grad():
        moe.gate.weight[:8, 0] = 4.0
    x_static = torch.randn(T, H, device=DEV).bfloat16()
    run = lambda x: moe(x, kernel_backend=KernelBackend.cuda)
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                run(x_static)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y_static, logits_static = run(x_static)
    for step, common in enumerate((8.0, 0.0, 8.0, 8.0, 0.0, 0.0)):  # 8: every token chooses the first eight experts
        x = torch.randn(T, H, device=DEV).bfloat16()
        x[:, 0] = common
        expect, expect_logits = run(x)  # the training forward, eager, between the replays
        x_static.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y_static, expect) and torch.equal(logits_static, expect_logits), step


def no_grad_sum(run, moe, x):
    with torch.no_grad():  # (inside the transform, where the grad mode outside does not count)
        return run(moe, x)[0].float().sum()


@pytest.mark.parametrize("T", [7, 100, 300])  # one native call; more than 64 and than 1024 (token, choice) slots
def test_layer_without_backward_in_other_forms(T):
    """what the general path takes or refuses is taken or refused on the kernels for a few rows as well: tracing without a
    graph break, weights of any strides, forward-mode AD and functorch transforms (refused), a subclass's own expert computation"""
    from fma import KernelBackend, MoE, swiglu_packed

    torch.manual_seed(T)
    E, k, H, I = 16, 4, 128, 64
    moe = MoE(E, k, H, I, swiglu_packed, True, True, 0.05).to(torch.bfloat16).to(DEV)
    x = torch.randn(T, H, device=DEV).bfloat16()
    run = lambda m, x: m(x, kernel_backend=KernelBackend.cuda)
    with torch.no_grad():
        y, logits = run(moe, x)
        for got in (torch.compile(lambda x: run(moe, x), fullgraph=True)(x),
                    torch.compile(lambda x: run(moe, x), fullgraph=True, dynamic=True)(x)):
            assert torch.equal(got[0], y) and torch.equal(got[1], logits)

        with forward_ad.dual_level():
            with pytest.raises(NotImplementedError):
                run(moe, forward_ad.make_dual(x, torch.ones_like(x)))
        for transform in (torch.func.grad, torch.vmap):
            with pytest.raises(RuntimeError):
                transform(lambda x: no_grad_sum(run, moe, x))(x[None] if transform is torch.vmap else x)

        class Doubled(MoE):
            def _compute_experts(self, *args, **kwargs):
                return 2 * super()._compute_experts(*args, **kwargs)

        moe.__class__ = Doubled
        assert torch.equal(run(moe, x)[0], 2 * y)  # (a power of two: exact)
        moe.__class__ = MoE

        moe._compute_experts = lambda *args, **kwargs: 2 * MoE._compute_experts(moe, *args, **kwargs)
        for call in (run, torch.compile(run, fullgraph=True)):
            assert torch.equal(call(moe, x)[0], 2 * y)
        del moe._compute_experts

        moe.fuse_swiglu_backward = False
        moe.c_proj.cuda_forward = lambda **kwargs: 2 * type(moe.c_proj).cuda_forward(moe.c_proj, **kwargs)
        assert torch.equal(run(moe, x)[0], 2 * y)
        moe.fuse_swiglu_backward = True
        assert torch.equal(run(moe, x)[0], y)
        del moe.c_proj.cuda_forward

        for p in moe.parameters():
            p.data = p.data.transpose(-1, -2).contiguous().transpose(-1, -2)
        assert not moe.c_fc.weight.is_contiguous()
        got = run(moe, x.t().contiguous().t().view(T, H))
        assert torch.equal(got[0], y) and torch.equal(got[1], logits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "T,H,E,k",
    # one and several workgroups, partial blocks of 16 tokens and experts, the split reduction (E <= 16), one to many steps of
    # 128 with a remainder, the most slots and experts
    [(1, 2048, 64, 8), (1, 8, 1, 1), (16, 4096, 8, 2), (17, 136, 17, 3), (65, 512, 16, 2), (128, 4096, 128, 8), (15, 1048, 256, 64),
     (1024, 128, 250, 1)],
)
def test_router_and_index_in_two_launches(T, H, E, k, dtype):
    from fma import _lib

    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    # two halves with the same experts: ties among the logits
    w = (torch.randn(E, H, generator=g) * 0.05).to(dtype)
    w[E // 2 :] = w[: E - E // 2].clone()
    w = w.to(DEV)
    expect_logits, expect_weights, selected, _ = ci.fused_router_with_histogram(x, w, k)
    expect = ci.build_routing_index(selected, E)
    logits, weights = torch.empty_like(expect_logits), torch.empty_like(expect_weights)
    counts, offsets = (torch.empty(E, dtype=torch.uint32, device=DEV) for _ in range(2))
    perm, inv = (torch.empty(T * k, dtype=torch.int32, device=DEV) for _ in range(2))
    rc = _lib.load().fma_router_topk_index(
        x.data_ptr(), w.data_ptr(), T, H, E, k, logits.data_ptr(), weights.data_ptr(), counts.data_ptr(), offsets.data_ptr(),
        perm.data_ptr(), inv.data_ptr(), _lib.dtype_code(dtype), _lib.current_stream(x.device),
    )
    _lib.check(rc, "router_topk_index")
    for got, want, name in zip((logits, weights, counts, offsets, perm, inv),
                               (expect_logits, expect_weights, expect[0], expect[1], expect[2], expect[4]),
                               ("logits", "weights", "counts", "offsets", "perm", "inv")):
        assert torch.equal(got.view(torch.int32) if got.dtype == torch.uint32 else got,
                           want.view(torch.int32) if want.dtype == torch.uint32 else want), name


def _same(got, want):
    """equal, NaN where NaN"""
    return torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0))


def _with_specials(t, g, value):
    """a few elements replaced by infinities, NaN or the type's lowest value"""
    at = torch.randint(0, t.numel(), (3,), generator=g, device="cpu")
    t.view(-1)[at.to(t.device)] = torch.tensor(value, dtype=torch.float64).to(t.dtype).to(t.device)
    return t


_SPECIALS = [[float("inf")] * 3, [float("inf"), float("-inf"), float("nan")], [float("nan")] * 3, [-3.0e38, 3.0e38, -3.0e38]]


@pytest.mark.parametrize("special", range(len(_SPECIALS)))
@pytest.mark.parametrize("swiglu", [False, True])
def test_thin_product_of_infinities_and_nan(special, swiglu):
    sizes, N, K = [33, 1, 0, 70, 17], 144, 136
    E, R = len(sizes), sum(sizes)
    g = torch.Generator().manual_seed(special)
    counts = torch.tensor(sizes, dtype=torch.int32, device=DEV).view(torch.uint32)
    offsets = torch.tensor(sizes).cumsum(0).to(torch.int32).to(DEV).view(torch.uint32)
    W = _with_specials(torch.randn(E, N, K, generator=g).bfloat16().to(DEV), g, _SPECIALS[special])
    x = _with_specials(torch.randn(R, K, generator=g).bfloat16().to(DEV), g, _SPECIALS[special])
    expect, got = (torch.empty(R, N // 2 if swiglu else N, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    if swiglu:
        ci.grouped_gemm_swiglu_cuda(x, W, counts, None, expect, None)
    else:
        ci.grouped_gemm_ragged_cuda(x, W, expect, counts, False, 0, N, K, False, True, None)
        at = 0
        for e, m in enumerate(sizes if special < 3 else []):  # which elements are finite is no matter of rounding
            assert torch.equal(torch.isnan(x[at : at + m].float() @ W[e].float().T), torch.isnan(expect[at : at + m]))
            at += m
    ci.grouped_gemm_thin_cuda(x, None, 1, W, None, counts, offsets, got, swiglu)
    assert _same(got, expect) and (special == 3 or not torch.isfinite(expect).all())


@pytest.mark.parametrize("special", range(len(_SPECIALS)))
@pytest.mark.parametrize("T,H,E,k", [(33, 136, 17, 3), (16, 512, 64, 8), (5, 264, 256, 64)])
def test_router_and_index_of_infinities_and_nan(special, T, H, E, k):
    from fma import _lib

    g = torch.Generator().manual_seed(special + T)
    x = _with_specials(torch.randn(T, H, generator=g).bfloat16().to(DEV), g, _SPECIALS[special])
    w = _with_specials((torch.randn(E, H, generator=g) * 0.05).bfloat16().to(DEV), g, _SPECIALS[special])
    expect_logits, expect_weights, selected, _ = ci.fused_router_with_histogram(x, w, k)
    expect = ci.build_routing_index(selected, E)
    logits, weights = torch.empty_like(expect_logits), torch.empty_like(expect_weights)
    counts, offsets = (torch.empty(E, dtype=torch.uint32, device=DEV) for _ in range(2))
    perm, inv = (torch.empty(T * k, dtype=torch.int32, device=DEV) for _ in range(2))
    rc = _lib.load().fma_router_topk_index(
        x.data_ptr(), w.data_ptr(), T, H, E, k, logits.data_ptr(), weights.data_ptr(), counts.data_ptr(), offsets.data_ptr(),
        perm.data_ptr(), inv.data_ptr(), _lib.dtype_code(x.dtype), _lib.current_stream(x.device),
    )
    _lib.check(rc, "router_topk_index")
    assert _same(logits, expect_logits) and _same(weights, expect_weights) and (special == 3 or not torch.isfinite(logits).all())
    for got, want in zip((counts, offsets, perm, inv), (expect[0], expect[1], expect[2], expect[4])):
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))


def test_layer_without_backward_where_the_training_forward_splits_its_reduction():
    """I >= 3072 and few tiles: the training forward adds the second projection up in parts, the streaming kernel does not. Both in
    fp32, so that an expert's output differs by one rounding to bf16 where the sums fall on two sides of a boundary: 2^-8 of it, and
    as much again for the combined output."""
    from fma import KernelBackend, MoE, _lib, swiglu_packed

    T, k, E, H, I = 64, 2, 8, 256, 4096
    assert _lib.load().fma_grouped_gemm_ragged_workspace_bytes(T * k, E, H, I, 1) > 0
    torch.manual_seed(0)
    moe = MoE(E, k, H, I, swiglu_packed, True, False, 0.05).to(torch.bfloat16).to(DEV)
    x = torch.randn(T, H, device=DEV).bfloat16()
    expect, expect_logits = (t.detach() for t in moe(x, kernel_backend=KernelBackend.cuda))
    with torch.no_grad():
        y, logits = moe(x, kernel_backend=KernelBackend.cuda)
    assert torch.equal(logits, expect_logits)
    assert float((y.double() - expect.double()).norm() / expect.double().norm()) <= 2.0**-7


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize(
    "T,k,E,H,inter",
    # units of 16 weight rows (reductions from 2048 on): one to 32 rows per expert (both token blocks), partial last units of 8 columns,
    # partial last steps; in the first projection, in the second, in both
    [(1, 1, 4, 2056, 24), (3, 2, 8, 2048, 104), (16, 2, 2, 40, 2056), (17, 2, 2, 2120, 2072), (32, 3, 3, 72, 2048)],
)
def test_units_of_sixteen_weight_rows(T, k, E, H, inter, bias, dtype):
    from fma import KernelBackend, MoE, swiglu_packed

    torch.manual_seed(T + inter)
    moe = MoE(E, k, H, inter, swiglu_packed, True, bias, 0.1).to(dtype).to(DEV)
    if bias:
        with torch.no_grad():
            moe.c_fc.bias.normal_(0, 0.5)
            moe.c_proj.bias.normal_(0, 0.5)
    x = torch.randn(T, H, device=DEV).to(dtype)
    expect = moe(x.clone().requires_grad_(), kernel_backend=KernelBackend.cuda)
    with torch.no_grad():
        got = moe(x, kernel_backend=KernelBackend.cuda)
    assert torch.equal(got[0], expect[0]) and torch.equal(got[1], expect[1])
