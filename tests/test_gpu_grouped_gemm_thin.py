"""The grouped product for a few rows per group (fma_grouped_gemm_thin) against the tile kernel's entry points, bit for bit:
both walk the reduction in the same order with the same instruction. Sizes around the edges of its units: 16 / 32 / 64 rows
of a pass, 32 / 64 weight rows of a wavefront, 64 reduction elements of a step, more than 64 groups."""

import pytest
import torch

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
