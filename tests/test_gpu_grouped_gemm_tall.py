"""GPU parity of the tiles of up to 288 rows, which launches of at most 256 groups with varying rows take where that makes fewer
tiles. The same groups followed by empty ones up to 257 run on tiles of 256 rows: the same bits from every kernel that has both
forms; the plain product also against a float64 product of integer operands."""

import pytest
import torch

from fma import _lib
from fma.modules.moe.cuda_implementation import (
    gather_rows_cuda,
    grouped_gemm_gathered_cuda,
    grouped_gemm_ragged_cuda,
    grouped_gemm_swiglu_bwd_cuda,
    grouped_gemm_swiglu_cuda,
)
from fma.ops.swiglu.cuda_implementation import swiglu_backward_cuda, swiglu_forward_cuda

from gpu_util import DEV

pytestmark = pytest.mark.gpu

MOST = 256  # groups of a launch on tall tiles

# rows per group around every edge of a tall tile: none or all rows past 256, of one wavefront or both, one to three tiles, the sizes
# from which on 256-row tiles are as few, between groups of few rows and empty ones
SIZES = [256, 257, 271, 272, 273, 287, 288, 289, 0, 512, 513, 544, 576, 577, 16, 64, 65, 800, 864, 865, 1152, 1, 300]
# N, K: whole tiles, an odd number of K steps; partial column tiles (columns of some wavefronts only), a partial K step; one K step.
# The groups are 52 row tiles of 256 rows, 40 tall ones: with up to four column tiles both are one round, which the 256-row tiles
# win; with five and six they are two rounds and one, and tall tiles are taken.
DIMS = [(512, 192), (264, 584), (40, 64), (1536, 192), (1400, 584), (1288, 64)]


def _u32(values):
    return torch.tensor(values, dtype=torch.int64).to(torch.uint32).to(DEV)


def _both(sizes):
    return [_u32(sizes), _u32(list(sizes) + [0] * (MOST + 1 - len(sizes)))]


def _inputs(sizes, N, K, dtype, b_shape):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randint(-3, 4, (sum(sizes), K), device=DEV, generator=g).to(dtype)
    w = torch.randint(-3, 4, (MOST + 1, *b_shape), device=DEV, generator=g).to(dtype)
    bias = torch.randint(-8, 9, (MOST + 1, N), device=DEV, generator=g).to(dtype)
    return x, w, bias


def _fresh(*shape, dtype):
    return torch.full(shape, 7.0, dtype=dtype, device=DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tB", [True, False])
@pytest.mark.parametrize("N,K", DIMS)
def test_plain(N, K, tB, dtype):
    x, w, bias = _inputs(SIZES, N, K, dtype, (N, K) if tB else (K, N))
    R = x.shape[0]
    for b in (None, bias) if tB else (None,):
        results = []
        for M in _both(SIZES):
            E = M.numel()
            out = _fresh(R, N, dtype=dtype)
            grouped_gemm_ragged_cuda(x, w[:E], out, M, False, 0, N, K, False, tB, None if b is None else b[:E])
            results.append(out)
        assert torch.equal(*results)
        at = 0
        for e, m in enumerate(SIZES):
            expect = (x[at : at + m].double() @ (w[e].T if tB else w[e]).double()).to(dtype)
            if b is not None:
                expect = (expect.float() + b[e].float()).to(dtype)
            assert torch.equal(results[0][at : at + m], expect), f"group {e} of {m} rows"
            at += m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("N,K", [(512, 192), (272, 584), (48, 64), (1536, 192), (1296, 584)])  # (tiles of 128 of N / 2 columns)
def test_swiglu_and_gather(N, K, with_bias, dtype):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    R, T, divisor = sum(SIZES), 700, 3
    x = torch.randn(T, K, device=DEV, generator=g).to(dtype)
    w = (torch.randn(MOST + 1, N, K, device=DEV, generator=g) * 0.1).to(dtype)
    bias = torch.randn(MOST + 1, N, device=DEV, generator=g).to(dtype)
    row_index = torch.randint(0, T * divisor, (R,), device=DEV, generator=g, dtype=torch.int32)
    row_index[::11] = -3  # rows of zeros
    xg = torch.zeros(R, K, device=DEV, dtype=dtype)
    gather_rows_cuda(x, row_index.clamp(min=0), divisor, xg)
    xg[::11] = 0
    results = []
    for M in _both(SIZES):
        E = M.numel()
        b = bias[:E].contiguous() if with_bias else None
        h, act, act_only, plain = (_fresh(R, n, dtype=dtype) for n in (N, N // 2, N // 2, N))
        gh, gact, gact_only = (_fresh(R, n, dtype=dtype) for n in (N, N // 2, N // 2))
        grouped_gemm_swiglu_cuda(xg, w[:E], M, h, act, b)
        grouped_gemm_swiglu_cuda(xg, w[:E], M, None, act_only, b)
        grouped_gemm_gathered_cuda(x, row_index, divisor, w[:E], b, M, gh, gact)
        grouped_gemm_gathered_cuda(x, row_index, divisor, w[:E], b, M, None, gact_only)
        grouped_gemm_gathered_cuda(x, row_index, divisor, w[:E], b, M, plain, None)
        assert torch.equal(act, act_only) and torch.equal(act, gact) and torch.equal(act, gact_only)
        assert torch.equal(h, gh) and torch.equal(h, plain)
        results.append((h, act))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("inter,K", [(512, 192), (136, 584), (40, 64), (1536, 192), (1288, 584)])
def test_swiglu_backward(inter, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(inter + K)
    R = sum(SIZES)
    dy = torch.randn(R, K, device=DEV, generator=g).to(dtype)
    w = (torch.randn(MOST + 1, K, inter, device=DEV, generator=g) * 0.1).to(dtype)
    h = (torch.randn(R, 2 * inter, device=DEV, generator=g) * 2).to(dtype)
    results = []
    for M in _both(SIZES):
        results.append(_fresh(R, 2 * inter, dtype=dtype))
        grouped_gemm_swiglu_bwd_cuda(dy, w[: M.numel()], h, M, results[-1])
    assert torch.equal(*results)


@pytest.mark.parametrize("N", [264, 2808])  # two parts of 12 x 11 tiles of 256 rows are two rounds, of 8 x 11 tall ones one
@pytest.mark.parametrize("tB", [True, False])
def test_split_reduction(tB, N):
    sizes, K = [257, 288, 289, 0, 270, 16, 530], 4104
    x, w, _ = _inputs(sizes, N, K, torch.bfloat16, (N, K) if tB else (K, N))
    lib, R = _lib.load(), sum(sizes)
    results = []
    for M in _both(sizes):
        E = M.numel()
        out = _fresh(R, N, dtype=x.dtype)
        nbytes = lib.fma_grouped_gemm_ragged_split_bytes(R, E, N, K, int(tB))
        workspace = torch.full((max(nbytes // 4, 1),), float("nan"), device=DEV)
        rc = lib.fma_grouped_gemm_ragged_split(
            x.data_ptr(), w.data_ptr(), out.data_ptr(), M.data_ptr(), None, E, _lib.FMA_VARY_M, 0, N, K, 0, int(tB), 1.0, R,
            workspace.data_ptr() if nbytes else None, nbytes, _lib.FMA_BF16, torch.cuda.current_stream().cuda_stream,
        )  # fmt: skip
        _lib.check(rc, "fma_grouped_gemm_ragged_split")
        results.append(out)
        if E <= MOST:  # this launch is split, and has written every sum
            assert nbytes > 0 and not bool(torch.isnan(workspace).any())
    assert torch.equal(*results)  # (integers below 2^24: exact in any order)


@pytest.mark.parametrize("sizes", [[257, 288, 289, 530, 3], [40, 0, 3, 64, 17]])
@pytest.mark.parametrize("N,K", [(257, 72), (72, 67), (501, 31), (6899, 31)])  # (27 column tiles: tall tiles save a round)
def test_element_wise_tiles(N, K, sizes):
    """sizes whose rows are no multiple of 16 bytes take the element-wise path: tall tiles, tiles in parts of their columns (some past
    the last column), half-width tiles"""
    x, w, _ = _inputs(sizes, N, K, torch.bfloat16, (N, K))
    out = _fresh(sum(sizes), N, dtype=x.dtype)
    grouped_gemm_ragged_cuda(x, w[: len(sizes)], out, _u32(sizes), False, 0, N, K, False, True, None)
    at = 0
    for e, m in enumerate(sizes):
        assert torch.equal(out[at : at + m], (x[at : at + m].double() @ w[e].T.double()).bfloat16()), f"group {e}"
        at += m


def test_many_tiles_per_workgroup():
    """tall and other tiles after each other in every workgroup, 256 groups"""
    sizes = [(250 + 7 * (e % 11)) if e % 5 else (e % 3) * 40 for e in range(MOST)]
    N, K = 512, 136
    x, w, _ = _inputs(sizes, N, K, torch.bfloat16, (N, K))
    results = []
    for M in _both(sizes):
        results.append(_fresh(x.shape[0], N, dtype=x.dtype))
        grouped_gemm_ragged_cuda(x, w[: M.numel()], results[-1], M, False, 0, N, K, False, True, None)
    assert torch.equal(*results)
    at = 0
    for e, m in enumerate(sizes):
        assert torch.equal(results[0][at : at + m], (x[at : at + m].double() @ w[e].T.double()).bfloat16()), f"group {e}"
        at += m


@pytest.mark.parametrize("K", [1984, 2040, 2048, 2120])  # 31 K steps: two LDS stages from 65 rows on; 32 (the last partial or whole), 34
@pytest.mark.parametrize("tB", [True, False])
def test_groups_around_the_three_stage_loop(tB, K):
    """groups on either side of 64 and 128 rows, after each other in every workgroup: packed, gathered and with the activation, against
    a float64 product of integer operands (|sum| <= 9 K < 2^24: exact in fp32)"""
    sizes = [64, 65, 128, 129, 1, 100, 0, 127, 300, 63, 80, 256, 112, 16, 113, 96] * 3
    N = 520
    x, w, bias = _inputs(sizes, N, K, torch.bfloat16, (N, K) if tB else (K, N))
    E, R = len(sizes), sum(sizes)
    w, bias = w[:E], bias[:E].contiguous()
    out = _fresh(R, N, dtype=x.dtype)
    grouped_gemm_ragged_cuda(x, w, out, _u32(sizes), False, 0, N, K, False, tB, None)
    at = 0
    for e, m in enumerate(sizes):
        assert torch.equal(out[at : at + m], (x[at : at + m].double() @ (w[e].T if tB else w[e]).double()).bfloat16()), f"group {e} of {m} rows"
        at += m
    if not tB:
        return
    row_index = torch.randperm(R, device=DEV).int()
    packed = torch.empty_like(x)
    gather_rows_cuda(x, row_index, 1, packed)
    h, act, gh, gact, gact_only = (_fresh(R, n, dtype=x.dtype) for n in (N - 8, (N - 8) // 2, N - 8, (N - 8) // 2, (N - 8) // 2))
    w, bias = w[:, : N - 8].contiguous(), bias[:, : N - 8].contiguous()
    grouped_gemm_ragged_cuda(packed, w, h, _u32(sizes), False, 0, N - 8, K, False, True, bias)
    grouped_gemm_gathered_cuda(x, row_index, 1, w, bias, _u32(sizes), gh, gact)
    grouped_gemm_gathered_cuda(x, row_index, 1, w, bias, _u32(sizes), None, gact_only)
    grouped_gemm_swiglu_cuda(packed, w, _u32(sizes), None, act, bias)
    assert torch.equal(h, gh) and torch.equal(act, gact) and torch.equal(act, gact_only)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [1984, 2040, 2048, 2120])  # 31 K steps: two LDS stages from 65 rows on; 32 (the last partial or whole), 34
@pytest.mark.parametrize("groups", [48, MOST + 1])  # the kernels of both forms
def test_every_kernel_with_the_three_stage_loop(groups, K, dtype):
    """groups on either side of 64 and 128 rows, after each other in every workgroup, through every kernel that has the loop: packed and
    gathered, with and without a bias (with one it ends at 64 rows), the activation and its gradient, both layouts. Against a float64
    product of operands that are whole numbers over 64 (|sum| <= 9 K / 64, a multiple of 1 / 64: exact in fp32) and, behind it, the
    activation's own kernels."""
    sizes = [64, 65, 128, 129, 1, 100, 0, 127, 300, 63, 80, 256, 112, 16, 113, 96] * 3
    sizes += [0] * (groups - len(sizes))
    N, R = 528, sum(sizes)
    x, w, bias = _inputs(sizes, N, K, dtype, (N, K))
    w, bias, M = w[:groups] / 64, bias[:groups].contiguous(), _u32(sizes)
    wt = w.transpose(1, 2).contiguous()
    product = torch.cat([part.double() @ w[e].T.double() for e, part in enumerate(x.split(sizes))]).to(dtype)
    row_index = torch.randperm(R, device=DEV).int()
    tokens = torch.empty_like(x)
    tokens[row_index.long()] = x

    out = _fresh(R, N, dtype=dtype)
    grouped_gemm_ragged_cuda(x, wt, out, M, False, 0, N, K, False, False, None)
    assert torch.equal(out, product), "NN"
    for b in (None, bias):
        want = product if b is None else (product.float() + b.repeat_interleave(torch.tensor(sizes, device=DEV), 0).float()).to(dtype)
        up, gate = want.chunk(2, dim=-1)
        act_want = torch.empty(R, N // 2, dtype=dtype, device=DEV)
        swiglu_forward_cuda(gate=gate, up=up, output=act_want, BLOCK_SIZE=1024)
        h, gh, gh2 = (_fresh(R, N, dtype=dtype) for _ in range(3))
        act, act_only, gact, gact_only = (_fresh(R, N // 2, dtype=dtype) for _ in range(4))
        grouped_gemm_ragged_cuda(x, w, h, M, False, 0, N, K, False, True, b)
        assert torch.equal(h, want), "NT"
        grouped_gemm_gathered_cuda(tokens, row_index, 1, w, b, M, gh, None)
        assert torch.equal(gh, want), "NT, gathered"
        h.fill_(7.0)
        grouped_gemm_swiglu_cuda(x, w, M, h, act, b)
        grouped_gemm_swiglu_cuda(x, w, M, None, act_only, b)
        assert torch.equal(h, want) and torch.equal(act, act_want) and torch.equal(act_only, act_want), "activation"
        grouped_gemm_gathered_cuda(tokens, row_index, 1, w, b, M, gh2, gact)
        grouped_gemm_gathered_cuda(tokens, row_index, 1, w, b, M, None, gact_only)
        assert torch.equal(gh2, want) and torch.equal(gact, act_want) and torch.equal(gact_only, act_want), "activation, gathered"

    pre = torch.randn(R, 2 * N, device=DEV, generator=torch.Generator(device=DEV).manual_seed(K)).to(dtype)
    got, expect = _fresh(R, 2 * N, dtype=dtype), _fresh(R, 2 * N, dtype=dtype)
    (up, gate), (up_grad, gate_grad) = pre.chunk(2, dim=-1), expect.chunk(2, dim=-1)
    swiglu_backward_cuda(gate=gate, up=up, output_grad=product, gate_grad=gate_grad, up_grad=up_grad, BLOCK_SIZE=1024)
    grouped_gemm_swiglu_bwd_cuda(x, wt, pre, M, got)
    assert torch.equal(got, expect), "gradient of the activation"
