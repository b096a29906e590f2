"""GPU parity of fma_grouped_gemm_ragged_split: launches with few tiles, whose reduction is computed in parts. Operands are
small integers, so that every fp32 sum is exact in any order (|sum| <= 9 K < 2^24) and the result has to equal the unsplit
one, and the float64 product rounded once, bit for bit."""

import pytest
import torch

from fma import _lib

from gpu_util import DEV

pytestmark = pytest.mark.gpu


def _call(A, B, sizes, rows, N, K, tB, bias, alpha, workspace_bytes):
    lib = _lib.load()
    out = torch.full((rows, N), 7.0, dtype=A.dtype, device=DEV)
    s = torch.tensor(sizes, dtype=torch.int64).to(torch.uint32).to(DEV)
    # never read before it is written: NaN would show
    workspace = torch.full((max(workspace_bytes // 4, 1),), float("nan"), device=DEV)
    rc = lib.fma_grouped_gemm_ragged_split(
        A.data_ptr(), B.data_ptr(), out.data_ptr(), s.data_ptr(), _lib.ptr(bias), len(sizes), _lib.FMA_VARY_M, 0, N, K, 0,
        int(tB), alpha, rows, workspace.data_ptr() if workspace_bytes else None, workspace_bytes, _lib.dtype_code(A.dtype),
        torch.cuda.current_stream().cuda_stream,
    )
    assert rc == 0, lib.fma_last_error_string()
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tB", [True, False])
@pytest.mark.parametrize(
    "sizes,N,K,bias,alpha",
    [
        ([250, 257, 0, 3, 64, 65, 512, 130], 2048, 8192, True, 1.0),  # ragged, empty, thin groups; whole K steps
        ([128] * 8, 2048, 4104, False, 1.0),  # 65 K steps, the last of 8 elements: an odd and partial last part
        ([1], 264, 3080, False, 0.5),  # the shortest split reduction, one row, a partial column tile
        ([600, 30], 520, 5000, True, 1.0),  # partial column tile of 8, K a multiple of 8 only
        ([16] * 40, 8, 16384, False, 1.0),  # one narrow column tile, many parts
    ],
)
def test_split_equals_unsplit(dtype, tB, sizes, N, K, bias, alpha):
    bias = bias and tB  # (added in the forward form only)
    E, R = len(sizes), sum(sizes)
    rows = R + 5  # rows past the groups stay as they are
    g = torch.Generator(device=DEV).manual_seed(K + N)
    A = torch.randint(-3, 4, (rows, K), device=DEV, generator=g).to(dtype)
    B = torch.randint(-3, 4, (E, N, K) if tB else (E, K, N), device=DEV, generator=g).to(dtype)
    b = torch.randint(-64, 65, (E, N), device=DEV, generator=g).to(dtype) if bias else None
    nbytes = _lib.load().fma_grouped_gemm_ragged_workspace_bytes(rows, E, N, K, int(tB))
    assert nbytes >= 2 * rows * N * 4, "the sizes are chosen to be split"
    got = _call(A, B, sizes, rows, N, K, tB, b, alpha, nbytes)
    assert torch.equal(got, _call(A, B, sizes, rows, N, K, tB, b, alpha, 0))
    assert (got[R:] == 7.0).all()
    at = 0
    for e, m in enumerate(sizes):
        expect = (alpha * (A[at : at + m].double() @ (B[e].T if tB else B[e]).double())).to(dtype)
        if bias:
            expect = (expect.float() + b[e].float()).to(dtype)
        assert torch.equal(got[at : at + m], expect), f"group {e}"
        at += m


@pytest.mark.parametrize("rows,E,N,K", [(65536, 128, 4096, 1536), (16, 8, 2048, 3000), (2042, 8, 2047, 8192), (0, 8, 2048, 8192)])
def test_no_split_where_it_cannot_pay_or_run(rows, E, N, K):
    assert _lib.load().fma_grouped_gemm_ragged_workspace_bytes(rows, E, N, K, 1) == 0


@pytest.mark.parametrize("tB", [True, False])
@pytest.mark.parametrize("values", [[float("inf")], [float("inf"), float("-inf")], [float("nan"), 1.0]])
def test_split_of_infinities_and_nan(values, tB):
    """in different parts of the reduction, and against each other"""
    sizes, N, K = [3, 130, 64], 264, 4104
    E, R = len(sizes), sum(sizes)
    g = torch.Generator(device=DEV).manual_seed(K)
    A = torch.randint(-3, 4, (R, K), device=DEV, generator=g).bfloat16()
    B = torch.randint(1, 4, (E, N, K) if tB else (E, K, N), device=DEV, generator=g).bfloat16()
    for row in (1, 60, 196):
        for i, v in enumerate(values):
            A[row, [5, K - 3][i]] = v  # the first and the last part
    nbytes = _lib.load().fma_grouped_gemm_ragged_workspace_bytes(R, E, N, K, int(tB))
    assert nbytes >= 2 * R * N * 4
    got, want = (_call(A, B, sizes, R, N, K, tB, None, 1.0, n) for n in (nbytes, 0))
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0))
    special = torch.zeros(R, dtype=torch.bool, device=DEV)
    special[[1, 60, 196]] = True
    assert torch.equal(torch.isfinite(got).all(1), ~special) and not torch.isfinite(got[special]).any()


def test_product_runs_unsplit_where_the_sums_find_no_memory():
    from fma.modules.moe import cuda_implementation as ci

    sizes, N, K = [512] * 8, 4096, 14336
    E, R = len(sizes), sum(sizes)
    nbytes = _lib.load().fma_grouped_gemm_ragged_workspace_bytes(R, E, N, K, 1)
    assert nbytes >= 64 << 20
    g = torch.Generator(device=DEV).manual_seed(1)
    A = torch.randint(-3, 4, (R, K), device=DEV, generator=g).bfloat16()
    B = torch.randint(-3, 4, (E, N, K), device=DEV, generator=g).bfloat16()
    s = torch.tensor(sizes, dtype=torch.int32, device=DEV).view(torch.uint32)
    outputs = [torch.empty(R, N, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    ci.grouped_gemm_ragged_cuda(A, B, outputs[0], s, False, 0, N, K, False, True)
    torch.cuda.empty_cache()
    try:  # a limit of this process's allocator that is below what it holds already: nothing more is to be had
        torch.cuda.set_per_process_memory_fraction(1e-4)
        held = []
        with pytest.raises(torch.OutOfMemoryError):  # what is free inside of it is used up
            for _ in range(200):
                held.append(torch.empty(nbytes, dtype=torch.uint8, device=DEV))
        ci.grouped_gemm_ragged_cuda(A, B, outputs[1], s, False, 0, N, K, False, True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(*outputs)
